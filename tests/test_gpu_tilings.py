"""The kernels that linears and groups of them run on where a neighbouring choice measured slower (the rules by themselves,
as far as the host can tell: test_host_tilings.py), bit for bit against an exact fp64 product on the device."""
import ctypes

import pytest
import torch

from test_gpu_panel_tiles import _run, _s8

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _family():
    import torch_int._CUDA as C
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    return C._lib.ti_last_kernel().decode()


@pytest.mark.parametrize("T,H,family", [(4096, 40, "pipe16_256x160_group"), (2560, 56, "pipe16_256x128_group"),
                                        (3700, 20, "pipe16_256x160_group"), (2112, 40, "pipe16_256x160_group")])
def test_three_projections(T, H, family):
    import torch_int._hip_ext as X
    gen = torch.Generator(device=DEV).manual_seed(T)
    N = H * 128
    x, ws, bs = _s8(gen, (T, N), 3.0), [_s8(gen, (N, N), 3.0) for _ in range(3)], [_s8(gen, (N,), 20.0) for _ in range(3)]
    al, be = [2.0 ** -8, 2.0 ** -7, 2.0 ** -9], [0.5, 1.0, 0.25]
    print(f"group {T}x{N}x{N}", flush=True)
    out = X.linear_a8_w8_b8_o8_group_heads(x, ws, bs, al, be, 1, T, H, 128)
    assert _family() == family
    for o, w, b, a, c in zip(out, ws, bs, al, be):
        want = torch.clamp(torch.round((x.double() @ w.double().t()) * a + c * b.double()), -128, 127).to(torch.int8)
        assert torch.equal(o, want.view(1, T, H, 128).transpose(1, 2))


@pytest.mark.parametrize("out_dtype", [torch.int8, torch.int32])
@pytest.mark.parametrize("M,N,K,family", [(1029, 16384, 4096, "pipe_256x256+stream"), (2064, 8192, 2048, "pipe_256x256+stream"),
                                          (1538, 20480, 5120, "pipe16_256x160+stream")])
def test_a_few_rows_beyond_a_multiple_of_256(M, N, K, family, out_dtype):
    print(f"rows cut off {M}x{N}x{K} {out_dtype}", flush=True)
    out, want = _run(M, N, K, out_dtype, M)
    assert _family() == family and torch.equal(out, want)


@pytest.mark.parametrize("out_dtype", [torch.int8, torch.int32])
@pytest.mark.parametrize("M,N,K,family", [(300, 20480, 5120, "pipe16_256x160"), (320, 20480, 5120, "pipe16_256x160"),
                                          (569, 16384, 4096, "pipe16_160x256"), (528, 8192, 2048, "pipe16_192x128")])
def test_two_rows_of_tiles(M, N, K, family, out_dtype):
    """Two rows of tiles keep every CU busy where they can, three and more go by their price."""
    print(f"rows of tiles {M}x{N}x{K} {out_dtype}", flush=True)
    out, want = _run(M, N, K, out_dtype, M)
    assert _family() == family and torch.equal(out, want)


@pytest.mark.parametrize("room", ["own", "the other epilogues'", "none"])
@pytest.mark.parametrize("M,N,K,family", [(376, 5120, 20480, "splitk_256x160"), (406, 4096, 16384, "splitk_256x256"),
                                          (588, 2560, 10240, "splitk_256x160")])
def test_slices_of_the_accumulating_epilogue(M, N, K, family, room):
    """They never meet in one launch, so they are not those that would; with less room than they want it takes what fits."""
    import torch_int._CUDA as C
    gen = torch.Generator(device=DEV).manual_seed(M)
    x, w, bias = _s8(gen, (M, K), 3.0), _s8(gen, (N, K), 3.0), torch.randint(-99, 99, (N,), device=DEV, generator=gen).float()
    before = torch.randint(-999, 999, (M, N), device=DEV, generator=gen).float()
    out, want = before.clone(), (before.double() + x.double() @ w.double().t() + bias.double()).float()    # integers below 2^24
    have = {"own": C._lib.ti_linear_acc_workspace_bytes(M, N, K), "none": 0}.get(room, C._lib.ti_linear_workspace_bytes(M, N, K))
    ws = torch.full((have + 4096,), 77, dtype=torch.uint8, device=DEV)
    print(f"accumulating {M}x{N}x{K} {room}", flush=True)
    rc = C._lib.ti_linear_a8_w8_bfp32_ofp32_acc(x.data_ptr(), w.data_ptr(), bias.data_ptr(), out.data_ptr(), M, N, K, 1.0, 1.0,
                                                ws.data_ptr() if have else None, have, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(out, want) and bool((ws[have:] == 77).all())
    assert room != "own" or _family() == family


def _form():
    import torch_int._CUDA as C
    C._lib.ti_last_kernel_form.restype = ctypes.c_char_p
    return C._lib.ti_last_kernel_form().decode()


@pytest.mark.parametrize("M,N,K,family,form8,form32", [
    (1025, 2048, 512, "pipe_128x128", "gemm_pipe", "gemm_pipe"), (2047, 2033, 2048, "pipe_128x128", "gemm_pipe16q", "gemm_pipe16q"),
    (2048, 2048, 640, "pipe_128x128", "gemm_pipe", "gemm_pipe"),
    (2048, 7168, 2048, "pipe_256x256", "gemm_pipe16q", "gemm_pipe2"), (4096, 2816, 192, "pipe_256x256", "gemm_pipe", "gemm_pipe"),
    (2048, 7168, 1920, "pipe_256x256", "gemm_pipe2", "gemm_pipe2")])
@pytest.mark.parametrize("out_dtype", [torch.int8, torch.int32])
def test_forms_of_one_tiling(M, N, K, family, form8, form32, out_dtype):
    print(f"form {M}x{N}x{K} {out_dtype}", flush=True)
    out, want = _run(M, N, K, out_dtype, M)
    assert (_family(), _form()) == (family, form8 if out_dtype == torch.int8 else form32) and torch.equal(out, want)


@pytest.mark.parametrize("M,N,K,family,form", [(130, 2048, 16384, "splitk_128x128", "gemm_pipe"), (100, 2048, 16384, "splitk_128x128", "gemm_pipe"), (100, 512, 16384, "splitk_128x128", "gemm_pipe16q"),
                                               (256, 1024, 8192, "splitk_128x128", "gemm_pipe16q"), (256, 2048, 8192, "fusedk_128x128", "gemm_pipe16q")])
def test_steps_of_split_products(M, N, K, family, form):
    """128-byte steps where slices meet in one launch or a quarter of the CUs is free, else 64-byte steps."""
    print(f"split steps {M}x{N}x{K}", flush=True)
    out, want = _run(M, N, K, torch.int32, M)
    assert (_family(), _form()) == (family, form) and torch.equal(out, want)


@pytest.mark.parametrize("M,N,K,family", [(2945, 2000, 1024, "pipe16_192x128"), (2241, 4096, 1280, "pipe16_160x256"),
                                          (2111, 5104, 1152, "pipe16_192x256"), (1500, 3008, 1024, "pipe16_192x128")])
def test_every_epilogue_of_the_tilings_by_rows(M, N, K, family):
    """Epilogues whose results are exact: scale a power of two, integers below 2^24."""
    import torch_int._CUDA as C
    import torch_int._hip_ext as X
    gen = torch.Generator(device=DEV).manual_seed(M)
    x, w, b8 = _s8(gen, (M, K), 3.0), _s8(gen, (N, K), 3.0), _s8(gen, (N,), 20.0)
    bf = torch.randint(-9999, 9999, (N,), device=DEV, generator=gen).float()
    before = torch.randint(-9999, 9999, (M, N), device=DEV, generator=gen).float()
    acc = x.double() @ w.double().t()
    sums = (acc + bf.double()).float()
    int8 = torch.round(acc * 2.0 ** -3 + 0.5 * b8.double())
    for name, call, want in (
            ("fp32", lambda: C.linear_a8_w8_bfp32_ofp32(x, w, bf, 1.0, 1.0), sums),
            ("accumulating", lambda: C._linear_a8_w8_bfp32_ofp32_acc(x, w, bf, 1.0, 1.0, before.clone()), sums + before),
            ("int32 scaled", lambda: C.linear_a8_w8_b32_o32_with_scaling(x, w, bf.int(), 1.0, 1.0), sums.int()),
            ("relu", lambda: C.linear_relu_a8_w8_b8_o8(x, w, b8, 2.0 ** -3, 0.5), int8.clamp(0, 127).to(torch.int8)),
            ("head-major", lambda: X.linear_a8_w8_b8_o8_heads(x, w, b8, 2.0 ** -3, 0.5, 1, M, N // 16, 16).permute(0, 2, 1, 3).reshape(M, N),
             int8.clamp(-128, 127).to(torch.int8))):
        print("epilogue", name, M, N, K, flush=True)
        out = call()
        assert _family() == family and torch.equal(out, want), name


@pytest.mark.parametrize("M,N,K", [(4101, 4096, 1024), (4097, 4096, 1024), (4112, 4096, 1024), (4113, 4096, 1024), (4160, 4096, 1024),
                                   (3168, 20480, 1024)])
def test_every_epilogue_of_rows_cut_off_the_end(M, N, K):
    import torch_int._CUDA as C
    import torch_int._hip_ext as X
    gen = torch.Generator(device=DEV).manual_seed(M)
    x, w, b8 = _s8(gen, (M, K), 3.0), _s8(gen, (N, K), 3.0), _s8(gen, (N,), 20.0)
    bf = torch.randint(-9999, 9999, (N,), device=DEV, generator=gen).float()
    before = torch.randint(-9999, 9999, (M, N), device=DEV, generator=gen).float()
    acc = x.double() @ w.double().t()
    sums = (acc + bf.double()).float()
    int8 = torch.round(acc * 2.0 ** -3 + 0.5 * b8.double())
    assert C._lib.ti_linear_row_split(ctypes.c_int64(M), ctypes.c_int64(N), ctypes.c_int64(K)) == M % 256
    for name, call, want in (
            ("int32", lambda: C.linear_a8_w8_b32_o32(x, w, bf.int()), sums.int()),
            ("int32 scaled", lambda: C.linear_a8_w8_b32_o32_with_scaling(x, w, bf.int(), 1.0, 1.0), sums.int()),
            ("fp32", lambda: C.linear_a8_w8_bfp32_ofp32(x, w, bf, 1.0, 1.0), sums),
            ("accumulating", lambda: C._linear_a8_w8_bfp32_ofp32_acc(x, w, bf, 1.0, 1.0, before.clone()), sums + before),
            ("int8", lambda: C.linear_a8_w8_b8_o8(x, w, b8, 2.0 ** -3, 0.5), int8.clamp(-128, 127).to(torch.int8)),
            ("relu", lambda: C.linear_relu_a8_w8_b8_o8(x, w, b8, 2.0 ** -3, 0.5), int8.clamp(0, 127).to(torch.int8)),
            ("head-major", lambda: X.linear_a8_w8_b8_o8_heads(x, w, b8, 2.0 ** -3, 0.5, 1, M, N // 128, 128).permute(0, 2, 1, 3).reshape(M, N),
             int8.clamp(-128, 127).to(torch.int8))):
        print("rows cut off", name, M, N, K, flush=True)
        out = call()
        assert "+" in _family() and torch.equal(out, want), (name, _family())


@pytest.mark.parametrize("K,reached", [(1 << 23, True), ((1 << 23) + 128, False)])
def test_rows_up_to_8_mib_apart_are_left_to_the_rules(K, reached):
    """Beyond that, no tiling with 32-bit panel offsets is a candidate."""
    print(f"rows apart {K}", flush=True)
    out, want = _run(20, 24, K, torch.int32, 5)
    assert (_form() != "gemm_pipe" or _family() != "pipe_128x128") == reached and torch.equal(out, want)
