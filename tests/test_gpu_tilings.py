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
