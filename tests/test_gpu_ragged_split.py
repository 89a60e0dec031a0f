"""Split products whose slices meet in one launch where M ends inside a tile (gemm_pipe16q_kernel, RAGGED): rows at the edges of
tiles, of a wave's rows and of a 16-row block, every epilogue and head-major outputs, against an exact product
on the device and the two-launch form."""
import ctypes

import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("N,K,tile", [(2048, 8192, "128x128"), (4096, 4096, "128x128"), (768, 3072, "128x192")])
@pytest.mark.parametrize("M", [257, 272, 288, 289, 303, 320, 383, 384, 385, 449, 481, 512])
def test_rows_that_end_inside_a_tile_are_exact(M, N, K, tile):
    import torch_int._CUDA as C
    import torch_int._hip_ext as X
    lib = C._lib
    lib.ti_last_kernel.restype = ctypes.c_char_p
    g = torch.Generator(device=DEV).manual_seed(M + N)
    s8 = lambda *shape: torch.randint(-127, 128, shape, dtype=torch.int8, device=DEV, generator=g)
    x, w, b8 = s8(M, K), s8(N, K), s8(N)
    b32 = torch.randint(-65536, 65536, (N,), dtype=torch.int32, device=DEV, generator=g)
    bf = torch.randn(N, device=DEV, generator=g)
    acc = torch.mm(x.double(), w.double().t().contiguous()).to(torch.int32).cpu()   # sums below 2^53
    al, be = 1e-4, 0.02
    one = tile == "128x128" or M % 128 == 0 or M > 320   # 128x192: from three rows of tiles on
    print("ragged split", M, N, K, flush=True)
    runs = [(lambda: C.linear_a8_w8_b32_o32(x, w, b32), orc.epi_b32_o32(acc, b32.cpu())),
            (lambda: C.linear_a8_w8_b32_o32_with_scaling(x, w, b32, al, be), orc.epi_b32_o32_scaled(acc, b32.cpu(), al, be)),
            (lambda: C.linear_a8_w8_bfp32_ofp32(x, w, bf, al, 1.0), orc.epi_bfp32_ofp32(acc, bf.cpu(), al, 1.0)),
            (lambda: C.linear_a8_w8_b8_o8(x, w, b8, al, be), orc.epi_b8_o8(acc, b8.cpu(), al, be)),
            (lambda: C.linear_relu_a8_w8_b8_o8(x, w, b8, al, be), orc.epi_b8_o8(acc, b8.cpu(), al, be, relu=True)),
            (lambda: X.linear_a8_w8_b8_o8_heads(x, w, b8, al, be, 1, M, N // 64, 64).permute(0, 2, 1, 3).reshape(M, N),
             orc.epi_b8_o8(acc, b8.cpu(), al, be))]
    try:
        for call, want in runs:
            for _ in range(2):
                out = call()
                assert lib.ti_last_kernel().decode() == ("fusedk_" if one else "splitk_") + tile, lib.ti_last_kernel()
                assert torch.equal(out.cpu(), want)
            lib.ti_fused_splitk(0)
            assert torch.equal(call().cpu(), want) and lib.ti_last_kernel().decode() == "splitk_" + tile
            lib.ti_fused_splitk(1)
    finally:
        lib.ti_fused_splitk(1)


@pytest.mark.parametrize("M,N,K", [(300, 2048, 8192), (512, 2048, 8192)])
def test_a_workspace_of_the_slices_alone_still_serves(M, N, K):
    """Tiles are parked whole: callers that bring no more than the slices' outputs get two launches."""
    import torch_int._CUDA as C
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    g = torch.Generator(device=DEV).manual_seed(M)
    s8 = lambda *shape: torch.randint(-127, 128, shape, dtype=torch.int8, device=DEV, generator=g)
    x, w, b8 = s8(M, K), s8(N, K), s8(N)
    want = C.linear_a8_w8_b8_o8(x, w, b8, 1e-4, 0.02)
    assert C._lib.ti_last_kernel().decode() == "fusedk_128x128"
    need = C._lib.ti_linear_workspace_bytes(M, N, K)
    slices = need // ((M + 127) // 128 * 128 * N * 4)
    ws = torch.full((need + 4096,), 77, dtype=torch.uint8, device=DEV)
    for given, form in ((need, "fusedk_128x128"), (slices * M * N * 4, "splitk_128x128" if M % 128 else "fusedk_128x128")):
        out = torch.empty_like(want)
        rc = C._lib.ti_linear_a8_w8_b8_o8(x.data_ptr(), w.data_ptr(), b8.data_ptr(), out.data_ptr(), M, N, K, 1e-4, 0.02,
                                          ws.data_ptr(), given, torch.cuda.current_stream().cuda_stream)
        assert rc == 0 and C._lib.ti_last_kernel().decode() == form
        assert torch.equal(out, want) and bool((ws[given:] == 77).all()), (M, given)   # nothing written beyond it
        ws.fill_(77)
