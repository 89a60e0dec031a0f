"""The 160x160 tiles of the split products: row counts at the edges of the range in which they save rows over 128-row
tiles (257 to 320), every element against an exact product on the device."""
import ctypes

import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M,square", [(256, False), (257, True), (300, True), (320, True), (321, False)])
def test_split_products_on_square_tiles_are_exact(M, square):
    import torch_int._CUDA as C
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    N, K, al, be = 5120, 20480, 1e-4, 0.02
    g = torch.Generator(device=DEV).manual_seed(M)
    s8 = lambda *shape: torch.randint(-127, 128, shape, dtype=torch.int8, device=DEV, generator=g)
    x, w, b8 = s8(M, K), s8(N, K), s8(N)
    bf = torch.randn(N, device=DEV, generator=g)
    acc = torch.mm(x.double(), w.double().t().contiguous()).to(torch.int32).cpu()   # sums below 2^53
    print("square tiles", M, N, K, flush=True)
    for out, want in ((C.linear_a8_w8_b8_o8(x, w, b8, al, be), orc.epi_b8_o8(acc, b8.cpu(), al, be)),
                      (C.linear_a8_w8_bfp32_ofp32(x, w, bf, al, 1.0), orc.epi_bfp32_ofp32(acc, bf.cpu(), al, 1.0))):
        assert (C._lib.ti_last_kernel().decode() == "splitk_160x160") == square, C._lib.ti_last_kernel()
        assert torch.equal(out.cpu(), want)


@pytest.mark.parametrize("M,N,K", [(300, 5120, 20480), (160, 20480, 5120)])
def test_without_their_workspace_the_other_tiles_run(M, N, K):
    """A workspace that does not hold the slices of the square tiles leaves the shape to what ran it before them."""
    import torch_int._CUDA as C
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    g = torch.Generator(device=DEV).manual_seed(M)
    s8 = lambda *shape: torch.randint(-127, 128, shape, dtype=torch.int8, device=DEV, generator=g)
    x, w, b8 = s8(M, K), s8(N, K), s8(N)
    print("without workspace", M, N, K, flush=True)
    want = C.linear_a8_w8_b8_o8(x, w, b8, 1e-4, 0.02)
    assert C._lib.ti_last_kernel().decode() == "splitk_160x160"
    need = C._lib.ti_linear_workspace_bytes(M, N, K)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    out = torch.empty_like(want)
    for given in (need - 256, 0):
        out.zero_()
        rc = C._lib.ti_linear_a8_w8_b8_o8(x.data_ptr(), w.data_ptr(), b8.data_ptr(), out.data_ptr(), M, N, K, 1e-4, 0.02,
                                          ws.data_ptr() if given else None, given, torch.cuda.current_stream().cuda_stream)
        assert rc == 0 and "160x160" not in C._lib.ti_last_kernel().decode()
        assert torch.equal(out, want)
