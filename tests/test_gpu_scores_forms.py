"""Every form of the batched products with 32-bit outputs and a short inner dimension (csrc/bmm_scores.h) by its name: pieces of rows, columns
and K inside and at the end of its blocks; and the sizes that stay with the tiled kernels.  Against the oracle bit for bit."""
import ctypes

import pytest
import torch

from oracle import oracle as orc
from test_gpu_scores import _case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _form():
    import torch_int._CUDA as C
    C._lib.ti_last_kernel_form.restype = ctypes.c_char_p
    return C._lib.ti_last_kernel_form().decode()


@pytest.mark.parametrize("batch,M,N,K", [(3, 17, 1, 16), (7, 130, 257, 64), (8, 244, 244, 128), (32, 116, 116, 128), (2, 129, 500, 112)])
def test_16_by_32(batch, M, N, K):
    _case(batch, M, N, K)
    assert _form() == "16x32 to a wave"


@pytest.mark.parametrize("batch,M,N,K", [(41, 131, 501, 64), (41, 131, 501, 48), (30, 200, 300, 80), (33, 177, 289, 96), (140, 100, 100, 128),
                                         (41, 257, 130, 112)])
def test_32_by_32(batch, M, N, K):
    _case(batch, M, N, K)
    assert _form() == "32x32 to a wave"


@pytest.mark.parametrize("batch,M,N,K", [(61, 701, 601, 64), (12, 1501, 1500, 48), (9, 900, 701, 80), (40, 200, 211, 128), (41, 300, 170, 112)])
def test_through_the_lds(batch, M, N, K):
    _case(batch, M, N, K)
    assert _form() == "rows through the LDS"


@pytest.mark.parametrize("batch,M,N,K", [(61, 1025, 1056, 64), (33, 1500, 1376, 48), (33, 1501, 1376, 80), (41, 1270, 1248, 128), (3, 17, 1280032, 16)])
def test_non_temporal_stores(batch, M, N, K):
    """Outputs that the last-level cache does not hold: rows, columns and K that end inside a tile; every byte of the fp32 product against
    exact sums (below 2^24), and what lies behind the outputs stays as it was."""
    import torch_int._CUDA as C
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    print(f"stream batch={batch} M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + N)
    a, b = (torch.randint(-127, 128, (batch, n, K), dtype=torch.int8, device=DEV, generator=g) for n in (M, N))
    out = torch.full((batch * M * N + 64,), 77.0, device=DEV)
    for call, dtype in ((C._lib.ti_bmm_s8t_s8n_f32t, torch.float32), (C._lib.ti_bmm_s8t_s8n_s32t, torch.int32)):
        c = out.view(dtype)
        c[batch * M * N:] = 77
        alpha = (ctypes.c_float(0.5),) if dtype is torch.float32 else ()
        rc = call(a.data_ptr(), b.data_ptr(), c.data_ptr(), batch, M, N, K, *alpha, torch.cuda.current_stream().cuda_stream)
        assert rc == 0 and C._lib.ti_last_kernel() == b"scores" and _form() == "rows through the LDS, non-temporal stores"
        for i in range(batch):
            want = a[i].float() @ b[i].float().t().contiguous()
            if dtype is torch.float32:
                want *= 0.5
            assert torch.equal(c[i * M * N:(i + 1) * M * N].view(M, N).float(), want), i
        assert bool((c[batch * M * N:] == 77).all())


@pytest.mark.parametrize("batch,M,N,K,kernel", [
    (1, 1151, 1151, 128, "tile_64x64"), (65, 116, 116, 128, "tile_64x64"), (6, 305, 305, 128, "tile_64x64"), (12, 368, 368, 128, "tile_64x64"),
    (14, 362, 362, 128, "tile_64x64"), (1, 1290, 1300, 112, "tile_64x64"), (204, 160, 160, 80, "tile_256x256"), (228, 223, 192, 80, "tile_256x256")])
def test_sizes_that_the_tiled_kernels_keep(batch, M, N, K, kernel):
    """1.05 to 1.3 times as fast there."""
    import torch_int._CUDA as C
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    print(f"tiled batch={batch} M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(batch + M)
    a, b = (torch.randint(-127, 128, (batch, n, K), dtype=torch.int8, generator=g) for n in (M, N))
    ref = orc.bmm_s8t_s8n_s32t(a, b)
    assert torch.equal(C.bmm_s8t_s8n_f32t(a.to(DEV), b.to(DEV), 0.0021).cpu(), orc.epi_f32t(ref, 0.0021))
    assert C._lib.ti_last_kernel().decode() == kernel
    assert torch.equal(C.bmm_s8t_s8n_s32t(a.to(DEV), b.to(DEV)).cpu(), ref) and C._lib.ti_last_kernel().decode() == kernel
