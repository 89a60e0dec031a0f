"""Batched products with a head size as the inner dimension and 32-bit outputs (csrc/bmm_scores.h) against the oracle bit for bit: the
three forms, head sizes inside and at the end of a slice, lengths at the edges of blocks, pieces of rows and tiles."""
import ctypes

import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(batch, M, N, K):
    import torch_int._CUDA as C
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    print(f"batch={batch} M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(batch + 3 * M + 5 * N + K)
    a, b = (torch.randint(-127, 128, (batch, n, K), dtype=torch.int8, generator=g) for n in (M, N))
    ref = orc.bmm_s8t_s8n_s32t(a, b)
    # outputs inside a larger tensor: what lies behind them stays as it was
    out = torch.full((batch * M * N + 64,), 77.0, device=DEV)
    lib = C._lib
    ad, bd = a.to(DEV), b.to(DEV)
    rc = lib.ti_bmm_s8t_s8n_f32t(ad.data_ptr(), bd.data_ptr(), out.data_ptr(), batch, M, N, K, 0.0021,
                                 torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and lib.ti_last_kernel() == b"scores"
    assert torch.equal(out[:batch * M * N].cpu().view(batch, M, N), orc.epi_f32t(ref, 0.0021))
    assert bool((out[batch * M * N:] == 77.0).all())
    assert torch.equal(C.bmm_s8t_s8n_s32t(ad, bd).cpu(), ref)
    assert lib.ti_last_kernel() == b"scores"


@pytest.mark.parametrize("K", [16, 48, 64, 80, 112, 128])
@pytest.mark.parametrize("M,N", [(17, 1), (33, 31), (64, 66), (127, 129), (130, 257)])
def test_few_outputs(M, N, K):
    _case(3, M, N, K)


@pytest.mark.parametrize("batch,M,N,K", [(200, 33, 130, 64), (210, 40, 67, 80), (70, 129, 65, 128)])
def test_waves_of_32_by_32(batch, M, N, K):
    _case(batch, M, N, K)


@pytest.mark.parametrize("batch,M,N,K", [(40, 200, 211, 128), (41, 257, 130, 112), (9, 17, 12000, 128), (27, 512, 512, 80), (120, 129, 387, 96),
                                         (12, 1000, 2050, 48)])
def test_rows_through_the_lds(batch, M, N, K):
    _case(batch, M, N, K)
