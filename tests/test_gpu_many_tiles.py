"""Batched products of more output tiles than one row of a grid can have threads for (2^32: a launch drops the rest silently): 65535
batches whose outputs are a column or a row.  All batches share an operand, so that one exact matrix product is the reference."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M,N,K,kernel", [(16448, 1, 49, b"any"), (1, 16400, 49, b"any_skinny"), (32896, 1, 16, b"scores")])
def test_more_than_2_to_32_threads(M, N, K, kernel):
    import torch_int._CUDA as C
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    batch = 65535
    print(f"many tiles {batch} x {M} x {N} x {K}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M)
    rows = max(M, N)
    one = torch.randint(-127, 128, (rows, K), dtype=torch.int8, device=DEV, generator=g)
    shared = torch.empty((batch, rows, K), dtype=torch.int8, device=DEV)
    shared.copy_(one.expand(batch, rows, K))
    own = torch.randint(-127, 128, (batch, 1, K), dtype=torch.int8, device=DEV, generator=g)
    out = C.bmm_s8t_s8n_s32t(shared, own) if M > 1 else C.bmm_s8t_s8n_s32t(own, shared)
    assert C._lib.ti_last_kernel() == kernel
    del shared
    for lo in range(0, batch, 8192):   # sums below 2^24: exact in fp32
        want = own[lo:lo + 8192, 0].float() @ one.float().t().contiguous()
        assert torch.equal(out[lo:lo + 8192].view(want.shape).float(), want), lo
    del out, want
    torch.cuda.empty_cache()
