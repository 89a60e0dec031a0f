"""Batched products whose rows are not whole aligned 16-byte chunks (csrc/bmm_any.h): inner dimensions that 16 does not divide and
operands that begin anywhere, against the oracle bit for bit: every tile and the few-row kernel, edges of chunks, steps, tiles."""
import ctypes

import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _operand(g, batch, rows, K, offset):
    """On the device at `offset` bytes from an aligned address, and on the host."""
    flat = torch.randint(-127, 128, (batch * rows * K + offset,), dtype=torch.int8, generator=g)
    t = flat.to(DEV)[offset:].view(batch, rows, K)
    assert t.data_ptr() % 16 == offset
    return t, flat[offset:].view(batch, rows, K)


def _case(batch, M, N, K, off_a=0, off_b=0):
    import torch_int._CUDA as C
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    print(f"batch={batch} M={M} N={N} K={K} offsets {off_a} {off_b}", flush=True)
    g = torch.Generator().manual_seed(batch * 7 + M * 5 + N * 3 + K)
    (ad, a), (bd, b) = _operand(g, batch, M, K, off_a), _operand(g, batch, N, K, off_b)
    ref = orc.bmm_s8t_s8n_s32t(a, b)
    assert torch.equal(C.bmm_s8t_s8n_s32t(ad, bd).cpu(), ref)
    kernel = C._lib.ti_last_kernel().decode()
    assert torch.equal(C.bmm_s8t_s8n_s8t(ad, bd, 0.0021).cpu(), orc.epi_s8t(ref, 0.0021))
    assert torch.equal(C.bmm_s8t_s8n_f32t(ad, bd, 0.0021).cpu(), orc.epi_f32t(ref, 0.0021))
    return kernel


@pytest.mark.parametrize("K", [1, 3, 15, 17, 30, 33, 127, 129, 143, 255, 257, 517, 2047])
def test_inner_dimensions(K):
    assert _case(5, 1, 66, K) == "any_skinny"       # one wave to many, ragged strips of rows
    assert _case(3, 16, 15, K) == "any_skinny"
    assert _case(3, 17, 33, K) == "any"
    assert _case(2, 65, 128, K) == "any"


@pytest.mark.parametrize("M,N", [(64, 64), (65, 63), (129, 130), (300, 80), (1, 1), (17, 1), (40, 500)])
def test_output_edges(M, N):
    assert _case(9, M, N, 75) == ("any_skinny" if M <= 16 else "any")


def test_every_tile_and_many_batches():
    assert _case(600, 1, 20, 37) == "any_skinny"
    assert _case(300, 33, 20, 37) == "any"          # 64x64
    assert _case(400, 60, 100, 150) == "any"        # 64x128
    assert _case(140, 250, 140, 150) == "any"       # 128x128


@pytest.mark.parametrize("off_a,off_b", [(1, 0), (0, 3), (2, 5), (8, 8), (15, 1)])
def test_operands_that_begin_anywhere(off_a, off_b):
    for K in (64, 100, 256):                        # 16 divides the first and the last
        assert _case(4, 3, 40, K, off_a, off_b) == "any_skinny"
        assert _case(3, 70, 40, K, off_a, off_b) == "any"


@pytest.mark.parametrize("batch,M,N,K", [(1, 2100, 2100, 77), (2, 256, 256, 4097), (1, 1500, 3400, 33)])
def test_products_that_are_padded(batch, M, N, K):
    assert not _case(batch, M, N, K).startswith("any")
