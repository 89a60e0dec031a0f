"""Batched products of a short inner dimension that 16 does not divide (csrc/bmm_any.h): rows shorter than a chunk, which begin at any
byte, and the line up to which a thread to an output has them, against the oracle bit for bit."""
import ctypes

import pytest
import torch

from test_gpu_any_rows import _case

pytestmark = pytest.mark.gpu


def _form():
    import torch_int._CUDA as C
    C._lib.ti_last_kernel_form.restype = ctypes.c_char_p
    return C._lib.ti_last_kernel_form().decode()


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 7, 8, 11, 13, 15, 17, 31])
def test_short_rows_of_many_outputs(K):
    """The tiles and the strips at such K: outputs enough that neither is left to a thread to an output."""
    for off_a, off_b in ((0, 0), (1, 2), (3, 1)):
        assert _case(2 if K > 4 else 6, 1100, 1100, K, off_a, off_b) == "any"
        assert K < 3 or _form() != "a thread to an output"
        assert _case(220, 16, 1600, K, off_a, off_b) == "any_skinny"
        assert K < 3 or _form() == "strips of 16"


@pytest.mark.parametrize("batch,M,N,K", [(5, 152, 80, 15), (13, 18, 80, 15), (8, 76, 80, 14), (4, 21, 128, 9), (2, 55, 80, 24), (18, 24, 128, 24),
                                         (64, 1, 128, 7), (300, 1, 128, 9), (3, 70, 70, 17), (234, 142, 1, 17)])
def test_a_short_k_of_few_outputs(batch, M, N, K):
    """1.1 to 3.8 times as fast with a thread to an output."""
    _case(batch, M, N, K)
    assert _form() == "a thread to an output"


@pytest.mark.parametrize("batch,M,N,K", [(36, 61, 61, 32), (9, 150, 64, 40), (40, 200, 80, 17), (2, 40, 128, 49), (4, 1, 128, 47), (300, 1, 128, 33)])
def test_more_outputs_or_a_longer_k(batch, M, N, K):
    _case(batch, M, N, K)
    assert _form() != "a thread to an output"


@pytest.mark.parametrize("batch,M,N,K,form", [(18, 130, 64, 130, "64x64"), (9, 129, 63, 143, "64x64"), (256, 129, 127, 53, "64x128"),
                                              (400, 60, 100, 150, "64x128"), (128, 129, 120, 53, "128x128"), (64, 777, 80, 777, "128x128")])
def test_every_tile(batch, M, N, K, form):
    """Each tiling over rows, columns and steps that end inside it."""
    _case(batch, M, N, K, 3, 1)
    assert _form() == form
