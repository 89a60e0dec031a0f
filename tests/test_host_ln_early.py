"""Where the LayerNorm-quantiser fetches gamma and beta with the row: not at the sizes that it made slower (up to 1.06 times the time)."""
import ctypes

import pytest

import torch_int._CUDA as C

DQ, ADD, READ, ADD_F32 = range(4)


@pytest.mark.parametrize("mode,half,rows,width,early", [
    (DQ, 0, 256, 5120, 1), (DQ, 0, 257, 5120, 0), (DQ, 0, 2048, 5120, 0), (ADD, 0, 4096, 2048, 0),
    (READ, 0, 4096, 2560, 0), (READ, 0, 7018, 3072, 0), (READ, 0, 2048, 4096, 0), (READ, 0, 1630, 5120, 0), (READ, 0, 1024, 2048, 1),
    (READ, 0, 1023, 2048, 0), (READ, 0, 2048, 768, 1), (READ, 1, 2560, 768, 0), (ADD, 1, 2560, 768, 0), (READ, 1, 4096, 768, 1), (DQ, 1, 2048, 768, 1),
    (ADD_F32, 1, 2048, 768, 1), (READ, 1, 2048, 1024, 1), (READ, 1, 2048, 2560, 0), (READ, 1, 2112, 2560, 1), (READ, 1, 1024, 2048, 1),
    (READ, 1, 1024, 3072, 1), (ADD, 1, 1024, 2560, 1), (ADD, 1, 512, 2560, 0)])
def test_gamma_and_beta_come_with_the_row(mode, half, rows, width, early):
    call = C._lib.ti_selftest_ln_early
    assert call(mode, half, ctypes.c_int64(rows), width, 256) == early
