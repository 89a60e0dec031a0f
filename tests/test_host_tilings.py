"""The tilings that linears and groups of them are given where a neighbouring choice measured slower, as far as the host
can tell: by the workspace of their slices and by the launches of a group."""
import ctypes

import pytest

import torch_int._CUDA as C

C._lib.ti_linear_workspace_bytes.restype = ctypes.c_int64
C._lib.ti_linear_workspace_bytes.argtypes = [ctypes.c_int64] * 3


def _slices(M, N, K):
    """Slices of a product on 128x128 tiles, whose workspace holds whole tiles when they meet in one launch (0: unsplit)."""
    rows = {M, (M + 127) // 128 * 128}
    need = C._lib.ti_linear_workspace_bytes(M, N, K)
    return {need / (r * N * 4) for r in rows}


@pytest.mark.parametrize("M,N,K", [(130, 1024, 1024), (256, 1024, 1024), (512, 1024, 1024), (384, 512, 1024), (1000, 512, 1280),
                                   (256, 2048, 1024), (240, 1408, 1280)])
def test_a_short_k_is_left_to_the_small_tiles(M, N, K):
    assert _slices(M, N, K) == {0}


@pytest.mark.parametrize("M,N", [(256, 1024), (512, 1024), (130, 2048), (384, 512)])
def test_from_1536_on_few_tiles_are_split(M, N):
    assert _slices(M, N, 1536) & {2, 3, 4}


@pytest.mark.parametrize("M,N,K,slices", [(130, 2048, 8192, 4), (256, 2048, 8192, 4), (256, 1024, 8192, 8), (256, 2048, 16384, 8),
                                          (900, 1024, 4096, 2), (1024, 1024, 4096, 2), (700, 1024, 4096, 4), (1000, 1024, 16384, 4)])
def test_slices_of_products_on_128x128_tiles(M, N, K, slices):
    """Four that meet in one launch rather than eight short ones on a full chip; two rather than four short ones on a full chip."""
    assert slices in _slices(M, N, K)


@pytest.mark.parametrize("M,N,one_launch", [(2112, 5120, 1), (2064, 5120, 1), (2048, 2048, 1), (5696, 7168, 0)])
def test_groups_that_are_one_launch(M, N, one_launch):
    assert C._lib.ti_linear_group_is_one_launch(ctypes.c_int64(M), ctypes.c_int64(N), ctypes.c_int64(N), 3) == one_launch


@pytest.mark.parametrize("M,N,K,cut", [(1538, 20480, 5120, 2), (2060, 5120, 20480, 12), (1029, 16384, 4096, 5), (2064, 8192, 2048, 16),
                                       (2112, 5120, 20480, 64), (2368, 5120, 5120, 0), (2112, 5120, 5120, 0)])
def test_rows_that_are_cut_off_the_end(M, N, K, cut):
    """A few rows stream the weights in less time than a further round of tiles takes; 64 on small weights do not."""
    assert C._lib.ti_linear_row_split(ctypes.c_int64(M), ctypes.c_int64(N), ctypes.c_int64(K)) == cut


@pytest.mark.parametrize("M,N,K,slices", [(376, 5120, 20480, 4), (368, 2560, 10240, 5), (406, 4096, 16384, 8)])
def test_room_for_the_slices_of_the_accumulating_epilogue(M, N, K, slices):
    need = C._lib.ti_linear_acc_workspace_bytes(M, N, K)
    assert need >= C._lib.ti_linear_workspace_bytes(M, N, K) and need == slices * M * N * 4
    for m in (1, 16, 40, 64, 512, 1024, 1030, 2112, 8192):     # never less than the others' room
        assert C._lib.ti_linear_acc_workspace_bytes(m, N, K) >= C._lib.ti_linear_workspace_bytes(m, N, K)
