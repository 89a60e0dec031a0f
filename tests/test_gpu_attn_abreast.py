"""Prefill attention of more heads than attn_rows_kernel takes abreast (those whose keys and values the L2 holds), at the edges of
their groups, against the chain of operators, bit for bit."""
import pytest

from test_gpu_attn_rows import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["none", "causal", "padded"])
@pytest.mark.parametrize("B,H,T,S,d", [(1, 32, 33, 2048, 128), (1, 33, 40, 2048, 128), (3, 13, 17, 2048, 128), (1, 64, 16, 2048, 128),
                                       (3, 23, 50, 1536, 80), (2, 65, 64, 1024, 128), (5, 52, 18, 512, 128)])
def test_more_heads_than_go_abreast(B, H, T, S, d, kind):
    _check(B, H, T, S, d, kind)
