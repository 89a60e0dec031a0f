"""The LayerNorm-quantiser on both sides of the row counts from which gamma and beta come with the row, and to which, against the oracle."""
import pytest

from test_gpu_ln_widths import test_every_form_is_exact as _every_form

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [256, 257, 1023, 1024, 2047, 2048])
@pytest.mark.parametrize("width", [768, 1024, 1028, 2048])
def test_where_gamma_and_beta_come_with_the_row(rows, width):
    _every_form(rows, width)
