"""The form that a prefill attention takes on both sides of the lines of the rule, where the neighbouring form measured
slower, and where the classes of a mask are made for it."""
import ctypes

import pytest

import torch_int._CUDA as C
from torch_int import _hip_ext as X

SINGLE, ROWS, SWEEPS = 1, 2, 3
C._lib.ti_attn_prefill_form.argtypes = [ctypes.c_int64] * 4 + [ctypes.c_int] * 2


@pytest.mark.parametrize("BH,T,S,d,mask,classes,form", [
    (128, 80, 80, 64, 1, 0, SINGLE), (12, 80, 80, 64, 1, 0, ROWS), (51, 80, 80, 64, 1, 0, ROWS), (80, 128, 128, 128, 1, 0, ROWS),
    (81, 128, 128, 128, 0, 0, SINGLE), (12, 64, 64, 64, 1, 0, SINGLE), (64, 256, 256, 64, 1, 0, ROWS), (65, 256, 256, 64, 1, 0, SINGLE),
    (256, 122, 368, 128, 1, 1, SINGLE), (80, 368, 368, 128, 1, 1, SINGLE), (256, 128, 384, 128, 1, 1, SINGLE),
    (160, 384, 384, 128, 1, 1, ROWS), (160, 384, 384, 128, 1, 0, SINGLE), (160, 384, 384, 128, 0, 0, SINGLE),
    (160, 512, 512, 128, 1, 1, ROWS), (160, 512, 512, 128, 1, 0, SINGLE), (160, 512, 512, 128, 0, 0, ROWS),
    (160, 192, 576, 128, 0, 0, SINGLE), (160, 192, 576, 128, 1, 1, ROWS), (64, 512, 512, 128, 0, 0, SINGLE),
    (160, 592, 592, 128, 1, 0, ROWS), (320, 2048, 2048, 128, 0, 0, ROWS), (8, 2064, 2064, 64, 1, 1, SWEEPS),
    (8, 100, 100, 64, 1, 0, 0)])
def test_forms(BH, T, S, d, mask, classes, form):
    assert C._lib.ti_attn_prefill_form(BH, T, S, d, mask, classes) == form


@pytest.mark.parametrize("BH,T,S,d,pv,wanted", [
    (160, 512, 512, 128, 1, 1), (160, 512, 512, 128, 0, 0), (160, 368, 368, 128, 1, 0), (160, 384, 384, 128, 1, 1),
    (12, 512, 512, 64, 1, 0), (12, 592, 592, 64, 1, 1), (12, 592, 592, 64, 0, 1), (12, 4096, 4096, 64, 1, 1), (12, 4112, 4112, 64, 1, 0),
    (12, 600, 600, 64, 1, 0), (256, 122, 368, 128, 1, 0)])
def test_classes_where_the_form_turns_on_them(BH, T, S, d, pv, wanted):
    assert X._lib.ti_attn_wants_mask_classes(BH, T, S, d, pv) == wanted
