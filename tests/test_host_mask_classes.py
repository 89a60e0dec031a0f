"""The class array of an attention mask belongs to the call that reads it: made on the stream of that call, from the mask as it is
then.  On the CPU, with stand-ins for the two launches."""
import contextlib

import pytest
import torch

from torch_int import _hip_ext as X


@pytest.fixture
def launches(monkeypatch):
    """What is launched, in order: ("classes" or "attention", stream, address of the class array)."""
    seen, stream = [], [1]
    monkeypatch.setattr(X, "_raw_stream", lambda index: stream[0])
    monkeypatch.setattr(X, "_on", lambda dev: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(X._lib, "ti_attn_mask_classes", lambda m, cls, b, t, s, st: seen.append(("classes", st, cls)) or 0)
    monkeypatch.setattr(X._lib, "ti_attn_prefill_s8_mc", lambda q, k, vt, m, cls, *a: seen.append(("attention", a[-1], cls)) or 0)
    monkeypatch.setattr(X._lib, "ti_attn_qk_softmax_q_mc", lambda q, k, m, cls, *a: seen.append(("attention", a[-1], cls)) or 0)
    return seen, stream


@pytest.mark.parametrize("with_v", [True, False])
def test_each_call_reads_classes_of_its_own_stream_and_time(launches, with_v):
    seen, stream = launches
    s8 = lambda *shape: torch.zeros(shape, dtype=torch.int8)
    q, k, vt, mask = s8(2, 592, 64), s8(2, 592, 64), s8(2, 64, 592), torch.zeros(1, 1, 592, 592)
    call = ((lambda: X.attn_prefill(q, k, vt, mask, 1e-3, 1e-2, 2, checked=True)) if with_v
            else (lambda: X.attn_qk_softmax_q(q, k, mask, 1e-3, 2, checked=True)))
    for step in range(3):
        stream[0] = 2 if step == 1 else 1          # the same mask on another stream
        if step == 2:
            version = mask._version
            mask.numpy()[...] = -1e30              # a write that does not show in the version, as a graph's replay
            assert mask._version == version
        before = len(seen)
        call()
        assert [(what, at) for what, at, _ in seen[before:]] == [("classes", stream[0]), ("attention", stream[0])]
        assert seen[-1][2] == seen[-2][2] is not None


def test_kept_classes_are_kept_for_their_stream(launches):
    seen, stream = launches
    mask = torch.zeros(1, 1, 592, 592)
    first = X.mask_classes(mask)
    assert X.mask_classes(mask) is first
    stream[0] = 2
    other = X.mask_classes(mask)
    assert other is not first and X.mask_classes(mask) is other
    stream[0] = 1
    assert X.mask_classes(mask) is first
    mask[0, 0, 0, 0] = 1.0
    assert X.mask_classes(mask) is not first and [at for _, at, _ in seen] == [1, 2, 1]
