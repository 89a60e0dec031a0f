"""Decode steps whose cache is as the step before left it: all layers from one C call.  Against the modules, logits and caches bit for
bit: steps past the end of the buffers, one cache continued twice, copied, cut and re-ordered caches, hooks,
padded batches, two threads on one stream."""
import copy
import threading

import pytest
import torch

from torch_int import _hip_ext
from torch_int.models.opt import Int8OPTDecoderLayer, Int8OPTForCausalLM, OPTConfigLite
from test_gpu_models import randomize_int8_layer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _model(half):
    torch.manual_seed(0)
    g = torch.Generator().manual_seed(1)
    lm = Int8OPTForCausalLM(OPTConfigLite(hidden_size=128, num_hidden_layers=3, ffn_dim=512, num_attention_heads=2, vocab_size=64,
                                          max_position_embeddings=512))
    for layer in lm.model.decoder.layers:
        randomize_int8_layer(layer, g)
    lm = lm.to(DEV)
    return lm.half() if half else lm


class _Modules:
    def __enter__(self):
        Int8OPTDecoderLayer.decode_in_one_call = False

    def __exit__(self, *exc):
        Int8OPTDecoderLayer.decode_in_one_call = True


def _same(a, b):
    assert torch.equal(a.logits, b.logits)
    for (ka, va), (kb, vb) in zip(a.past_key_values, b.past_key_values):
        assert torch.equal(ka, kb) and torch.equal(va, vb)


@torch.no_grad()
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("bsz", [1, 4, 5, 17])
def test_steps_continue_each_other(bsz, half, monkeypatch):
    lm = _model(half)
    seen = []
    real = _hip_ext.opt_layers_decode
    monkeypatch.setattr(_hip_ext, "opt_layers_decode", lambda *a: (seen.append(a[6]), real(*a)) and None)
    ids = torch.randint(2, 64, (bsz, 120), device=DEV)
    print("continue", bsz, half, flush=True)
    one = mod = lm(ids[:, :32], use_cache=True)
    for step in range(32, 120):   # buffers of 112 positions, then larger ones
        one = lm(ids[:, step:step + 1], past_key_values=one.past_key_values, use_cache=True)
        with _Modules():
            mod = lm(ids[:, step:step + 1], past_key_values=mod.past_key_values, use_cache=True)
        _same(one, mod)
    moved = [S for S in range(34, 121) if S not in seen]
    assert len(moved) <= 1, moved   # the step that found its buffers full

    fork, past = [], one.past_key_values
    for token in (3, 4):   # one cache continued twice: the second finds the position taken
        a = lm(torch.full_like(ids[:, :1], token), past_key_values=past, use_cache=True)
        with _Modules():
            b = lm(torch.full_like(ids[:, :1], token), past_key_values=mod.past_key_values, use_cache=True)
        _same(a, b)
        fork.append((a, b))
    _same(*fork[0])   # what the first holds is still there
    order = torch.arange(bsz - 1, -1, -1, device=DEV)
    past = fork[1][0].past_key_values
    for other in (copy.deepcopy(past), tuple(tuple(t[:, :, :100] for t in kv) for kv in past), lm._reorder_cache(past, order),
                  (past[1], past[0], past[2])):
        n = len(seen)
        a = lm(ids[:, :1], past_key_values=other, use_cache=True)
        assert len(seen) == n   # not what the buffers hold
        with _Modules():
            _same(a, lm(ids[:, :1], past_key_values=other, use_cache=True))
    handle = lm.model.decoder.layers[1].fc1.register_forward_hook(lambda *a: None)
    n = len(seen)
    a = lm(ids[:, :1], past_key_values=past, use_cache=True)
    handle.remove()
    assert len(seen) == n
    with _Modules():
        _same(a, lm(ids[:, :1], past_key_values=past, use_cache=True))


@torch.no_grad()
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("bsz", [3, 9])
def test_steps_of_a_padded_batch_continue_each_other(bsz, half, monkeypatch):
    lm = _model(half)
    masked = []
    real = _hip_ext.opt_layers_decode
    monkeypatch.setattr(_hip_ext, "opt_layers_decode", lambda *a: (masked.append(a[2] is not None), real(*a)) and None)
    ids = torch.randint(2, 64, (bsz, 64), device=DEV)
    keep = torch.arange(64, device=DEV) >= torch.arange(bsz, device=DEV)[:, None] * 7 % 31   # padding on the left, none to 30 tokens
    print("continue padded", bsz, half, flush=True)
    one = mod = lm(ids[:, :32], attention_mask=keep[:, :32], use_cache=True)
    for step in range(32, 64):
        mask = keep[:, :step + 1]
        one = lm(ids[:, step:step + 1], attention_mask=mask, past_key_values=one.past_key_values, use_cache=True)
        with _Modules():
            mod = lm(ids[:, step:step + 1], attention_mask=mask, past_key_values=mod.past_key_values, use_cache=True)
        _same(one, mod)
    assert masked == [True] * 31   # all but the first step, which moves the cache


@torch.no_grad()
@pytest.mark.parametrize("half", [False, True])
def test_two_threads_on_one_stream_do_not_meet(half):
    """Two caches continued at once by two threads on the default stream, against the same steps one thread after the other."""
    lm = _model(half)
    prompts = [torch.randint(2, 64, (5, 32), device=DEV) for _ in range(2)]
    tokens = [torch.randint(2, 64, (5, 60), device=DEV) for _ in range(2)]

    @torch.no_grad()
    def steps(i, out):
        step = lm(prompts[i], use_cache=True)
        for n in range(tokens[i].shape[1]):
            step = lm(tokens[i][:, n:n + 1], past_key_values=step.past_key_values, use_cache=True)
            out.append(step.logits)
        out.append(step)

    print("two threads", half, flush=True)
    alone, together = [[], []], [[], []]
    for i in range(2):
        steps(i, alone[i])
    threads = [threading.Thread(target=steps, args=(i, together[i])) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, together):
        assert len(a) == len(b) == 61 and all(torch.equal(x, y) for x, y in zip(a[:-1], b[:-1]))
        _same(a[-1], b[-1])
