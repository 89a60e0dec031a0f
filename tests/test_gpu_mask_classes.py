"""One mask used from two streams and rewritten by a graph's replay, and one class array to a prefill of many layers."""
import pytest
import torch

from test_gpu_attn_rows import _mask
from test_gpu_models import randomize_int8_layer
from torch_int.models.opt import Int8OPTForCausalLM, OPTConfigLite

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _call(S=640):
    import torch_int._hip_ext as X
    gen = torch.Generator(device=DEV).manual_seed(9)
    s8 = lambda *shape: torch.randn(shape, device=DEV, generator=gen).mul_(30).round_().clamp_(-127, 127).to(torch.int8)
    q, k, vt = s8(4, S, 64), s8(4, S, 64), s8(4, 64, S)
    return (lambda m: X.attn_prefill(q, k, vt, m, 0.0003, 2.0 / 127, 4)), gen


def test_one_mask_on_two_streams():
    call, gen = _call()
    mask = _mask("causal", 1, 640, 640, gen)
    want = call(mask.clone())
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    print("mask on two streams", flush=True)
    torch.cuda._sleep(20_000_000)      # this stream's kernels wait behind some milliseconds; the other's do not
    first = call(mask)
    with torch.cuda.stream(side):
        second = call(mask)
    torch.cuda.synchronize()
    assert torch.equal(first, want) and torch.equal(second, want)


def test_a_mask_that_a_replay_rewrote():
    call, gen = _call()
    mask, fresh = _mask("causal", 1, 640, 640, gen), torch.zeros(1, 1, 640, 640, device=DEV)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=side):
        mask.copy_(fresh)
    for kind in ("causal", "none", "padded"):
        print("mask from a replay", kind, flush=True)
        fresh.copy_(_mask(kind, 1, 640, 640, gen)) if kind != "none" else fresh.zero_()
        graph.replay()
        assert torch.equal(call(mask), call(fresh.clone())), kind


@pytest.mark.parametrize("mode", [torch.no_grad, torch.inference_mode])
def test_one_class_array_to_a_pass(mode, monkeypatch):
    import torch_int._hip_ext as X
    lm = Int8OPTForCausalLM(OPTConfigLite(hidden_size=128, num_hidden_layers=3, ffn_dim=512, num_attention_heads=2, vocab_size=64,
                                          max_position_embeddings=640))
    g = torch.Generator().manual_seed(2)
    for layer in lm.model.decoder.layers:
        randomize_int8_layer(layer, g)
    lm = lm.to(DEV)
    made, real = [], X.make_mask_classes
    monkeypatch.setattr(X, "make_mask_classes", lambda m: made.append(1) or real(m))
    ids = torch.randint(2, 60, (1, 600), device=DEV, generator=torch.Generator(device=DEV).manual_seed(3))
    results = []
    for classes in (True, False):
        if not classes:
            monkeypatch.setattr(X, "_classes", lambda *a: None)
        print("classes to a pass", mode.__name__, classes, flush=True)
        with mode():
            results.append(lm.model(ids).last_hidden_state)
    assert len(made) == 1 and torch.equal(*results)
