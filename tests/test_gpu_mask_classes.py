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


def _summed_mask(kind, B, T, S, gen):
    """Causal part and padding of a 16-bit (or 32-bit) model as they add up: the lowest value, and -infinity where both say no."""
    dtype = torch.float32 if kind.startswith("fp32") else torch.float16
    low = torch.finfo(dtype).min
    m = torch.zeros(B, 1, T, S, device=DEV, dtype=dtype)
    causal = torch.zeros(T, S, device=DEV, dtype=dtype).masked_fill_(torch.ones(T, S, dtype=torch.bool, device=DEV).triu(1 + S - T), low)
    for b in range(B):
        cut = S - 13 - (b * S) // (2 * B)          # keys that are tokens
        if kind.endswith("left"):
            m[b, ..., :S - cut] = low              # queries in the padding are masked throughout
        else:
            m[b, ..., cut:] = low
    m = (m + causal).float()
    assert (m == low).any() and (torch.isinf(m).any() or kind.endswith("left"))
    return m


@pytest.mark.parametrize("kind", ["fp16 right", "fp16 left", "fp32 right", "fp32 left"])
@pytest.mark.parametrize("B,H,T,S,d", [(2, 2, 384, 384, 80), (3, 1, 528, 528, 128), (2, 2, 1040, 1040, 64), (2, 1, 500, 768, 128),
                                       (1, 2, 2048, 2048, 128), (2, 1, 2064, 2064, 64)])
def test_padding_on_a_causal_mask(B, H, T, S, d, kind, monkeypatch):
    import test_gpu_attn_rows as rows
    monkeypatch.setattr(rows, "_mask", _summed_mask)
    rows._check(B, H, T, S, d, kind)


@pytest.mark.parametrize("kind", ["fp16 right", "fp32 right"])
def test_masked_tiles_are_known_where_padding_meets_them(kind):
    import torch_int._hip_ext as X
    mask = _summed_mask(kind, 2, 512, 512, None)
    classes = X.make_mask_classes(mask).view(2, 8, 2).cpu()
    tiles = mask.view(2, 8, 64, 2, 256).cpu()
    for b in range(2):
        for i in range(8):
            for j in range(2):
                t = tiles[b, i, :, j]
                want = 1 if (t == 0).all() else 0 if (t > -6e4).any() else 3 if (t != t[0, 0]).any() or t[0, 0] > -1e30 else 2
                assert classes[b, i, j] == want, (b, i, j)
    assert (classes[:, :4, 1] == 3).all()          # above the diagonal
