"""The layers of a model chained, one C call each with the last addition left to the next layer's first kernel, against the
same model going through its modules: logits and key / value caches bit for bit."""
import gc
import pytest
import torch

from torch_int.models.opt import Int8OPTDecoderLayer, Int8OPTForCausalLM, OPTConfigLite
from test_gpu_models import randomize_int8_layer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _generate(lm, ids, attention_mask, steps):
    results = []
    out = lm(ids, attention_mask=attention_mask, use_cache=True)
    for step in range(steps):
        results.append(out)
        if attention_mask is not None:
            attention_mask = torch.cat([attention_mask, attention_mask.new_ones(ids.shape[0], 1)], dim=1)
        out = lm(ids[:, step:step + 1], attention_mask=attention_mask, past_key_values=out.past_key_values, use_cache=True)
    return results + [out]


# rows of the prefill up to and past the 4096 at which fp32 streams change how they add fc2's output; 1, 3 and 17 sequences in
# the decode steps; with and without padding
@torch.no_grad()
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("bsz,T,layers,pad", [(1, 48, 1, False), (3, 16, 3, True), (17, 33, 2, False), (4, 1024, 2, True),
                                              (3, 1376, 3, True), (5, 1000, 2, False)])
def test_chained_layers_give_the_modules_values(bsz, T, layers, pad, half):
    torch.manual_seed(0)
    g = torch.Generator().manual_seed(T)
    lm = Int8OPTForCausalLM(OPTConfigLite(hidden_size=128, num_hidden_layers=layers, ffn_dim=512, num_attention_heads=2, vocab_size=64,
                                          max_position_embeddings=2048))
    for layer in lm.model.decoder.layers:
        randomize_int8_layer(layer, g)
    lm = lm.to(DEV)
    lm = lm.half() if half else lm
    ids = torch.randint(2, 64, (bsz, T), generator=g).to(DEV)
    keep = torch.ones(bsz, T, dtype=torch.long, device=DEV) if pad else None
    if pad:
        keep[1, :5] = 0
        keep[2, T // 2:] = 0
    print("chained", bsz, T, layers, pad, half, flush=True)
    chained = _generate(lm, ids, keep, 3)
    seen = []
    hook = lm.model.decoder.layers[-1].register_forward_hook(lambda *a: seen.append(1))
    hooked = _generate(lm, ids, keep, 3)     # the hooked layer is called as a module
    hook.remove()
    assert len(seen) == 4
    try:
        Int8OPTDecoderLayer.prefill_in_one_call = Int8OPTDecoderLayer.decode_in_one_call = False
        modules = _generate(lm, ids, keep, 3)
    finally:
        Int8OPTDecoderLayer.prefill_in_one_call = Int8OPTDecoderLayer.decode_in_one_call = True
    for a, h, b in zip(chained, hooked, modules):
        assert torch.equal(a.logits, b.logits) and torch.equal(h.logits, b.logits)
        for (ka, va), (kb, vb) in zip(a.past_key_values, b.past_key_values):
            assert torch.equal(ka, kb) and torch.equal(va, vb)


def _against_the_modules(lm, ids):
    """A cached prefill and three decode steps, chained and through the modules: logits and caches bit for bit."""
    chained = _generate(lm, ids, None, 3)
    try:
        Int8OPTDecoderLayer.prefill_in_one_call = Int8OPTDecoderLayer.decode_in_one_call = False
        modules = _generate(lm, ids, None, 3)
    finally:
        Int8OPTDecoderLayer.prefill_in_one_call = Int8OPTDecoderLayer.decode_in_one_call = True
    for a, b in zip(chained, modules):
        assert torch.equal(a.logits, b.logits)
        for (ka, va), (kb, vb) in zip(a.past_key_values, b.past_key_values):
            assert torch.equal(ka, kb) and torch.equal(va, vb)


@torch.no_grad()
@pytest.mark.parametrize("widths,bsz,T", [((256, 2048, 1024), 2, 160), ((1024, 256), 20, 48), ((128, 8192), 5, 32)])
def test_layers_of_different_widths(widths, bsz, T):
    """Layers whose fc1 has been pruned or widened one by one: the memory of a pass is that of the widest."""
    g = torch.Generator().manual_seed(T)
    lm = Int8OPTForCausalLM(OPTConfigLite(hidden_size=128, num_hidden_layers=len(widths), ffn_dim=512, num_attention_heads=2,
                                          vocab_size=64, max_position_embeddings=512))
    layers = lm.model.decoder.layers
    for i, width in enumerate(widths):
        layers[i] = randomize_int8_layer(Int8OPTDecoderLayer(128, 2, width), g)
    lm = lm.to(DEV).half()
    print("widths", widths, bsz, T, flush=True)
    _against_the_modules(lm, torch.randint(2, 64, (bsz, T), generator=g).to(DEV))


@torch.no_grad()
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("bsz,T", [(2, 512), (16, 1024)])   # scratch of the stream and of the pass
def test_a_chained_prefill_needs_hardly_more_memory_than_the_modules(bsz, T, half):
    """A byte per token and channel more, where the scratch is not the stream's: 9 (x 1, h 4, the carry 4) against 8 (h and
    fc2's output; x is gone by then)."""
    lm = Int8OPTForCausalLM(OPTConfigLite(hidden_size=1024, num_hidden_layers=3, ffn_dim=4096, num_attention_heads=8, vocab_size=64,
                                          max_position_embeddings=1024)).to(DEV)
    model = (lm.half() if half else lm).model
    ids = torch.randint(2, 64, (bsz, T), device=DEV)
    peak = {}
    try:
        for chained in (False, True):
            Int8OPTDecoderLayer.prefill_in_one_call = chained
            print("memory", bsz, T, half, chained, flush=True)
            model(ids, use_cache=True)   # the stream's kept buffers are there
            torch.cuda.synchronize()
            gc.collect()   # what earlier tests left in reference cycles would be freed during the pass, and hide as much of its peak
            torch.cuda.reset_peak_memory_stats()
            before = torch.cuda.memory_allocated()
            model(ids, use_cache=True)
            peak[chained] = torch.cuda.max_memory_allocated() - before
    finally:
        Int8OPTDecoderLayer.prefill_in_one_call = True
    assert peak[True] <= peak[False] + (bsz * T * 1024 if bsz * T > 4096 else 0)


@torch.no_grad()
def test_layers_handed_one_cache_keep_their_own_rows():
    g = torch.Generator().manual_seed(1)
    lm = Int8OPTForCausalLM(OPTConfigLite(hidden_size=128, num_hidden_layers=3, ffn_dim=512, num_attention_heads=2, vocab_size=64,
                                          max_position_embeddings=64))
    for layer in lm.model.decoder.layers:
        randomize_int8_layer(layer, g)
    lm = lm.to(DEV)
    ids = torch.randint(2, 64, (2, 21), generator=g).to(DEV)
    # the cache of a decode step has room behind it, and all layers would append there
    first = lm(ids[:, 19:20], past_key_values=lm(ids[:, :19], use_cache=True).past_key_values, use_cache=True).past_key_values[0]
    out = lm(ids[:, 20:], past_key_values=[first] * 3, use_cache=True)
    alone = lm(ids[:, 20:], past_key_values=[tuple(t.clone() for t in first) for _ in range(3)], use_cache=True)
    assert torch.equal(out.logits, alone.logits)
    for kept, want in zip(out.past_key_values, alone.past_key_values):
        assert all(torch.equal(a, b) for a, b in zip(kept, want))


@torch.no_grad()
@pytest.mark.parametrize("bsz", [1638, 1639])   # 40 heads: 65520 and 65560 matrices of values to transpose
def test_prefills_around_65535_sequences_times_heads(bsz):
    g = torch.Generator().manual_seed(bsz)
    lm = Int8OPTForCausalLM(OPTConfigLite(hidden_size=640, num_hidden_layers=2, ffn_dim=64, num_attention_heads=40, vocab_size=64,
                                          max_position_embeddings=64))
    for layer in lm.model.decoder.layers:
        randomize_int8_layer(layer, g)
    lm = lm.to(DEV).half()
    print("sequences", bsz, flush=True)
    assert (lm.model.decoder.layers[0]._prefill_checks(torch.empty((bsz, 32, 640), dtype=torch.float16, device=DEV), None)
            is not None) == (bsz * 40 <= 65535)
    _against_the_modules(lm, torch.randint(2, 64, (bsz, 32), generator=g).to(DEV))


@pytest.mark.parametrize("bsz,T,taken", [(64, 16, True), (65536, 16, False), (1025, 1024, False)])
def test_prefills_beyond_what_the_c_call_takes_go_to_the_modules(bsz, T, taken):
    layer = randomize_int8_layer(Int8OPTDecoderLayer(128, 2, 512), torch.Generator().manual_seed(2)).to(DEV)
    hidden = torch.empty((1, 1, 128), device=DEV).expand(bsz, T, 128)
    assert (layer._prefill_checks(hidden, None) is not None) == taken


@torch.no_grad()
def test_recorded_passes_keep_their_memory():
    """The layers of a prefill and of a decode step recorded into a graph after eager passes on the recording stream: later
    eager passes there need more scratch and workspace, which replaces the stream's buffers, and run between the replays."""
    g = torch.Generator().manual_seed(3)
    lm = Int8OPTForCausalLM(OPTConfigLite(hidden_size=512, num_hidden_layers=2, ffn_dim=8192, num_attention_heads=4, vocab_size=64,
                                          max_position_embeddings=512))
    for layer in lm.model.decoder.layers:
        randomize_int8_layer(layer, g)
    lm = lm.to(DEV).half()
    dec = lm.model.decoder
    prompt, one, more = (torch.randn(*shape, 512, generator=g).to(DEV).half() for shape in ((2, 80), (20, 1), (8, 128)))
    past = dec._chain_layers(torch.randn(20, 48, 512, generator=g).to(DEV).half(), None, None, True)

    def layers(hidden, cache):
        hidden = hidden.clone()
        return (hidden, *(t for kv in dec._chain_layers(hidden, None, cache, True) for t in kv))
    want, want_more = layers(prompt, None) + layers(one, past), layers(more, None)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        layers(prompt, None) + layers(one, past)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    print("recording", flush=True)
    with torch.cuda.graph(graph, stream=side):
        got = layers(prompt, None) + layers(one, past)
    for replay in range(4):
        print("replay", replay, flush=True)
        with torch.cuda.stream(side):
            eager = layers(more, None)
            filled = [torch.full((1 << 20,), 7, dtype=torch.uint8, device=DEV) for _ in range(16)]
        side.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(eager, want_more)) and all(bool((f == 7).all()) for f in filled)
        assert all(torch.equal(a, b) for a, b in zip(got, want))


@torch.no_grad()
@pytest.mark.parametrize("where", ["instance", "class", "layer"])
@pytest.mark.parametrize("bsz,T", [(20, 32), (3, 1376)])
def test_replaced_forwards_are_called(bsz, T, where, monkeypatch):
    g = torch.Generator().manual_seed(7)
    lm = Int8OPTForCausalLM(OPTConfigLite(hidden_size=128, num_hidden_layers=2, ffn_dim=512, num_attention_heads=2, vocab_size=64,
                                          max_position_embeddings=2048))
    for layer in lm.model.decoder.layers:
        randomize_int8_layer(layer, g)
    lm = lm.to(DEV).half()
    ids = torch.randint(2, 64, (bsz, T), generator=g).to(DEV)
    fc1, seen = lm.model.decoder.layers[1].fc1, []
    want = _generate(lm, ids, None, 1)
    holder = {"instance": fc1, "class": type(fc1), "layer": Int8OPTDecoderLayer}[where]
    stock = holder.forward

    def forward(*a, **k):
        seen.append(1)
        return stock(*a, **k)
    monkeypatch.setattr(holder, "forward", forward)
    print("replaced", where, bsz, T, flush=True)
    got = _generate(lm, ids, None, 1)
    assert len(seen) == (2 if where == "instance" else 4)   # a prefill and a decode step of one layer or both
    assert all(torch.equal(a.logits, b.logits) for a, b in zip(got, want))
