"""Passes without an attention mask against the same passes with the positions and the mask made from a mask of ones: hidden
states, logits and caches bit for bit, as chained layers, through the modules (a hook) and with every hidden state returned."""
import pytest
import torch

from torch_int.models.opt import Int8OPTDecoder, Int8OPTForCausalLM, OPTConfigLite
from test_gpu_models import randomize_int8_layer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("way", ["chained", "modules", "states"])
def test_no_mask_is_a_mask_of_ones(way, dtype, monkeypatch):
    g = torch.Generator().manual_seed(7)
    lm = Int8OPTForCausalLM(OPTConfigLite(hidden_size=128, num_hidden_layers=3, ffn_dim=512, num_attention_heads=2, vocab_size=64,
                                          max_position_embeddings=64))
    for layer in lm.model.decoder.layers:
        randomize_int8_layer(layer, g)
    lm = lm.to(DEV).to(dtype)
    if way == "modules":
        lm.model.decoder.layers[0].self_attn.register_forward_hook(lambda *a: None)
    more = {"output_hidden_states": True} if way == "states" else {}
    ids = torch.randint(2, 60, (2, 37), device=DEV, generator=torch.Generator(device=DEV).manual_seed(3))
    results = []
    for masked in (False, True):
        if masked:
            monkeypatch.setattr(Int8OPTDecoder, "_positions_in_order", lambda *a: None)
        print("in order", way, dtype, masked, flush=True)
        with torch.no_grad():
            out = lm.model(ids, use_cache=True, **more)
            past = [tuple(t[:, :, :37].contiguous() for t in kv) for kv in out.past_key_values]
            kept = [out.last_hidden_state, *(out.hidden_states or ()), *(t for kv in out.past_key_values for t in kv)]
            for step in range(3):
                out = lm(ids[:, step:step + 1], past_key_values=past, use_cache=True, **more)
                past = out.past_key_values
                kept += [out.logits, *(out.hidden_states or ())]
        results.append(kept + [t for kv in past for t in kv])
    assert len(results[0]) == len(results[1]) and all(torch.equal(a, b) for a, b in zip(*results))
