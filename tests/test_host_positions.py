"""Passes without an attention mask: the positions and the causal mask they use against those of a mask of ones, and when the
position table's own forward is called instead."""
import pytest
import torch

from torch_int.models import opt
from torch_int.models.opt import Int8OPTDecoder, OPTConfigLite


def _decoder():
    torch.manual_seed(0)
    return Int8OPTDecoder(OPTConfigLite(vocab_size=64, hidden_size=32, num_attention_heads=2, ffn_dim=64, num_hidden_layers=1,
                                        max_position_embeddings=40))


@pytest.mark.parametrize("past,count", [(0, 1), (0, 16), (7, 1), (39, 1), (0, 40)])
def test_positions_are_those_of_a_mask_of_ones(past, count):
    dec = _decoder()
    want = dec.embed_positions(torch.ones(3, past + count, dtype=torch.bool), past)
    got = dec._positions_in_order(past, count)
    assert got.shape == (1, count, 32) and torch.equal(got.expand_as(want), want)


def test_positions_past_the_table_are_left_to_the_lookup():
    dec = _decoder()
    assert dec._positions_in_order(0, 41) is None and dec._positions_in_order(40, 1) is None
    with pytest.raises(IndexError):
        dec.embed_positions(torch.ones(1, 41, dtype=torch.bool), 0)


def test_a_changed_position_module_is_called(monkeypatch):
    dec = _decoder()
    handle = dec.embed_positions.register_forward_hook(lambda *a: None)
    assert dec._positions_in_order(0, 4) is None
    handle.remove()
    assert dec._positions_in_order(0, 4) is not None
    dec.embed_positions.max_norm = 1.0
    assert dec._positions_in_order(0, 4) is None
    dec.embed_positions.max_norm = None
    dec.embed_positions.forward = lambda mask, past=0: None
    assert dec._positions_in_order(0, 4) is None
    del dec.embed_positions.forward
    monkeypatch.setattr(opt.OPTLearnedPositionalEmbedding, "forward", lambda self, mask, past=0: None)
    assert dec._positions_in_order(0, 4) is None


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_causal_mask(dtype):
    want = opt._additive_decoder_mask(torch.ones(2, 48, dtype=torch.bool), 48, 0, dtype, "cpu").float()
    got = opt._causal_mask(2, 48, dtype, "cpu")
    assert got.dtype is torch.float32 and got.is_contiguous() and torch.equal(got, want)
