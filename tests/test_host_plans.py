"""What the one-call paths of torch_int.models.opt stand for and what they leave to the modules, on the CPU (nothing is
launched: a plan is built from CPU tensors, and the checks before a call take stand-ins)."""
import types

import pytest
import torch

from torch_int import _hip_ext
from torch_int.models.opt import Int8OPTAttention, Int8OPTDecoderLayer
from torch_int.nn.fused import LayerNormQ
from torch_int.nn.linear import W8A8B8O8LinearReLU


def _layer():
    g = torch.Generator().manual_seed(6)
    layer = Int8OPTDecoderLayer(128, 2, 512)
    for lin in (layer.self_attn.q_proj, layer.self_attn.k_proj, layer.self_attn.v_proj, layer.self_attn.out_proj, layer.fc1, layer.fc2):
        lin.weight = torch.randint(-127, 128, lin.weight.shape, dtype=torch.int8, generator=g)
    return layer


@pytest.mark.parametrize("name", ["self_attn", "fc1", "fc2", "self_attn_layer_norm", "final_layer_norm", "self_attn.q_proj",
                                  "self_attn.out_proj", "self_attn.qk_bmm"])
@pytest.mark.parametrize("native", [True, False])
def test_a_forward_of_a_modules_own_is_not_passed_by(name, native, monkeypatch):
    """The plan behind the one-call paths (CPU tensors do for building it) does not stand for a layer one of whose modules has
    had its forward replaced, and does again once it is taken back."""
    if not native:
        monkeypatch.setattr(_hip_ext, "plan_current", _hip_ext._plan_current)
    layer, dev = _layer(), torch.device("cpu")
    mod = layer.get_submodule(name)
    assert layer._decode_plan(False, dev) is not None
    mod.forward = lambda *a, **k: None
    assert layer._decode_plan(False, dev) is None and layer._decode_plan(False, dev) is None
    del mod.forward
    assert layer._decode_plan(False, dev) is not None
    mod.forward = lambda *a, **k: None   # ... also where no plan was there before
    del layer.__dict__["_ti_decode_plan"]
    assert layer._decode_plan(False, dev) is None
    del mod.forward
    hook = mod.register_forward_hook(lambda *a: None)
    assert layer._decode_plan(False, dev) is None
    hook.remove()
    assert layer._decode_plan(False, dev) is not None


@pytest.mark.parametrize("cls", [Int8OPTAttention, LayerNormQ, W8A8B8O8LinearReLU])
def test_a_forward_replaced_on_a_class_is_not_passed_by(cls, monkeypatch):
    stream = types.SimpleNamespace(is_cuda=True, is_contiguous=lambda: True, dtype=torch.float32)
    assert Int8OPTDecoderLayer._one_call_tensors(stream, None) == (True, None)
    monkeypatch.setattr(cls, "forward", lambda *a, **k: None)
    assert Int8OPTDecoderLayer._one_call_tensors(stream, None)[0] is False


def test_two_continuations_of_one_past_get_rooms_of_their_own():
    """A decode step takes the position behind a past before its launches, not after them: another thread that continues the same
    past meanwhile, or another layer handed the same cache, gets a copy; a step that is not taken gives the position back."""
    from torch_int.models import opt
    past = tuple(opt._kv_view(opt._KVBuffer(torch.zeros(2, 3, 32, 16, dtype=torch.int8), 10), 10) for _ in range(2))
    first, second = opt._kv_rooms(past), opt._kv_rooms(past)
    assert first[0] is past[0]._ti_kv and first[1] is past[1]._ti_kv
    assert len({id(kv) for kv in first + second}) == 4 and all(kv.filled == 11 for kv in first + second)
    both = opt._kv_rooms((past[0], past[0]))   # a key tensor handed as the value tensor too
    assert both[0] is not both[1]
    opt._kv_give_back(first)
    assert opt._kv_rooms(past)[0] is first[0]


def test_a_cache_without_room_is_left_to_the_kernel_only_where_it_lies_as_the_kernel_reads_it():
    """Bare buffers only for both halves of a cache and for one pitch from row to row, head to head and sequence to sequence; any other
    cache is copied first."""
    from torch_int.models import opt
    flat = torch.arange(2 * 3 * 10 * 16, dtype=torch.int32).to(torch.int8)
    plain = flat.view(2, 3, 10, 16)
    long = torch.cat([plain, plain], 2)[:, :, :10]
    others = [torch.cat([plain, plain], 1)[:, :3], plain.transpose(0, 1).contiguous().transpose(0, 1), plain[:, :1].expand(2, 3, 10, 16),
              plain.transpose(2, 3).contiguous().transpose(2, 3), torch.cat([flat[:3], flat])[3:].view(2, 3, 10, 16), plain[:, :, :0]]
    for past, bare in ([((plain, plain), True), ((long, long), True), ((plain, long), False)]
                       + [(pair, False) for o in others for pair in ((o, o), (plain[:, :, :o.shape[2]], o))]):
        kk, vv = opt._kv_rooms(past)
        S = past[0].shape[2]
        assert kk.bare is vv.bare is bare and kk.filled == vv.filled == S + 1 and kk.buf.shape[2] > S
        if not bare:
            assert torch.equal(kk.buf[:, :, :S], past[0]) and torch.equal(vv.buf[:, :, :S], past[1])
    kept = opt._kv_view(opt._KVBuffer(torch.zeros(2, 3, 80, 16, dtype=torch.int8), 10), 10)
    assert [kv.bare for kv in opt._kv_rooms((kept, plain))] == [False, False]


def test_a_16_bit_mask_is_converted_by_every_call():
    """A layer's fp32 copy of an fp16 mask is not kept on the mask: another stream would not wait for it, a graph that is recorded
    would not make it, a replay that rewrites the mask does not show in its version, and a tensor of inference mode has none."""
    from torch_int.models import opt

    class Mask:
        is_cuda, dtype = True, torch.float16
        value = 1.0

        def float(self):
            return torch.full((1,), self.value)

        @property
        def _version(self):
            raise RuntimeError("Inference tensors do not track version counter.")

    mask = Mask()
    first = opt._mask_as_fp32(mask)
    mask.value = 2.0
    second = opt._mask_as_fp32(mask)
    assert first is not second and first.item() == 1.0 and second.item() == 2.0
