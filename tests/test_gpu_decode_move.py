"""A decode step that moves its cache to other buffers on the way (ti_decode_attn_s8_from, csrc/decode_attn.hip): the context, the
rows in the buffers and the source left as it was, against the step that appends in place, bit for bit, at the edges of
every form; and a model's first step after a prefill against the module path."""
import ctypes

import pytest
import torch

from torch_int.models.opt import Int8OPTForCausalLM, OPTConfigLite
from test_gpu_models import randomize_int8_layer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _cases():
    for d, rows in ((128, 8), (64, 16)):
        for groups in (8, 16, 32, 64, 96, 128, 192, 256):
            yield 6, d, groups * rows, 0
            yield 6, d, groups * rows + 1, 3
    yield 4, 80, 509, 0        # rows that do not fill the lanes
    yield 4, 48, 63, 16
    yield 260, 64, 2001, 1     # eight waves of 16 groups
    yield 516, 16, 2050, 5     # streaming, more than 512 heads
    yield 3, 128, 2, 0         # one row to move


@pytest.mark.parametrize("heads,d,S,spare", list(_cases()))
def test_a_moved_cache_gives_the_same_bits(heads, d, S, spare):
    import torch_int._hip_ext as X
    print("decode move", heads, d, S, spare, flush=True)
    g = torch.Generator(device=DEV).manual_seed(heads + 3 * d + 7 * S)

    def s8(*shape):
        return torch.randint(-127, 128, shape, dtype=torch.int8, device=DEV, generator=g)

    cap, past_cap = S + 16, S - 1 + spare
    q, kn, vn, kp, vp = s8(heads, 1, 1, d), s8(heads, 1, 1, d), s8(heads, 1, 1, d), s8(heads, 1, past_cap, d), s8(heads, 1, past_cap, d)
    mask = torch.randn(heads, 1, 1, S, device=DEV, generator=g)
    mask[0, ..., : S // 2] = torch.finfo(torch.float32).min
    mask[-1] = float("-inf")
    kb, vb = s8(heads, 1, cap, d), s8(heads, 1, cap, d)
    k_ref, v_ref = kb.clone(), vb.clone()
    k_ref[:, :, :S - 1], v_ref[:, :, :S - 1] = kp[:, :, :S - 1], vp[:, :, :S - 1]
    want, _ = X.decode_attention(q, kn, vn, k_ref, v_ref, S - 1, mask, 3e-4, 4e-3)
    before = kp.clone(), vp.clone()
    ctx = torch.empty(heads, 1, d, dtype=torch.int8, device=DEV)
    f = X._lib.ti_decode_attn_s8_from
    p, n = ctypes.c_void_p, ctypes.c_int64
    f.argtypes, f.restype = [p] * 5 + [n] + [p] * 4 + [n] * 6 + [ctypes.c_float] * 2 + [p], ctypes.c_int
    args = (heads, 1, d, cap, S, 1, 3e-4, 4e-3, torch.cuda.current_stream().cuda_stream)
    ptrs = [t.data_ptr() for t in (q, kn, vn, kp, vp)]
    bufs = [t.data_ptr() for t in (kb, vb, mask, ctx)]
    assert f(*ptrs, past_cap, *bufs, *args) == 0
    assert torch.equal(ctx.view(-1), want.reshape(-1))
    assert torch.equal(kb, k_ref) and torch.equal(vb, v_ref)   # rows beyond the new one keep their bytes too
    assert torch.equal(kp, before[0]) and torch.equal(vp, before[1])
    assert f(*ptrs, S - 2, *bufs, *args) != 0                  # refused: fewer rows than the step continues
    assert f(*ptrs[:4], 0, past_cap, *bufs, *args) != 0        # refused: one cache moved, the other not


def _strided(t):      # every second head of a wider tensor: rows 2 x 21 positions apart from head to head
    return torch.stack([t, t + 1], 2).flatten(1, 2)[:, ::2]


def _cut(t):          # the first heads of more: no single pitch from head to head
    return torch.cat([t, t], 1)[:, :t.shape[1]]


def _narrowed(t):     # the first positions of longer rows
    return torch.cat([t, t], 2)[:, :, :t.shape[2]]


def _misaligned(t):
    flat = torch.zeros(t.numel() + 3, dtype=t.dtype, device=t.device)[3:]
    return flat.copy_(t.reshape(-1)).view(t.shape)


@torch.no_grad()
@pytest.mark.parametrize("form", [torch.Tensor.contiguous, _strided, _cut, _narrowed, _misaligned])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_first_steps_over_any_cache_are_those_of_the_modules(form, dtype):
    g = torch.Generator().manual_seed(3)
    lm = Int8OPTForCausalLM(OPTConfigLite(hidden_size=128, num_hidden_layers=3, ffn_dim=512, num_attention_heads=2, vocab_size=64))
    for layer in lm.model.decoder.layers:
        randomize_int8_layer(layer, g)
    lm = lm.to(DEV).to(dtype)
    past = [tuple(form(torch.randint(-127, 128, (2, 2, 21, 64), dtype=torch.int8, generator=g).to(DEV)) for _ in range(2))
            for _ in range(3)]
    token = torch.tensor([[5], [9]], device=DEV)

    def two_steps():
        out = lm(token, past_key_values=past, use_cache=True)
        end = lm(token, past_key_values=out.past_key_values, use_cache=True)
        return [end.logits, out.logits, *(t.clone() for kv in end.past_key_values for t in kv)]

    got = two_steps()
    for layer in lm.model.decoder.layers:
        layer.decode_in_one_call = False
    for a, b in zip(got, two_steps()):
        assert torch.equal(a, b)
