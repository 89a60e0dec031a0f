"""ti_decode_attn_s8_from with two to four new tokens at the edges of its forms, against the step that appends in place: the
context, the rows in the buffers and the source left as it was, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T", [2, 3, 4])
@pytest.mark.parametrize("heads,d,S,spare", [(6, 128, 9, 0), (6, 128, 640, 2), (5, 128, 641, 0), (6, 64, 1280, 1), (3, 64, 1300, 0),
                                             (4, 80, 333, 5), (4, 48, 70, 0), (3, 128, 5, 0)])
def test_tokens_over_a_moved_cache(heads, d, S, spare, T):
    import torch_int._CUDA as C
    print("decode move", T, heads, d, S, spare, flush=True)
    g = torch.Generator(device=DEV).manual_seed(heads + 3 * d + 7 * S + T)
    s8 = lambda *shape: torch.randint(-127, 128, shape, dtype=torch.int8, device=DEV, generator=g)
    cap, past_cap = S + 16, S - T + spare
    q, kn, vn, kp, vp = s8(heads, T, d), s8(heads, T, d), s8(heads, T, d), s8(heads, past_cap, d), s8(heads, past_cap, d)
    mask = torch.randn(heads, T, S, device=DEV, generator=g)
    stream = torch.cuda.current_stream().cuda_stream
    kept, results = (kp.clone(), vp.clone()), []
    for moved in (True, False):
        kb, vb, ctx = s8(heads, cap, d).fill_(3), s8(heads, cap, d).fill_(4), s8(heads, T, d)
        if not moved:
            kb[:, :S - T], vb[:, :S - T] = kp[:, :S - T], vp[:, :S - T]
        head = [t.data_ptr() for t in (q, kn, vn)]
        tail = [kb.data_ptr(), vb.data_ptr(), mask.data_ptr(), ctx.data_ptr()]
        if moved:
            rc = C._lib.ti_decode_attn_s8_from(*_args(head + [kp.data_ptr(), vp.data_ptr()], past_cap, tail, heads, T, d, cap, S, stream))
        else:
            rc = C._lib.ti_decode_attn_s8(*_args(head, None, tail + [None], heads, T, d, cap, S, stream))
        assert rc == 0, C._lib.ti_last_error()
        results.append((ctx, kb, vb))
    assert all(torch.equal(a, b) for a, b in zip(*results)) and torch.equal(kp, kept[0]) and torch.equal(vp, kept[1])


def _args(first, past_cap, tail, heads, T, d, cap, S, stream):
    import ctypes
    vp, i64, f32 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_float
    middle = [] if past_cap is None else [i64(past_cap)]
    return [vp(p) for p in first] + middle + [vp(p) for p in tail] + [i64(n) for n in (heads, T, d, cap, S, 1)] + [f32(1e-3), f32(2.0 / 127), vp(stream)]
