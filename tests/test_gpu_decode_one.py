"""The decode attention of one new token (decode_attn_one_kernel, csrc/decode_attn.hip) against the oracle, bit for bit: cache
lengths on both sides of every form's limit, head sizes that fill the lanes of a row and that do not, masks with the
lowest finite value, minus infinity and whole masked rows, an empty cache, and the two rules that depend on the number
of heads."""
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LIMITS = [8, 16, 32, 64, 96, 128, 192, 256]   # row groups a form holds; a group is 8 rows (head size > 64) or 16


def _cases():
    for d in (128, 64):
        rows = 8 if d == 128 else 16
        for i, g in enumerate(LIMITS):
            for s in (g * rows - 3, g * rows, g * rows + 1):
                yield 2, 3, d, s, i % 2 == 0
    for d, s in ((80, 509), (80, 1), (96, 257), (16, 1025), (48, 63), (112, 100)):
        yield 2, 2, d, s, True
    yield 1, 1, 128, 1, False            # nothing cached
    yield 65, 4, 64, 2001, True          # more than 256 heads between 96 and 128 groups
    yield 129, 4, 16, 2050, False        # more than 512 heads beyond 128 groups


@pytest.mark.parametrize("B,H,d,S,masked", list(_cases()))
def test_one_new_token_is_exact(B, H, d, S, masked):
    import torch_int._hip_ext as X
    print("decode one", B, H, d, S, masked, flush=True)
    g = torch.Generator().manual_seed(B + 3 * d + 7 * S)

    def s8(*shape):
        return torch.randint(-127, 128, shape, dtype=torch.int8, generator=g)

    cap = (S + 31) // 16 * 16
    q, kn, vn = s8(B * H, 1, d), s8(B * H, 1, d), s8(B * H, 1, d)
    kb, vb = s8(B * H, cap, d), s8(B * H, cap, d)
    mask = None
    if masked:
        mask = torch.randn(B, 1, 1, S, generator=g)
        mask[0, ..., : S // 2] = torch.finfo(torch.float32).min
        mask[-1, ..., S // 3:S // 2] = float("-inf")
        if B > 2:
            mask[1] = torch.finfo(torch.float32).min
    a_qk, a_pv = 3e-4, 4e-3
    ctx, probs, k_ref, v_ref = orc.decode_attn_s8(q, kn, vn, kb, vb, S - 1, mask, H, a_qk, a_pv)
    kd, vd = kb.view(B, H, cap, d).to(DEV), vb.view(B, H, cap, d).to(DEV)
    args = (q.view(B, H, 1, d).to(DEV), kn.view(B, H, 1, d).to(DEV), vn.view(B, H, 1, d).to(DEV), kd, vd, S - 1,
            mask.to(DEV) if masked else None)
    got, got_p = X.decode_attention(*args, a_qk, a_pv, want_probs=True)
    assert torch.equal(got_p.cpu(), probs)
    assert torch.equal(got.cpu(), ctx)
    assert torch.equal(kd.cpu().view(B * H, cap, d), k_ref) and torch.equal(vd.cpu().view(B * H, cap, d), v_ref)
    again, none = X.decode_attention(*args, a_qk, a_pv)
    assert none is None and torch.equal(again.cpu(), ctx)


@pytest.mark.parametrize("d,heads", [(128, 256), (128, 260), (80, 260)])   # the rule for a length on the device: 256 heads, d > 96
def test_a_length_on_the_device_gives_the_values_of_one_on_the_host(d, heads):
    import torch_int._hip_ext as X
    g = torch.Generator(device=DEV).manual_seed(d + heads)
    cap, bound = 1056, 1049

    def s8(*shape):
        return torch.randint(-127, 128, shape, dtype=torch.int8, device=DEV, generator=g)

    q, kn, vn = (s8(heads // 4, 4, 1, d) for _ in range(3))
    kb, vb = s8(heads // 4, 4, cap, d), s8(heads // 4, 4, cap, d)
    length = torch.zeros(1, dtype=torch.int32, device=DEV)
    for n in (1, 20, 513, bound):
        print("length on the device", d, heads, n, flush=True)
        length.fill_(n)
        caches = [(kb.clone(), vb.clone()) for _ in range(2)]
        got = X.decode_attention_devlen(q, kn, vn, *caches[0], length, bound, 3e-4, 4e-3)
        want, _ = X.decode_attention(q, kn, vn, *caches[1], n - 1, None, 3e-4, 4e-3)
        assert torch.equal(got, want)
        assert torch.equal(caches[0][0], caches[1][0]) and torch.equal(caches[0][1], caches[1][1])
