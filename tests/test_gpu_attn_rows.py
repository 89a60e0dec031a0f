"""Prefill attention with a row's scores in registers (attn_rows_kernel): at the edges of its tiles of 256 keys, of its blocks of
16 rows and of the rule that chooses it, with every kind of mask, with and without the mask's classes, against the chain
of operators (product, softmax-quantise, product), bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LOW = torch.finfo(torch.float32).min


def _mask(kind, B, T, S, gen):
    if kind == "none":
        return None
    m = torch.zeros(B, 1, T, S, device=DEV)
    if kind in ("causal", "padded", "infinite", "half"):
        low = {"infinite": float("-inf"), "half": -65504.0}.get(kind, LOW)
        m.masked_fill_(torch.ones(T, S, dtype=torch.bool, device=DEV).triu(1 + S - T), low)
    if kind == "half":            # as an fp16 model's, with padding in front of some rows and rows masked throughout
        m[:, :, T // 3:T // 3 + 17] = -65504.0
        m[-1, ..., :S // 3] = -65504.0
    if kind == "padded":          # the last keys of every sequence, and every key of the last sequence's
        for b in range(B):
            m[b, ..., max(1, S - (b + 1) * S // (B + 1)):] = LOW
        m[-1] = LOW
    if kind == "random":
        m = torch.randn(B, 1, T, S, device=DEV, generator=gen) * 3
    if kind == "rows":            # every third row is masked throughout, some by values below -1e30 that differ per tile
        m[:, :, ::3] = LOW
        m[:, :, 1::3, S // 2:] = -2e30
    return m.contiguous()


def _check(B, H, T, S, d, kind, alpha=None):
    import torch_int._CUDA as C
    import torch_int._hip_ext as X
    print(f"attn rows {B}x{H} T={T} S={S} d={d} {kind}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(S + T)
    s8 = lambda *shape: torch.randn(shape, device=DEV, generator=gen).mul_(30).round_().clamp_(-127, 127).to(torch.int8)
    q, k, vt, mask = s8(B * H, T, d), s8(B * H, S, d), s8(B * H, d, S), _mask(kind, B, T, S, gen)
    alpha = alpha or 2.0 / (d ** 0.5 * 900)
    probs = X.attn_softmax_q(C.bmm_s8t_s8n_f32t(q, k, alpha), mask, H)
    want = C.bmm_s8t_s8n_s8t(probs, vt, 2.0 / 127).view(B, H, T, d).transpose(1, 2).reshape(B, T, H * d)
    ctx = torch.empty_like(want)
    for classes in ((None, X.mask_classes(mask)) if mask is not None else (None,)):
        ctx.fill_(99)
        rc = C._lib.ti_attn_prefill_s8_mc(q.data_ptr(), k.data_ptr(), vt.data_ptr(), X._ptr(mask), X._ptr(classes), ctx.data_ptr(),
                                          B * H, T, S, d, T * d, S * d, H, alpha, 2.0 / 127,
                                          torch.cuda.current_stream().cuda_stream)
        assert rc == 0 and torch.equal(ctx, want), (kind, classes is not None)


@pytest.mark.parametrize("kind", ["none", "causal", "padded", "random", "rows", "infinite", "half"])
@pytest.mark.parametrize("B,H,T,S,d", [(1, 3, 80, 80, 64), (2, 2, 256, 256, 128), (1, 2, 257, 272, 16), (1, 3, 500, 512, 80),
                                       (2, 1, 528, 528, 128), (1, 2, 592, 592, 64), (1, 1, 33, 768, 112), (2, 1, 1024, 1024, 128),
                                       (1, 2, 1025, 1040, 48), (1, 1, 1, 1280, 128), (1, 2, 700, 1296, 64), (1, 1, 1792, 1792, 96),
                                       (1, 2, 1900, 1904, 128), (1, 1, 2048, 2048, 64)])
def test_against_the_chain(B, H, T, S, d, kind):
    _check(B, H, T, S, d, kind)


@pytest.mark.parametrize("S", [352, 368])
def test_many_heads_at_the_edge_of_the_rule(S):
    _check(8, 32, S, S, 64, "causal")


@pytest.mark.parametrize("kind", ["causal", "half"])
@pytest.mark.parametrize("alpha", [float("inf"), float("nan"), 1e13, -0.01, 0.02, 0.05])
def test_odd_scales(alpha, kind):
    _check(1, 2, 300, 304, 64, kind, alpha)      # 0.02 and 0.05: products of a few thousand, on both sides of the room there is
    _check(1, 1, 600, 608, 128, kind, alpha)


def test_recorded_prefill_reads_the_mask_as_it_is():
    import torch_int._hip_ext as X
    gen = torch.Generator(device=DEV).manual_seed(5)
    s8 = lambda *shape: torch.randn(shape, device=DEV, generator=gen).mul_(30).round_().clamp_(-127, 127).to(torch.int8)
    q, k, vt = s8(4, 640, 64), s8(4, 640, 64), s8(4, 64, 640)
    mask = _mask("causal", 1, 640, 640, gen)
    call = lambda m: X.attn_prefill(q, k, vt, m, 0.0003, 2.0 / 127, 4)
    call(mask)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=side):
        ctx = call(mask)
    for kind in ("padded", "none", "causal"):
        mask.copy_(_mask(kind, 1, 640, 640, gen) if kind != "none" else torch.zeros_like(mask))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(ctx, call(mask.clone())), kind
    with torch.inference_mode():
        fresh = mask + 0.0
        assert torch.equal(call(fresh), ctx)
