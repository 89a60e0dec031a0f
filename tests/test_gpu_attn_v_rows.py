"""Prefill attention on V as the cache holds it against the same on V transposed (which other tests compare with the operators): key
counts at the edges of both forms, head sizes inside and at the end of the LDS rows, rows that end inside a block, masks."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("D", [16, 48, 64, 80, 112, 128])
@pytest.mark.parametrize("BH,T,S", [(4, 7, 16), (3, 33, 32), (2, 48, 48), (12, 48, 64), (300, 64, 64), (5, 80, 80), (200, 112, 112), (8, 128, 128),
                                    (300, 130, 144), (160, 256, 256), (24, 17, 272), (160, 320, 320), (4, 512, 512), (170, 384, 560),
                                    (60, 576, 576), (3, 100, 592), (2, 768, 768), (2, 40, 1040), (1, 1280, 1280), (1, 64, 1552),
                                    (1, 1800, 1808), (1, 33, 2048)])
def test_both_orders_of_v_give_the_same(BH, T, S, D):
    import torch_int._CUDA as C
    old, new = C._lib.ti_attn_prefill_s8_mc, C._lib.ti_attn_prefill_s8_v
    new.argtypes = old.argtypes = [ctypes.c_void_p] * 6 + [ctypes.c_int64] * 7 + [ctypes.c_float] * 2 + [ctypes.c_void_p]
    form = C._lib.ti_attn_prefill_form
    form.argtypes = [ctypes.c_int64] * 4 + [ctypes.c_int] * 2
    g = torch.Generator(device=DEV).manual_seed(S * 7 + D + T)
    q, k, v = (torch.randint(-127, 128, (BH, n, D), dtype=torch.int8, device=DEV, generator=g) for n in (T, S, S))
    vt = v.transpose(1, 2).contiguous()
    low = torch.finfo(torch.float32).min
    triangle = torch.zeros(1, 1, T, S, device=DEV).masked_fill_(torch.ones(T, S, dtype=torch.bool, device=DEV).triu(1), low)
    some = torch.randn(1, 1, T, S, device=DEV, generator=g)
    stream = torch.cuda.current_stream().cuda_stream
    for name, mask in (("none", None), ("causal", triangle), ("values", some)):
        classes = None
        if name == "causal":
            classes = torch.empty(C._lib.ti_attn_mask_classes_bytes(1, T, S), dtype=torch.uint8, device=DEV)
            assert C._lib.ti_attn_mask_classes(mask.data_ptr(), classes.data_ptr(), 1, T, S, stream) == 0
        print("v rows", BH, T, S, D, name, form(BH, T, S, D, mask is not None, classes is not None), flush=True)
        out = [torch.full((BH * T * D + 64,), 99, dtype=torch.int8, device=DEV) for _ in range(2)]
        for fn, value, o in ((old, vt, out[0]), (new, v, out[1])):
            rc = fn(q.data_ptr(), k.data_ptr(), value.data_ptr(), None if mask is None else mask.data_ptr(),
                    None if classes is None else classes.data_ptr(), o.data_ptr(), BH, T, S, D, T * D, S * D, BH, 0.002, 0.02, stream)
            assert rc == 0, C._lib.ti_last_error()
        assert torch.equal(out[0], out[1]) and (out[1][BH * T * D:] == 99).all()
        assert out[0][:BH * T * D].unique().numel() > 3
