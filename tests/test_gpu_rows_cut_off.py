"""The last rows of a linear, run as a problem of their own (ti_linear_row_split), where that problem needs no workspace: with and without
one, the same kernels and the same bytes."""
import ctypes

import pytest
import torch

from test_gpu_kwaves import _name

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M,N,K", [(8257, 2048, 8192), (8320, 2048, 7680)])
@pytest.mark.parametrize("kind", ["b8_o8", "of32_acc", "of16_acc"])
def test_rows_that_need_no_workspace(M, N, K, kind):
    import torch_int._CUDA as C
    r = C._lib.ti_linear_row_split(ctypes.c_int64(M), ctypes.c_int64(N), ctypes.c_int64(K))
    assert r == M % 256
    g = torch.Generator(device=DEV).manual_seed(M)
    x, w, b8 = (torch.randint(-127, 128, s, dtype=torch.int8, device=DEV, generator=g) for s in ((M, K), (N, K), (N,)))
    bf = torch.randn(N, device=DEV, generator=g)
    dtype = {"b8_o8": torch.int8, "of32_acc": torch.float32, "of16_acc": torch.float16}[kind]
    call = {"b8_o8": C._lib.ti_linear_a8_w8_b8_o8, "of32_acc": C._lib.ti_linear_a8_w8_bfp32_ofp32_acc,
            "of16_acc": C._lib.ti_linear_a8_w8_bfp32_of16_acc}[kind]
    need = C._lib.ti_linear_acc_workspace_bytes(ctypes.c_int64(M), ctypes.c_int64(N), ctypes.c_int64(K))
    ws = torch.empty(need + 256, dtype=torch.uint8, device=DEV)
    outs = []
    vp, i64, f32 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_float
    for given in (need, 0):
        out = torch.zeros((M, N), dtype=dtype, device=DEV)
        print("rows cut off", M, N, K, kind, given, flush=True)
        rc = call(vp(x.data_ptr()), vp(w.data_ptr()), vp((b8 if kind == "b8_o8" else bf).data_ptr()), vp(out.data_ptr()), i64(M), i64(N), i64(K),
                  f32(2e-5), f32(1.0), vp(ws.data_ptr() if given else None), i64(given), vp(torch.cuda.current_stream().cuda_stream))
        assert rc == 0 and "+mid_waves_" in _name(), _name()
        outs.append(out)
    assert torch.equal(*outs)
    rows = torch.arange(M - r - 3, M, device=DEV)   # both sides of the cut
    want = torch.mm(x[rows].double(), w.double().t().contiguous()).to(torch.float32)
    if kind == "b8_o8":
        return
    fresh = torch.addcmul(bf.double(), want.double(), torch.tensor(2e-5, dtype=torch.float32, device=DEV).double()).float()   # one rounding, as fmaf
    assert torch.equal(outs[0][rows], fresh.to(dtype))
