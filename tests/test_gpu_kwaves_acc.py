"""The fp32 epilogue of the linears whose waves share K (csrc/gemm_kwaves.h) that adds to what is there: all units of a wave fetched before the
sums, on every tile, over rows that end inside a unit, and outputs and biases that begin on any multiple of four bytes.  Exact."""
import pytest
import torch

from oracle import oracle as orc
from test_gpu_kwaves import _name
from test_gpu_rows import _s8

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("off_out,off_bias", [(0, 0), (1, 0), (0, 3), (2, 1)])
@pytest.mark.parametrize("M,N,K,tile", [(67, 2048, 8192, "32x32"), (97, 2560, 2560, "32x64"), (260, 2048, 2048, "48x64"), (391, 2048, 2048, "64x64"),
                                        (253, 5120, 5120, "64x80"), (515, 2048, 2048, "96x64"), (293, 5120, 5120, "80x80"), (331, 5120, 5120, "96x80"),
                                        (801, 2048, 2048, "128x64"), (1910, 768, 768, "96x64")])
def test_added_to_outputs_that_begin_anywhere(M, N, K, tile, off_out, off_bias):
    import torch_int._CUDA as C
    g = torch.Generator().manual_seed(M + N + off_out)
    x, w, bias, resid = _s8(g, M, K), _s8(g, N, K), torch.randn(N, generator=g), torch.randn(M, N, generator=g) * 3
    xd, wd = x.to(DEV), w.to(DEV)
    acc = torch.mm(xd.double(), wd.double().t().contiguous()).to(torch.int32).cpu()   # sums below 2^53
    out = torch.full((M * N + 64,), 77.0, device=DEV)
    at = out[off_out:off_out + M * N].view(M, N)
    at.copy_(resid)
    bd = torch.zeros(N + 8, device=DEV)[off_bias:off_bias + N]
    bd.copy_(bias)
    print("added to, waves that share K", M, N, K, off_out, off_bias, flush=True)
    rc = C._lib.ti_linear_a8_w8_bfp32_ofp32_acc(xd.data_ptr(), wd.data_ptr(), bd.data_ptr(), at.data_ptr(), M, N, K, 3e-4, 1.0, None, 0,
                                                torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and _name() == "mid_waves_" + tile
    assert torch.equal(at.cpu(), orc.linear_a8_w8_bfp32_ofp32_acc(x, w, bias, 3e-4, 1.0, resid, acc_fn=lambda *_: acc))
    assert bool((out[:off_out] == 77).all()) and bool((out[off_out + M * N:] == 77).all())   # nothing beside it
