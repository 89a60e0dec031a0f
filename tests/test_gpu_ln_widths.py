"""The LayerNorm-quantiser where a row ends inside, at the end of or just past the last chunk of its lanes (256 lanes x 4
elements), with few rows (gamma and beta fetched with the row) and with many, every form, against the oracle."""
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rows", [3, 70])
@pytest.mark.parametrize("width", [4, 1020, 1024, 1028, 2044, 5116, 5124, 16380, 16384])
def test_every_form_is_exact(rows, width):
    import torch_int._CUDA as C
    import torch_int._hip_ext as X
    print("ln widths", rows, width, flush=True)
    g = torch.Generator().manual_seed(rows * 17 + width)
    x32 = torch.randint(-30000, 30001, (rows, width), dtype=torch.int32, generator=g)
    x = torch.randn(rows, width, generator=g)
    res, gamma, beta = torch.randn(rows, width, generator=g), 30 * torch.randn(width, generator=g), torch.randn(width, generator=g)
    for half in (False, True):
        r, ga, be = (t.half() if half else t for t in (res, gamma, beta))
        dq, add = (orc.dq_add_layernorm_q_f16, orc.add_layernorm_q_f16) if half else (orc.dq_add_layernorm_q, orc.add_layernorm_q)
        gd, bd = ga.to(DEV), be.to(DEV)
        want_r, want_q = dq(x32, 1e-4, r, ga, be, 1e-5)
        got_r, got_q = C.dq_add_layernorm_q(x32.to(DEV), 1e-4, r.to(DEV), gd, bd, 1e-5)
        assert torch.equal(got_r.cpu(), want_r) and torch.equal(got_q.cpu(), want_q)
        # added in place (to an fp16 stream also from an fp32 tensor), and without an addend
        for y in ([x.half(), x] if half else [x]):
            want_r, want_q = add(y, r, ga, be, 1e-5)
            stream = r.to(DEV)
            assert torch.equal(X.add_layernorm_q(y.to(DEV), stream, gd, bd, 1e-5).cpu(), want_q)
            assert torch.equal(stream.cpu(), want_r)
        assert torch.equal(X.add_layernorm_q(None, r.to(DEV), gd, bd, 1e-5).cpu(), add(None, r, ga, be, 1e-5)[1])
