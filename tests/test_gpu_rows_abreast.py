"""Narrow outputs of 17 to 512 rows, whose 16-row blocks lie in several workgroups (csrc/gemm_rows.h, rows_blocks_each): one, two and
three blocks to a workgroup, last groups that are cut off or hold fewer blocks, outputs at the lines of the rule, an fp16 and an fp32 stream
that is added to, head-major stores and groups.  Integer sums: exact."""
import ctypes

import pytest
import torch

from oracle import oracle as orc
from test_gpu_ln_linear import _add_f16
from test_gpu_rows import _last, _s8

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _adds_into_an_fp16_stream(x, w, bias, acc, resid, alpha):
    fresh, old = orc.epi_bfp32_ofp32(acc, bias.cpu(), alpha, 1.0), resid.half()
    got = old.to(DEV)
    _add_f16(x, w, bias, got, alpha)
    assert _last()[0] == 1 and torch.equal(got.cpu(), (old.float() + fresh.half().float()).half())


@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 63, 64])
@pytest.mark.parametrize("N,K", [(16, 768), (50, 1024), (768, 3072), (1024, 5120), (1040, 2048), (2048, 4096), (2064, 2560)])
def test_rows_in_several_workgroups(M, N, K):
    import torch_int._CUDA as C
    g = torch.Generator().manual_seed(M * 7 + N + K)
    x, w, b8, bf = _s8(g, M, K), _s8(g, N, K), _s8(g, N), torch.randn(N, generator=g)
    resid = torch.randn(M, N, generator=g) * 3
    al, be = 3e-4, 0.02
    acc = orc.gemm_acc_torch(x, w)
    xd, wd, b8d, bfd = (t.to(DEV) for t in (x, w, b8, bf))
    print("rows abreast", M, N, K, flush=True)
    out = C.linear_a8_w8_b8_o8(xd, wd, b8d, al, be)
    assert _last()[0] == 1
    assert torch.equal(out.cpu(), orc.epi_b8_o8(acc, b8, al, be))
    assert torch.equal(C.linear_a8_w8_bfp32_ofp32(xd, wd, bfd, al, 1.0).cpu(), orc.epi_bfp32_ofp32(acc, bf, al, 1.0))
    assert torch.equal(C._linear_a8_w8_bfp32_ofp32_acc(xd, wd, bfd, al, 1.0, resid.to(DEV)).cpu(),
                       orc.linear_a8_w8_bfp32_ofp32_acc(x, w, bf, al, 1.0, resid, acc_fn=lambda *_: acc))
    _adds_into_an_fp16_stream(xd, wd, bfd, acc, resid, al)
    if N % 16 == 0:
        import torch_int._hip_ext as X
        want = orc.epi_b8_o8(acc, b8, al, be).view(1, M, N // 16, 16).transpose(1, 2)
        assert torch.equal(X.linear_a8_w8_b8_o8_heads(xd, wd, b8d, al, be, 1, M, N // 16, 16).cpu(), want)


@pytest.mark.parametrize("M,N,K", [(48, 512, 1024), (33, 400, 768), (64, 272, 4096)])
def test_groups_in_several_workgroups(M, N, K):
    import torch_int._hip_ext as X
    g = torch.Generator().manual_seed(M + N + K)
    x, ws, bs = _s8(g, M, K), [_s8(g, N, K) for _ in range(3)], [_s8(g, N) for _ in range(3)]
    al, be = [3e-4, 2e-4, 5e-4], [0.02, 0.1, 0.05]
    print("rows abreast group", M, N, K, flush=True)
    out = X.linear_a8_w8_b8_o8_group(x.to(DEV), [w.to(DEV) for w in ws], [b.to(DEV) for b in bs], al, be)
    for o, w, b, a, c in zip(out, ws, bs, al, be):
        assert torch.equal(o.cpu(), orc.linear_a8_w8_b8_o8(x, w, b, a, c, acc_fn=orc.gemm_acc_torch)), (M, N, K)


@pytest.mark.parametrize("K,want", [(768, "E1"), (1024, "B1"), (2048, "A1"), (2560, "D1"), (3072, "G1"), (3584, "H1"), (4096, "F1"),
                                    (5120, "C1")])
def test_every_tiling_with_all_rows_in_a_workgroup(K, want):
    """Outputs of more strips than there are CUs: one to four blocks of 16 rows to a workgroup, a kernel of its own each."""
    import torch_int._CUDA as C
    N = 4112
    g = torch.Generator().manual_seed(K)
    x, w, b = _s8(g, 64, K), _s8(g, N, K), _s8(g, N)
    ref = orc.linear_a8_w8_b8_o8(x, w, b, 3e-4, 0.02, acc_fn=orc.gemm_acc_torch)
    xd, wd, bd = x.to(DEV), w.to(DEV), b.to(DEV)
    for M in (16, 17, 32, 33, 48, 49, 64):
        print("rows whole", want, M, N, K, flush=True)
        assert torch.equal(C.linear_a8_w8_b8_o8(xd[:M], wd, bd, 3e-4, 0.02).cpu(), ref[:M]), M
        assert _last() == (1, want), M


@pytest.mark.parametrize("M,N,K", [(65, 768, 768), (320, 768, 768), (512, 768, 768), (96, 3072, 768), (128, 2304, 768), (81, 768, 3072), (256, 768, 3072),
                                   (511, 1024, 1024), (127, 4096, 1024), (65, 1000, 2048), (95, 2048, 2048), (256, 2048, 2048),
                                   (179, 2560, 2560), (160, 784, 3584), (128, 1040, 5120)])
def test_more_than_64_rows(M, N, K):
    """From the first to the last row count of a rule's range, two workgroups to a CU among them."""
    import torch_int._CUDA as C
    import torch_int._hip_ext as X
    g = torch.Generator().manual_seed(M + N + K)
    x, w, b8, bf = _s8(g, M, K), _s8(g, N, K), _s8(g, N), torch.randn(N, generator=g)
    resid = torch.randn(M, N, generator=g) * 3
    al, be = 3e-4, 0.02
    acc = orc.gemm_acc_torch(x, w)
    xd, wd, b8d, bfd = (t.to(DEV) for t in (x, w, b8, bf))
    print("rows beyond 64", M, N, K, flush=True)
    want = orc.epi_b8_o8(acc, b8, al, be)
    assert torch.equal(C.linear_a8_w8_b8_o8(xd, wd, b8d, al, be).cpu(), want)
    assert _last()[0] == 1
    assert torch.equal(C.linear_relu_a8_w8_b8_o8(xd, wd, b8d, al, be).cpu(), orc.epi_b8_o8(acc, b8, al, be, relu=True))
    assert torch.equal(C.linear_a8_w8_bfp32_ofp32(xd, wd, bfd, al, 1.0).cpu(), orc.epi_bfp32_ofp32(acc, bf, al, 1.0))
    assert torch.equal(C._linear_a8_w8_bfp32_ofp32_acc(xd, wd, bfd, al, 1.0, resid.to(DEV)).cpu(),
                       orc.linear_a8_w8_bfp32_ofp32_acc(x, w, bf, al, 1.0, resid, acc_fn=lambda *_: acc))
    _adds_into_an_fp16_stream(xd, wd, bfd, acc, resid, al)
    if N % 16 == 0:
        heads = want.view(1, M, N // 16, 16).transpose(1, 2)
        assert torch.equal(X.linear_a8_w8_b8_o8_heads(xd, wd, b8d, al, be, 1, M, N // 16, 16).cpu(), heads)


@pytest.mark.parametrize("M,N,K", [(192, 768, 768), (65, 768, 1024), (96, 1024, 2048), (80, 800, 2560)])
def test_groups_of_more_than_64_rows(M, N, K):
    import torch_int._hip_ext as X
    test_groups_in_several_workgroups(M, N, K)
    assert _last()[0] == 1 and X.linear_group_is_one_launch(M, N, K)


def test_where_more_than_64_rows_end():
    """One row further the tiled kernels have them, and the group says so before it is launched."""
    import torch_int._CUDA as C
    import torch_int._hip_ext as X
    g = torch.Generator().manual_seed(1)
    for M, N, K in ((513, 768, 768), (129, 3072, 768), (257, 768, 3072), (257, 2048, 2048), (193, 2560, 2560), (128, 752, 768)):
        x, w, b = _s8(g, M, K), _s8(g, N, K), _s8(g, N)
        print("rows end", M, N, K, flush=True)
        out = C.linear_a8_w8_b8_o8(x.to(DEV), w.to(DEV), b.to(DEV), 3e-4, 0.02)
        assert _last()[0] == 0 and torch.equal(out.cpu(), orc.linear_a8_w8_b8_o8(x, w, b, 3e-4, 0.02, acc_fn=orc.gemm_acc_torch))
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    for M in (192, 193):   # three 768 x 768
        test_groups_in_several_workgroups(M, 768, 768)
        one = X.linear_group_is_one_launch(M, 768, 768)
        assert one == (M == 192) == C._lib.ti_last_kernel().endswith(b"_group"), (M, C._lib.ti_last_kernel())
        assert not one or _last()[0] == 1
