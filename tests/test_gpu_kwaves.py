"""Linears whose waves share K (csrc/gemm_kwaves.h): every tile at the first and last row count it has, rows that end inside a block, K of steps
that the waves do not share evenly (6 and 20), every epilogue, groups, where the rule ends.  Integer sums: exact."""
import ctypes

import pytest
import torch

from oracle import oracle as orc
from test_gpu_ln_linear import _add_f16
from test_gpu_rows import _s8

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _name():
    import torch_int._CUDA as C
    C._lib.ti_last_kernel.restype = C._lib.ti_last_kernel_form.restype = ctypes.c_char_p
    return C._lib.ti_last_kernel().decode() + (" pairs" if C._lib.ti_last_kernel_form().endswith(b"pairs") else "")


@pytest.mark.parametrize("M,N,K,tile", [
    (65, 2048, 8192, "32x32"), (127, 2048, 8192, "32x32"), (96, 2560, 2560, "32x32"), (255, 2048, 8192, "32x64"), (97, 2560, 2560, "32x64"),
    (129, 3072, 768, "32x64"), (513, 768, 768, "32x64"), (65, 4096, 4096, "32x64"), (257, 2048, 2048, "48x64"), (384, 2048, 2048, "48x64"),
    (768, 768, 768, "48x64"), (129, 5120, 5120, "48x64"), (385, 2048, 2048, "64x64"), (512, 2048, 2048, "64x64"), (1280, 768, 3072, "64x64"),
    (193, 4096, 4096, "64x64"), (97, 10240, 2560, "64x80"), (497, 2560, 2560, "64x80"), (256, 5120, 5120, "64x80"),
    (513, 2048, 2048, "96x64"), (768, 2048, 2048, "96x64"), (384, 3072, 768, "96x64"), (65, 16384, 4096, "96x64"), (289, 5120, 5120, "80x80"),
    (640, 2560, 2560, "80x80"), (321, 5120, 5120, "96x80"), (96, 20480, 5120, "96x80"), (769, 2048, 2048, "128x64"), (1024, 2048, 2048, "128x64"),
    (2047, 768, 3072, "128x64"), (128, 16384, 4096, "128x64")])
def test_every_tile_is_exact(M, N, K, tile):
    import torch_int._CUDA as C
    import torch_int._hip_ext as X
    g = torch.Generator().manual_seed(M * 7 + N + K)
    x, w, b8, bf = _s8(g, M, K), _s8(g, N, K), _s8(g, N), torch.randn(N, generator=g)
    b32, resid = torch.randint(-65535, 65535, (N,), dtype=torch.int32, generator=g), torch.randn(M, N, generator=g) * 3
    al, be = 3e-4, 0.02
    xd, wd, b8d, bfd = (t.to(DEV) for t in (x, w, b8, bf))
    acc = torch.mm(xd.double(), wd.double().t().contiguous()).to(torch.int32).cpu()   # sums below 2^53
    fresh = orc.epi_bfp32_ofp32(acc, bf, al, 1.0)
    print("waves that share K", M, N, K, tile, flush=True)
    for call, want in (
            (lambda: C.linear_a8_w8_b32_o32(xd, wd, b32.to(DEV)), orc.epi_b32_o32(acc, b32)),
            (lambda: C.linear_a8_w8_b32_o32_with_scaling(xd, wd, b32.to(DEV), al, be), orc.epi_b32_o32_scaled(acc, b32, al, be)),
            (lambda: C.linear_a8_w8_bfp32_ofp32(xd, wd, bfd, al, 1.0), fresh),
            (lambda: C.linear_a8_w8_b8_o8(xd, wd, b8d, al, be), orc.epi_b8_o8(acc, b8, al, be)),
            (lambda: C.linear_relu_a8_w8_b8_o8(xd, wd, b8d, al, be), orc.epi_b8_o8(acc, b8, al, be, relu=True)),
            (lambda: C._linear_a8_w8_bfp32_ofp32_acc(xd, wd, bfd, al, 1.0, resid.to(DEV)),
             orc.linear_a8_w8_bfp32_ofp32_acc(x, w, bf, al, 1.0, resid, acc_fn=lambda *_: acc)),
            (lambda: X.linear_a8_w8_b8_o8_heads(xd, wd, b8d, al, be, 1, M, N // 64, 64).permute(0, 2, 1, 3).reshape(M, N),
             orc.epi_b8_o8(acc, b8, al, be))):
        assert torch.equal(call().cpu(), want) and _name() == "mid_waves_" + tile, _name()
    old = resid.half()
    got = old.to(DEV)
    _add_f16(xd, wd, bfd, got, al)
    assert _name() == "mid_waves_" + tile and torch.equal(got.cpu(), (old.float() + fresh.half().float()).half())


@pytest.mark.parametrize("M,N,K", [(257, 4096, 4096), (512, 4096, 4096), (320, 2048, 8192), (512, 2048, 8192), (384, 5120, 5120), (512, 768, 3072)])
def test_accumulating_epilogues_of_257_to_512_rows(M, N, K):
    import torch_int._CUDA as C
    g = torch.Generator().manual_seed(M * 7 + N + K)
    x, w, bf, resid = _s8(g, M, K).to(DEV), _s8(g, N, K).to(DEV), torch.randn(N, generator=g), torch.randn(M, N, generator=g) * 3
    acc = torch.mm(x.double(), w.double().t().contiguous()).to(torch.int32).cpu()
    print("accumulating, waves that share K", M, N, K, flush=True)
    got = C._linear_a8_w8_bfp32_ofp32_acc(x, w, bf.to(DEV), 3e-4, 1.0, resid.to(DEV)).cpu()
    assert _name().startswith("mid_waves_")
    assert torch.equal(got, orc.linear_a8_w8_bfp32_ofp32_acc(x.cpu(), w.cpu(), bf, 3e-4, 1.0, resid, acc_fn=lambda *_: acc))
    old = resid.half()
    got = old.to(DEV)
    _add_f16(x, w, bf.to(DEV), got, 3e-4)
    assert _name().startswith("mid_waves_")
    assert torch.equal(got.cpu(), (old.float() + orc.epi_bfp32_ofp32(acc, bf, 3e-4, 1.0).half().float()).half())


@pytest.mark.parametrize("M,N,K", [(65, 2048, 2048), (128, 2048, 2048), (191, 2048, 2048), (256, 2048, 2048), (257, 2048, 2048), (319, 2048, 2048),
                                   (128, 2560, 2560), (255, 2560, 2560), (66, 5120, 5120), (128, 5120, 5120), (97, 4096, 4096)])
def test_groups(M, N, K):
    import torch_int._hip_ext as X
    g = torch.Generator().manual_seed(M + N)
    x, ws, bs = _s8(g, M, K).to(DEV), [_s8(g, N, K).to(DEV) for _ in range(3)], [_s8(g, N) for _ in range(3)]
    al, be = [3e-4, 2e-4, 5e-4], [0.02, 0.1, 0.05]
    print("group of waves that share K", M, N, K, flush=True)
    out = X.linear_a8_w8_b8_o8_group(x, ws, [b.to(DEV) for b in bs], al, be)
    assert X.linear_group_is_one_launch(M, N, K) and _name().startswith("mid_waves_group")
    for o, w, b, a, c in zip(out, ws, bs, al, be):
        acc = torch.mm(x.double(), w.double().t().contiguous()).to(torch.int32).cpu()
        assert torch.equal(o.cpu(), orc.epi_b8_o8(acc, b, a, c)), (M, N, K)


@pytest.mark.parametrize("M,N,K", [(64, 4096, 4096), (96, 2048, 2048), (1025, 2048, 2048), (257, 4096, 4096), (256, 2048, 8192), (512, 2560, 1024),
                                   (128, 1024, 4096), (481, 3072, 768), (257, 768, 3072)])
def test_where_it_ends(M, N, K):
    import torch_int._CUDA as C
    g = torch.Generator().manual_seed(M)
    x, w, b = _s8(g, M, K), _s8(g, N, K), _s8(g, N)
    print("other kernels", M, N, K, flush=True)
    out = C.linear_a8_w8_b8_o8(x.to(DEV), w.to(DEV), b.to(DEV), 3e-4, 0.02)
    assert "mid_waves" not in _name() and torch.equal(out.cpu(), orc.linear_a8_w8_b8_o8(x, w, b, 3e-4, 0.02, acc_fn=orc.gemm_acc_torch))
