"""LayerNorm-quantise and the linears behind it in one launch, against the oracle: rows that end inside, at the end of or past the
last chunk of their lanes, every count of rows and of problems, weight rows that leave waves idle or take several rounds.  And the
linears that add into an fp16 stream, which leave those LayerNorms nothing to add."""
import ctypes

import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PP = ctypes.c_void_p * 3
FF = ctypes.c_float * 3


def _s8(g, *shape):
    return torch.randint(-127, 128, shape, dtype=torch.int8, generator=g)


def _pp(tensors):
    return PP(*(t.data_ptr() for t in tensors))


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("K,N,count", [(16, 3, 1), (768, 768, 3), (768, 3072, 1), (1008, 40, 2), (1024, 1024, 3), (1040, 5, 3),
                                       (2048, 8192, 1), (2560, 2560, 3), (4096, 4096, 3), (5120, 20480, 1), (5136, 64, 3),
                                       (6144, 100, 2), (7168, 2048, 3), (7184, 33, 1), (9216, 4096, 1)])
def test_one_launch_has_the_values_of_two(K, N, count, half):
    import torch_int._CUDA as C
    fn = C._lib.ti_layernorm_q_linear_a8_w8_b8_o8
    fn.argtypes = ([ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_float, PP, PP, PP, FF, FF]
                   + [ctypes.c_int64, ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_void_p])
    g = torch.Generator().manual_seed(K + N + count)
    dtype = torch.float16 if half else torch.float32
    hidden = (torch.randn(4, K, generator=g) * 2 + 0.3).to(dtype)
    gamma, beta = (30 * torch.randn(K, generator=g)).to(dtype), torch.randn(K, generator=g).to(dtype)
    w, b = [_s8(g, N, K) for _ in range(count)], [_s8(g, N) for _ in range(count)]
    al, be = [1e-3, 2e-3, 5e-4], [0.1, 0.3, 1.0]
    q = (orc.add_layernorm_q_f16 if half else orc.add_layernorm_q)(None, hidden, gamma, beta, 1e-5)[1]
    accs = [orc.gemm_acc_torch(q, wi) for wi in w]
    hd, gd, bd = hidden.to(DEV), gamma.to(DEV), beta.to(DEV)
    wd, biasd = [t.to(DEV) for t in w], [t.to(DEV) for t in b]
    stream = torch.cuda.current_stream().cuda_stream
    for M in (1, 2, 3, 4) if K <= 5120 else (1, 2):
        for relu in (False, True):
            print("ln linear", K, N, count, half, M, relu, flush=True)
            outs = [torch.full((M + 1, N), 77, dtype=torch.int8, device=DEV) for _ in range(count)]
            rc = fn(hd.data_ptr(), int(half), gd.data_ptr(), bd.data_ptr(), 1e-5, _pp(wd), _pp(biasd), _pp(outs), FF(*al), FF(*be),
                    count, int(relu), M, N, K, stream)
            assert rc == 0, C._lib.ti_last_error()
            for i in range(count):
                want = orc.epi_b8_o8(accs[i][:M], b[i], al[i], be[i], relu=relu)
                assert torch.equal(outs[i][:M].cpu(), want), (i, M, relu)
                assert (outs[i][M] == 77).all()   # nothing beyond the rows
    assert torch.equal(hd.cpu(), hidden)


def _add_f16(x, w, bias, inout, alpha, ws=None):
    import torch_int._CUDA as C
    fn = C._lib.ti_linear_a8_w8_bfp32_of16_acc
    fn.argtypes = ([ctypes.c_void_p] * 4 + [ctypes.c_int64] * 3 + [ctypes.c_float] * 2 + [ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p])
    rc = fn(x.data_ptr(), w.data_ptr(), bias.data_ptr(), inout.data_ptr(), x.shape[0], w.shape[0], x.shape[1], alpha, 1.0,
            None if ws is None else ws.data_ptr(), 0 if ws is None else ws.numel(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0, C._lib.ti_last_error()


# tiles whole and cut off in rows and in columns, rows cut off the end, slices, widths and addresses that no vector store fits
@pytest.mark.parametrize("M,N,K", [(17, 768, 768), (100, 768, 3072), (300, 5120, 20480), (512, 5120, 5120), (512, 12288, 12288),
                                   (1024, 2048, 8192), (2048, 2048, 2048), (2047, 2048, 8192), (1900, 4096, 4096), (1921, 4096, 16384),
                                   (2112, 5120, 5120), (2112, 5120, 20480), (2048, 9216, 9216), (3300, 2560, 10240), (1600, 5120, 5120),
                                   (1040, 5120, 20480), (4096, 768, 3072), (8192, 1000, 4096), (2049, 2052, 1024), (1500, 768, 768),
                                   (130, 1001, 96), (700, 4096, 1088), (2304, 8192, 2048), (512, 5120, 20480),
                                   (400, 4096, 4096)])
def test_prefills_add_into_an_fp16_stream(M, N, K):
    import torch_int._CUDA as C
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = (torch.randint(-127, 128, s, dtype=torch.int8, device=DEV, generator=g) for s in ((M, K), (N, K)))
    bias = torch.randn(N, device=DEV, generator=g)
    old = (torch.randn(M + 1, N, device=DEV, generator=g) * 3).half()
    alpha = 1e-3 / K ** 0.5
    fresh = C.linear_a8_w8_bfp32_ofp32(x, w, bias, alpha, 1.0)   # checked against the oracle elsewhere
    want = (old[:M].float() + fresh.half().float()).half()
    for shift, slices in ((0, True), (0, False), (1, True)):   # shift: a stream that lies between two vectors
        ws = torch.empty(C._lib.ti_linear_acc_workspace_bytes(M, N, K), dtype=torch.uint8, device=DEV) if slices else None
        got = torch.empty((M + 1) * N + 8, dtype=torch.float16, device=DEV)[shift:shift + (M + 1) * N].view(M + 1, N)
        got.copy_(old)
        print("acc f16", M, N, K, shift, slices, flush=True)
        _add_f16(x, w, bias, got[:M], alpha, ws)
        print(C._lib.ti_last_kernel().decode(), flush=True)
        assert torch.equal(got[:M], want) and torch.equal(got[M], old[M])


@pytest.mark.parametrize("M,N,K", [(1, 768, 768), (1, 5120, 5120), (1, 5120, 20480), (1, 9216, 36864), (1, 50, 1024), (2, 5120, 20480),
                                   (3, 768, 3072), (4, 4096, 16384), (16, 4099, 1024), (16, 5120, 10240), (7, 33, 48), (5, 19, 33)])
def test_linears_add_into_an_fp16_stream(M, N, K):
    g = torch.Generator().manual_seed(M * 31 + N + K)
    x, w, bias = _s8(g, M, K), _s8(g, N, K), torch.randn(N, generator=g)
    old = (torch.randn(M, N, generator=g) * 3).half()
    fresh = orc.epi_bfp32_ofp32(orc.gemm_acc_torch(x, w), bias, 3e-5, 1.0)
    want = (old.float() + fresh.half().float()).half()
    got, xd, wd, bd = (t.to(DEV) for t in (old, x, w, bias))
    for _ in range(2):   # the second time on what the first left behind: slices that meet clean up after themselves
        print("acc f16", M, N, K, flush=True)
        got.copy_(old)
        _add_f16(xd, wd, bd, got, 3e-5)
        assert torch.equal(got.cpu(), want)
