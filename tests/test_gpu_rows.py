"""The weight-streaming kernel for 2 to 64 rows of activations (csrc/gemm_rows.h) against the oracle: every tiling of the
inner dimension with one slice and with several, row counts at the edges of the 16-row blocks, widths that end inside a
strip of 16, every epilogue, head-major stores, groups, and the two-launch form of the sliced products."""
import ctypes

import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (M, N, K): tiling and slices
SHAPES = {
    (17, 16384, 2048): "A1",
    (33, 8192, 4096): "F1",
    (64, 4096, 8192): "A4",
    (2, 2048, 1024): "B1",
    (5, 50, 1024): "B1",       # a width inside one group of strips that ends inside a strip
    (16, 4099, 1024): "B1",    # a width that no vector store fits
    (64, 2064, 3072): "G1",    # a strip past a multiple of 64
    (48, 8192, 5120): "C1",
    (16, 5120, 10240): "C2",
    (40, 2560, 2560): "D1",
    (3, 640, 7680): "D3",
    (31, 768, 768): "E1",
    (8, 784, 2304): "E3",
    (49, 16, 768): "E1",       # one strip
    (64, 1024, 4096): "F1",    # 49 to 64 rows: eight waves instead of sixteen
    (24, 5120, 20480): "C4",
    (20, 1040, 3584): "H1",
    (33, 1024, 7168): "H2",
    (48, 1024, 9216): "G3",
    (17, 1024, 11264): "B11",
}


def _last():
    """The weight-streaming kernel's last launch: (form, tiling and slices)."""
    import torch_int._CUDA as C
    t, s = ctypes.c_int(0), ctypes.c_int(0)
    form = C._lib.ti_last_rows(ctypes.byref(t), ctypes.byref(s))
    return form, " ABCDEFGH"[t.value].strip() + str(s.value)


def _s8(g, *shape):
    return torch.randint(-127, 128, shape, dtype=torch.int8, generator=g)


@pytest.mark.parametrize("M,N,K", list(SHAPES))
def test_every_epilogue_is_exact(M, N, K):
    import torch_int._CUDA as C
    import torch_int._hip_ext as X
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    g = torch.Generator().manual_seed(M * 7 + N + K)
    x, w = _s8(g, M, K), _s8(g, N, K)
    b8, bf = _s8(g, N), torch.randn(N, generator=g)
    b32 = torch.randint(-65535, 65535, (N,), dtype=torch.int32, generator=g)
    resid = torch.randn(M, N, generator=g) * 3
    al, be = 3e-4, 0.02
    acc = orc.gemm_acc_torch(x, w)
    xd, wd, b8d, bfd, b32d = (t.to(DEV) for t in (x, w, b8, bf, b32))
    runs = [(lambda: C.linear_a8_w8_b32_o32(xd, wd, b32d), orc.epi_b32_o32(acc, b32)),
            (lambda: C.linear_a8_w8_b32_o32_with_scaling(xd, wd, b32d, al, be), orc.epi_b32_o32_scaled(acc, b32, al, be)),
            (lambda: C.linear_a8_w8_bfp32_ofp32(xd, wd, bfd, al, 1.0), orc.epi_bfp32_ofp32(acc, bf, al, 1.0)),
            (lambda: C.linear_a8_w8_b8_o8(xd, wd, b8d, al, be), orc.epi_b8_o8(acc, b8, al, be)),
            (lambda: C.linear_relu_a8_w8_b8_o8(xd, wd, b8d, al, be), orc.epi_b8_o8(acc, b8, al, be, relu=True)),
            (lambda: C._linear_a8_w8_bfp32_ofp32_acc(xd, wd, bfd, al, 1.0, resid.to(DEV)),
             orc.linear_a8_w8_bfp32_ofp32_acc(x, w, bf, al, 1.0, resid, acc_fn=lambda *_: acc))]
    for i, (run, want) in enumerate(runs):
        print("rows epilogue", i, M, N, K, flush=True)
        outs = [run() for _ in range(2)]
        assert C._lib.ti_last_kernel().decode() == ("stream" if M <= 16 else "mid_stream")
        assert _last() == (1 if SHAPES[M, N, K][1:] == "1" else 2, SHAPES[M, N, K])
        for o in outs:   # twice: the arrival counters and the accumulation buffers are left as they were found
            assert torch.equal(o.cpu(), want), (i, M, N, K)
    before = C._lib.ti_fused_splitk(0)   # several slices: the two-launch form, or another kernel where there is no workspace
    try:
        assert torch.equal(C.linear_a8_w8_b8_o8(xd, wd, b8d, al, be).cpu(), orc.epi_b8_o8(acc, b8, al, be))
    finally:
        C._lib.ti_fused_splitk(before)
    d = 16 if N % 16 == 0 else 0
    if d:
        want = orc.epi_b8_o8(acc, b8, al, be).view(1, M, N // d, d).transpose(1, 2)
        assert torch.equal(X.linear_a8_w8_b8_o8_heads(xd, wd, b8d, al, be, 1, M, N // d, d).cpu(), want)


@pytest.mark.parametrize("M,N,K,tiling", [(5, 768, 12288, "F3"), (17, 1024, 12288, "F3"), (24, 4096, 16384, "F4"), (64, 784, 16384, "F4"),
                                          (49, 2048, 16384, "F4"), (16, 5120, 16384, "F4")])
def test_slices_of_sixteen_waves(M, N, K, tiling, monkeypatch):
    monkeypatch.setitem(SHAPES, (M, N, K), tiling)
    test_every_epilogue_is_exact(M, N, K)


@pytest.mark.parametrize("N,K,want", [(272, 768, "E1"), (272, 1024, "B1"), (272, 2048, "A1"), (272, 2560, "D1"), (272, 3072, "G1"),
                                      (272, 3584, "H1"), (272, 4096, "F1"), (272, 5120, "C1"), (272, 2304, "E3"),
                                      (272, 6144, "A3"), (272, 7168, "H2"), (272, 7680, "D3"), (272, 9216, "G3"),
                                      (272, 11264, "B11"), (272, 20480, "C4")])
def test_every_tiling_at_every_number_of_row_blocks(N, K, want):
    """One to four blocks of 16 rows, the last one full and with a single row: a kernel of its own each."""
    import torch_int._CUDA as C
    g = torch.Generator().manual_seed(N + K)
    x, w, b = _s8(g, 64, K), _s8(g, N, K), _s8(g, N)
    ref = orc.linear_a8_w8_b8_o8(x, w, b, 3e-4, 0.02, acc_fn=orc.gemm_acc_torch)
    xd, wd, bd = x.to(DEV), w.to(DEV), b.to(DEV)
    for M in (9, 16, 17, 32, 33, 48, 49, 64):
        print("rows tiling", want, M, N, K, flush=True)
        for _ in range(2):
            assert torch.equal(C.linear_a8_w8_b8_o8(xd[:M], wd, bd, 3e-4, 0.02).cpu(), ref[:M]), M
        assert _last() == (1 if want[1:] == "1" else 2, want), M


@pytest.mark.parametrize("M,N,K", [(24, 4096, 4096), (16, 1024, 4096), (7, 2560, 2560), (48, 768, 768), (2, 100, 1024)])
def test_groups_are_exact(M, N, K):
    import torch_int._hip_ext as X
    g = torch.Generator().manual_seed(M + N + K)
    x, ws, bs = _s8(g, M, K), [_s8(g, N, K) for _ in range(3)], [_s8(g, N) for _ in range(3)]
    al, be = [3e-4, 2e-4, 5e-4], [0.02, 0.1, 0.05]
    ref = [orc.linear_a8_w8_b8_o8(x, w, b, a, c, acc_fn=orc.gemm_acc_torch) for w, b, a, c in zip(ws, bs, al, be)]
    print("rows group", M, N, K, flush=True)
    for _ in range(2):
        out = X.linear_a8_w8_b8_o8_group(x.to(DEV), [w.to(DEV) for w in ws], [b.to(DEV) for b in bs], al, be)
        for o, r in zip(out, ref):
            assert torch.equal(o.cpu(), r), (M, N, K)


@torch.no_grad()
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("D,H,bsz", [(768, 12, 17), (1024, 8, 64), (320, 4, 33), (2048, 16, 24)])
def test_decode_step_of_a_large_batch_from_one_call(D, H, bsz, half):
    """17 to 64 sequences, one new token each: residual stream and caches of the one C call bit for bit those of the
    modules, with the projections grouped (768, 1024, 2048), fc2 in four slices (2048) and on the split-K kernels (320)."""
    from test_gpu_models import causal_mask, randomize_int8_layer
    from torch_int.models.opt import Int8OPTDecoderLayer
    g = torch.Generator().manual_seed(D + bsz)
    layer = randomize_int8_layer(Int8OPTDecoderLayer(D, H, 4 * D), g).to(DEV)
    layer = layer.half() if half else layer
    dt = torch.float16 if half else torch.float32
    hidden = torch.randn(bsz, 32, D, generator=g).to(DEV).to(dt)
    out = layer(hidden.clone(), attention_mask=causal_mask(bsz, 32, 32).to(DEV).to(dt), use_cache=True)
    caches = {True: out[-1], False: tuple(t.clone() for t in out[-1])}
    for step in range(3):
        x = torch.randn(bsz, 1, D, generator=g).to(DEV).to(dt)
        res = {}
        for one_call in (True, False):
            layer.decode_in_one_call = one_call
            print("rows decode", D, bsz, half, step, one_call, flush=True)
            res[one_call] = layer(x.clone(), past_key_value=caches[one_call], use_cache=True)
            caches[one_call] = res[one_call][-1]
            if one_call and not (half or D == 320):   # fc2 comes last
                assert _last() == {768: (1, "G1"), 1024: (1, "F1"), 2048: (2, "A4")}[D]
        assert torch.equal(res[True][0], res[False][0])
        for a, b in zip(caches[True], caches[False]):
            assert torch.equal(a, b)


def test_a_group_too_wide_for_its_bias_in_the_lds():
    """The biases of a workgroup's strips (64 bytes each) lie beside the weight rings, which leave 24 to 30 KiB where a workgroup
    has a CU to itself: the widest groups of four go problem by problem."""
    import torch_int._hip_ext as X
    M, N, K = 2, 524272, 4096
    g = torch.Generator(device=DEV).manual_seed(5)
    x = torch.randint(-127, 128, (M, K), dtype=torch.int8, device=DEV, generator=g)
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=DEV, generator=g)
    bs = [torch.randint(-127, 128, (N,), dtype=torch.int8, device=DEV, generator=g) for _ in range(4)]
    al, be = [3e-4, 2e-4, 5e-4, 1e-4], [0.02, 0.1, 0.05, 0.3]
    print("rows wide group", M, N, K, flush=True)
    out = X.linear_a8_w8_b8_o8_group(x, [w] * 4, bs, al, be)
    some = torch.cat([torch.arange(2048), torch.arange(N - 2048, N)]).to(DEV)
    for o, b, a, c in zip(out, bs, al, be):
        want = orc.linear_a8_w8_b8_o8(x.cpu(), w[some].cpu(), b[some].cpu(), a, c, acc_fn=orc.gemm_acc_torch)
        assert torch.equal(o[:, some].cpu(), want)


@pytest.mark.parametrize("N,K,sliced", [(1000, 2560, True), (1008, 2560, False), (1000, 2048, False)])
def test_workspace_is_that_of_the_kernel_that_runs(N, K, sliced):
    """Widths that 16 does not divide go to the tiled kernels where 1024 does not divide the inner dimension, which slice it."""
    import torch_int._CUDA as C
    assert (C._lib.ti_linear_workspace_bytes(48, N, K) > 0) == sliced


def _sliced(M, N, K, seed):
    """A sliced linear of M rows: (call, the oracle's output)."""
    import torch_int._CUDA as C
    g = torch.Generator().manual_seed(seed)
    x, w, b = _s8(g, M, K), _s8(g, N, K), _s8(g, N)
    want = orc.linear_a8_w8_b8_o8(x, w, b, 3e-4, 0.02, acc_fn=orc.gemm_acc_torch).to(DEV)
    xd, wd, bd = x.to(DEV), w.to(DEV), b.to(DEV)
    return lambda: C.linear_a8_w8_b8_o8(xd, wd, bd, 3e-4, 0.02), want


def _form():
    return _last()[0]


@pytest.mark.parametrize("M,recorded", [(8, 0), (24, 3)])
def test_graphs_of_sliced_linears_replay_on_two_streams_beside_eager_work(M, recorded):
    """Two graphs recorded on one stream, replayed on two others while the recording stream runs the same linears eagerly:
    what is recorded keeps no state of the stream."""
    call, want = _sliced(M, 2560, 10240, 1)
    side, others = torch.cuda.Stream(), [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(2):
            call()
        assert _form() == 2    # eagerly the slices meet in one launch
    torch.cuda.synchronize()
    graphs, outs = [torch.cuda.CUDAGraph() for _ in range(2)], []
    for graph in graphs:
        print("recording", M, flush=True)
        with torch.cuda.graph(graph, stream=side):
            outs.append([call() for _ in range(6)])
            assert _form() == recorded
    torch.cuda.synchronize()
    for round_ in range(3):
        print("replays", M, round_, flush=True)
        eager = []
        for _ in range(8):
            for graph, stream in zip(graphs, others):
                with torch.cuda.stream(stream):
                    graph.replay()
            with torch.cuda.stream(side):
                eager.append(call())
        torch.cuda.synchronize()
        assert all(torch.equal(o, want) for o in outs[0] + outs[1] + eager)


def test_a_first_call_on_a_stream_while_another_thread_records():
    """A thread that records a graph does not disturb another one's linears on a stream that has no block of state yet, nor do
    they disturb the recording."""
    import threading
    import torch_int._CUDA as C
    cases = []
    for M, N, K in ((8, 2560, 10240), (40, 2048, 8192)):
        g = torch.Generator().manual_seed(M)
        x, w, b = _s8(g, M, K).to(DEV), _s8(g, N, K).to(DEV), _s8(g, N).to(DEV)
        need = C._lib.ti_linear_workspace_bytes(M, N, K)
        cases.append((M, N, K, x, w, b, torch.empty((M, N), dtype=torch.int8, device=DEV), need,
                      torch.empty(max(need, 1), dtype=torch.uint8, device=DEV), C.linear_a8_w8_b8_o8(x, w, b, 3e-4, 0.02)))
    h = ctypes.c_void_p()
    assert C._lib.hipStreamCreate(ctypes.byref(h)) == 0
    recording, done, status = threading.Event(), threading.Event(), []

    def other():
        recording.wait(60)
        for M, N, K, x, w, b, out, need, ws, _ in cases:
            status.append(C._lib.ti_linear_a8_w8_b8_o8(x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), M, N, K, 3e-4, 0.02,
                                                       ws.data_ptr() if need else None, need, h.value))
        done.set()

    thread = threading.Thread(target=other)
    thread.start()
    graph, y = torch.cuda.CUDAGraph(), torch.ones(64, device=DEV)
    torch.cuda.synchronize()
    print("recording beside another thread", flush=True)
    with torch.cuda.graph(graph):
        y.add_(1)
        recording.set()
        assert done.wait(60)
        y.add_(1)
    thread.join()
    torch.cuda.synchronize()
    assert status == [0, 0]
    assert all(torch.equal(c[6], c[9]) for c in cases)
    for turn in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, torch.full_like(y, 3 + 2 * turn))


def test_forty_streams_of_sliced_linears():
    """More streams than there are blocks of state, all with work queued at once, twice over: exact on every one."""
    import torch_int._CUDA as C
    call, want = _sliced(8, 2560, 10240, 2)
    big, want_big = _sliced(40, 2048, 8192, 3)
    streams = []
    for _ in range(40):
        h = ctypes.c_void_p()
        assert C._lib.hipStreamCreate(ctypes.byref(h)) == 0   # the HIP runtime that the library is linked to
        streams.append(torch.cuda.ExternalStream(h.value))
    torch.cuda.synchronize()
    forms = set()
    for turn in range(2):
        print("forty streams", turn, flush=True)
        outs = []
        for s in streams:
            with torch.cuda.stream(s):
                outs.append((call(), want))
                forms.add((8, _form()))
                outs.append((big(), want_big))
                forms.add((40, _form()))
        torch.cuda.synchronize()
        assert all(torch.equal(o, w) for o, w in outs)
    assert forms == {(8, 0), (8, 2), (40, 3), (40, 2)}


def test_a_stream_of_every_thread_keeps_no_state():
    """hipStreamPerThread is one handle for a stream of each thread."""
    import torch_int._CUDA as C
    g = torch.Generator().manual_seed(4)
    x, w, b = _s8(g, 40, 8192).to(DEV), _s8(g, 2048, 8192).to(DEV), _s8(g, 2048).to(DEV)
    out, want = torch.empty((40, 2048), dtype=torch.int8, device=DEV), C.linear_a8_w8_b8_o8(x, w, b, 3e-4, 0.02)
    need = C._lib.ti_linear_workspace_bytes(40, 2048, 8192)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    for _ in range(2):
        rc = C._lib.ti_linear_a8_w8_b8_o8(x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), 40, 2048, 8192, 3e-4, 0.02,
                                          ws.data_ptr(), need, 2)
        assert rc == 0 and _form() == 3
    torch.cuda.synchronize()
    assert torch.equal(out, want)
