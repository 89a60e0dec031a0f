"""Who holds the device memory whose address a launch is handed: scratch and workspaces of the Python layer, with the
allocations done in host memory (no kernel runs)."""
import ctypes
import threading
import types
import weakref

import pytest
import torch

from torch_int import _CUDA, _hip_ext


@pytest.fixture
def host_memory(monkeypatch):
    """torch.empty and the stream queries of the two modules without a HIP device."""
    def empty(*shape, device=None, **kw):
        return torch.zeros(*shape, **kw)
    fake = types.SimpleNamespace(**{n: getattr(torch, n) for n in ("uint8", "int8", "float32", "device", "Tensor")}, empty=empty,
                                 cuda=types.SimpleNamespace(is_current_stream_capturing=lambda: fake.capturing), capturing=False)
    for mod in (_CUDA, _hip_ext):
        monkeypatch.setattr(mod, "torch", fake)
        monkeypatch.setattr(mod, "_raw_stream", lambda index: 7)
    monkeypatch.setattr(_hip_ext, "_current_device", lambda: 0)
    monkeypatch.setattr(_CUDA, "_workspaces", {})
    monkeypatch.setattr(_hip_ext, "_layer_scratch", {})
    monkeypatch.setattr(_hip_ext, "_layer_scratch_need", {})
    return fake


def _hidden(rows, width):
    return types.SimpleNamespace(device=types.SimpleNamespace(index=0), shape=(1, rows, width))


def test_a_prefill_holds_its_workspace_while_another_thread_replaces_the_streams(host_memory):
    # 256 rows at these widths are split over K, so the pass has a workspace; a second thread on the same stream asks for
    # a larger one between two layers
    plan = types.SimpleNamespace(embed=5120, ffn=20480)
    memory = _hip_ext.opt_prefill_scratch([plan], _hidden(256, 5120))
    held = weakref.ref(_CUDA._workspaces[(0, 7)])
    address = held().data_ptr()
    assert address in [v for v in memory if type(v) is int]
    _CUDA._workspace(0, 7, held().numel() + 1)
    assert held() is not None and held().data_ptr() == address and held() is not _CUDA._workspaces[(0, 7)]
    del memory
    assert held() is None


@pytest.mark.parametrize("get", [lambda n: _CUDA._workspace(0, 7, n)[0],
                                 lambda n: _hip_ext._scratch_for(types.SimpleNamespace(index=0), 7, n)])
def test_a_recording_gets_memory_that_the_stream_does_not_keep(host_memory, get):
    # a graph holds the address for its life; the stream's buffer goes back to the allocator when a call needs a larger one,
    # and is written by every eager call beside a replay
    eager = get(4096)
    host_memory.capturing = True
    first, second = get(1024), get(1024)
    assert len({eager.data_ptr(), first.data_ptr(), second.data_ptr()}) == 3
    held = weakref.ref(first)
    del first
    assert held() is None
    host_memory.capturing = False
    assert get(1024) is eager


def test_memory_of_a_pass_fits_its_widest_layer(host_memory):
    # 304 rows of a 20480 wide layer are split over K and need a workspace; the narrow first layer needs none
    plans = [types.SimpleNamespace(embed=5120, ffn=f) for f in (512, 20480, 1024)]
    scratch, _, _, ws_bytes = _hip_ext.opt_prefill_scratch(plans, _hidden(304, 5120))
    assert scratch.numel() >= _hip_ext._lib.ti_opt_decoder_layer_prefill_chained_scratch_bytes(304, 5120, 20480)
    assert ws_bytes >= _CUDA._ws_bytes(304, 5120, 20480) > 0
    one = types.SimpleNamespace(device=types.SimpleNamespace(index=0), shape=(40, 1, 5120))
    assert _hip_ext.opt_decode_scratch(plans, one).numel() >= _hip_ext._lib.ti_opt_decoder_layer_decode_scratch_bytes(40, 5120, 20480)


@pytest.mark.parametrize("half", [False, True])
def test_passes_of_two_threads_on_one_stream_have_memory_of_their_own(host_memory, monkeypatch, half):
    # all layers of a decode step come from one C call that gives up the interpreter lock: two threads are inside at once, and
    # what one layer hands to its next kernel must not lie where the other thread's layer does (the fp16 stream's carry neither)
    both_inside, calls = threading.Barrier(2, timeout=20), []

    def call(layers, count, hidden, mask, k_bufs, v_bufs, bsz, cap, S, carry, scratch, nbytes, stream):
        calls.append((scratch, nbytes, carry))
        both_inside.wait()
        return 0
    monkeypatch.setattr(_hip_ext, "_layers_decode", call)
    plans = [types.SimpleNamespace(embed=64, ffn=256, addr=16, half=half)] * 3
    hidden = types.SimpleNamespace(device=types.SimpleNamespace(index=0), shape=(5, 1, 64), data_ptr=lambda: 256)
    threads = [threading.Thread(target=_hip_ext.opt_layers_decode, args=(plans, hidden, None, None, None, 64, 9)) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    need, carried = _hip_ext._lib.ti_opt_decoder_layer_decode_scratch_bytes(5, 64, 256), 4 * 5 * 64
    ranges = sorted((at, at + n) for scratch, n, carry in calls for at, n in [(scratch, n)] + ([(carry, carried)] if half else []))
    assert len(calls) == 2 and all(n >= need for _, n, _ in calls) and len(ranges) == (4 if half else 2)
    assert all(carry is None or carry % 16 == 0 for *_, carry in calls) and all((carry is None) == (not half) for *_, carry in calls)
    assert all(end <= start for (_, end), (start, _) in zip(ranges, ranges[1:])), ranges
    assert not _hip_ext._layer_scratch


def test_calls_that_are_handed_memory_of_the_stream_keep_the_interpreter_lock():
    # split-K products and layers issued one by one are several launches, which hand one another tiles in the stream's workspace or
    # scratch: another thread must not launch between them.  (The forwarder in C keeps the lock as it is.)
    kept = [*_CUDA._LINEAR_CTYPES.values(), *_CUDA._BMM_CTYPES.values(), *_CUDA._BMM_WS_CTYPES.values()]
    kept += [getattr(_hip_ext._lib, name) for name in ("ti_linear_a8_w8_b8_o8_heads", "ti_opt_decoder_layer_decode_from",
                                                       "ti_opt_decoder_layer_prefill_chained")]
    flag = type(ctypes.pythonapi.Py_IncRef)._flags_ & ~ctypes.CDLL(None)._FuncPtr._flags_
    assert flag and all(type(fn)._flags_ & flag for fn in kept)
    # the call whose memory is its own lets other threads run
    assert not type(_hip_ext._layers_decode)._flags_ & flag
