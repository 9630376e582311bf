"""Calls beside a stream capture, of the capturing thread and of another: what HIP allows there
leaves the capture whole, and the captured work runs."""
import ctypes
import threading

import numpy as np
import pytest

from _util import interval_mask, pack_rows

pytestmark = pytest.mark.gpu

GLOBAL, THREAD_LOCAL, RELAXED = 0, 1, 2
N = 300_000


def captured_beside(eng, mode, other_thread, call):
    """Captures two scans on a stream with `call` between them, then replays them."""
    rng = np.random.default_rng(4)
    x = rng.integers(0, 2 ** 32, N, dtype=np.uint64).astype(np.uint32)
    d = eng.DeviceBuffer.from_numpy(x)
    words = (N + 31) // 32
    outs = [eng.DeviceBuffer(4 * words) for _ in range(2)]
    stream = eng.Stream()
    hip = ctypes.CDLL("libamdhip64.so.7")
    s = ctypes.c_void_p(stream.handle)
    graph, instance = ctypes.c_void_p(), ctypes.c_void_p()
    eng.scan_range(d, N, 1, 2, outs[0], stream=stream)
    eng.synchronize()
    assert hip.hipStreamBeginCapture(s, mode) == 0
    eng.scan_range(d, N, 1 << 30, 1 << 31, outs[0], stream=stream)
    if other_thread:
        t = threading.Thread(target=call)
        t.start()
        t.join()
    else:
        call()
    second = eng.lib().rts_scan_range(d.ptr, N, 1 << 31, 3 << 30, outs[1].ptr, None, stream.handle)
    end = hip.hipStreamEndCapture(s, ctypes.byref(graph))
    hip.hipGetLastError()
    assert (second, end) == (0, 0)
    assert hip.hipGraphInstantiate(ctypes.byref(instance), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        for o in outs:
            o.fill(0xA5)
        eng.synchronize()
        assert hip.hipGraphLaunch(instance, s) == 0
        stream.synchronize()
        for o, (lo, hi) in zip(outs, [(1 << 30, 1 << 31), (1 << 31, 3 << 30)]):
            assert np.array_equal(o.to_numpy(np.uint32, words), pack_rows(interval_mask(x, lo, hi)))
    assert hip.hipGraphExecDestroy(instance) == 0 and hip.hipGraphDestroy(graph) == 0


# hipFree, with which an index goes, is refused in the other two modes' capturing threads
@pytest.mark.parametrize("mode,other_thread", [(THREAD_LOCAL, True), (RELAXED, False), (RELAXED, True)])
def test_an_index_freed(eng, mode, other_thread):
    rng = np.random.default_rng(5)
    d = eng.DeviceBuffer.from_numpy(rng.integers(0, 2 ** 32, N, dtype=np.uint64).astype(np.uint32))
    index = eng.BinDexIndex(d, N)
    captured_beside(eng, mode, other_thread, index.free)


@pytest.mark.parametrize("mode", [GLOBAL, THREAD_LOCAL, RELAXED])
@pytest.mark.parametrize("other_thread", [False, True])
def test_free_memory_asked_for(eng, mode, other_thread):
    """While the library keeps memory of a freed index."""
    rng = np.random.default_rng(5)
    d = eng.DeviceBuffer.from_numpy(rng.integers(0, 2 ** 32, N, dtype=np.uint64).astype(np.uint32))
    eng.BinDexIndex(d, N).free()
    captured_beside(eng, mode, other_thread, eng.device_free_bytes)
