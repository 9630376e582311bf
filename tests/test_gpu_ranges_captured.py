"""Counted range sets in a captured graph, replayed on another stream beside launches of the stream
that it was captured on: the counts of both, then and afterwards."""
import ctypes

import numpy as np
import pytest

from test_gpu_ranges import _column, _ranges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npred", [5, 64, 70])
def test_replays_beside_launches(eng, npred):
    n = 3_000_001
    x = _column(n, 7)
    col = eng.DeviceBuffer.from_numpy(x)
    words = (n + 31) // 32
    sets = [_ranges(x, npred, 1), _ranges(x, npred, 2)]
    want = [[int(((x >= lo) & (x <= hi)).sum()) for lo, hi in preds] for preds in sets]
    outs = [eng.DeviceBuffer(4 * npred * words) for _ in range(2)]
    a, b = eng.Stream(), eng.Stream()

    def scan(k, counts):
        eng.scan_ranges(col, n, [p[0] for p in sets[k]], [p[1] for p in sets[k]], outs[k], words, counts, a)

    replayed, launched = eng.DeviceBuffer(8 * npred), [eng.DeviceBuffer(8 * npred) for _ in range(20)]
    scan(0, replayed)  # the first call of a stream allocates
    a.synchronize()
    hip = ctypes.CDLL("libamdhip64.so.7")
    sa, sb = ctypes.c_void_p(a.handle), ctypes.c_void_p(b.handle)
    graph, instance = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(sa, 1) == 0
    scan(1, replayed)
    assert hip.hipStreamEndCapture(sa, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(instance), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        replayed.fill(0xFF)
        for c in launched:
            c.fill(0xFF)
        eng.synchronize()
        for c in launched:
            assert hip.hipGraphLaunch(instance, sb) == 0  # one after another, on the other stream
            scan(0, c)
        a.synchronize()
        b.synchronize()
        assert replayed.to_numpy(np.uint64, npred).tolist() == want[1]
        for c in launched:
            assert c.to_numpy(np.uint64, npred).tolist() == want[0]
    assert hip.hipGraphExecDestroy(instance) == 0 and hip.hipGraphDestroy(graph) == 0


@pytest.mark.parametrize("npred", [5, 64])
def test_first_call_of_a_stream_in_a_relaxed_capture(eng, npred):
    """It allocates, which that mode allows; the launches of the stream before and after the first
    replay count right, and so do the replays."""
    n = 1_100_003
    x = _column(n, 3)
    col = eng.DeviceBuffer.from_numpy(x)
    words = (n + 31) // 32
    preds = _ranges(x, npred, 1)
    want = [int(((x >= lo) & (x <= hi)).sum()) for lo, hi in preds]
    out, counts = eng.DeviceBuffer(4 * npred * words), eng.DeviceBuffer(8 * npred)
    junk = eng.DeviceBuffer(64 << 10).fill(0x77)  # what a new buffer may hold
    eng.synchronize()
    del junk
    stream = eng.Stream()
    s = ctypes.c_void_p(stream.handle)
    hip = ctypes.CDLL("libamdhip64.so.7")
    graph, instance = ctypes.c_void_p(), ctypes.c_void_p()

    def scan():
        eng.scan_ranges(col, n, [p[0] for p in preds], [p[1] for p in preds], out, words, counts, stream)

    assert hip.hipStreamBeginCapture(s, 2) == 0
    scan()
    assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(instance), graph, None, None, ctypes.c_size_t(0)) == 0
    for launch in (scan, scan, lambda: hip.hipGraphLaunch(instance, s), scan, lambda: hip.hipGraphLaunch(instance, s)):
        counts.fill(0xFF)
        eng.synchronize()
        launch()
        stream.synchronize()
        assert counts.to_numpy(np.uint64, npred).tolist() == want
    assert hip.hipGraphExecDestroy(instance) == 0 and hip.hipGraphDestroy(graph) == 0
