"""A batch launch in the caller's own graph, replayed with more and with fewer queries than it was
captured with: every bitmap, the counts that it was captured for, and the counts of the
launches after it."""
import ctypes

import numpy as np
import pytest

from test_gpu_batch_rank import AUTO, BINDEX, make_columns, make_plan, make_queries, verify

pytestmark = pytest.mark.gpu

POISON = 0x5A5A5A5A5A5A5A5A


# captured with queries that are evaluated together, and with queries that keep to their indexes
@pytest.mark.parametrize("first", [AUTO, BINDEX])
@pytest.mark.parametrize("modes", [(AUTO,), (AUTO, BINDEX)])
@pytest.mark.parametrize("captured", [16, 100])
def test_replays_with_more_and_fewer_queries(eng, captured, modes, first):
    n, most = 100003, 300
    cols = make_columns(n, 3, 8)
    plan = make_plan(eng, cols, most)
    stream = eng.Stream()
    words = (n + 31) // 32
    stride = (words + 3) // 4 * 4
    out = eng.DeviceBuffer(4 * stride * most)
    counts = eng.DeviceBuffer(8 * most)
    sets = {nq: make_queries(cols, nq, nq, modes if nq > 64 else (AUTO,), most=2) for nq in (16, 64, 100, 300, 9)}
    hip = ctypes.CDLL("libamdhip64.so.7")
    graph, instance = ctypes.c_void_p(), ctypes.c_void_p()
    s = ctypes.c_void_p(stream.handle)
    plan.set_queries(make_queries(cols, captured, captured, (first,), most=2), stream)
    assert plan.stats()["together"] == (captured if first == AUTO else 0)
    plan.launch(out, stride, counts, stream)
    stream.synchronize()
    assert hip.hipStreamBeginCapture(s, 1) == 0
    plan.launch(out, stride, counts, stream)
    assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(instance), graph, None, None, ctypes.c_size_t(0)) == 0
    for nq in (captured, 300, 64, 9, 300, 100, 16, 300):
        queries = sets[nq]
        plan.set_queries(queries, stream)
        # a graph that has the indexes' kernel alone takes nothing from the launches beside it
        assert plan.stats()["together"] == sum(all(m == AUTO for *_, m in q) for q in queries) or nq > 64 and BINDEX in modes
        for launch in ("replay", "replay", "launch", "graph_launch", "replay", "launch"):
            out.fill(0x5A)
            counts.fill(0x5A)
            eng.synchronize()
            if launch == "replay":
                assert hip.hipGraphLaunch(instance, s) == 0
            else:
                getattr(plan, launch)(out, stride, counts, stream)
            stream.synchronize()
            got = out.to_numpy(np.uint32, stride * most).reshape(most, stride)
            cnt = counts.to_numpy(np.uint64, most)
            written = min(nq, captured) if launch == "replay" else nq
            first_unwritten = captured if launch == "replay" and first == BINDEX else written
            assert (cnt[first_unwritten:] == POISON).all(), (nq, launch)
            assert (got[nq:] == POISON & 0xFFFFFFFF).all(), (nq, launch)
            verify(cols, queries[:written], got[:written, :words], cnt[:written])
            verify(cols, queries, got[:nq, :words], None)
    assert hip.hipGraphExecDestroy(instance) == 0 and hip.hipGraphDestroy(graph) == 0
    plan.free()
