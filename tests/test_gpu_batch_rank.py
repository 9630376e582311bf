"""Batches whose queries are evaluated together from the columns (k_batch_ranked): bitmaps and
counts against numpy, at the edges of its steps, groups, blocks of queries and bound tables,
and next to queries that keep to their columns' own forms."""
import ctypes

import numpy as np
import pytest

from _util import MAXU, interval_mask, pack_rows

pytestmark = pytest.mark.gpu

AUTO, BINDEX, DIRECT = 0, 1, 2


def make_columns(n, ncols, seed):
    """Columns of which some values repeat and some sit at the ends of the domain."""
    rng = np.random.default_rng(seed)
    cols = []
    for c in range(ncols):
        x = rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)
        x[c::7] = MAXU
        x[c + 3::11] = 0
        x[5::13] &= np.uint32(0xFFFF0000)
        cols.append(x)
    return cols


def make_queries(cols, nq, seed, modes=(AUTO,), most=4):
    """1..4 ranges each, on any columns (also two of one column): random ones, empty ones, whole
    ones, single values, repeated ones, bounds at the domain's ends."""
    rng = np.random.default_rng(seed)
    out = []
    for i in range(nq):
        q = []
        for c in rng.integers(0, len(cols), int(rng.integers(1, most + 1))):
            lo, hi = sorted(int(v) for v in rng.integers(0, 2 ** 32, 2))
            kind = int(rng.integers(0, 12))
            if kind == 0:
                lo = 0
            elif kind == 1:
                hi = MAXU
            elif kind == 2:
                lo, hi = 0, MAXU
            elif kind == 3:
                lo = hi = int(cols[c][rng.integers(0, cols[c].size)])
            elif kind == 4:
                lo = hi = MAXU if i % 2 else 0
            elif kind == 5 and out:
                c, lo, hi, _ = out[-1][0]
            q.append((int(c), lo, hi, int(rng.choice(modes))))
        if i % 29 == 11:
            q[-1] = (q[-1][0], 9, 3, q[-1][3])  # empty
        out.append(q)
    return out


def make_plan(eng, cols, nq, indexed=True):
    n = cols[0].size
    dcols = [eng.DeviceBuffer.from_numpy(c) for c in cols]
    idx = [eng.BinDexIndex(d, n) if indexed else None for d in dcols]
    return eng.BatchPlan(dcols, idx, n, nq)


def check(eng, plan, cols, queries, counted=True, launch=None):
    n = cols[0].size
    words = (n + 31) // 32
    stride = (words + 3) // 4 * 4
    out = eng.DeviceBuffer(4 * (stride * len(queries) + 8)).fill(0xA5)
    counts = eng.DeviceBuffer(8 * len(queries)).fill(0xFF) if counted else None
    for _ in range(2):  # the second finds what the first left behind
        (launch or plan.launch)(out, stride, counts)
        eng.synchronize()
        got = out.to_numpy(np.uint32, stride * len(queries) + 8)
        assert (got[stride * len(queries):] == 0xA5A5A5A5).all()
        got = got[:-8].reshape(len(queries), stride)[:, :words]
        cnt = counts.to_numpy(np.uint64, len(queries)) if counted else None
        verify(cols, queries, got, cnt)


def verify(cols, queries, got, cnt):
    memo = {}
    for i, q in enumerate(queries):
        m = True
        for c, lo, hi, _ in q:
            if (c, lo, hi) not in memo:
                memo[c, lo, hi] = interval_mask(cols[c], lo, hi)
            m = m & memo[c, lo, hi]
        assert np.array_equal(got[i], pack_rows(m)), (i, q)
        assert cnt is None or int(cnt[i]) == int(m.sum()), (i, q)


# rows on both sides of a word, a lane's four words, a wave's and a workgroup's rows
@pytest.mark.parametrize("n", [1, 31, 33, 127, 2047, 2049, 8191, 8192, 8193, 16384 + 2048, 70001])
@pytest.mark.parametrize("nq,ncols", [(8, 1), (33, 2), (64, 3), (65, 4), (300, 4)])
def test_rows_and_blocks(eng, n, nq, ncols):
    cols = make_columns(n, ncols, n + nq)
    plan = make_plan(eng, cols, nq, indexed=n >= 128)
    queries = make_queries(cols, nq, n)
    plan.set_queries(queries)
    check(eng, plan, cols, queries, counted=nq != 65)
    plan.free()


# one group of 254 bounds; the last query into a second; 13 and 40 groups, which no XCD's
# workgroups divide evenly, so that a workgroup changes its group; the most queries of a group
# (repeated bounds); more columns than a group has
@pytest.mark.parametrize("n,nq,ncols,kind", [(20000, 40 * 127, 1, "own")] + [
    (n, *case) for n in (20000, 300001)
    for case in [(127, 1, "own"), (128, 1, "own"), (13 * 127, 1, "own"), (256, 2, "repeated"), (257, 4, "repeated"),
                 (200, 7, "own")]])
def test_groups(eng, n, nq, ncols, kind):
    cols = make_columns(n, ncols, nq)
    rng = np.random.default_rng(nq)
    queries = []
    for i in range(nq):
        c = i % ncols
        lo, hi = sorted(int(v) for v in rng.integers(1, 2 ** 32 - 1, 2))
        if kind == "repeated":
            lo, hi = (i * 7 % 10) << 28, ((i * 7 % 10) << 28) + (1 << 29)
        queries.append([(c, lo, hi, AUTO)])
    plan = make_plan(eng, cols, nq, indexed=n > 20000)
    plan.set_queries(queries)
    check(eng, plan, cols, queries)
    plan.free()


@pytest.mark.parametrize("modes", [(AUTO, DIRECT), (AUTO, BINDEX), (BINDEX,), (DIRECT,), (AUTO, BINDEX, DIRECT)])
@pytest.mark.parametrize("n", [40003, 1 << 20])
def test_modes(eng, modes, n):
    """Queries with a column that has to be read from its index keep out of the groups."""
    cols = make_columns(n, 4, 5)
    plan = make_plan(eng, cols, 150)
    for nq in (150, 40, 9, 7):
        queries = make_queries(cols, nq, nq, modes, most=2)
        plan.set_queries(queries)
        check(eng, plan, cols, queries)
    plan.free()


def test_unaligned_column_is_left_to_its_index(eng):
    n, nq = 50001, 64
    cols = make_columns(n, 2, 3)
    store = eng.DeviceBuffer.from_numpy(np.concatenate([np.zeros(1, np.uint32), cols[1]]))

    class View:
        ptr = store.ptr + 4

    dcols = [eng.DeviceBuffer.from_numpy(cols[0]), View]
    plan = eng.BatchPlan(dcols, [eng.BinDexIndex(d, n) for d in dcols], n, nq)
    queries = make_queries(cols, nq, 4)
    plan.set_queries(queries)
    check(eng, plan, cols, queries)
    plan.free()


@pytest.mark.parametrize("n", [8192 * 3, 40001])
def test_own_bitmaps(eng, n):
    """Bitmaps of the queries' own at 16-byte offsets, each just as long as it has to be."""
    cols = make_columns(n, 3, n)
    nq, words = 70, (n + 31) // 32
    queries = make_queries(cols, nq, 6)
    plan = make_plan(eng, cols, nq)
    pitch = (words + 4 + 3) // 4 * 4 + 4
    out = eng.DeviceBuffer(4 * pitch * nq).fill(0xA5)
    counts = eng.DeviceBuffer(8 * nq)
    outs = (ctypes.c_void_p * nq)(*[out.ptr + 4 * pitch * i for i in range(nq)])
    L = eng.lib()
    assert L.rts_batch_plan_set_queries_out(plan.h, eng.query_specs(queries), outs, nq, None) == 0
    assert L.rts_batch_plan_launch(plan.h, None, 0, counts.ptr, None) == 0
    eng.synchronize()
    got = out.to_numpy(np.uint32, pitch * nq).reshape(nq, pitch)
    assert (got[:, words:] == 0xA5A5A5A5).all()
    verify(cols, queries, got[:, :words], counts.to_numpy(np.uint64, nq))
    plan.free()


def test_captured_launches_follow_the_queries(eng):
    """A launch in the caller's own graph, and graph_launch, evaluate the queries that are set
    after the capture, whichever form they take, with eager work in between."""
    n, nq = 100003, 64
    cols = make_columns(n, 3, 8)
    plan = make_plan(eng, cols, nq)
    stream = eng.Stream()
    words = (n + 31) // 32
    stride = (words + 3) // 4 * 4
    out = eng.DeviceBuffer(4 * stride * nq)
    counts = eng.DeviceBuffer(8 * nq)
    sets = [make_queries(cols, nq, 10 + i, m) for i, m in enumerate([(AUTO,), (BINDEX,), (AUTO,), (AUTO, BINDEX), (DIRECT,)])]
    hip = ctypes.CDLL("libamdhip64.so.7")
    graph, instance = ctypes.c_void_p(), ctypes.c_void_p()
    s = ctypes.c_void_p(stream.handle)
    plan.set_queries(sets[1], stream)
    plan.launch(out, stride, counts, stream)
    stream.synchronize()
    assert hip.hipStreamBeginCapture(s, 1) == 0
    plan.launch(out, stride, counts, stream)
    assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(instance), graph, None, None, ctypes.c_size_t(0)) == 0
    for queries in sets * 2:
        plan.set_queries(queries, stream)
        for replay in (lambda: hip.hipGraphLaunch(instance, s), lambda: plan.graph_launch(out, stride, counts, stream),
                       lambda: plan.launch(out, stride, counts, stream)):
            out.fill(0x5A)
            counts.fill(0x5A)
            eng.synchronize()
            assert not replay()
            stream.synchronize()
            verify(cols, queries, out.to_numpy(np.uint32, stride * nq).reshape(nq, stride)[:, :words],
                   counts.to_numpy(np.uint64, nq))
    assert hip.hipGraphExecDestroy(instance) == 0 and hip.hipGraphDestroy(graph) == 0
    plan.free()
