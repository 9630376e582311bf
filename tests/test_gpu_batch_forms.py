"""Batches evaluated by their columns' forms (k_batch): every query has a column that is read from
its index, or there are too few queries to be evaluated together, and the plan says so.  All
tile, group and workgroup shapes, packed groups, list-form ranges, index sets and direct
columns beside indexed ones, against numpy.  And where queries are evaluated together, the plan
says that."""
import numpy as np
import pytest

from _util import MAXU
from test_gpu_batch import check_results, make_table, random_queries
from test_gpu_batch_rank import make_columns, make_plan, make_queries
from test_gpu_bins import datasets, engine_bin_starts

pytestmark = pytest.mark.gpu

AUTO, BINDEX, DIRECT = 0, 1, 2
SHAPES = [(1024, 16, 1, 512), (1024, 4, 0, 512), (1024, 1, 1, 512), (1024, 64, 0, 256), (2048, 8, 1, 512),
          (2048, 64, 0, 512), (2048, 16, 1, 256), (2048, 1, 0, 256), (512, 32, 1, 512), (512, 64, 0, 512),
          (512, 3, 1, 512), (512, 8, 1, 256)]


def pinned(queries, rest=AUTO):
    """The queries with one column each that is read from its index, the others' mode `rest`."""
    return [[(c, lo, hi, BINDEX if k == i % len(q) else rest) for k, (c, lo, hi, _) in enumerate(q)]
            for i, q in enumerate(queries)]


def buffers(eng, n, nq):
    stride = ((n + 31) // 32 + 3) // 4 * 4
    return stride, eng.DeviceBuffer(4 * stride * nq), eng.DeviceBuffer(8 * nq)


def launch_and_check(eng, plan, cols, queries, out, counts, stride):
    assert plan.stats()["together"] == 0
    out.fill(0xEE)
    counts.fill(0xFF)
    eng.synchronize()
    plan.launch(out, stride, counts)
    eng.synchronize()
    check_results(eng, cols, queries, out, counts, stride)


@pytest.mark.parametrize("tile_words,qgroup,order,threads", SHAPES)
def test_shapes(eng, tile_words, qgroup, order, threads):
    n = (1 << 20) + 12345  # partial last tile, partial last word
    cols, dcols, idx, sc = make_table(eng, n)
    rng = np.random.default_rng(tile_words + qgroup)
    plan = eng.BatchPlan(dcols, idx, n, 150, eng.batch_config(tile_words, qgroup, 4, order, threads))
    stride, out, counts = buffers(eng, n, 150)
    for queries in (pinned(random_queries(rng, sc, 150)), pinned(random_queries(rng, sc, 33), DIRECT),
                    random_queries(rng, sc, 7, direct_share=1.0), random_queries(rng, sc, 5, direct_share=0.4)):
        plan.set_queries(queries)
        launch_and_check(eng, plan, cols, queries, out, counts, stride)
    plan.free()


@pytest.mark.parametrize("n", [31 * 128, 5000, 70001])
def test_small_tables_with_shapes_in_turn(eng, n):
    cols, dcols, idx, sc = make_table(eng, n, seed=n % 97)
    rng = np.random.default_rng(n)
    plan = eng.BatchPlan(dcols, idx, n, 70)
    stride, out, counts = buffers(eng, n, 70)
    for nq in (70, 8, 1):
        queries = pinned(random_queries(rng, sc, nq))
        plan.set_queries(queries)
        for shape in [(2048, 32, 4, 1, 256), (512, 8, 2, 0, 512), (2048, 32, 4, 1, 256), (1024, 64, 1, 1, 256)]:
            plan.set_config(eng.batch_config(*shape))
            launch_and_check(eng, plan, cols, queries, out, counts, stride)
    plan.free()


@pytest.mark.parametrize("threads,order", [(256, 1), (256, 0), (512, 1)])
def test_packed_groups(eng, threads, order):
    """Queries of 1..4 columns fill the groups' slots: 4 | 3 + 1 | 2 + 2."""
    n = (1 << 18) + 77
    cols, dcols, idx, sc = make_table(eng, n, seed=29)
    rng = np.random.default_rng(threads + order)
    shape = [4] * 9 + [3] * 14 + [2] * 11 + [1] * 14
    rng.shuffle(shape)
    queries = []
    for k in shape:
        q = random_queries(rng, sc, 1, with_edges=False)[0]
        while len(q) != k:
            q = random_queries(rng, sc, 1, with_edges=False)[0]
        queries.append(q)
    queries = pinned(queries)
    plan = eng.BatchPlan(dcols, idx, n, len(queries), eng.batch_config(2048, 64, 4, order, threads))
    plan.set_queries(queries)
    assert plan.stats()["groups"] == -(-sum(shape) // (32 * threads // 2048))
    stride, out, counts = buffers(eng, n, len(queries))
    launch_and_check(eng, plan, cols, queries, out, counts, stride)
    plan.free()


def test_index_sets_and_direct_columns_by_cost(eng):
    n, nq = 1 << 20, 120
    cols, dcols, idx, sc = make_table(eng, n, seed=17)
    sets = [[eng.BinDexIndex(d, n, bins=b) for d in dcols] for b in (256, 512)]
    queries = pinned(random_queries(np.random.default_rng(6), sc, nq))
    plan = eng.BatchPlan(dcols, idx, n, nq)
    for s in sets:
        plan.add_indexes(s)
    plan.set_queries(queries)
    stride, out, counts = buffers(eng, n, nq)
    direct = 0
    for bins in (0, 256, 512, 128):
        for weight in (0, 40):
            plan.set_config(eng.batch_config(bins=bins, direct_weight=weight))
            direct += plan.stats()["auto_direct_cols"]
            launch_and_check(eng, plan, cols, queries, out, counts, stride)
    assert direct > 0
    plan.free()


@pytest.mark.parametrize("name", ["uniform", "zipf15", "small_range", "split_heavy"])
def test_list_form_ranges_at_bin_edges(eng, name):
    """Ranges from a bin's start, or one past it, to the ends of the next bins."""
    n = 1_000_003
    x = datasets(eng, n)[name]
    d = eng.DeviceBuffer.from_numpy(x)
    ix = eng.BinDexIndex(d, n, bins=256)
    st = engine_bin_starts(ix, np.sort(x), 256) + [MAXU + 1]
    queries = []
    for b in (0, 1, 2, 17, 63, 100, 127, 128, 200, 253, 254, 255):
        lo, nxt = st[b], st[min(b + 1, 256)]
        for hi_bin in (b + 1, b + 2, b + 3):
            hi = min(st[min(hi_bin, 256)] - 1, MAXU)
            queries += [[(0, at, hi, BINDEX)] for at in (lo, lo + 1) if at <= hi]
            if nxt <= MAXU and lo < nxt - 1:
                queries.append([(0, lo + 1, nxt, BINDEX)])
    stride, out, counts = buffers(eng, n, len(queries))
    for shape in ((2048, 64, 4, 1, 256), (512, 64, 4, 0, 512)):
        plan = eng.BatchPlan([d], [ix], n, len(queries), eng.batch_config(*shape))
        plan.set_queries(queries)
        if name == "uniform":
            assert plan.stats()["list_cols"] >= len(queries) // 3
        launch_and_check(eng, plan, [x], queries, out, counts, stride)
        plan.free()


def test_graph_replays_and_requeries(eng):
    n, nq = 1 << 20, 64
    cols, dcols, idx, sc = make_table(eng, n, seed=9)
    rng = np.random.default_rng(2)
    plan = eng.BatchPlan(dcols, idx, n, nq)
    stride, out, counts = buffers(eng, n, nq)
    stream = eng.Stream()
    scratch = eng.DeviceBuffer(4 * stride)
    for _ in range(3):
        queries = pinned(random_queries(rng, sc, nq))
        plan.set_queries(queries, stream)
        assert plan.stats()["together"] == 0
        for _ in range(2):
            out.fill(0x5A)
            eng.synchronize()
            plan.graph_launch(out, stride, counts, stream)
            stream.synchronize()
            check_results(eng, cols, queries, out, counts, stride)
            eng.scan_range(dcols[0], n, 5, 1 << 31, scratch, None, stream)
            stream.synchronize()
    plan.free()


@pytest.mark.parametrize("n", [1, 31, 8191, 8193, 20000, 70001, 300001])
@pytest.mark.parametrize("nq,ncols", [(8, 1), (33, 2), (64, 3), (65, 4), (300, 4)])
def test_queries_together(eng, n, nq, ncols):
    """Tables and sets that the evaluation together is tested with take it; a column that has to
    be read from its index keeps its query out, and fewer than eight queries stay apart."""
    cols = make_columns(n, ncols, n + nq)
    plan = make_plan(eng, cols, nq, indexed=n >= 128)
    queries = make_queries(cols, nq, n)
    plan.set_queries(queries)
    assert plan.stats()["together"] == nq
    plan.set_queries(queries[:7])
    assert plan.stats()["together"] == 0
    if n >= 128:
        plan.set_queries(pinned(queries))
        assert plan.stats()["together"] == 0
    plan.free()
