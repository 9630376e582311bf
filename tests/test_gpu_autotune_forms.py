"""The autotuner times the launch shapes on the kernel that they belong to, also with queries that
the plan evaluates together."""
import numpy as np
import pytest

from test_gpu_batch import check_results
from test_gpu_batch_rank import DIRECT, make_columns

pytestmark = pytest.mark.gpu


def test_shapes_are_timed_by_the_columns_forms(eng):
    n, nq = 4_000_000, 256
    cols = make_columns(n, 2, 1)
    rng = np.random.default_rng(2)
    queries = [[(c, *sorted(int(v) for v in rng.integers(0, 2 ** 32, 2)), DIRECT) for c in (0, 1)] for _ in range(nq)]
    plan = eng.BatchPlan([eng.DeviceBuffer.from_numpy(c) for c in cols], [None, None], n, nq)
    plan.set_queries(queries)
    assert plan.stats()["together"] == nq
    stride = n // 32
    out, counts = eng.DeviceBuffer(4 * stride * nq), eng.DeviceBuffer(8 * nq)
    stream = eng.Stream()
    a, b = eng.Event(), eng.Event()
    plan.launch(out, stride, counts, stream)
    times = []
    for _ in range(5):
        a.record(stream)
        plan.launch(out, stride, counts, stream)
        b.record(stream)
        b.synchronize()
        times.append(a.elapsed_ms(b))
    together_ms = sorted(times)[2]
    good, bad = eng.batch_config(2048, 32, 4, 1, 256), eng.batch_config(512, 1, 1, 1, 256)
    for candidates in ([good, bad], [bad, good]):
        chosen, ms = plan.autotune(out, stride, candidates, reps=3, stream=stream)
        # a query a work item on one workgroup a compute unit; every row tested for every
        # query-column where together it is searched once a column
        assert chosen.astuple() == good.astuple()
        assert ms > 2 * together_ms, (ms, together_ms)
        assert plan.stats()["together"] == nq
    plan.launch(out, stride, counts, stream)
    stream.synchronize()
    check_results(eng, cols, queries, out, counts, stride)
    plan.free()
