"""Batches of which some queries have to be read from an index: the others are evaluated together
only where both kernels take less time than one, and every bitmap and count is right either way."""
import numpy as np
import pytest

from test_gpu_batch_rank import AUTO, BINDEX, DIRECT, check, make_columns, make_plan, make_queries

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ncols,nq,every,rest,together", [
    (100_000, 4, 16, 2, AUTO, False),  # two kernels of 20 and 28 us for one of 29
    (1_000_003, 4, 64, 2, AUTO, False),
    (4_200_000, 4, 128, 2, AUTO, False),
    (100_000, 2, 1024, 2, AUTO, False),
    (1_000_003, 4, 256, 8, DIRECT, True)])  # the columns' forms test the rows of every direct column
def test_some_queries_from_their_indexes(eng, n, ncols, nq, every, rest, together):
    cols = make_columns(n, ncols, nq)
    queries = make_queries(cols, nq, 3, most=ncols)
    queries = [[(c, lo, hi, BINDEX if i % every == 0 else rest) for c, lo, hi, _ in q] for i, q in enumerate(queries)]
    plan = make_plan(eng, cols, nq)
    plan.set_queries(queries)
    assert plan.stats()["together"] == (sum(q[0][3] == rest for q in queries) if together else 0)
    check(eng, plan, cols, queries)
    plan.free()
