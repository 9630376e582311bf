"""Queries evaluated together over tables that give a workgroup several work items: of one group,
of groups whose number divides the workgroups (it stays with its group), and of groups whose
number does not (it changes its group, whose tables and counts it then exchanges)."""
import numpy as np
import pytest

from _util import pack_rows
from test_gpu_batch_rank import AUTO, make_columns

pytestmark = pytest.mark.gpu

STEP = 8192  # rows of a workgroup's step


class _Part:
    def __init__(self, buf, off):
        self.ptr = buf.ptr + off


@pytest.mark.parametrize("n,nq,ngroups,run", [(9_000_011, 40, 1, 1), (4_000_003, 4 * 127, 4, 1), (5_000_033, 13 * 127, 13, 4)])
@pytest.mark.parametrize("counted", [True, False])
def test_several_items_a_workgroup(eng, n, nq, ngroups, run, counted):
    per_xcd = 2 * eng.device_info()["cus"] // 8
    even = per_xcd // ngroups * ngroups
    stays = 16 * even >= 15 * per_xcd
    assert stays == (run == 1)
    runs = -(-(-(-n // STEP)) // run)
    items = -(-runs // 8) * ngroups  # of an XCD
    assert items > 2 * per_xcd  # three rounds and more
    x = make_columns(n, 1, nq)[0]
    rng = np.random.default_rng(nq)
    bounds = rng.choice(2 ** 32 - 2, 2 * nq, replace=False).astype(np.uint64) + 1  # all distinct: 254 a group
    queries = [[(0, int(min(a, b)), int(max(a, b)), AUTO)] for a, b in bounds.reshape(nq, 2)]
    col = eng.DeviceBuffer.from_numpy(x)
    plan = eng.BatchPlan([col], [None], n, nq)
    plan.set_queries(queries)
    assert plan.stats()["together"] == nq
    words = (n + 31) // 32
    stride = (words + 3) // 4 * 4
    out, counts = eng.DeviceBuffer(4 * stride * nq), eng.DeviceBuffer(8 * nq).fill(0xFF)
    ordered = np.sort(x)
    want = [int(np.searchsorted(ordered, hi, "right") - np.searchsorted(ordered, lo, "left")) for [(_, lo, hi, _)] in queries]
    one = eng.DeviceBuffer(4 * words)
    for _ in range(2):  # the second finds the sums that the first left behind
        out.fill(0xA5)
        eng.synchronize()
        plan.launch(out, stride, counts if counted else None)
        eng.synchronize()
        if counted:
            assert counts.to_numpy(np.uint64, nq).tolist() == want
    for i, [(_, lo, hi, _)] in enumerate(queries):
        eng.scan_range(col, n, lo, hi, one)
        eng.synchronize()
        r = eng.bitmap_compare(one, _Part(out, 4 * i * stride), n)
        assert r["first_mismatch"] == -1 and r["got_count"] == want[i], (i, r)
        if i % 97 == 5:
            got = np.empty(words, np.uint32)
            eng.check(eng.lib().rts_memcpy_dtoh(got.ctypes.data, out.ptr + 4 * i * stride, 4 * words), "dtoh")
            assert np.array_equal(got, pack_rows((x >= lo) & (x <= hi))), i
    plan.free()
