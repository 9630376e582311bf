"""Range sets whose bitmaps pass through LDS (more bytes than the caches hold, not on cache lines):
bitmaps at 16-byte offsets, which take 16-byte stores, and at 4-byte ones, whole halves of 32
predicates and parts, against one range a call."""
import numpy as np
import pytest

from _util import interval_mask, pack_rows
from test_gpu_ranges import _column, _ranges

pytestmark = pytest.mark.gpu


class _Part:
    def __init__(self, buf, off):
        self.ptr = buf.ptr + off


@pytest.mark.parametrize("counted", [True, False])
@pytest.mark.parametrize("n,npred,pad,wide", [(45_000_003, 64, 1, True), (45_000_003, 63, 1, True),
                                              (90_000_001, 31, 3, True), (90_000_001, 32, 7, True),
                                              (45_000_003, 64, 0, False)])
def test_store_widths(eng, n, npred, pad, wide, counted):
    words = (n + 31) // 32
    stride = words + pad
    assert 4 * words * npred >= 320 << 20 and stride % 32 and (stride % 4 == 0) == wide
    x = _column(n, n % 1000)
    preds = _ranges(x, npred, npred)
    col = eng.DeviceBuffer.from_numpy(x)
    out = eng.DeviceBuffer(4 * npred * stride).fill(0xA5)
    counts = eng.DeviceBuffer(8 * npred) if counted else None
    eng.scan_ranges(col, n, [p[0] for p in preds], [p[1] for p in preds], out, stride, counts)
    eng.synchronize()
    one, c1 = eng.DeviceBuffer(4 * words), eng.DeviceBuffer(8)
    for p, (lo, hi) in enumerate(preds):
        eng.scan_range(col, n, lo, hi, one, c1)
        eng.synchronize()
        r = eng.bitmap_compare(one, _Part(out, 4 * p * stride), n)
        assert r["first_mismatch"] == -1 and r["truth_count"] == r["got_count"], (p, r)
        if counted:
            assert counts.to_numpy(np.uint64, npred)[p] == c1.to_numpy(np.uint64, 1)[0], p
    got = out.to_numpy(np.uint32, npred * stride).reshape(npred, stride)
    assert (got[:, words:] == 0xA5A5A5A5).all()
    for p in (2, npred - 1):
        lo, hi = preds[p]
        assert np.array_equal(got[p, :words], pack_rows(interval_mask(x, lo, hi) if lo <= hi else np.zeros(n, bool))), p
