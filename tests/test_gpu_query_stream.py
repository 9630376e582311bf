"""BinDex queries whose filter vectors and result pass the caches by (long columns): bitmaps and
counts against numpy, on both sides of the size from which they do, for one to five columns,
with a last word and a last four words that are not whole, and a result off 16 bytes."""
import numpy as np
import pytest

from _util import MAXU, interval_mask, pack_rows

pytestmark = pytest.mark.gpu

BYTES = 9 << 20


def _edge(ncols):
    """The rows from which filter vectors and result of `ncols` columns have that many bytes."""
    return 32 * -(-BYTES // (4 * (2 * ncols + 1)))


@pytest.mark.parametrize("ncols", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("rows", [-33, 0, 32 * 1024 * 3 + 7, 32 * 2 + 1])
def test_queries(eng, ncols, rows):
    n = _edge(min(ncols, 4)) + rows
    rng = np.random.default_rng(n)
    cols = [rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(ncols)]
    dcols = [eng.DeviceBuffer.from_numpy(c) for c in cols]
    idx = [eng.BinDexIndex(d, n) for d in dcols]
    words = (n + 31) // 32
    store, count = eng.DeviceBuffer(4 * (words + 3)), eng.DeviceBuffer(8)
    for i, kind in enumerate(("wide", "narrow", "ends", "wide")):
        lo, hi = [], []
        for c in range(ncols):
            a, b = sorted(int(v) for v in rng.integers(0, 2 ** 32, 2))
            if kind == "narrow":
                b = min(MAXU, a + (1 << 22))
            elif kind == "ends":
                a, b = (0, b) if c % 2 else (a, MAXU)
            lo.append(a)
            hi.append(b)
        offset = i % 2 * (1 + ncols % 3)

        class Out:
            ptr = store.ptr + 4 * offset

        store.fill(0xA5)
        eng.bindex_query(idx, lo, hi, Out, count)
        eng.synchronize()
        m = np.ones(n, bool)
        for c in range(ncols):
            m &= interval_mask(cols[c], lo[c], hi[c])
        got = store.to_numpy(np.uint32, words + 3)
        assert np.array_equal(got[offset:offset + words], pack_rows(m)), kind
        assert (got[:offset] == 0xA5A5A5A5).all() and (got[offset + words:] == 0xA5A5A5A5).all(), kind
        assert int(count.to_numpy(np.uint64, 1)[0]) == int(m.sum()), kind
    for x in idx:
        x.free()
