"""rts_scan_ranges by searching the predicates' bounds (long columns, many predicates): bitmaps
and counts against numpy, at the edges of its tiles, halves and tables."""
import numpy as np
import pytest

from _util import MAXU, interval_mask, pack_rows

pytestmark = pytest.mark.gpu


def _column(n, seed):
    """Values of which some repeat and some sit at the ends of the domain."""
    rng = np.random.default_rng(seed)
    x = rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)
    x[::7] = MAXU
    x[3::11] = 0
    x[5::13] = x[5::13] & np.uint32(0xFFFF0000)
    return x


def _ranges(x, npred, seed):
    """Random ranges with empty ones, whole ones, single values, repeated ones and bounds at
    the domain's ends and at values of the column."""
    rng = np.random.default_rng(seed)
    out = []
    for i in range(npred):
        lo, hi = sorted(int(v) for v in rng.integers(0, 2 ** 32, 2))
        kind = i % 9
        if kind == 1:
            lo, hi = hi, lo  # empty (or one value)
        elif kind == 2:
            lo = 0
        elif kind == 3:
            hi = MAXU
        elif kind == 4:
            lo, hi = 0, MAXU
        elif kind == 5:
            lo = hi = int(x[rng.integers(0, x.size)])
        elif kind == 6 and out:
            lo, hi = out[-3]
        elif kind == 7:
            lo = hi = MAXU
        out.append((lo, hi))
    return out


def _check(eng, x, preds, offset=0, counted=True, pad=0):
    n, k, words = x.size, len(preds), (x.size + 31) // 32
    stride = words + pad
    store = eng.DeviceBuffer.from_numpy(np.concatenate([np.zeros(offset, np.uint32), x]))

    class View:
        ptr = store.ptr + 4 * offset

    out = eng.DeviceBuffer(4 * k * stride).fill(0xA5)
    counts = eng.DeviceBuffer(8 * k).fill(0xFF) if counted else None
    eng.scan_ranges(View, n, [p[0] for p in preds], [p[1] for p in preds], out, stride, counts)
    eng.synchronize()
    got = out.to_numpy(np.uint32, k * stride).reshape(k, stride)
    for p, (lo, hi) in enumerate(preds):
        mask = interval_mask(x, lo, hi) if lo <= hi else np.zeros(n, bool)
        assert np.array_equal(got[p, :words], pack_rows(mask)), p
        if counted:
            assert int(counts.to_numpy(np.uint64, k)[p]) == int(mask.sum()), p
    if pad:
        assert (got[:, words:] == 0xA5A5A5A5).all()


@pytest.mark.parametrize("n", [(1 << 18) - 1, (3 << 17) - 1, 3 << 17, (3 << 17) + 2047, (1 << 20) + 1])
@pytest.mark.parametrize("npred", [17, 40, 41, 63, 64, 107])
def test_many_ranges_sizes(eng, n, npred):
    x = _column(n, n)
    _check(eng, x, _ranges(x, npred, npred), pad=npred % 3)


@pytest.mark.parametrize("npred", [8, 9, 31, 32, 33])
def test_ranges_of_a_long_column(eng, npred):
    n = (1 << 22) + 2049
    x = _column(n, npred)
    _check(eng, x, _ranges(x, npred, npred))


@pytest.mark.parametrize("offset", [1, 2, 3])
@pytest.mark.parametrize("counted", [False, True])
def test_many_ranges_of_an_unaligned_column(eng, offset, counted):
    x = _column((3 << 17) + 77, offset)
    _check(eng, x, _ranges(x, 64, offset), offset=offset, counted=counted)


def test_ranges_with_128_distinct_bounds_and_with_none(eng):
    """Every node of the search in use (64 disjoint ranges), and no bound at all (64 empty
    ranges)."""
    x = _column(1 << 20, 5)
    cuts = [int(v) for v in np.linspace(7, MAXU - 7, 128).astype(np.uint64)]
    _check(eng, x, [(cuts[2 * i], cuts[2 * i + 1]) for i in range(64)])
    _check(eng, x, [(9, 3)] * 64)


def test_ranges_of_a_column_of_one_value(eng):
    """All rows in one range of the search: the row counts' worst case."""
    for value in (0, 12345, MAXU):
        x = np.full((1 << 20) + 5, value, np.uint32)
        _check(eng, x, _ranges(x, 64, 1) + [(value, value)] * 3)


@pytest.mark.parametrize("n,npred,pad", [(45_000_003, 63, 0), (45_000_003, 64, 2), (90_000_001, 31, 1)])
def test_bitmaps_of_many_bytes_off_cache_lines(eng, n, npred, pad):
    """Bitmaps of more bytes than the caches hold that don't start on cache lines, at 4- and at
    16-byte offsets: against one range a call, and numpy for some."""
    words = (n + 31) // 32
    stride = words + pad
    assert 4 * words * npred >= 320 << 20 and stride % 32
    x = _column(n, n % 1000)
    preds = _ranges(x, npred, npred)
    col = eng.DeviceBuffer.from_numpy(x)
    out = eng.DeviceBuffer(4 * npred * stride).fill(0xA5)
    counts = eng.DeviceBuffer(8 * npred)
    eng.scan_ranges(col, n, [p[0] for p in preds], [p[1] for p in preds], out, stride, counts)
    eng.synchronize()
    got = out.to_numpy(np.uint32, npred * stride).reshape(npred, stride)
    cnt = counts.to_numpy(np.uint64, npred)
    one, c1 = eng.DeviceBuffer(4 * words), eng.DeviceBuffer(8)
    for p, (lo, hi) in enumerate(preds):
        eng.scan_range(col, n, lo, hi, one, c1)
        eng.synchronize()
        assert np.array_equal(got[p, :words], one.to_numpy(np.uint32, words)), p
        assert cnt[p] == c1.to_numpy(np.uint64, 1)[0], p
        if p % 29 == 2 and lo <= hi:
            assert np.array_equal(got[p, :words], pack_rows(interval_mask(x, lo, hi))), p
    if pad:
        assert (got[:, words:] == 0xA5A5A5A5).all()


@pytest.mark.parametrize("npred", [1, 33, 64, 130])
def test_counts_again_and_again_on_streams(eng, npred):
    """Counts of launches of one to a few thousand workgroups, after each other on one stream and
    in turn with another's: each finds the accumulators that the one before left."""
    streams = [None, eng.Stream()]
    for rep, n in enumerate([1, 700, 4097, 100_003, 1 << 20, 100_003, 9_000_001, 5, 1 << 20]):
        x = _column(n, n % 1009)
        preds = _ranges(x, npred, rep)
        col = eng.DeviceBuffer.from_numpy(x)
        words = (n + 31) // 32
        out = eng.DeviceBuffer(4 * npred * words)
        counts = [eng.DeviceBuffer(8 * npred).fill(0xFF) for _ in range(4)]
        for i, c in enumerate(counts):
            eng.scan_ranges(col, n, [p[0] for p in preds], [p[1] for p in preds], out, words, c, streams[i % 2])
            streams[1].synchronize() if i % 2 else eng.synchronize()
        want = [int(((x >= lo) & (x <= hi)).sum()) for lo, hi in preds]
        for c in counts:
            assert c.to_numpy(np.uint64, npred).tolist() == want, n
