"""The encoders' codes written to row order through groups of rows (long columns), at the edges
of the windows, groups and tiles, against numpy."""
import numpy as np
import pytest

import rtscan_amd as R

pytestmark = pytest.mark.gpu


def _column(kind, n):
    rng = np.random.default_rng(n)
    if kind == "uniform":
        return rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)
    if kind == "few":
        return rng.integers(0, 1000, n, dtype=np.uint64).astype(np.uint32)
    return np.full(n, 4_000_000_000, np.uint32)


# one window a group; a last window of one row; 513 windows, so two windows a group
@pytest.mark.parametrize("n", [1 << 22, (1 << 22) + 1, (1 << 22) + 32768 + 5, 512 * 32768 + 3])
@pytest.mark.parametrize("kind", ["uniform", "few", "one"])
def test_codes_of_long_columns(eng, n, kind):
    x = _column(kind, n)
    order = np.argsort(x, kind="stable")
    values, first = np.unique(x[order], return_index=True)
    d = R.DeviceBuffer.from_numpy(x)
    lo, hi = 5, 2 ** 32 - 1
    step = (hi - lo) // n
    codes, mv, ms, sp, sc = R.encode_column(d, n, lo, hi, want_sorted=True)
    want = ((lo + np.arange(n, dtype=np.uint64) * step) & 0xFFFFFFFF).astype(np.uint32)
    assert np.array_equal(mv, values) and np.array_equal(ms, want[first])
    assert np.array_equal(sp.to_numpy(np.int32, n), order)
    assert np.array_equal(sc.to_numpy(np.uint32, n), want)
    assert np.array_equal(codes.to_numpy(np.uint32, n)[order], want)
    # dispersed, over the column itself: every row's code in its value's range
    counts = np.diff(np.append(first, n))
    steps = (counts * ((hi - lo) / n)).astype(np.int64)
    starts = (lo + np.cumsum(steps) - steps) & 0xFFFFFFFF
    codes, mv, ms = R.encode_column_dispersed(d, n, lo, hi, seed=3, codes=d)
    assert np.array_equal(mv, values) and np.array_equal(ms, starts.astype(np.uint32))
    run = np.repeat(np.arange(values.size), counts)
    off = (codes.to_numpy(np.uint32, n)[order].astype(np.int64) - starts[run]) & 0xFFFFFFFF
    assert (off < np.where(steps >= 2, steps - 1, 1)[run]).all()
