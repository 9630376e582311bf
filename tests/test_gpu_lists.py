"""The refine lists and the tile directory of a GPU build against numpy: every bin's rows in row
order, at the edges of the partition's chunks, tiles and tile parts."""
import numpy as np
import pytest

import snapshot_format as S

pytestmark = pytest.mark.gpu

LIGHT = 64  # a bin start of at most this many rows is in its bin's list


def _column(kind, n, rng):
    if kind == "uniform":
        return rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)
    if kind == "few":  # a few hundred values: heavy bin starts, equal starts, empty lists
        return rng.integers(0, 300, n, dtype=np.uint64).astype(np.uint32) * np.uint32(9999991)
    if kind == "sorted":  # a tile's rows in one or two bins
        return np.sort(rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32))
    return np.full(n, 77, np.uint32)


@pytest.mark.parametrize("n", [128, 4095, 4097, 32767, 32768, 32769, 3 * 32768 + 4096, 300_001])
@pytest.mark.parametrize("bins", [128, 256, 512, 1024])
def test_lists(eng, tmp_path, n, bins):
    rng = np.random.default_rng(n + bins)
    for kind in ("uniform", "few", "sorted", "one"):
        x = _column(kind, n, rng)
        d = eng.DeviceBuffer.from_numpy(x)
        index = eng.BinDexIndex(d, n, bins=bins)
        path = tmp_path / "index"
        index.save(str(path))
        raw = path.read_bytes()
        f, a, off = S.parse(raw)
        off += 8 * n + 4 * (bins - 1) * f["fv_stride"]
        bent = np.frombuffer(raw, np.uint32, 2 * f["nb"], off).reshape(-1, 2)
        starts = a["estarts"]
        # bin of a value: the number of k in [1, bins) with starts[k] <= value
        of = np.searchsorted(starts[1:], x, side="right")
        rows_of_start = np.searchsorted(np.sort(x), starts, side="right") - np.searchsorted(np.sort(x), starts)
        listed = (x > starts[of]) | (rows_of_start[of] <= LIGHT)
        rows = np.flatnonzero(listed)
        rows = rows[np.argsort(of[rows], kind="stable")]
        assert np.array_equal(bent[:, 0], rows), (kind, "rows")
        assert np.array_equal(bent[:, 1], x[rows]), (kind, "values")
        assert np.array_equal(a["boff"], np.searchsorted(of[rows], np.arange(bins + 1))), (kind, "offsets")
        # the directory is read by queries only: ranges with bounds inside bins
        lo, hi = sorted(int(v) for v in rng.choice(x, 2))
        lo, hi = min(lo + 1, hi), max(lo, hi - 1)
        out, count = eng.DeviceBuffer(4 * ((n + 31) // 32)), eng.DeviceBuffer(8)
        eng.bindex_query([index, index], [lo, lo], [hi, hi], out, count)
        want = (x >= lo) & (x <= hi)
        got = np.unpackbits(out.to_numpy(np.uint32).astype(">u4").view(np.uint8))[:n].astype(bool)
        assert np.array_equal(got, want), (kind, "query")
        assert int(count.to_numpy(np.uint64, 1)[0]) == int(want.sum()), (kind, "count")
        index.free()
