"""Area and bin starts, block bounds and the rest that a GPU build keeps on the host, against
numpy: runs of one value over no, some and all bin starts, the smallest columns, areas of whole
blocks, and a column whose block bounds are copied apart."""
import numpy as np
import pytest

import snapshot_format as S

pytestmark = pytest.mark.gpu

AREAS, BLOCK = 128, 3276


def _column(kind, n, rng):
    if kind == "distinct":
        return rng.permutation(n).astype(np.uint32) * np.uint32(3)
    if kind == "runs":  # runs of 1 to n / 10 rows
        cuts = np.sort(rng.integers(0, n, 40))
        return rng.permutation(np.searchsorted(cuts, np.arange(n)).astype(np.uint32) * np.uint32(0x05000001))
    if kind == "ends":  # half the rows at one end of the domain, some at the other
        x = rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)
        x[::2], x[1::16] = 0xFFFFFFFF, 0
        return x
    return np.full(n, 0xFFFFFFFF, np.uint32)


def _starts(s, sub):
    """First sorted slots of the areas and values of the bins' first slots."""
    n, avg = s.size, s.size // AREAS
    idx = np.zeros(AREAS, np.int64)
    for i in range(1, AREAS):
        v = s[i * avg]
        idx[i] = i * avg if v == s[(i - 1) * avg] else np.searchsorted(s, v)
    ends = np.append(idx[1:], n)
    slots = [idx[a] + j * (ends[a] - idx[a]) // sub for a in range(AREAS) for j in range(sub)]
    return idx, ends, s[slots]


@pytest.mark.parametrize("n", [128, 129, 255, 5000, AREAS * BLOCK, AREAS * BLOCK + 1, AREAS * (BLOCK + 1), 4_000_003])
@pytest.mark.parametrize("sub", [1, 2, 8])
def test_starts(eng, tmp_path, n, sub):
    rng = np.random.default_rng(n + sub)
    for kind in ("distinct", "runs", "ends", "one"):
        x = _column(kind, n, rng)
        s = np.sort(x)
        d = eng.DeviceBuffer.from_numpy(x)
        index = eng.BinDexIndex(d, n, bins=AREAS * sub)
        idx, ends, estarts = _starts(s, sub)
        assert np.array_equal(index.area_counts(), ends), kind
        assert np.array_equal(np.array(index.s.areaStartValues[:], np.uint32), s[np.arange(AREAS) * (n // AREAS)]), kind
        assert index.s.data_min == s[0] and index.s.data_max == s[-1], kind
        for k in range(AREAS):
            a = index.s.areas[k].contents
            first = np.arange(idx[k], ends[k], BLOCK)
            assert (a.start, a.length, a.blockNum) == (idx[k], ends[k] - idx[k], first.size), (kind, k)
            assert a.blockFirst[:a.blockNum] == list(s[first]), (kind, k)
            assert a.blockLast[:a.blockNum] == list(s[np.minimum(first + BLOCK, ends[k]) - 1]), (kind, k)
        if n < 1_000_000:
            path = tmp_path / "index"
            index.save(str(path))
            _, arrays, _ = S.parse(path.read_bytes())
            assert np.array_equal(arrays["estarts"], estarts), kind
        # counts go by the rank samples
        out, count = eng.DeviceBuffer(4 * ((n + 31) // 32)), eng.DeviceBuffer(8)
        for lo, hi in ((s[n // 3], s[n // 2]), (s[0], s[-1]), (s[-1], s[-1])):
            eng.bindex_query([index], [int(lo)], [int(hi)], out, count)
            eng.synchronize()
            assert int(count.to_numpy(np.uint64, 1)[0]) == int(((x >= lo) & (x <= hi)).sum()), (kind, lo, hi)
        index.free()
