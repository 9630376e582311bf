"""The value sort behind index builds and encoders against numpy's stable argsort, at the edges
of its tiles, of the ranges that take tiles of one size, and of the runs of tiles an XCD takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _columns(n):
    rng = np.random.default_rng(n)
    yield "uniform", rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)
    yield "bytes", rng.integers(0, 256, n, dtype=np.uint64).astype(np.uint32) << np.uint32(8)
    yield "descending", np.arange(n, 0, -1, dtype=np.uint64).astype(np.uint32) * np.uint32(257)
    yield "one", np.full(n, 0xFFFFFFFF, np.uint32)


@pytest.mark.parametrize("n", [128, (1 << 16) - 1, 1 << 16, (1 << 16) + 1, (1 << 17) + 1, (1 << 18) - 1, 1 << 18,
                               (1 << 18) + 1, 5 << 18, (5 << 18) + 1, 1 << 21, (1 << 21) + 1, 256 * 8192 + 5, 3_000_001,
                               3 << 17, (3 << 17) + 1, 3 << 19, (3 << 19) + 1, 7 << 19, (7 << 19) + 1])
@pytest.mark.parametrize("offset", [0, 3])
def test_sorted_values_and_rows(eng, n, offset):
    for name, x in _columns(n):
        store = eng.DeviceBuffer.from_numpy(np.concatenate([np.zeros(offset, np.uint32), x]))

        class Column:
            ptr = store.ptr + 4 * offset

        index = eng.BinDexIndex(Column, n)
        values, rows = index.sorted()
        order = np.argsort(x, kind="stable")
        assert np.array_equal(rows, order), name
        assert np.array_equal(values, x[order]), name
        index.free()


@pytest.mark.parametrize("n", [1, 2, 127, 8193])
def test_short_columns_through_the_encoder(eng, n):
    for name, x in _columns(n):
        d = eng.DeviceBuffer.from_numpy(x)
        _, _, _, pos, _ = eng.encode_column(d, n, 0, n, want_sorted=True)
        assert np.array_equal(pos.to_numpy(np.int32, n), np.argsort(x, kind="stable")), name
