"""The filter vectors of a GPU build against numpy, every word of every vector, at the edges of
the waves' rows and words, for columns off 16 bytes and starts at the ends of the domain."""
import numpy as np
import pytest

import snapshot_format as S

pytestmark = pytest.mark.gpu


def _column(kind, n, rng):
    x = rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)
    if kind == "few":
        x = x % np.uint32(200) * np.uint32(21474836)
    elif kind == "ends":  # few enough of either end to be listed, in a short column
        x[: min(60, n // 3)], x[n - min(60, n // 3):] = 0, 0xFFFFFFFF
    return x


@pytest.mark.parametrize("n", [128, 2047, 2048, 2049, 2048 + 33, 4 * 2048, 4 * 2048 + 31, 60_001])
@pytest.mark.parametrize("bins", [128, 256, 512, 1024])
def test_filter_vectors(eng, tmp_path, n, bins):
    rng = np.random.default_rng(n * bins)
    for i, kind in enumerate(("any", "few", "ends")):
        x = _column(kind, n, rng)
        offset = (n + i) % 4
        store = eng.DeviceBuffer.from_numpy(np.concatenate([np.zeros(offset, np.uint32), x]))

        class View:
            ptr = store.ptr + 4 * offset

        index = eng.BinDexIndex(View, n, bins=bins)
        path = tmp_path / "index"
        index.save(str(path))
        raw = path.read_bytes()
        f, a, off = S.parse(raw)
        fvs = np.frombuffer(raw, np.uint32, (bins - 1) * f["fv_stride"], off + 8 * n).reshape(bins - 1, -1)
        bits = np.zeros((bins - 1, 32 * f["fv_stride"]), bool)
        bits[:, :n] = x < a["estarts"][1:, None]
        want = np.packbits(bits, axis=1).view(">u4").astype(np.uint32)
        assert np.array_equal(fvs, want), kind
        index.free()
