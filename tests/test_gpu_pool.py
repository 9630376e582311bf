"""Device memory kept between calls: index arrays and workspaces are reused by later builds and
encodings of any thread and stream, and given back when memory is asked for."""
import threading

import numpy as np
import pytest

from _util import interval_mask, pack_rows

pytestmark = pytest.mark.gpu


def _query(eng, index, x, lo, hi, stream=None):
    out = eng.DeviceBuffer(4 * ((x.size + 31) // 32))
    eng.bindex_query([index], [lo], [hi], out, stream=stream)
    eng.synchronize()
    return np.array_equal(out.to_numpy(np.uint32), pack_rows(interval_mask(x, lo, hi)))


def test_threads_and_streams_share_kept_memory(eng):
    """Four threads, each on a stream of its own, build, query, free and encode columns of
    different sizes in a loop: every result is right."""
    errors = []

    def worker(k):
        try:
            rng = np.random.default_rng(k)
            stream = eng.Stream()
            for i in range(6):
                n = int(rng.integers(200_000, 1_500_000))
                x = rng.integers(0, 1 << int(rng.integers(8, 33)), n, dtype=np.uint64).astype(np.uint32)
                d = eng.DeviceBuffer.from_numpy(x)
                index = eng.BinDexIndex(d, n, stream=stream, bins=int(rng.choice([128, 256, 512])))
                lo, hi = sorted(int(v) for v in rng.integers(0, int(x.max()) + 1, 2))
                if not _query(eng, index, x, lo, hi, stream):
                    errors.append(("query", k, i, n))
                index.free()
                codes, values, starts = eng.encode_column(d, n, 0, 1 << 31, stream=stream)
                step = (1 << 31) // n
                want_values, first = np.unique(np.sort(x), return_index=True)
                if not (np.array_equal(values, want_values) and np.array_equal(starts, first.astype(np.uint64) * step)):
                    errors.append(("map", k, i, n))
                order = np.argsort(x, kind="stable")
                got = codes.to_numpy(np.uint32, n)
                if not np.array_equal(got[order], (np.arange(n, dtype=np.uint64) * step).astype(np.uint32)):
                    errors.append(("codes", k, i, n))
        except Exception as e:  # noqa: BLE001
            errors.append(repr(e))

    threads = [threading.Thread(target=worker, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[:3]


def test_an_index_freed_under_queued_queries(eng):
    """An index freed while queries of it are queued on another stream: they finish on its
    arrays before the next index takes them."""
    n = 3_000_000
    rng = np.random.default_rng(2)
    a, b = (rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(2))
    da, db = eng.DeviceBuffer.from_numpy(a), eng.DeviceBuffer.from_numpy(b)
    stream = eng.Stream()
    lo, hi = 1 << 30, 3 << 30
    want = pack_rows(interval_mask(a, lo, hi))
    index = eng.BinDexIndex(da, n)
    outs = [eng.DeviceBuffer(4 * want.size) for _ in range(40)]
    for out in outs:
        eng.bindex_query([index], [lo], [hi], out, stream=stream)
    index.free()
    other = eng.BinDexIndex(db, n)
    stream.synchronize()
    assert all(np.array_equal(out.to_numpy(np.uint32), want) for out in outs)
    assert _query(eng, other, b, lo, hi)


def test_kept_memory_is_given_back(eng):
    """What freed indexes leave is bounded, and comes back when the free memory is asked for."""
    n = 40_000_000
    rng = np.random.default_rng(3)
    d = eng.DeviceBuffer.from_numpy(rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32))
    eng.BinDexIndex(d, n).free()
    free = eng.device_free_bytes()
    for _ in range(3):
        indexes = [eng.BinDexIndex(d, n, bins=512) for _ in range(4)]  # 3.2 GB each
        for index in indexes:
            index.free()
    assert eng.device_free_bytes() >= free - (64 << 20)
