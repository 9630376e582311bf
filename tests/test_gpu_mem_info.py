"""The free memory that the library reports, and what it keeps for later calls."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def device_free():
    hip = ctypes.CDLL("libamdhip64.so.7")
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value


def test_asking_for_the_free_memory_keeps_it(eng):
    """Kept memory counts as free and stays with the library, until it is asked to give it back."""
    n = 20_000_000
    rng = np.random.default_rng(3)
    d = eng.DeviceBuffer.from_numpy(rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32))
    eng.BinDexIndex(d, n).free()
    eng.device_mem_trim()
    free = device_free()
    assert eng.device_free_bytes() == free
    for _ in range(3):
        eng.BinDexIndex(d, n).free()
        kept = free - device_free()
        assert kept > 400 << 20  # sorted values and rows, filter vectors, lists
        assert abs(eng.device_free_bytes() - free) <= 4 << 20
        assert free - device_free() == kept
    eng.device_mem_trim()
    assert abs(device_free() - free) <= 4 << 20
