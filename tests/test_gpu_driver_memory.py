"""The query driver's line of device memory: the indexes' bytes, whatever the library keeps of the
workspaces of builds and encodings."""
import os
import re

import pytest

from test_gpu_driver import GOLDEN, run

pytestmark = pytest.mark.gpu


def used(n, cols, encode):
    rc, out, err = run(["-b", str(cols), "-p", os.path.join(GOLDEN, "scan_cmd_1e8-2c.txt"), "-n", str(n), "-s", "7"]
                       + ["-e"] * encode)
    assert rc == 0, (rc, err[-2000:], out[-2000:])
    return float(re.search(r"Device memory used\(MB\): (-?[\d.]+)", out).group(1)) * 2 ** 20


@pytest.mark.parametrize("encode", [False, True])
def test_memory_of_the_indexes(eng, encode):
    """Against a short column's run, which has the process's own memory (code, queues) in it too."""
    cols, rows = 2, (200_000, 20_000_000)
    want = []
    for n in rows:
        x = eng.DeviceBuffer.from_numpy(eng.generate_column(0, 7, 0, n))
        want.append(cols * eng.BinDexIndex(x, n).device_bytes())
    got = used(rows[1], cols, encode) - used(rows[0], cols, encode)
    # arrays in whole blocks, and codes in place of the values (other lists): 5 %; the
    # workspaces are 15 % and more
    assert abs(got - (want[1] - want[0])) <= 0.05 * (want[1] - want[0]), (got, want)
