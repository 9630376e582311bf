"""The pool of device memory on the host: device_pool.cpp with a device that the test plays, which
runs out of memory, refuses to take blocks back, and has no host memory beside it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include/hip"),
                    reason="needs g++ and the HIP headers")
def test_pool_of_device_memory(tmp_path):
    exe = str(tmp_path / "pool_test")
    csrc = os.path.join(ROOT, "rtscan_amd", "csrc")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + csrc, "-o", exe, os.path.join(ROOT, "tests", "host_logic", "pool_test.cpp"),
                    os.path.join(csrc, "device_pool.cpp")], check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "pool ok" in r.stdout, (r.returncode, r.stdout, r.stderr)
