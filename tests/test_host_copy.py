"""CPU: the copies of the host-array entry points (liteqt_amd/csrc/rgf_hostcopy.hpp, compiled
with g++ against the stand-in tests/hostcopy/hip), with pinned areas and where these cannot be
allocated.  Sizes: below an area, across both, and empty."""
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MIB = 1 << 20


@pytest.fixture(scope="module")
def hostcopy(tmp_path_factory):
    d = tmp_path_factory.mktemp("hostcopy")
    here = os.path.join(ROOT, "tests", "hostcopy")
    shutil.copy(os.path.join(ROOT, "liteqt_amd", "csrc", "rgf_hostcopy.hpp"), d)
    so = d / "libhostcopy.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-pthread", "-I", here, "-I", str(d), "-o", str(so),
                    os.path.join(here, "host_copy.cpp")], check=True)
    return str(so)


CODE = """
import ctypes, sys
import numpy as np
L = ctypes.CDLL(sys.argv[1])
fail, sizes = int(sys.argv[2]), np.array([int(s) for s in sys.argv[3].split(",")], np.uint64)
n = int(sizes.sum())
src = np.random.default_rng(1).integers(0, 256, n, dtype=np.uint8)
dev, dst = np.zeros(n, np.uint8), np.zeros(n, np.uint8)
p = lambda a: ctypes.c_void_p(a.ctypes.data)
rc = L.host_copy(fail, 2, len(sizes), p(sizes), p(src), p(dev), p(dst))
assert rc == 0, rc
assert np.array_equal(dev, src) and np.array_equal(dst, src)
"""


# a process of its own with a time limit: copies that make no progress would not end
@pytest.mark.parametrize("fail", [0, 1])
@pytest.mark.parametrize("sizes", [(1,), (8, 0, 4096, 100), (300 * 1024, 7, 513 * 1024), (5 * MIB, 3, 40 * MIB + 1, 16 * MIB)])
def test_host_copies(hostcopy, fail, sizes):
    r = subprocess.run([sys.executable, "-c", CODE, hostcopy, str(fail), ",".join(map(str, sizes))], capture_output=True,
                       text=True, timeout=20)
    assert r.returncode == 0, r.stderr
