"""pf_perft_batch_noalloc when a launch does not start: the call reports it, and
returns only once what it had queued, which reads the caller's positions and
writes the caller's counts, has ended (host side only, with replaced launches)."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "noalloc_check.cpp")
LIB = os.path.join(HERE, "native", "_build", "libnoalloc_check.so")
CSRC = os.path.join(HERE, "..", "perft_gpu_amd", "csrc")


@pytest.fixture(scope="module")
def noalloc():
    deps = [SRC] + [os.path.join(CSRC, f) for f in ("noalloc.hip", "engine.h", "kernels.h", "tt_kernels.h")]
    if not (os.path.exists(LIB) and all(os.path.getmtime(LIB) >= os.path.getmtime(d) for d in deps)):
        os.makedirs(os.path.dirname(LIB), exist_ok=True)
        subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-fPIC", "-shared", "--offload-arch=gfx950",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-x", "hip", SRC, "-o", LIB],
                       check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    return ctypes.CDLL(LIB)


@pytest.mark.parametrize("n,depth", [(1, 1), (100, 4), (1024, 2), (1025, 2), (2000, 4), (5, 0)])
def test_failed_launch_waits(pg, noalloc, n, depth):
    queued, unfinished = ctypes.c_int(), ctypes.c_int()
    assert noalloc.nc_call(n, depth, 0, ctypes.byref(queued), ctypes.byref(unfinished)) == 0
    steps = queued.value
    assert steps >= 1 and not unfinished.value
    for fail in range(1, steps + 1):
        assert noalloc.nc_call(n, depth, fail, ctypes.byref(queued), ctypes.byref(unfinished)) == pg.PF_EDEVICE
        assert queued.value == fail - 1
        assert not unfinished.value, fail
