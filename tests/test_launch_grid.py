"""The grid of kernels that have a workgroup per frame or run of frames: every
workgroup is there, and no dimension holds 2^32 work-items, where a launch's
count wraps."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(ROOT, "mdtraj_amd", "_build", "launch_grid_host.so")


@pytest.fixture(scope="module")
def grid():
    src = os.path.join(HERE, "launch_grid_host.hip")
    deps = [src, os.path.join(ROOT, "mdtraj_amd", "csrc", "common.h")]
    if not os.path.exists(LIB) or os.path.getmtime(LIB) < max(os.path.getmtime(d) for d in deps):
        os.makedirs(os.path.dirname(LIB), exist_ok=True)
        cmd = ["hipcc", "--offload-arch=gfx950", "-O2", "-std=c++17", "-fPIC", "-shared",
               "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
               "-I" + os.path.join(ROOT, "include"),
               "-I" + os.path.join(ROOT, "mdtraj_amd", "csrc"), src, "-o", LIB]
        try:
            subprocess.run(cmd, check=True, capture_output=True, timeout=600)
        except (OSError, subprocess.CalledProcessError) as e:
            pytest.skip(f"hipcc unavailable for the host build of the launch grid: {e}")
    fn = ctypes.CDLL(LIB).launch_grid_host
    fn.argtypes = [ctypes.c_longlong, ctypes.c_int, ctypes.POINTER(ctypes.c_uint)]

    def call(groups, threads):
        out = (ctypes.c_uint * 3)()
        fn(groups, threads, out)
        return tuple(out)
    return call


@pytest.mark.parametrize("threads", [64, 128, 256])
@pytest.mark.parametrize("groups", [1, 2, 1000003, 2**24 - 1, 2**24, 2**25 - 1, 2**25, 2**25 + 1,
                                    2**26, 2**31 - 1, 2**31, 2**32 - 2**16])
def test_every_workgroup_within_the_launch_limits(grid, groups, threads):
    x, y, z = grid(groups, threads)
    assert z == 1 and x * threads < 2**32 and x < 2**31 and y < 2**16
    assert groups <= x * y < groups + 2**16  # at most one row's remainder past the end
    if groups * threads < 2**32:
        assert (x, y) == (groups, 1)
    else:
        assert x == 2**16  # what workgroup_index() counts a row as
