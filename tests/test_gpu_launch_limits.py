"""Calls whose frames, at a lane or a row of lanes each, make 2^32 work-items
and more, where one dimension of a launch wraps: every frame is computed."""
import pytest

from mdtraj_amd import _lib

pytestmark = pytest.mark.gpu


def room(gpu, nbytes):
    gpu.cuda.empty_cache()
    if gpu.cuda.mem_get_info()[0] < nbytes + (8 << 30):
        pytest.skip(f"needs {nbytes >> 30} GiB of device memory")


def stream(gpu):
    return gpu.cuda.current_stream().cuda_stream


def test_short_frames(gpu):
    """One-atom frames at a lane each; their RMSD is 0."""
    F = 2**32 + 65
    room(gpu, 16 * F)
    x = gpu.zeros(3 * F, device="cuda")
    out = gpu.full((F,), -1.0, device="cuda")
    ws = gpu.empty(_lib.load().hr_rmsd_workspace_bytes(1), dtype=gpu.uint8, device="cuda")
    _lib.call("hr_rmsd_one_vs_all", x.data_ptr(), F, 1, None, 1, x.data_ptr(), None, 0,
              out.data_ptr(), ws.data_ptr(), stream(gpu))
    wrong = sum(int(gpu.count_nonzero(out[a:a + 2**28])) for a in range(0, F, 2**28))
    del x, out
    gpu.cuda.empty_cache()
    assert wrong == 0
