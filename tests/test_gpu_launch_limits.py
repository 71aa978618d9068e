"""Calls whose frames, at a lane or a row of lanes each, make 2^32 work-items
and more, where one dimension of a launch wraps: every frame is computed."""
import struct

import numpy as np
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


def test_xtc_frames(gpu):
    """Frames of one atom at a row of eight lanes each.  The offsets name one
    frame's bytes again and again, so that every other frame, whose bytes would
    end before they begin, is refused."""
    F = 2**29 + 9
    room(gpu, 72 * F)
    rec = struct.pack(">3if9fi3f", 1995, 1, 7, 0.5, *range(9), 1, 1.0, 2.0, 3.0)
    data = gpu.from_numpy(np.frombuffer(2 * rec, np.uint8).copy()).cuda()
    offs = gpu.tensor([0, len(rec)], device="cuda").repeat(F // 2 + 1)[:F].contiguous()
    xyz = gpu.zeros((F, 3), device="cuda")
    time, prec = (gpu.empty(F, device="cuda") for _ in range(2))
    step, status = (gpu.full((F,), -1, dtype=gpu.int32, device="cuda") for _ in range(2))
    box = gpu.empty((F, 9), device="cuda")
    _lib.call("hr_xtc_decode", data.data_ptr(), data.numel(), offs.data_ptr(), F, 1,
              xyz.data_ptr(), time.data_ptr(), step.data_ptr(), box.data_ptr(), prec.data_ptr(),
              status.data_ptr(), stream(gpu))
    assert F % 2 == 1  # the last frame ends with the data
    good = int((status[::2] == 0).sum()) == F // 2 + 1
    refused = int((status[1::2] == 3).sum()) == F // 2
    steps = int((step[::2] == 7).sum()) == F // 2 + 1
    want = gpu.tensor([1.0, 2.0, 3.0], device="cuda")
    right = all(bool((xyz[a:a + 2**27:2] == want).all()) for a in range(0, F, 2**27))
    del offs, xyz, time, prec, step, status, box
    gpu.cuda.empty_cache()
    assert good and refused and steps and right
