"""XTC frames of up to nine atoms, which are stored uncompressed: every atom
count, frame counts around a workgroup's 32 and 64 frames, and frames whose
header or length is wrong beside good ones.  Bytes are copied, so everything is
equal to what was written."""
import numpy as np
import pytest

from mdtraj_amd import _lib

pytestmark = pytest.mark.gpu


def decode(gpu, data, offs, n_atoms):
    F = len(offs)
    d = gpu.from_numpy(np.frombuffer(data, np.uint8).copy()).cuda()
    o = gpu.from_numpy(offs).cuda()
    xyz = gpu.full((F + 1, n_atoms, 3), -9.0, device="cuda")
    time, prec = (gpu.full((F + 1,), -9.0, device="cuda") for _ in range(2))
    step, status = (gpu.full((F + 1,), -9, dtype=gpu.int32, device="cuda") for _ in range(2))
    box = gpu.full((F + 1, 9), -9.0, device="cuda")
    _lib.call("hr_xtc_decode", d.data_ptr(), d.numel(), o.data_ptr(), F, n_atoms, xyz.data_ptr(),
              time.data_ptr(), step.data_ptr(), box.data_ptr(), prec.data_ptr(), status.data_ptr(),
              gpu.cuda.current_stream().cuda_stream)
    return [t.cpu().numpy() for t in (xyz, time, step, box, prec, status)]


def records(rng, n_frames, n_atoms):
    rec = np.zeros((n_frames, 14 + 3 * n_atoms), ">i4")
    rec[:, 0] = 1995
    rec[:, 1] = rec[:, 13] = n_atoms
    rec[:, 2] = np.arange(n_frames) + 5
    rec[:, 3:13] = rng.random((n_frames, 10)).astype(">f4").view(">i4")
    rec[:, 14:] = rng.random((n_frames, 3 * n_atoms)).astype(">f4").view(">i4")
    return rec


@pytest.mark.parametrize("n_frames", [1, 31, 32, 33, 63, 64, 65, 1000])
@pytest.mark.parametrize("n_atoms", range(1, 10))
def test_frames_are_copied(gpu, n_frames, n_atoms):
    rec = records(np.random.default_rng(n_atoms), n_frames, n_atoms)
    offs = np.arange(n_frames, dtype=np.int64) * rec.shape[1] * 4
    xyz, time, step, box, prec, status = decode(gpu, rec.tobytes(), offs, n_atoms)
    real = rec.view(">f4").astype(np.float32)
    assert np.array_equal(xyz[:-1].reshape(n_frames, -1), real[:, 14:])
    assert np.array_equal(time[:-1], real[:, 3]) and np.array_equal(box[:-1], real[:, 4:13])
    assert np.array_equal(step[:-1], rec[:, 2])
    assert not status[:-1].any() and not prec[:-1].any()
    for out in (xyz, time, step, box, prec, status):  # nothing past the last frame
        assert (out[-1] == -9).all()


@pytest.mark.parametrize("n_atoms", [1, 3, 4, 9])
def test_refused_frames(gpu, n_atoms):
    rec = records(np.random.default_rng(3), 40, n_atoms)
    size = rec.shape[1] * 4
    offs = np.arange(40, dtype=np.int64) * size
    rec[7, 0] = 1994
    rec[11, 1] = n_atoms + 1
    rec[12, 13] = n_atoms + 1
    offs[20] += 2  # unaligned
    data = rec.tobytes()[:-4]  # the last frame ends early
    xyz, time, step, box, prec, status = decode(gpu, data, offs, n_atoms)
    want = np.zeros(40, np.int32)
    want[[7, 11, 12, 20, 39]] = [1, 2, 2, 3, 3]
    want[19] = 0  # its bytes end two later
    assert np.array_equal(status[:-1], want)
    good = want == 0
    real = rec.view(">f4").astype(np.float32)
    assert np.array_equal(xyz[:-1].reshape(40, -1)[good], real[good, 14:])
    assert (xyz[:-1][~good] == -9).all()
    assert np.array_equal(step[:-1][good], rec[good, 2])
