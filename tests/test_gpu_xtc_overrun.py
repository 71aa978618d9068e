"""A group whose run of small atoms reaches past the frame's last atom, its length
set by the group's own run code or kept from the group before: the frame is
refused, the groups before it are decoded, and the next frame's coordinates are
not written to.  At every row width."""
import random
import struct

import numpy as np
import pytest

from mdtraj_amd import _lib
from oracle import xtc as oracle
from tests.test_gpu_xtc_streams import stream, write

pytestmark = pytest.mark.gpu

N, IDX, SIZES = 200, 14, (900, 1000, 1100)


def frame(rng, runs):
    """Groups of the given runs of small atoms, each with a flag where its run is
    another than the last group's; smallidx stays."""
    bits, last = [], 0

    def field(bound, nbits):
        v = rng.randrange(bound)
        while nbits > 8:
            bits.append(format(v & 255, "08b"))
            v >>= 8
            nbits -= 8
        bits.append(format(v, f"0{nbits}b"))

    prod = SIZES[0] * SIZES[1] * SIZES[2]
    for run in runs:
        field(prod, prod.bit_length())
        bits.append("0" if run == last else "1" + format(3 * run + 1, "05b"))
        last = run
        for _ in range(run):
            field(oracle.MAGICINTS[IDX] ** 3, IDX)
    text = "".join(bits)
    text += "0" * (-len(text) % 8)
    data = int(text, 2).to_bytes(len(text) // 8, "big")
    return (struct.pack(">if6i", N, 1000.0, 0, 0, 0, *(s - 1 for s in SIZES))
            + struct.pack(">2i", IDX, len(data)) + data + b"\0" * (-len(data) % 4))


@pytest.mark.parametrize("n_frames", [1, 3001, 6001, 16001])
@pytest.mark.parametrize("runs,whole", [
    ([4] * 39 + [10], 195),   # five atoms left, eleven in the last group, by its run code
    ([6] * 28 + [6], 196),    # four left, seven by the run kept
    ([3] * 49 + [4], 196),    # four left, five by the run code: one too many
    ([10] * 18 + [1], 200)])  # and a frame that ends just so
def test_run_past_the_last_atom(gpu, tmp_path, n_frames, runs, whole):
    rng = random.Random(1)
    good = stream(rng, N, SIZES, IDX, 0.3)
    odd = frame(rng, runs)
    frames = [good] * n_frames + [odd] + [good]
    _, data = write(tmp_path, frames, N)
    F = len(frames)
    size = [52 + len(f) for f in frames]
    offs = gpu.from_numpy(np.concatenate([[0], np.cumsum(size)[:-1]]).astype(np.int64)).cuda()
    d = gpu.frombuffer(bytearray(data), dtype=gpu.uint8).cuda()
    xyz = gpu.full((F + 1, N, 3), -9.0, device="cuda")
    tm, pr = (gpu.zeros(F, device="cuda") for _ in range(2))
    sp, st = (gpu.zeros(F, dtype=gpu.int32, device="cuda") for _ in range(2))
    bx = gpu.zeros((F, 9), device="cuda")
    _lib.call("hr_xtc_decode", d.data_ptr(), d.numel(), offs.data_ptr(), F, N, xyz.data_ptr(),
              tm.data_ptr(), sp.data_ptr(), bx.data_ptr(), pr.data_ptr(), st.data_ptr(),
              gpu.cuda.current_stream().cuda_stream)
    st, xyz = st.cpu().numpy(), xyz.cpu().numpy()
    broken = sum(r + 1 for r in runs) > N
    want = np.zeros(F, np.int32)
    want[n_frames] = 4 if broken else 0
    assert np.array_equal(st, want)
    fine = oracle.read(write(tmp_path, [good], N)[1])[0][0]
    assert np.array_equal(xyz[0], fine) and np.array_equal(xyz[n_frames - 1], fine)
    assert np.array_equal(xyz[n_frames + 1], fine)
    # what lies past the last whole group was not touched
    assert (xyz[n_frames, whole:] == -9).all() and not (xyz[n_frames, :whole] == -9).any()
    assert (xyz[F] == -9).all()
