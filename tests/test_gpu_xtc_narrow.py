"""XTC frames of a few atoms, many of them: decoded by rows of four lanes, on both
sides of the rule's frame and atom counts.  Coordinates must equal the oracle's
bit for bit."""
import random

import numpy as np
import pytest

from mdtraj_amd.xtc import XTCTrajectoryFile
from oracle import xtc as oracle
from tests.test_gpu_xtc_streams import stream, write

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_frames", [65535, 65536, 65537, 65551])
@pytest.mark.parametrize("n_atoms", [10, 11, 20, 21])
@pytest.mark.parametrize("sizes,idx,flag_rate", [
    ((900, 1000, 1100), 14, 0.0), ((900, 1000, 1100), 14, 1.0),
    ((1 << 25, 1 << 30, 77), 60, 0.5), ((0xFFFFFF, 0xFFFFFF, 0xFFFFFF), 71, 0.4)])
def test_short_frames(gpu, tmp_path, n_frames, n_atoms, sizes, idx, flag_rate):
    rng = random.Random(n_frames + n_atoms)
    some = [stream(rng, n_atoms, sizes, idx, flag_rate) for _ in range(37)]
    want = oracle.read(write(tmp_path, some, n_atoms)[1])[0]
    pick = [rng.randrange(len(some)) for _ in range(n_frames)]
    name, _ = write(tmp_path, [some[k] for k in pick], n_atoms)
    with XTCTrajectoryFile(name) as f:
        xyz = f.read()[0]
    assert np.array_equal(xyz, want[pick])
