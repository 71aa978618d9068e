"""Trajectory.superpose at frame sizes around the one-pass kernel's rules: runs
of many short frames (flat and wave-wise moves), of four, three, two and one
frames, sizes that go to the two-kernel path, runs cut short by the last frame,
and arrays that start off a 16-byte boundary.  Against the FP64 oracle: float32
coordinates of up to 20 nm, moved and rotated in float32, are within 1e-5 nm."""
import numpy as np
import pytest

import mdtraj_amd as md
from mdtraj_amd import gen
from oracle import fp64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_atoms", [1, 2, 3, 21, 22, 27, 28, 112, 191, 192, 400, 416, 420, 700,
                                     830, 1000, 1111, 1400, 1650, 1700, 2000, 2700, 3001, 3320,
                                     3400, 4450, 6600, 6700])
@pytest.mark.parametrize("n_frames", [1, 7, 301])
def test_sizes(gpu, n_atoms, n_frames):
    if n_atoms * n_frames > 300000:
        n_frames = 50
    x = gen.walk(seed=n_atoms, n_frames=n_frames + 1, n_atoms=n_atoms)
    d = gpu.from_numpy(x).cuda()[1:]  # off the allocation's start by one frame
    for n_sel in (0, max(1, n_atoms // 8), max(1, 3 * n_atoms // 4)):
        sel = gen.subset(3, n_atoms, n_sel) if n_sel else None
        n_fit = n_sel or n_atoms
        t = md.Trajectory(d.clone())
        t.xyz = gpu.empty((n_frames + 1, n_atoms, 3), device="cuda")[1:].copy_(d)
        before = t.xyz.data_ptr()
        t.superpose(md.Trajectory(x[:1]), 0, atom_indices=sel)
        assert t.xyz.data_ptr() == before
        got = t.xyz.cpu().numpy()
        if n_fit < 3:  # the rotation is not determined: only the fit's RMSD is
            part = slice(None) if sel is None else sel
            want = fp64.rmsd(x[1:], x[:1], 0, sel)
            left = np.sqrt(((got[:, part] - x[0][part]) ** 2).sum(2).mean(1))
            assert np.abs(left - want).max() < 1e-5
        else:
            want = fp64.superpose(x[1:], x[:1], 0, sel)
            assert np.abs(got - want).max() < 1e-5
