"""RMSF at selection and frame counts around its passes' splits: 16 atoms a
workgroup and 16 waves of chunks in the finish, 256 atoms a workgroup and up to
1,024 chunks of frames, eight frames at a time, in the accumulation.  Against
the FP64 oracle; the bar is one rounding of the result to float32."""
import numpy as np
import pytest

import mdtraj_amd as md
from mdtraj_amd import gen
from oracle import fp64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_frames", [1, 2, 7, 9, 64, 65, 1100])
@pytest.mark.parametrize("n_atoms,n_sel", [(4, 0), (15, 0), (16, 0), (17, 0), (40, 31), (255, 0),
                                           (300, 257), (530, 0)])
def test_sizes(gpu, n_frames, n_atoms, n_sel):
    x = gen.walk(seed=n_atoms + n_frames, n_frames=n_frames, n_atoms=n_atoms)
    sel = gen.subset(5, n_atoms, n_sel) if n_sel else None
    for ref in (x, None):
        want = fp64.rmsf(x, ref, 0, sel)
        got = md.rmsf(x, x if ref is not None else None, 0, atom_indices=sel)
        assert np.abs(got - want).max() <= 1e-6 * max(1.0, want.max())
