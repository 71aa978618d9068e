"""RMSF of few frames: chunks of one frame, and the finish that takes a thread per
atom for up to 16 chunks, on both sides of that line and of a workgroup's atoms.
Against the FP64 oracle; the bar is one rounding of the result to float32."""
import numpy as np
import pytest

import mdtraj_amd as md
from mdtraj_amd import gen
from oracle import fp64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_frames", [1, 2, 15, 16, 17, 40])
@pytest.mark.parametrize("n_atoms", [5, 256, 257, 6000])
def test_sizes(gpu, n_frames, n_atoms):
    x = gen.walk(seed=n_atoms + n_frames, n_frames=n_frames, n_atoms=n_atoms)
    for ref in (x, None):
        want = fp64.rmsf(x, ref, 0, None)
        got = md.rmsf(x, ref, 0)
        assert np.abs(got - want).max() <= 1e-6 * max(1.0, want.max())


def test_many_atoms_few_chunks(gpu):
    """40,000 atoms leave 14 chunks, of up to 30 frames each."""
    x = gen.walk(seed=1, n_frames=400, n_atoms=40000)
    want = fp64.rmsf(x, None, 0, None)
    got = md.rmsf(x, None, 0)
    assert np.abs(got - want).max() <= 1e-6 * max(1.0, want.max())
