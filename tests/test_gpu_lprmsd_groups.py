"""LP-RMSD's assignment at group sizes around its loops (columns in fours, 64
rows a wave, 320 rows a sweep) from its greedy start: nearly every row matched
at once (little noise), most rows searched for (noise as wide as the group),
and groups whose atoms coincide.  Against the FP64 oracle; the bar is the
float32 coordinates' rounding, as in the other LP-RMSD tests (2e-5 nm)."""
import numpy as np
import pytest

import mdtraj_amd as md
from oracle import lprmsd as olp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("noise", [0.02, 0.6])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 63, 64, 65, 67, 128, 319, 320, 321, 641])
def test_group_sizes(gpu, k, noise):
    rng = np.random.default_rng(k)
    base = np.concatenate([rng.normal(0, 0.6, (7, 3)), rng.uniform(-1, 1, (k, 3))])
    x = base[None] + rng.normal(0, noise, (4, k + 7, 3))
    for f in range(4):
        x[f, 7:] = x[f, 7 + rng.permutation(k)]
    x = x.astype(np.float32)
    groups = [np.arange(7, 7 + k)]
    want = olp.lprmsd(x, base[None].astype(np.float32), 0, None, groups)
    got = md.lprmsd(x, base[None].astype(np.float32), 0, None, groups)
    assert np.abs(got - want).max() < 2e-5


@pytest.mark.parametrize("k", [6, 70, 200])
def test_coinciding_atoms(gpu, k):
    """Several atoms of the group at each point, in two groups beside each
    other: any order among them is the same structure, and the solute, drawn
    anew, keeps the RMSD away from 0 (where float32 coordinates allow less)."""
    rng = np.random.default_rng(k)
    points = rng.uniform(-1, 1, (k // 3 + 1, 3))
    base = np.concatenate([rng.normal(0, 0.6, (5, 3)), points[rng.integers(0, len(points), k)],
                           rng.uniform(-1, 1, (9, 3))])
    x = np.repeat(base[None], 3, 0)
    x[:, :5] += rng.normal(0, 0.3, (3, 5, 3))
    for f in range(3):
        x[f, 5:5 + k] = x[f, 5 + rng.permutation(k)]
        x[f, 5 + k:] = x[f, 5 + k + rng.permutation(9)]
    x = x.astype(np.float32)
    groups = [np.arange(5, 5 + k), np.arange(5 + k, 14 + k)]
    want = olp.lprmsd(x, base[None].astype(np.float32), 0, None, groups)
    got = md.lprmsd(x, base[None].astype(np.float32), 0, None, groups)
    assert want.min() > 1e-2 and np.abs(got - want).max() < 2e-5


def test_largest_group(gpu):
    """1,073 atoms in one group: 65,486 of the 65,536 bytes of LDS allowed."""
    rng = np.random.default_rng(8)
    base = rng.uniform(-2, 2, (1073, 3))
    x = base[None] + rng.normal(0, 0.05, (2, 1073, 3))
    for f in range(2):
        x[f] = x[f, rng.permutation(1073)]
    x = x.astype(np.float32)
    want = olp.lprmsd(x, base[None].astype(np.float32), 0)
    got = md.lprmsd(x, base[None].astype(np.float32), 0)
    assert np.abs(got - want).max() < 2e-5
