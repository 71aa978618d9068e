"""Centroid scores at frame counts around the score tiles (256 columns by 32 or
64 rows) against numpy on the full matrix; relative error below 1e-9, the bar
of the other centroid tests."""
import numpy as np
import pytest

from mdtraj_amd import allpairs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 31, 32, 33, 63, 64, 65, 255, 256, 257, 258, 300, 511, 513,
                               1000, 8063, 8064, 8065, 8321])
def test_sizes(gpu, n):
    rng = np.random.default_rng(n)
    d = rng.uniform(0.05, 1.0, n * (n - 1) // 2).astype(np.float32)
    full = np.zeros((n, n))
    iu = np.triu_indices(n, 1)
    full[iu] = d
    full += full.T
    std = full.std()
    want = np.exp(-full / std).sum(1) if std > 0 else np.ones(n)
    got = allpairs.centroid_scores(gpu.from_numpy(d).cuda() if n > 1 else d, n)
    assert np.abs(got / want - 1).max() < 1e-9
