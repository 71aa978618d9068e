"""LP-RMSD at the edges of its group search, against the FP64 oracle."""
import numpy as np
import pytest

import mdtraj_amd as md
from oracle import lprmsd as olp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1e16, 1e-17])
@pytest.mark.parametrize("k,noise", [(33, 0.02), (63, 0.02), (63, 0.6), (70, 0.02)])
def test_coordinates_of_any_size(gpu, k, noise, scale):
    """Squared distances beyond the value that fills up the search's last tile
    of targets (63 atoms leave one such place, 33 leave 31), and below what its
    float products resolve.  The bar is the 2e-5 of coordinates of order 1."""
    rng = np.random.default_rng(k)
    base = np.concatenate([rng.normal(0, 0.6, (7, 3)), rng.uniform(-1, 1, (k, 3))])
    x = base[None] + rng.normal(0, noise, (3, k + 7, 3))
    for f in range(3):
        x[f, 7:] = x[f, 7 + rng.permutation(k)]
    x = (scale * x).astype(np.float32)
    ref = (scale * base[None]).astype(np.float32)
    groups = [np.arange(7, 7 + k)]
    want = olp.lprmsd(x, ref, 0, None, groups)
    got = md.lprmsd(x, ref, 0, None, groups)
    assert np.abs(got - want).max() < 2e-5 * scale


@pytest.mark.parametrize("groups", [[[]], [[], []]])
def test_groups_without_atoms(gpu, groups):
    """No group between the fit on the solute and the final RMSD and rotation,
    which read it from LDS: the plain RMSD, every frame turned by its own fit."""
    rng = np.random.default_rng(5)
    base = rng.normal(0, 0.6, (41, 3))
    x = base[None] + rng.normal(0, 0.05, (67, 41, 3))
    for f in range(67):
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        x[f] = x[f] @ (q if np.linalg.det(q) > 0 else -q)
    x = x.astype(np.float32)
    ref = base[None].astype(np.float32)
    want, moved = olp.lprmsd(x, ref, 0, None, groups, superpose=True)
    y = x.copy()
    got = md.lprmsd(y, ref, 0, permute_groups=groups, superpose=True)
    assert np.abs(got - want).max() < 2e-5
    assert np.abs(y - moved).max() < 2e-5


@pytest.mark.parametrize("sizes", [(1,), (1, 1, 1), (2, 1, 2), (31, 1), (32, 33, 32), (33, 1, 2, 64),
                                   (129, 2, 192), (200, 1), (256,), (320, 40), (385,)])
@pytest.mark.parametrize("noise", [0.02, 0.5])
def test_several_groups(gpu, sizes, noise):
    """Groups of one wave beside groups of both, single atoms beside them, and
    searches of one, two and five columns a lane at a time, with superposition."""
    rng = np.random.default_rng(sum(sizes))
    n = 9 + sum(sizes)
    base = np.concatenate([rng.normal(0, 0.6, (9, 3)), rng.uniform(-1, 1, (n - 9, 3))])
    x = base[None] + rng.normal(0, noise, (3, n, 3))
    groups, at = [], 9
    for k in sizes:
        groups.append(np.arange(at, at + k))
        for f in range(3):
            x[f, at:at + k] = x[f, at + rng.permutation(k)]
        at += k
    x = x.astype(np.float32)
    ref = base[None].astype(np.float32)
    want, moved = olp.lprmsd(x, ref, 0, None, groups, superpose=True)
    y = x.copy()
    got = md.lprmsd(y, ref, 0, permute_groups=groups, superpose=True)
    assert np.abs(got - want).max() < 2e-5
    assert np.abs(y - moved).max() < 2e-5


def test_more_frames_than_one_launch_dimension(gpu):
    """2^25 + 3 frames of two waves each: above 2^32 work-items.  The frames
    repeat, so every result is one of a few."""
    free, _ = gpu.cuda.mem_get_info()
    F, N, some = 2**25 + 3, 3, 7
    if free < 4 * 12 * F * N:
        pytest.skip("needs 5 GB of device memory")
    rng = np.random.default_rng(2)
    base = rng.uniform(-1, 1, (some, N, 3)).astype(np.float32)
    x = gpu.from_numpy(base).cuda().repeat(F // some + 1, 1, 1)[:F].contiguous()
    got = md.lprmsd(x, x[:1], 0, permute_groups=[[1, 2]])
    few = md.lprmsd(x[:some].clone(), x[:1], 0, permute_groups=[[1, 2]])
    want = few.repeat(F // some + 1)[:F]
    assert got.shape == (F,) and bool((got == want).all())
    assert np.abs(few.cpu().numpy() - olp.lprmsd(base, base[:1], 0, None, [[1, 2]]))[1:].max() < 2e-5
