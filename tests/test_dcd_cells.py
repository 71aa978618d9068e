"""Unit cells of a whole file, constant, changing, or the same in the first and the
last frame only: as each frame's cell by itself."""
import numpy as np
import pytest

from mdtraj_amd.dcd import cell_lengths_angles


@pytest.mark.parametrize("n", [0, 1, 2, 50, 511, 512, 600])
@pytest.mark.parametrize("kind", ["constant", "changing", "ends_alike", "last_differs", "nan"])
def test_cells(n, kind):
    rng = np.random.default_rng(n)
    row = np.array([60, 0.1, 61, -0.2, 0.3, 62], np.float32)
    c = np.tile(row, (n, 1))
    if kind == "changing":
        c = c + rng.random((n, 6)).astype(np.float32)
    elif kind == "ends_alike":
        c[1:-1] += rng.random((max(0, n - 2), 6)).astype(np.float32)
    elif kind == "last_differs" and n:
        c[-1, 5] = 70
    elif kind == "nan" and n:
        c[n // 2, 1] = np.nan
    lengths, angles = cell_lengths_angles(c)
    assert lengths.shape == angles.shape == (n, 3)
    for f in range(n):
        want = cell_lengths_angles(c[f:f + 1])
        assert np.array_equal(lengths[f:f + 1], want[0], equal_nan=True)
        assert np.array_equal(angles[f:f + 1], want[1], equal_nan=True)
