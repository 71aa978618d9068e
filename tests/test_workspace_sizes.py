"""Workspace sizes never fall as the problem grows, so a buffer sized for the
largest problem serves the smaller ones."""
import pytest

from mdtraj_amd import _lib


@pytest.mark.parametrize("lo,hi", [(1, 600), (7900, 8200), (10700, 10900), (16000, 16600)])
def test_centroid_workspace_never_shrinks(lo, hi):
    """The score tiles' height changes at 8,064 frames."""
    lib = _lib.load()
    size = [lib.hr_centroid_workspace_bytes(n) for n in range(lo, hi)]
    assert size == sorted(size)
