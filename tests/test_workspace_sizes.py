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


@pytest.mark.parametrize("n_frames", [1, 3, 700, 1000, 1024, 1025, 100000])
def test_rmsf_workspace_never_shrinks(n_frames):
    """The accumulation's chunks of frames become fewer with every block of
    256 atoms."""
    lib = _lib.load()
    size = [lib.hr_rmsf_workspace_bytes(n_frames, n) for n in range(1, 5000)]
    assert size == sorted(size)
    size = [lib.hr_rmsf_workspace_bytes(f, 1500) for f in range(1, 3000)]
    assert size == sorted(size)
    # and holds the chunks' sums, of four doubles an atom, beside what a
    # superposition needs
    for n in range(1, 5000):
        blocks = -(-n // 256)
        chunks = min(-(-2048 // blocks), 1024, n_frames)
        need = lib.hr_superpose_workspace_bytes(n_frames, n) + 32 * chunks * n
        assert lib.hr_rmsf_workspace_bytes(n_frames, n) >= need
