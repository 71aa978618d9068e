"""hr_superpose's fit and rotation kernels, which serve frames too long for LDS and
separate alignment arrays: chunks of frames, every row width of the fit, and
agreement with the one pass that serves all other frames."""
import numpy as np
import pytest

import mdtraj_amd as md
from mdtraj_amd import _lib, gen
from oracle import fp64

pytestmark = pytest.mark.gpu


def superpose(gpu, w, frame, sel, translate=1, chunk_mib=0, separate=False, outputs=True):
    """Moved coordinates, rotations and RMSDs of hr_superpose."""
    F, N = w.shape[:2]
    x = gpu.from_numpy(w).cuda()
    ref = x[frame].clone()
    idx = None if sel is None else gpu.from_numpy(np.asarray(sel, np.int32)).cuda()
    n_sel = N if sel is None else len(sel)
    p = None if idx is None else idx.data_ptr()
    align = x.clone() if separate else None
    rot, out = gpu.full((F + 1, 9), -9.0, device="cuda"), gpu.full((F + 1,), -9.0, device="cuda")
    ws = gpu.empty(_lib.load().hr_superpose_workspace_bytes(F, n_sel), dtype=gpu.uint8,
                   device="cuda")
    _lib.call("hr_set_tuning", _lib.HR_TUNE_SUPERPOSE_CHUNK_MIB, chunk_mib)
    try:
        _lib.call("hr_superpose", x.data_ptr(), F, N, None if align is None else align.data_ptr(),
                  N, p, n_sel, ref.data_ptr(), p, translate, rot.data_ptr() if outputs else None,
                  out.data_ptr() if outputs else None, ws.data_ptr(),
                  gpu.cuda.current_stream().cuda_stream)
    finally:
        _lib.call("hr_set_tuning", _lib.HR_TUNE_SUPERPOSE_CHUNK_MIB, 0)
    rot, out = rot.cpu().numpy(), out.cpu().numpy()
    assert (rot[F] == -9).all() and out[F] == -9
    return x.cpu().numpy(), rot[:F], out[:F]


@pytest.mark.parametrize("n_frames", [12, 13, 29])
@pytest.mark.parametrize("selected", [False, True])
def test_chunks_of_long_frames(gpu, n_frames, selected):
    """7,000 atoms: 84,000 B a frame, 12 frames a MiB, the last chunk whole or
    ragged.  Every frame's fit is its own, so chunks change no bit, with the
    rotations in the caller's array and in the workspace."""
    N = 7000
    w = gen.walk(seed=n_frames, n_frames=n_frames, n_atoms=N)
    sel = np.arange(1, N, 3) if selected else None
    whole = superpose(gpu, w, 5, sel, chunk_mib=4096)
    parts = superpose(gpu, w, 5, sel, chunk_mib=1)
    for a, b in zip(whole, parts):
        assert np.array_equal(a, b)
    assert np.array_equal(superpose(gpu, w, 5, sel, chunk_mib=1, outputs=False)[0], whole[0])
    assert np.abs(parts[0] - fp64.superpose(w, w, 5, sel)).max() < 2e-5
    assert np.abs(parts[2] - fp64.rmsd(w, w, 5, sel)).max() < 1e-6


@pytest.mark.parametrize("n_atoms", [1, 5, 22, 100, 191, 192, 300, 1700, 3001, 6600])
@pytest.mark.parametrize("translate", [0, 1])
def test_one_pass_agrees_with_two_kernels(gpu, n_atoms, translate):
    """The same frames as their own alignment array.  The sums' order differs, so
    rotations may differ by a rounding to float32 of entries up to 1 (6e-8, of
    coordinates up to 20 nm) and centroids not at all at that size."""
    F = 70 if n_atoms < 1000 else 9
    w = gen.walk(seed=n_atoms, n_frames=F, n_atoms=n_atoms)
    for sel in (None, gen.subset(2, n_atoms, max(1, n_atoms // 3))):
        one = superpose(gpu, w, 2, sel, translate)
        two = superpose(gpu, w, 2, sel, translate, separate=True)
        assert np.abs(one[2] - two[2]).max() < 1e-6
        if (n_atoms if sel is None else len(sel)) >= 4:  # the rotation is determined
            assert np.abs(one[1] - two[1]).max() <= 1.2e-7
            assert np.abs(one[0] - two[0]).max() < 1e-5


@pytest.mark.parametrize("row_lanes", [4, 8, 16, 32, 64])
def test_row_widths_of_the_fit(gpu, row_lanes):
    """16 to 1 frames a wave, through RMSF and a separate alignment array."""
    _lib.call("hr_set_tuning", _lib.HR_TUNE_FRAMES_ROW_LANES, row_lanes)
    try:
        for n_frames, n_atoms, n_sel in [(131, 300, 220), (67, 2000, None), (5, 40, 17),
                                         (70, 1001, None)]:
            x = gen.walk(seed=n_frames * 7 + n_atoms, n_frames=n_frames, n_atoms=n_atoms)
            sel = None if n_sel is None else gen.subset(n_atoms, n_atoms, n_sel)
            f = n_frames // 3
            moved, _, rmsd = superpose(gpu, x, f, sel, separate=True)
            assert np.abs(moved - fp64.superpose(x, x, f, sel)).max() < 2e-5
            assert np.abs(rmsd - fp64.rmsd(x, x, f, sel)).max() < 1e-6
            want = fp64.rmsf(x, x, f, sel)
            got = md.rmsf(x, x, f, atom_indices=sel)
            assert np.abs(got - want).max() <= 1e-6 * max(1.0, want.max())
    finally:
        _lib.call("hr_set_tuning", _lib.HR_TUNE_FRAMES_ROW_LANES, 0)
