"""Measured cases: what users of this package have it do, through its public calls.

Every case is a dict of plain values with a ``kind``:

  rmsd       md.rmsd of a trajectory to one of its frames (numpy or device)
  superpose  Trajectory.superpose in place, in HBM
  rmsf       md.rmsf of a device trajectory
  matrix     rmsd_matrix, the condensed all-pairs matrix
  centroid   rmsd_matrix, then centroid_scores (the centroid notebook)
  leaders    nearest leader of every frame, from raw coordinates
  batch      BatchRMSD over uneven systems, one plan launched again and again
  xtc, dcd   reading every frame of a trajectory file into HBM
  lprmsd     md.lprmsd with one group of interchangeable atoms

Coordinates are nanometres: a reference structure plus a random walk or
independent noise, every frame rigidly moved, as a simulation's frames drift
and tumble.
"""
import math
import os
import struct
import tempfile

import numpy as np
import torch

import mdtraj_amd as md
from mdtraj_amd import allpairs, batch, dcd, xtc

_DEV = "cuda"


# ------------------------------------------------------------------- cases
def listed():
    return [
        # a peptide's trajectory as numpy arrays (alanine dipeptide's 22
        # atoms): one call of a script, all latency
        {"name": "rmsd_host_small", "kind": "rmsd", "where": "host", "frames": 1000, "atoms": 22,
         "sel": 0, "motion": "noise", "superpose": True},
        # a long peptide simulation kept in HBM: a million short frames
        {"name": "rmsd_peptide", "kind": "rmsd", "where": "device", "frames": 1000003, "atoms": 22,
         "sel": 0, "motion": "noise", "superpose": True},
        # a protein's trajectory, a subset of its atoms scored to frame 0
        {"name": "rmsd_protein", "kind": "rmsd", "where": "device", "frames": 100000,
         "atoms": 2000, "sel": 1500, "motion": "walk", "superpose": True},
        # aligning a trajectory on a subset (alpha carbons) before analysis
        {"name": "superpose", "kind": "superpose", "frames": 20000, "atoms": 3001, "sel": 375},
        # per-atom fluctuations after a fit
        {"name": "rmsf", "kind": "rmsf", "frames": 20000, "atoms": 2000, "sel": 1500},
        # clustering: the distance matrix of a whole trajectory
        {"name": "matrix_large", "kind": "matrix", "frames": 20000, "atoms": 500},
        # the centroid of a few thousand frames: matrix and scores
        {"name": "centroid", "kind": "centroid", "frames": 4001, "atoms": 301},
        # two-pass clustering: every frame to its nearest leader
        {"name": "leaders", "kind": "leaders", "frames": 100000, "atoms": 500, "leaders": 250},
        # independent systems of uneven size scored as one batch
        {"name": "batch_uneven", "kind": "batch", "systems": 64, "min_atoms": 50,
         "max_atoms": 5000, "min_frames": 10, "max_frames": 8000},
        # compressed trajectory of a solvated chain, read into HBM
        {"name": "xtc_read", "kind": "xtc", "frames": 10000, "atoms": 3001},
        # uncompressed trajectory with a unit cell, read into HBM
        {"name": "dcd_read", "kind": "dcd", "frames": 10001, "atoms": 2500},
        # a solute among interchangeable water oxygens
        {"name": "lprmsd", "kind": "lprmsd", "frames": 20000, "solute": 100, "group": 300},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rmsd", "rmsd", "superpose", "rmsf", "matrix", "centroid", "leaders",
                       "batch", "xtc", "dcd", "lprmsd"])
    if kind == "rmsd":
        where = rng.choice(["host", "device", "device"])
        atoms = _log_int(rng, 8, 6000)
        most = 2e6 if where == "host" else 1.5e8
        frames = _log_int(rng, 100, max(200, min(2000000, int(most / atoms))))
        return {"kind": kind, "where": where, "frames": frames, "atoms": atoms,
                "sel": rng.choice([0, 0, max(4, atoms // 4), max(5, 3 * atoms // 4)]),
                "motion": rng.choice(["noise", "walk"]), "superpose": rng.random() < 0.85}
    if kind in ("superpose", "rmsf"):
        atoms = _log_int(rng, 20, 8000)
        frames = _log_int(rng, 50, max(100, min(1000000, int(6e7 / atoms))))
        return {"kind": kind, "frames": frames, "atoms": atoms,
                "sel": rng.choice([0, max(4, atoms // 8), max(5, 3 * atoms // 4)])}
    if kind in ("matrix", "centroid"):
        return {"kind": kind, "frames": _log_int(rng, 100, 12000 if kind == "matrix" else 6000),
                "atoms": _log_int(rng, 20, 800)}
    if kind == "leaders":
        atoms = _log_int(rng, 20, 800)
        return {"kind": kind, "frames": _log_int(rng, 500, int(4.5e7 / max(atoms, 450))),
                "atoms": atoms, "leaders": _log_int(rng, 5, 250)}
    if kind == "batch":
        return {"kind": kind, "systems": _log_int(rng, 3, 60),
                "min_atoms": rng.randint(10, 100), "max_atoms": _log_int(rng, 200, 5000),
                "min_frames": rng.randint(1, 20), "max_frames": _log_int(rng, 50, 8000)}
    if kind in ("xtc", "dcd"):
        atoms = _log_int(rng, 30, 12000)
        return {"kind": kind, "frames": _log_int(rng, 20, max(50, min(60000, int(2.5e7 / atoms)))),
                "atoms": atoms}
    group = _log_int(rng, 8, 300)
    return {"kind": kind, "frames": _log_int(rng, 100, int(4e6 / max(group, 250))),
            "solute": _log_int(rng, 4, 150), "group": group}


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device=_DEV)
    g.manual_seed(seed)
    return g


def _rotations(g, n):
    """Uniform random rotation matrices (n, 3, 3), float64."""
    q = torch.randn((n, 4), generator=g, device=_DEV, dtype=torch.float64)
    w, x, y, z = (q / q.norm(dim=1, keepdim=True)).unbind(1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)],
                       1).reshape(n, 3, 3)


def _frames(g, n_frames, n_atoms, motion):
    """Trajectory (n_frames, n_atoms, 3), float32 in HBM: a box of atoms of
    about a protein's extent, moved by noise or a walk, each frame turned and
    shifted as a whole."""
    box = max(1.0, 0.4 * n_atoms ** (1.0 / 3.0))
    ref = torch.rand((n_atoms, 3), generator=g, device=_DEV, dtype=torch.float64) * box
    out = torch.empty((n_frames, n_atoms, 3), device=_DEV, dtype=torch.float32)
    chunk = max(1, 16000000 // n_atoms)
    for a in range(0, n_frames, chunk):
        b = min(n_frames, a + chunk)
        step = torch.randn((b - a, n_atoms, 3), generator=g, device=_DEV, dtype=torch.float64)
        if motion == "walk":
            pos = ref + torch.cumsum(0.005 * step, 0)
            ref = pos[-1]
        else:
            pos = ref + 0.03 * step
        R = _rotations(g, b - a)
        t = torch.rand((b - a, 1, 3), generator=g, device=_DEV, dtype=torch.float64) * 4 - 2
        out[a:b] = ((pos[:, :, :1] * R[:, :1] + pos[:, :, 1:2] * R[:, 1:2]
                     + pos[:, :, 2:] * R[:, 2:]) + t).float()
    return out


def _selection(case, seed):
    if not case["sel"]:
        return None
    rng = np.random.default_rng(seed + 77)
    return np.sort(rng.choice(case["atoms"], size=case["sel"], replace=False))


def _batch_sizes(case, seed):
    # the sizes belong to the case (a plan's launch is timed), the frames to the seed
    rng = np.random.default_rng(3)
    n = case["systems"]
    def sizes(lo, hi):
        return np.exp(rng.uniform(np.log(lo), np.log(hi + 1), n)).astype(int).clip(lo, hi)
    atoms = sizes(case["min_atoms"], case["max_atoms"])
    return list(zip(sizes(case["min_frames"], case["max_frames"]).tolist(), atoms.tolist()))


def _lprmsd_frames(case, seed):
    """A solute and water oxygens that drift and trade places."""
    g = _generator(seed)
    F, s, k = case["frames"], case["solute"], case["group"]
    base = torch.cat([torch.randn((s, 3), generator=g, device=_DEV, dtype=torch.float64) * 0.6,
                      torch.rand((k, 3), generator=g, device=_DEV, dtype=torch.float64) * 3 - 1.5])
    x = base + 0.02 * torch.randn((F, s + k, 3), generator=g, device=_DEV, dtype=torch.float64)
    p = torch.argsort(torch.rand((F, k), generator=g, device=_DEV), dim=1) + s
    x[:, s:] = torch.gather(x, 1, p[:, :, None].expand(F, k, 3))
    return x.float().contiguous()


# the format's table of small-delta ranges: entry i holds three digits in i bits
_XTC_RANGE = [0] * 9 + [
    8, 10, 12, 16, 20, 25, 32, 40, 50, 64, 80, 101, 128, 161, 203, 256, 322, 406, 512, 645, 812,
    1024, 1290, 1625, 2048, 2580, 3250, 4096, 5060, 6501, 8192]


def _xtc_field(v, bits):
    """v as the format's bit field: whole low bytes first, then the rest."""
    s = ""
    while bits > 8:
        s += format(v & 255, "08b")
        v >>= 8
        bits -= 8
    return s + format(v, "0%db" % bits)


def _xtc_stream(q):
    """One frame's integer coordinates (N, 3) in XTC's bytes, from the precision
    on: runs of up to eight near atoms after each full one, the first stored
    swapped with it, the range of the deltas following the data."""
    n = len(q)
    lo, hi = q.min(0), q.max(0)
    size = [int(v) for v in hi - lo + 1]
    bits = (size[0] * size[1] * size[2]).bit_length()
    atoms = q.tolist()
    first = int(np.median(np.abs(np.diff(q, axis=0)).max(1)))
    idx = 9
    while idx + 9 < len(_XTC_RANGE) and _XTC_RANGE[idx] // 2 <= first:
        idx += 1
    low, high, start = max(9, idx - 4), min(idx + 4, len(_XTC_RANGE) - 1), idx
    m0, m1, m2 = (int(v) for v in lo)
    out, i, last = [], 0, 0
    while i < n:
        half, span = _XTC_RANGE[idx] // 2, _XTC_RANGE[idx]
        run, worst = [], 0
        if i + 1 < n:
            frm, to = atoms[i + 1], atoms[i]
            j = i + 1
            while len(run) < 8:
                d = [to[c] - frm[c] for c in range(3)]
                big = max(abs(d[0]), abs(d[1]), abs(d[2]))
                if big >= half:
                    near = big < _XTC_RANGE[min(idx + 1, high)] // 2
                    break
                worst = max(worst, big)
                run.append((d[0] + half) * span * span + (d[1] + half) * span + d[2] + half)
                j += 1
                if j >= n:
                    break
                frm, to = to, atoms[j]
        full = atoms[i + 1] if run else atoms[i]
        out.append(_xtc_field(((full[0] - m0) * size[1] + full[1] - m1) * size[2] + full[2] - m2,
                              bits))
        change = 0
        if run and idx > low and worst < _XTC_RANGE[idx - 1] // 2 and len(run) > 2:
            change = -1
        elif not run and i + 1 < n and near and idx < high:
            change = 1
        if change or 3 * len(run) != last:
            out.append("1" + format(3 * len(run) + change + 1, "05b"))
            last = 3 * len(run)
        else:
            out.append("0")
        out.extend(_xtc_field(v, idx) for v in run)
        i += 1 + len(run)
        idx += change
    s = "".join(out)
    s += "0" * (-len(s) % 8)
    data = int(s, 2).to_bytes(len(s) // 8, "big")
    return (struct.pack(">f6iii", 1000.0, *[int(v) for v in lo], *[int(v) for v in hi], start,
                        len(data)) + data + b"\0" * (-len(data) % 4))


def _xtc_frames(case, seed):
    """A few distinct frames of a chain (a third of the atoms) in water, in
    thousandths of a nanometre, and the order in which the file repeats them."""
    rng = np.random.default_rng(seed)
    n = case["atoms"]
    chain = max(1, n // 3)
    some = min(case["frames"], max(2, 30000 // n))
    box = max(2.0, (n / 100.0) ** (1.0 / 3.0))
    walk = rng.normal(0, 0.09, (chain, 3)).cumsum(0) * 0.6 + box / 2
    n_wat = -(-(n - chain) // 3)
    oxy = rng.uniform(0, box, (n_wat, 1, 3))
    wat = np.concatenate([oxy, oxy + rng.normal(0, 0.06, (n_wat, 2, 3))], 1).reshape(-1, 3)
    base = np.concatenate([walk, wat[: n - chain]])
    q = np.rint(1000 * (base + rng.normal(0, 0.01, (some, n, 3)))).astype(np.int64)
    return q, rng.integers(0, some, case["frames"]), box


def _xtc_file(case, seed):
    q, order, box = _xtc_frames(case, seed)
    n = case["atoms"]
    cell = struct.pack(">9f", box, 0, 0, 0, box, 0, 0, 0, box)
    body = [_xtc_stream(f) for f in q]
    return b"".join(struct.pack(">iiif", 1995, n, 10 * k, 2.0 * k) + cell
                    + struct.pack(">i", n) + body[o] for k, o in enumerate(order.tolist()))


def _dcd_frames(case, seed):
    g = _generator(seed)
    return 10 * _frames(g, case["frames"], case["atoms"], "noise")


def _dcd_file(case, seed):
    """CHARMM layout: control record, titles, atom count, then per frame the
    cell and the X, Y and Z records."""
    x = _dcd_frames(case, seed)
    F, n = case["frames"], case["atoms"]
    ctl = bytearray(80)
    struct.pack_into("<iii", ctl, 0, F, 0, 1)
    struct.pack_into("<f", ctl, 36, 1.0)
    struct.pack_into("<i", ctl, 40, 1)
    struct.pack_into("<i", ctl, 76, 24)
    head = (struct.pack("<i", 84) + b"CORD" + bytes(ctl) + struct.pack("<iii", 84, 164, 2)
            + b" " * 160 + struct.pack("<iiii", 164, 4, n, 4))
    rec = torch.empty((F, 14 + 3 * (n + 2)), dtype=torch.int32, device=_DEV)
    rec[:, 0] = rec[:, 13] = 48
    cell = np.array([60.0, 0, 61.0, 0, 0, 62.0]).view(np.int32)
    rec[:, 1:13] = torch.from_numpy(cell).to(_DEV)
    for k in range(3):
        o = 14 + k * (n + 2)
        rec[:, o] = rec[:, o + n + 1] = 4 * n
        rec[:, o + 1:o + 1 + n] = x[:, :, k].contiguous().view(torch.int32)
    return head + rec.cpu().numpy().tobytes()


def _open(reader, data, suffix):
    fd, name = tempfile.mkstemp(suffix=suffix)
    try:
        with os.fdopen(fd, "wb") as f:
            f.write(data)
        return reader(name)
    finally:
        os.unlink(name)


# ----------------------------------------------------------------- the pass
def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "rmsd":
        x = _frames(_generator(seed), case["frames"], case["atoms"], case["motion"])
        state["traj"] = md.Trajectory(x.cpu().numpy() if case["where"] == "host" else x)
        state["sel"] = _selection(case, seed)
    elif kind in ("superpose", "rmsf"):
        x = _frames(_generator(seed), case["frames"], case["atoms"], "walk")
        state["traj"] = md.Trajectory(x)
        state["ref"] = md.Trajectory(x[:1].clone())
        state["sel"] = _selection(case, seed)
    elif kind in ("matrix", "centroid"):
        state["traj"] = md.Trajectory(_frames(_generator(seed), case["frames"], case["atoms"], "walk"))
    elif kind == "leaders":
        x = _frames(_generator(seed), case["frames"], case["atoms"], "walk")
        state["frames"] = x
        state["leaders"] = x[:: max(1, case["frames"] // case["leaders"])][: case["leaders"]].contiguous()
    elif kind == "batch":
        g = _generator(seed)
        xs = [_frames(g, f, n, "noise") for f, n in _batch_sizes(case, seed)]
        # the library's own defaults, without the tuner's timing runs
        state["batch"] = batch.BatchRMSD(xs, frames_per_unit=64, waves=3, unit_kib=0)
    elif kind == "xtc":
        state["file"] = _open(xtc.XTCTrajectoryFile, _xtc_file(case, seed), ".xtc")
    elif kind == "dcd":
        state["file"] = _open(dcd.DCDTrajectoryFile, _dcd_file(case, seed), ".dcd")
    else:
        x = _lprmsd_frames(case, seed)
        state["traj"] = md.Trajectory(x)
        state["ref"] = md.Trajectory(x[:1].clone())
        state["groups"] = [np.arange(case["solute"], case["solute"] + case["group"])]
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "rmsd":
        t = state["traj"]
        return md.rmsd(t, t, 0, atom_indices=state["sel"], superpose=case["superpose"])
    if kind == "superpose":
        return state["traj"].superpose(state["ref"], 0, atom_indices=state["sel"]).xyz
    if kind == "rmsf":
        return md.rmsf(state["traj"], state["ref"], 0, atom_indices=state["sel"])
    if kind == "matrix":
        return md.rmsd_matrix(state["traj"])
    if kind == "centroid":
        d = md.rmsd_matrix(state["traj"])
        return d, allpairs.centroid_scores(d, case["frames"])
    if kind == "leaders":
        return allpairs.nearest(allpairs.SplitSet(state["frames"]),
                                allpairs.SplitSet(state["leaders"]))
    if kind == "batch":
        return state["batch"].run()
    if kind in ("xtc", "dcd"):
        state["file"].seek(0)
        return [v for v in state["file"].read(device=True) if v is not None]
    return md.lprmsd(state["traj"], state["ref"], 0, permute_groups=state["groups"])


def work(case):
    """Coordinates and files read once, results written once; per atom and
    frame 18 operations for the correlation, 12 for sums and trace."""
    kind = case["kind"]
    if kind == "batch":
        sizes = _batch_sizes(case, 0)
        return {"bytes": sum(12 * f * n + 4 * f for f, n in sizes),
                "flops": sum(30 * f * n for f, n in sizes)}
    F = case["frames"]
    if kind == "lprmsd":
        n, k = case["solute"] + case["group"], case["group"]
        return {"bytes": 12 * F * n + 4 * F, "flops": F * (8 * k * k + 30 * n)}
    n = case["atoms"]
    if kind == "rmsd":
        s = case["sel"] or n
        return {"bytes": 12 * F * s + 4 * F, "flops": (30 if case["superpose"] else 8) * F * s}
    if kind == "superpose":
        return {"bytes": 24 * F * n, "flops": F * (30 * (case["sel"] or n) + 18 * n)}
    if kind == "rmsf":
        s = case["sel"] or n
        return {"bytes": 12 * F * s + 4 * s, "flops": F * s * (30 + 18 + 6)}
    pairs = F * (F - 1) // 2
    if kind in ("matrix", "centroid"):
        return {"bytes": 12 * F * n + 4 * pairs, "flops": 18 * n * pairs}
    if kind == "leaders":
        return {"bytes": 12 * (F + case["leaders"]) * n + 8 * F,
                "flops": 18 * n * F * case["leaders"]}
    if kind == "xtc":
        # about 30 compressed bits an atom
        return {"bytes": F * (4 * n + 92 + 12 * n + 48), "flops": 10 * F * n}
    return {"bytes": F * (24 * n + 80 + 28), "flops": 3 * F * n}


# ------------------------------------------------------- 64-bit expectations
def _lambda_max(M):
    """Largest eigenvalue of the quaternion key matrix of M (..., 3, 3), by
    Newton's method from its Frobenius bound on the characteristic quartic."""
    a, b, c, d, e, f, g, h, i = M.reshape(-1, 9).unbind(1)
    c2 = -2 * (M.reshape(-1, 9) ** 2).sum(1)
    c1 = -8 * (a * (e * i - f * h) - b * (d * i - f * g) + c * (d * h - e * g))
    K = torch.stack([a + e + i, f - h, g - c, b - d, f - h, a - e - i, b + d, g + c,
                     g - c, b + d, e - a - i, f + h, b - d, g + c, f + h, i - a - e], 1)
    k = K.unbind(1)
    def minor(x, y, z):
        return (k[4 + x] * (k[8 + y] * k[12 + z] - k[8 + z] * k[12 + y])
                - k[4 + y] * (k[8 + x] * k[12 + z] - k[8 + z] * k[12 + x])
                + k[4 + z] * (k[8 + x] * k[12 + y] - k[8 + y] * k[12 + x]))
    c0 = (k[0] * minor(1, 2, 3) - k[1] * minor(0, 2, 3)
          + k[2] * minor(0, 1, 3) - k[3] * minor(0, 1, 2))
    x = torch.sqrt(-1.5 * c2)
    for _ in range(30):
        p = ((x * x + c2) * x + c1) * x + c0
        dp = (4 * x * x + 2 * c2) * x + c1
        x = torch.where(dp > 0, x - p / dp, x)
    return x


def _moments(x):
    """Centred float64 coordinates and their sums of squares."""
    c = x.double()
    c = c - c.mean(-2, keepdim=True)
    return c, (c * c).sum((-1, -2))


def _rmsd_to(x, ref):
    """RMSD of every frame of x to ref (n, 3) after the best fit."""
    r, gr = _moments(ref)
    out = []
    chunk = max(1, 30000000 // x.shape[1])
    for a in range(0, x.shape[0], chunk):
        c, g = _moments(x[a:a + chunk])
        M = torch.stack([(c[:, :, i, None] * r).sum(1) for i in range(3)], 1)
        out.append(torch.sqrt(((g + gr - 2 * _lambda_max(M)) / x.shape[1]).clamp(min=0)))
    return torch.cat(out)


def _rmsd_between(x, y):
    """RMSD of every frame of x to every frame of y, (len(x), len(y))."""
    c, g = _moments(x)
    r, gr = _moments(y)
    n = x.shape[1]
    X = c.permute(0, 2, 1).reshape(-1, n)
    Y = r.permute(0, 2, 1).reshape(-1, n)
    M = (X @ Y.T).reshape(len(x), 3, len(y), 3).permute(0, 2, 1, 3).reshape(-1, 3, 3)
    lam = _lambda_max(M).reshape(len(x), len(y))
    return torch.sqrt(((g[:, None] + gr - 2 * lam) / n).clamp(min=0))


def _matrix(x):
    F = len(x)
    rows, step = [], max(1, 4000000 // F)
    cols = torch.arange(F, device=_DEV)
    for a in range(0, F, step):
        d = _rmsd_between(x[a:a + step], x)
        rows.append(d[cols[None] > torch.arange(a, a + len(d), device=_DEV)[:, None]])
    return torch.cat(rows)


def _fit(x, ref):
    """Rotations R with (x - mean) R nearest to ref - mean, per frame."""
    r, _ = _moments(ref)
    out = []
    chunk = max(1, 30000000 // x.shape[1])
    for a in range(0, x.shape[0], chunk):
        c, _ = _moments(x[a:a + chunk])
        out.append(torch.stack([(c[:, :, i, None] * r).sum(1) for i in range(3)], 1).cpu())
    U, _, V = np.linalg.svd(torch.cat(out).numpy())
    U[np.linalg.det(U) * np.linalg.det(V) < 0, :, 2] *= -1
    return torch.from_numpy(U @ V).to(_DEV)


def _turn(x, R):
    return sum(x[:, :, i, None] * R[:, None, i] for i in range(3))


def _numpy(x):
    return x.cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "rmsd":
        x = _frames(_generator(seed), case["frames"], case["atoms"], case["motion"])
        sel = _selection(case, seed)
        ref = x[0].clone()
        if sel is not None:
            x, ref = x[:, sel], ref[sel]
        if case["superpose"]:
            d = _rmsd_to(x, ref)
            d[0] = 0
            return _numpy(d)
        step = max(1, 30000000 // x.shape[1])
        return _numpy(torch.cat([((x[a:a + step].double() - ref.double()) ** 2).sum(2).mean(1).sqrt()
                                 for a in range(0, len(x), step)]))
    if kind in ("superpose", "rmsf"):
        x = _frames(_generator(seed), case["frames"], case["atoms"], "walk")
        sel = _selection(case, seed)
        part = x if sel is None else x[:, sel]
        R = _fit(part, part[0])
        if kind == "superpose":
            mid, to = part.double().mean(1, keepdim=True), part[0].double().mean(0)
            return _numpy(_turn(x.double() - mid, R) + to)
        y = part.double()
        if sel is None:
            y = y - y.mean(1, keepdim=True)
        y = _turn(y, R)
        return _numpy(((y - y.mean(0)) ** 2).sum(2).mean(0).sqrt())
    if kind in ("matrix", "centroid"):
        x = _frames(_generator(seed), case["frames"], case["atoms"], "walk")
        d = _matrix(x)
        if kind == "matrix":
            return _numpy(d)
        F = len(x)
        full = torch.zeros((F, F), dtype=torch.float64, device=_DEV)
        full[tuple(torch.triu_indices(F, F, 1, device=_DEV))] = d
        full += full.T.clone()
        return _numpy(d), _numpy(torch.exp(-full / full.std(unbiased=False)).sum(1))
    if kind == "leaders":
        x = _frames(_generator(seed), case["frames"], case["atoms"], "walk")
        s = x[:: max(1, case["frames"] // case["leaders"])][: case["leaders"]]
        step = max(1, 4000000 // len(s))
        return None, _numpy(torch.cat([_rmsd_between(x[a:a + step], s).min(1).values
                                       for a in range(0, len(x), step)]))
    if kind == "batch":
        g = _generator(seed)
        out = []
        for f, n in _batch_sizes(case, seed):
            x = _frames(g, f, n, "noise")
            d = _rmsd_to(x, x[0])
            d[0] = 0
            out.append(_numpy(d))
        return out
    if kind == "xtc":
        q, order, box = _xtc_frames(case, seed)
        k = np.arange(case["frames"])
        return [q[order] / 1000.0, 2.0 * k, None, np.tile(np.eye(3) * np.float32(box), (len(k), 1, 1))]
    if kind == "dcd":
        F = case["frames"]
        return [_numpy(_dcd_frames(case, seed).double()), np.tile([60.0, 61.0, 62.0], (F, 1)),
                np.full((F, 3), 90.0)]
    return None
