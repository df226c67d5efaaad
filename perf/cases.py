"""Timed calls of the RMSD framework: what a trajectory analysis asks of it,
through the public entry points of cpptraj_amd, from the smallest calls to the
largest.

A case is a dict of plain values.  `kind` names the call:

  rms2d    rms2d(): the all-pairs matrix of one trajectory (or against a second)
  cluster  cluster_cache(): the pairwise-distance cache over a sieved frame list
  batch    Batch.run(): one matrix per trajectory, a plan kept by the program
  fit      rmsd_fit(): every frame to a reference structure
  grad     RmsdToReference, forward and backward
  block    PairwiseRmsd, forward and backward over a block of frame pairs
  perres   rmsd_fit() and rmsd_perres() with the fit's update
  avgcorr  rms_avgcorr(): every window size
  symm     rmsd_symm(): symmetric atoms re-paired per frame

Trajectories are a 3.8 A random-walk chain with Gaussian displacements (for
`drift` an autoregressive walk, so that neighbouring frames are alike), each
frame rotated and moved at random as a freely tumbling molecule is; masses are
those of H, C, N, O and S.  Everything is made from the seed on the GPU.
"""
import itertools
import math

import numpy as np
import torch

import cpptraj_amd as ca

DEV = "cuda"


# ---- cases ----------------------------------------------------------------------
def listed():
    return [
        # The regression suite's trajectory, a backbone mask: launches and latency.
        dict(name="rms2d_small", kind="rms2d", frames=101, atoms=223, sel=66, precision="fp64",
             mode="fit", mass=False, ref_frames=0, soa=False, drift=False),
        # An ordinary rms2d of C-alpha atoms at the default precision, ragged sizes.
        dict(name="rms2d_ca", kind="rms2d", frames=3001, atoms=305, sel=305, precision="fp64",
             mode="fit", mass=False, ref_frames=0, soa=False, drift=False),
        # The headline matrix: 50,000 frames x 1,200 atoms of a drifting trajectory.
        dict(name="rms2d_large", kind="rms2d", frames=50000, atoms=1200, sel=1200,
             precision="bf16x3", mode="fit", mass=False, ref_frames=0, soa=False, drift=True),
        # Clustering on pre-aligned frames: every third frame, every second atom, no fit.
        dict(name="cluster_nofit", kind="cluster", frames=12000, atoms=500, sel=250, sieve=3,
             nofit=True, mass=False, precision="fp64"),
        # Many trajectories of uneven size in one plan.
        dict(name="batch_mixed", kind="batch", sets=16, fmin=500, fmax=8000, nmin=50, nmax=3000,
             precision="bf16x3", soa=True),
        # One small chunk of the rmsd action with a mask: launches and latency.
        dict(name="fit_small", kind="fit", frames=100, atoms=223, sel=66, mass=False,
             modify="rottrans", save=True, soa=False),
        # The rmsd action's default over a long trajectory: fit, rotate, rewrite.
        dict(name="fit_stream", kind="fit", frames=100000, atoms=3000, sel=3000, mass=False,
             modify="rottrans", save=False, soa=False),
        # RMSD to a reference as a loss: forward and gradient, mass-weighted.
        dict(name="fit_grad", kind="grad", frames=4096, atoms=2000, mass=True),
        # A block of pairwise RMSDs as a loss: forward and both gradients.
        dict(name="block_grad", kind="block", frames_a=512, frames_b=512, atoms=2000, mass=True),
        # rms ... perres over residues of uneven length, after the fit's update.
        dict(name="perres_stream", kind="perres", frames=50000, atoms=3000, rmin=7, rmax=24,
             mass=True, center=False, soa=False),
        # RMS average correlation of a fitted C-alpha trajectory, all windows.
        dict(name="avgcorr_all", kind="avgcorr", frames=10000, atoms=300, mass=False,
             maxwindow=-1, offset=1),
        # Symmetry-corrected RMSD of a protein: methyls, carboxylates, rings.
        dict(name="symm_protein", kind="symm", frames=50000, atoms=2000, groups=250, gmax=3,
             mass=False, want_map=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rms2d", "cluster", "batch", "fit", "grad", "block", "perres", "avgcorr",
                       "symm"])
    if kind == "rms2d":
        prec = rng.choice(["fp64", "fp32", "bf16x3"])
        f, n = _log(rng, 100, 20000), _log(rng, 20, 3000)
        most = {"fp64": 4e10, "fp32": 8e10, "bf16x3": 2e11}[prec]
        every = rng.choice([1, 1, 2, 3])
        sel = max(10, n // every)
        while f * f / 2.0 * sel > most:
            f = f * 3 // 4
        full = rng.random() < 0.25
        return dict(kind=kind, frames=f, atoms=every * sel, sel=sel, precision=prec,
                    mode=rng.choice(["fit", "fit", "qrmsd", "nofit"]), mass=rng.random() < 0.4,
                    ref_frames=max(2, f // 3) if full else 0, soa=rng.random() < 0.3,
                    drift=rng.random() < 0.5)
    if kind == "cluster":
        f, n = _log(rng, 300, 20000), _log(rng, 30, 1500)
        sieve = rng.choice([1, 2, 3, 5, 10])
        while (f / sieve) ** 2 / 2 * n > 2e10:
            f = f * 3 // 4
        return dict(kind=kind, frames=max(f, 2 * sieve), atoms=2 * n, sel=n, sieve=sieve,
                    nofit=rng.random() < 0.4, mass=rng.random() < 0.4,
                    precision=rng.choice(["fp64", "fp32", "bf16x3"]))
    if kind == "batch":
        fmax, nmax = _log(rng, 600, 10000), _log(rng, 100, 3000)
        return dict(kind=kind, sets=rng.randint(2, 24), fmin=max(100, fmax // 16), fmax=fmax,
                    nmin=max(20, nmax // 30), nmax=nmax,
                    precision=rng.choice(["fp32", "bf16x3", "bf16x3"]), soa=rng.random() < 0.5)
    if kind == "fit":
        n = _log(rng, 20, 5000)
        f = min(_log(rng, 1, 200000), int(3e8 / n))
        every = rng.choice([1, 1, 2, 10]) if n >= 100 else 1
        return dict(kind=kind, frames=f, atoms=n, sel=n // every,
                    mass=rng.random() < 0.4, modify=rng.choice(["rottrans", "nomod", "norotate"]),
                    save=rng.random() < 0.4, soa=rng.random() < 0.3)
    if kind == "grad":
        n = _log(rng, 20, 4000)
        return dict(kind=kind, frames=min(_log(rng, 8, 16384), int(8e6 / n)), atoms=n,
                    mass=rng.random() < 0.5)
    if kind == "block":
        n = _log(rng, 20, 3000)
        fa, fb = _log(rng, 8, 768), _log(rng, 8, 768)
        while fa * fb * n > 5.2e8:
            fa, fb = max(1, fa * 3 // 4), max(1, fb * 3 // 4)
        return dict(kind=kind, frames_a=fa, frames_b=fb, atoms=n, mass=rng.random() < 0.5)
    if kind == "perres":
        n = _log(rng, 150, 5000)
        return dict(kind=kind, frames=min(_log(rng, 50, 100000), int(1.5e8 / n)), atoms=n, rmin=5,
                    rmax=rng.randint(8, 30), mass=rng.random() < 0.6, center=rng.random() < 0.4,
                    soa=rng.random() < 0.4)
    if kind == "avgcorr":
        f, n = _log(rng, 100, 8000), _log(rng, 20, 500)
        while f * f * n > 2.8e10:
            f = f * 3 // 4
        return dict(kind=kind, frames=f, atoms=n, mass=rng.random() < 0.4,
                    maxwindow=rng.choice([-1, -1, f // 2]), offset=rng.choice([1, 1, 3, 10]))
    n = _log(rng, 60, 4000)
    return dict(kind="symm", frames=min(_log(rng, 20, 60000), int(1e8 / n)), atoms=n,
                groups=max(1, n // rng.randint(8, 20)), gmax=rng.choice([2, 3, 4]),
                mass=rng.random() < 0.4, want_map=rng.random() < 0.6)


# ---- inputs ---------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device=DEV, dtype=dtype)


def _rotations(g, k):
    """k uniform random rotations, from random unit quaternions."""
    q = _randn(g, k, 4, dtype=torch.float64)
    w, x, y, z = (q / q.norm(dim=1, keepdim=True)).unbind(1)
    R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], 1)
    return R.reshape(k, 3, 3).float()


def _chain(g, n):
    u = _randn(g, n, 3, dtype=torch.float64)
    return torch.cumsum(3.8 * u / u.norm(dim=1, keepdim=True), 0).float()


def _tumble(g, X):
    """X rotated and moved at random, frame by frame, in place."""
    for s in range(0, X.shape[0], 16384):
        k = min(16384, X.shape[0] - s)
        t = 40.0 * torch.rand((k, 1, 3), generator=g, device=DEV) - 20.0
        X[s:s + k] = torch.bmm(X[s:s + k], _rotations(g, k)) + t
    return X


def _noisy(g, frames, chain, sigma, rigid=True):
    X = _randn(g, frames, chain.shape[0], 3).mul_(sigma).add_(chain)
    return _tumble(g, X) if rigid else X


def _drift(g, frames, chain, rho=0.99, sigma=0.3):
    """Frames chain + d_f, d_f = rho d_(f-1) + N(0, sigma^2), 128 frames a step."""
    B, n = 128, chain.shape[0]
    e = torch.arange(B, device=DEV, dtype=torch.float64)
    L = torch.tril(rho ** (e[:, None] - e[None, :])).float() * sigma
    carry = (rho ** (e + 1)).float()[:, None]
    X = _randn(g, frames, n, 3)
    d = _randn(g, 1, 3 * n) * (sigma / math.sqrt(1 - rho * rho))
    for s in range(0, frames, B):
        k = min(B, frames - s)
        blk = torch.addmm(carry[:k] @ d, L[:k, :k], X[s:s + k].reshape(k, -1))
        d = blk[-1:]
        X[s:s + k] = blk.reshape(k, n, 3) + chain
    return _tumble(g, X)


def _masses(g, n):
    p = torch.tensor([0.50, 0.30, 0.08, 0.10, 0.02], device=DEV)
    m = torch.tensor([1.0, 12.0, 14.0, 16.0, 32.0], device=DEV, dtype=torch.float64)
    return m[torch.multinomial(p, n, replacement=True, generator=g)]


def _mask(c):
    if c["sel"] == c["atoms"]:
        return None
    step = c["atoms"] // c["sel"]
    return torch.arange(0, step * c["sel"], step, device=DEV, dtype=torch.int32)


def _lay(X, soa):
    """(F, n, 3) as the program stores it: AoS rows, or SoA rows of n atoms."""
    return X.permute(0, 2, 1).contiguous() if soa else X.reshape(X.shape[0], -1)


def _batch_sizes(c):
    """Evenly spread sizes (logarithmic), frame counts and atom counts unalike."""
    k = c["sets"]
    t = [(i + 0.5) / k for i in range(k)]
    F = [int(c["fmin"] * (c["fmax"] / c["fmin"]) ** x) for x in t]
    N = [int(c["nmin"] * (c["nmax"] / c["nmin"]) ** ((x * 7.31) % 1.0)) for x in t]
    return F, N


def _residues(c):
    """Offsets of consecutive residues whose lengths run over rmin .. rmax."""
    span = c["rmax"] - c["rmin"] + 1
    off, k = [0], 0
    while off[-1] < c["atoms"]:
        off.append(min(c["atoms"], off[-1] + c["rmin"] + (k * 5) % span))
        k += 1
    return np.asarray(off, np.int32)


def _groups(c):
    """Disjoint runs of 2 .. gmax neighbouring atoms, evenly spread."""
    step = c["atoms"] // c["groups"]
    return [list(range(i * step, i * step + 2 + i % (c["gmax"] - 1))) for i in range(c["groups"])]


def prepare(case, seed):
    c, g = case, _gen(seed)
    kind = c["kind"]
    s = {"case": c}
    if kind == "rms2d":
        chain = _chain(g, c["atoms"])
        make = _drift if c["drift"] else (lambda g_, f, x: _noisy(g_, f, x, 0.5))
        rigid = c["mode"] != "nofit"
        if not rigid:
            make = lambda g_, f, x: _noisy(g_, f, x, 0.5, False)  # noqa: E731
        s["X"] = _lay(make(g, c["frames"], chain), c["soa"])
        s["ref"] = _lay(make(g, c["ref_frames"], chain), c["soa"]) if c["ref_frames"] else None
        s["mask"] = _mask(c)
        s["mass"] = _masses(g, c["sel"]) if c["mass"] else None
    elif kind == "cluster":
        s["X"] = _lay(_noisy(g, c["frames"], _chain(g, c["atoms"]), 0.5, not c["nofit"]), False)
        s["list"] = torch.arange(0, c["frames"], c["sieve"], device=DEV, dtype=torch.int32)
        s["mask"] = _mask(c)
        s["mass"] = _masses(g, c["sel"]) if c["mass"] else None
    elif kind == "batch":
        F, N = _batch_sizes(c)
        s["sets"] = [_lay(_noisy(g, f, _chain(g, n), 0.5), c["soa"]) for f, n in zip(F, N)]
        s["outs"] = [torch.empty(f * (f - 1) // 2, dtype=torch.float32, device=DEV) for f in F]
        s["ctx"] = ca.Context(0)
        s["plan"] = ca.Batch(s["ctx"], [ca.frames_desc(x, soa=c["soa"]) for x in s["sets"]],
                             s["outs"], "fit", False, c["precision"], graph=True)
    elif kind == "fit":
        chain = _chain(g, c["atoms"])
        s["X"] = _lay(_noisy(g, c["frames"], chain, 1.0), c["soa"])
        s["ref"] = _lay(_noisy(g, 1, chain, 1.0), c["soa"])
        s["mask"] = _mask(c)
        s["mass"] = _masses(g, c["sel"]) if c["mass"] else None
    elif kind == "grad":
        chain = _chain(g, c["atoms"])
        s["X"] = _noisy(g, c["frames"], chain, 1.0).requires_grad_(True)
        s["ref"] = _noisy(g, 1, chain, 1.0)
        s["G"] = _randn(g, c["frames"], dtype=torch.float64)
        s["mass"] = _masses(g, c["atoms"]) if c["mass"] else None
    elif kind == "block":
        chain = _chain(g, c["atoms"])
        s["A"] = _noisy(g, c["frames_a"], chain, 1.0).requires_grad_(True)
        s["B"] = _noisy(g, c["frames_b"], chain, 1.0).requires_grad_(True)
        s["G"] = _randn(g, c["frames_a"], c["frames_b"])
        s["mass"] = _masses(g, c["atoms"]) if c["mass"] else None
    elif kind == "perres":
        chain = _chain(g, c["atoms"])
        s["X"] = _lay(_noisy(g, c["frames"], chain, 1.0), c["soa"])
        s["ref"] = _lay(_noisy(g, 1, chain, 1.0), c["soa"])
        s["mass"] = _masses(g, c["atoms"]) if c["mass"] else None
        s["hmass"] = s["mass"].cpu().numpy() if c["mass"] else None
        s["off"] = _residues(c)
        s["entries"] = np.arange(c["atoms"], dtype=np.int32)
    elif kind == "avgcorr":
        chain = _chain(g, c["atoms"])
        s["X"] = _lay(_noisy(g, c["frames"], chain, 0.6, False), False)
        s["ref"] = _lay(_noisy(g, 1, chain, 0.3), False)
        s["mass"] = _masses(g, c["atoms"]) if c["mass"] else None
    else:
        groups = _groups(c)
        chain = _chain(g, c["atoms"])
        m = _masses(g, c["atoms"])
        for a in groups:  # symmetric atoms: equal masses, 1.5 A from the first
            u = _randn(g, len(a), 3)
            chain[a] = chain[a[0]] + 1.5 * u / u.norm(dim=1, keepdim=True)
            m[a] = m[a[0]].item()
        X = _randn(g, c["frames"], c["atoms"], 3).mul_(0.3).add_(chain)
        for size in range(2, c["gmax"] + 1):  # every frame's groups in an order of its own
            at = torch.tensor([a for a in groups if len(a) == size], device=DEV)
            if at.numel():
                pick = torch.rand((c["frames"], *at.shape), generator=g, device=DEV).argsort(-1)
                src = at.expand(c["frames"], -1, -1).gather(2, pick).reshape(c["frames"], -1, 1)
                X[:, at.reshape(-1)] = X.gather(1, src.expand(-1, -1, 3))
        s["X"] = _lay(_tumble(g, X), False)
        s["ref"] = _lay(_noisy(g, 1, chain, 0.3), False)
        s["mass"] = m if c["mass"] else None
        s["groups"] = ca.symm_groups(groups)
    return s


# ---- the calls ------------------------------------------------------------------
def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "rms2d":
        return ca.rms2d(s["X"], mask=s["mask"], mass=s["mass"], mode=c["mode"],
                        use_mass=c["mass"], precision=c["precision"], ref_frames=s["ref"],
                        soa=c["soa"])
    if kind == "cluster":
        return ca.cluster_cache(s["X"], s["list"], mask=s["mask"], mass=s["mass"],
                                nofit=c["nofit"], use_mass=c["mass"], precision=c["precision"])
    if kind == "batch":
        s["plan"].run()
        return s["outs"]
    if kind == "fit":
        r, U, t = ca.rmsd_fit(s["X"], s["ref"], mask=s["mask"], mass=s["mass"],
                              use_mass=c["mass"], modify=c["modify"], save_matrices=c["save"],
                              save_vectors=c["save"], soa=c["soa"])
        out = {"rmsd": r}
        if c["save"]:
            out.update(U=U, tvec=t)
        if c["modify"] != "nomod":
            out["frames"] = s["X"]
        return out
    if kind == "grad":
        from cpptraj_amd.autograd import RmsdToReference
        r = RmsdToReference.apply(s["X"], s["ref"], s["mass"], c["mass"])
        return r, torch.autograd.grad(r, s["X"], s["G"])[0]
    if kind == "block":
        from cpptraj_amd.autograd import PairwiseRmsd
        r = PairwiseRmsd.apply(s["A"], s["B"], s["mass"], c["mass"])
        return r, *torch.autograd.grad(r, (s["A"], s["B"]), s["G"])
    if kind == "perres":
        r, U, t = ca.rmsd_fit(s["X"], s["ref"], mass=s["mass"], use_mass=c["mass"],
                              modify="nomod", save_matrices=True, save_vectors=True,
                              soa=c["soa"])
        return r, ca.rmsd_perres(s["X"], s["off"], s["entries"], s["ref"], tmass=s["hmass"],
                                 use_mass=c["mass"], center=c["center"], modify="rottrans", U=U,
                                 tvec=t, soa=c["soa"])
    if kind == "avgcorr":
        return ca.rms_avgcorr(s["X"], mass=s["mass"], ref_frames=s["ref"], use_mass=c["mass"],
                              maxwindow=c["maxwindow"], offset=c["offset"])
    r, amap, _, _ = ca.rmsd_symm(s["X"], s["groups"], s["ref"], mass=s["mass"],
                                 use_mass=c["mass"], want_map=c["want_map"])
    return (r, amap) if c["want_map"] else r


def _windows(c):
    top = c["frames"] if c["maxwindow"] == -1 else min(c["maxwindow"] + 1, c["frames"])
    return [1] + list(range(1 + c["offset"], top, c["offset"]))


def work(case):
    """Inputs read once, outputs written once; 18 flops per atom and pair for a
    3 x 3 covariance, 9 for a squared distance."""
    c = case
    kind = c["kind"]
    if kind in ("rms2d", "cluster"):
        full = c.get("ref_frames", 0)
        f = -(-c["frames"] // c.get("sieve", 1))
        pairs = f * full if full else f * (f - 1) / 2
        per = 9 if c.get("nofit") or c.get("mode") == "nofit" else 18
        return {"bytes": 12.0 * c["sel"] * (f + full) + 4.0 * pairs,
                "flops": float(per * c["sel"] * pairs)}
    if kind == "batch":
        F, N = _batch_sizes(c)
        return {"bytes": sum(12.0 * f * n + 2.0 * f * (f - 1) for f, n in zip(F, N)),
                "flops": sum(9.0 * n * f * (f - 1) for f, n in zip(F, N))}
    if kind == "block":
        fa, fb, n = c["frames_a"], c["frames_b"], c["atoms"]
        return {"bytes": 24.0 * n * (fa + fb) + 8.0 * fa * fb, "flops": 3.0 * 18 * n * fa * fb}
    if kind == "avgcorr":
        f, n = c["frames"], c["atoms"]
        fits = sum(f - w + 1 for w in _windows(c))
        return {"bytes": 12.0 * f * n + 20.0 * len(_windows(c)),
                "flops": 9.0 * fits * n}
    f, n = c["frames"], c["atoms"]
    if kind == "fit":
        moved = 24.0 * n if c["modify"] != "nomod" else 12.0 * c["sel"]
        return {"bytes": f * (moved + 8.0 + (120.0 if c["save"] else 0.0)),
                "flops": f * (30.0 * c["sel"] + (18.0 * n if c["modify"] == "rottrans" else 0.0))}
    if kind == "grad":
        return {"bytes": f * (24.0 * n + 16.0), "flops": f * 54.0 * n}
    if kind == "perres":
        return {"bytes": f * (12.0 * n + 8.0 * (len(_residues(c)) - 1) + 8.0),
                "flops": f * 58.0 * n}
    atoms = sum(len(a) for a in _groups(c))
    return {"bytes": f * (12.0 * n + 8.0 + (4.0 * n if c["want_map"] else 0.0)),
            "flops": f * (30.0 * n + 30.0 * atoms)}


# ---- the same results in 64 bits --------------------------------------------------
def _key_lambda(S, E0):
    """Largest eigenvalue of the quaternion key matrix of S (..., 3, 3), that is
    the trace of U^T S at the best rotation, by Newton's method on its
    characteristic polynomial, downwards from E0."""
    rows = S.unbind(-2)
    dots = [[(a * b).sum(-1) for b in rows] for a in rows]  # S S^T
    S2 = dots[0][0] + dots[1][1] + dots[2][2]
    G2 = sum(d * d for row in dots for d in row)
    det = (torch.linalg.cross(rows[0], rows[1]) * rows[2]).sum(-1)
    c2, c1, c0 = -2.0 * S2, -8.0 * det, 2.0 * G2 - S2 * S2
    lam = E0.clone()
    for _ in range(60):
        l2 = lam * lam
        p = (l2 + c2) * l2 + c1 * lam + c0
        dp = 4.0 * l2 * lam + 2.0 * c2 * lam + c1
        step = torch.where(dp != 0, p / dp, torch.zeros_like(p))
        lam -= step
        if bool((step.abs() <= 1e-13 * lam.abs()).all()):
            break
    return lam


def _centre(X, w):
    return (X * w[:, None]).sum(-2, keepdim=True) / w.sum()


def _pairs_exact(A, B, w, fit, tri):
    """RMSDs of frames A (Fa, n, 3) x B (Fb, n, 3), rows of A a block at a time."""
    M, sw = w.sum(), w.sqrt()[:, None]
    if fit:
        A, B = A - _centre(A, w), (B - _centre(B, w) if B is not A else None)
        B = A if B is None else B
    A, B = A * sw, (B * sw if B is not A else None)
    B = A if B is None else B
    n, fb = A.shape[1], B.shape[0]
    ga, gb = (A * A).sum((1, 2)), (B * B).sum((1, 2))
    cols = B.permute(1, 0, 2).reshape(n, 3 * fb)
    out = []
    step = max(1, int(4e7) // fb)
    for s in range(0, A.shape[0], step):
        a = A[s:s + step]
        k = a.shape[0]
        j0 = s + 1 if tri else 0
        if j0 >= fb:
            break
        if fit:
            S = a.permute(0, 2, 1).reshape(3 * k, n) @ cols[:, 3 * j0:]
            S = S.reshape(k, 3, fb - j0, 3).permute(0, 2, 1, 3)
            E0 = 0.5 * (ga[s:s + k, None] + gb[None, j0:])
            r = (2.0 * (E0 - _key_lambda(S, E0)) / M).clamp_min(0.0).sqrt()
        else:
            r = torch.cdist(a.reshape(k, -1), B[j0:].reshape(fb - j0, -1),
                            compute_mode="donot_use_mm_for_euclid_dist") / M.sqrt()
        if tri:
            i = torch.arange(s, s + k, device=DEV)[:, None]
            out.append(r[torch.arange(j0, fb, device=DEV)[None] > i])
        else:
            out.append(r)
    return torch.cat(out)


def _rotations_exact(S):
    """U with x' = U x from S = sum w x y^T (..., 3, 3)."""
    V, _, W = torch.linalg.svd(S.reshape(-1, 3, 3).cpu())
    d = torch.det(V) * torch.det(W)
    V[:, :, 2] *= d[:, None]
    return (V @ W).transpose(1, 2).reshape(S.shape).to(S.device)


def _aos(X, soa, n):
    return X.reshape(X.shape[0], 3, n).permute(0, 2, 1) if soa else X.reshape(X.shape[0], n, 3)


def _fit_exact(X, ref, idx, w):
    """(rmsd, U, Trans, refTrans) of frames X (F, n, 3) on atoms idx."""
    y = ref.double()[0][idx]
    cy = _centre(y, w)
    y, out = y - cy, []
    for s in range(0, X.shape[0], 16384):
        x = X[s:s + 16384, idx].double()
        cx = _centre(x, w)
        x = x - cx
        S = (x * w[:, None]).transpose(1, 2) @ y
        U = _rotations_exact(S)
        d = x @ U.transpose(1, 2) - y
        out.append(((w[:, None] * d * d).sum((1, 2)).div(w.sum()).sqrt(), U, -cx[:, 0]))
    r, U, t = (torch.cat(v) for v in zip(*out))
    return r, U, t, cy[0]


def _moved_exact(X, U, t, cy):
    return (X.double() + t[:, None]) @ U.transpose(1, 2) + cy


def exact(case, seed):
    c = case
    kind = c["kind"]
    s = prepare(c, seed)
    w = s.get("mass")
    if kind in ("rms2d", "cluster"):
        idx = s["mask"].long() if s["mask"] is not None else slice(None)
        X = _aos(s["X"], c.get("soa", False), c["atoms"])[:, idx]
        X = (X[s["list"].long()] if kind == "cluster" else X).double()
        w = torch.ones(c["sel"], dtype=torch.float64, device=DEV) if w is None else w
        fit = not c["nofit"] if kind == "cluster" else c["mode"] != "nofit"
        if s.get("ref") is None:
            return _pairs_exact(X, X, w, fit, True)
        R = _aos(s["ref"], c["soa"], c["atoms"])[:, idx].double()
        return _pairs_exact(X, R, w, fit, False)
    if kind == "batch":
        out = []
        for x, n in zip(s["sets"], _batch_sizes(c)[1]):
            X = _aos(x, c["soa"], n).double()
            out.append(_pairs_exact(X, X, torch.ones(n, dtype=torch.float64, device=DEV), True,
                                    True))
        return out
    w = torch.ones(c.get("sel", c["atoms"]), dtype=torch.float64, device=DEV) if w is None else w
    if kind == "fit":
        X = _aos(s["X"], c["soa"], c["atoms"])
        idx = s["mask"].long() if s["mask"] is not None else slice(None)
        r, U, t, cy = _fit_exact(X, _aos(s["ref"], c["soa"], c["atoms"]), idx, w)
        out = {"rmsd": r}
        if c["save"]:
            out.update(U=U, tvec=torch.cat([t, cy.expand(len(t), 3)], 1))
        if c["modify"] != "nomod":
            Y = _moved_exact(X, U, t, cy) if c["modify"] == "rottrans" else \
                X.double() + (t + cy)[:, None]
            out["frames"] = _lay(Y, c["soa"])
        return out
    if kind == "grad":
        X = s["X"].detach()
        r, U, t, cy = _fit_exact(X, s["ref"], slice(None), w)
        y = s["ref"].double()[0] - cy
        d = (X.double() + t[:, None]) - y @ U
        return r, d * (s["G"] / r / w.sum())[:, None, None] * w[:, None]
    if kind == "block":
        A, B = s["A"].detach().double(), s["B"].detach().double()
        r = _pairs_exact(A, B, w, True, False)
        A, B = A - _centre(A, w), B - _centre(B, w)
        n, fa, fb = A.shape[1], A.shape[0], B.shape[0]
        S = (A * w[:, None]).permute(0, 2, 1).reshape(3 * fa, n) @ B.permute(1, 0, 2).reshape(n, -1)
        U = _rotations_exact(S.reshape(fa, 3, fb, 3).permute(0, 2, 1, 3))
        k = s["G"].double() / r / w.sum()
        kU = (k[..., None, None] * U).permute(0, 2, 1, 3)  # (fa, 3 of B, fb, 3 of A)
        ga = k.sum(1)[:, None, None] * A - (kU.permute(0, 3, 2, 1).reshape(3 * fa, 3 * fb) @
                                            B.permute(0, 2, 1).reshape(3 * fb, n)
                                            ).reshape(fa, 3, n).transpose(1, 2)
        gb = k.sum(0)[:, None, None] * B - (kU.permute(2, 1, 0, 3).reshape(3 * fb, 3 * fa) @
                                            A.permute(0, 2, 1).reshape(3 * fa, n)
                                            ).reshape(fb, 3, n).transpose(1, 2)
        return r, ga * w[:, None], gb * w[:, None]
    if kind == "perres":
        X = _aos(s["X"], c["soa"], c["atoms"])
        ref = _aos(s["ref"], c["soa"], c["atoms"])
        r, U, t, cy = _fit_exact(X, ref, slice(None), w)
        off = torch.as_tensor(s["off"].astype(np.int64), device=DEV)
        size = off[1:] - off[:-1]
        k = torch.arange(int(size.max()), device=DEV)
        at = (off[:-1, None] + k).clamp_max(c["atoms"] - 1)  # (residues, longest)
        wr = w[at] * (k < size[:, None])
        mean = lambda Z: (Z * wr[..., None]).sum(-2, keepdim=True) / wr.sum(-1)[:, None, None]  # noqa: E731
        yr = ref.double()[0][at]
        yr = yr - mean(yr) if c["center"] else yr
        out = []
        for f in range(0, len(r), 8192):
            e = slice(f, f + 8192)
            x = _moved_exact(X[e], U[e], t[e], cy)[:, at]
            x = x - mean(x) if c["center"] else x
            out.append((((x - yr) ** 2).sum(-1) * wr).sum(-1).div(wr.sum(-1)).sqrt())
        return r, torch.cat(out)
    if kind == "avgcorr":
        return _avgcorr_exact(c, s, w)
    X, ref = _aos(s["X"], False, c["atoms"]), _aos(s["ref"], False, c["atoms"])
    _, U, t, cy = _fit_exact(X, ref, slice(None), w)
    y, out = ref.double()[0] - cy, []
    groups = _groups(c)
    for f in range(0, len(U), 8192):
        e = slice(f, f + 8192)
        x, z = _moved_exact(X[e], U[e], t[e], 0.0), X[e].clone()
        for size in range(2, c["gmax"] + 1):  # the cheapest of all orders of a group
            at = torch.tensor([a for a in groups if len(a) == size], device=DEV)
            if at.numel():
                perms = torch.tensor(list(itertools.permutations(range(size))), device=DEV)
                cost = torch.stack([((x[:, at[:, p]] - y[at]) ** 2).sum((-1, -2)) for p in perms])
                pick = at[None].expand(len(x), -1, -1).gather(2, perms[cost.argmin(0)])
                z[:, at.reshape(-1)] = X[e].gather(1, pick.reshape(len(x), -1, 1).expand(-1, -1, 3))
        out.append(_fit_exact(z, ref, slice(None), w)[0])
    r = torch.cat(out)
    return (r, None) if c["want_map"] else r


def _avgcorr_exact(c, s, w):
    """Running averages as differences of prefix sums of the frames about their
    mean, fitted diagonal by diagonal of the (end, begin) matrix."""
    F, n = c["frames"], c["atoms"]
    X = s["X"].reshape(F, n, 3).double()
    mu = X.mean(0)
    P = torch.cat([torch.zeros_like(X[:1]), torch.cumsum(X - mu, 0)])
    y = s["ref"].reshape(n, 3).double()
    y = y - _centre(y, w)
    gy, y = (y * y).sum(-1) @ w, y * w[:, None]
    M, ct, sd, sizes = w.sum(), [], [], _windows(c)
    for k in sizes:
        a = (P[k:] - P[:-k]) / k + mu
        a -= _centre(a, w)
        E0 = 0.5 * ((a * a).sum(-1) @ w + gy)
        S = (a.permute(0, 2, 1).reshape(-1, n) @ y).reshape(-1, 3, 3)
        r = (2.0 * (E0 - _key_lambda(S, E0)) / M).clamp_min(0.0).sqrt()
        ct.append(r.mean())
        sd.append(r.var(unbiased=False))
    return (np.asarray(sizes, np.int32), torch.stack(ct),
            torch.stack(sd).sqrt())
