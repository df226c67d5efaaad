"""RMS average correlation (rmsd_avgcorr) against the oracle.

The library fits every averaged frame by single-pass FP64 moments and QCP,
the oracle by the reference's two-pass Kabsch; the running sums are the same
FP64 sequence.  Bar: 1e-9 A on the mean and the SD of every window with a
fixed reference.  With 'first', every window fits its first averaged frame
to itself: the true RMSD is 0, where the reference's Kabsch eigenvalue
formula returns rounding noise up to ~sqrt(eps E0 / M) ~ 1e-7 A and QCP
~1e-8 A, so that one sample moves the window's mean and SD by up to ~1e-7 A:
the bar there is 5e-7 A.  Cases:
fixed reference and 'first', mass weighting, 'stop' and 'offset', a
selection, SoA frames, and the argument errors.

Both methods of rmsd_avgcorr_set_method run every case: the running sum (one
wavefront per window) and the prefix form (window sums as differences of
prefix sums of the mean-subtracted coordinates, every averaged frame fitted
independently in tiles of prefix rows: 64 x 64 with a fixed reference,
32 x 32 with 'first', whose window references are staged per diagonal).
Both meet the same bars; the prefix form also past the running method's LDS
atom limit, across many tiles, on a drifting trajectory, and against the
running method on 3,000 frames.
"""
import numpy as np
import pytest

from cpptraj_amd import synth

pytestmark = pytest.mark.gpu

TOL = 1e-9


def _avgcorr(ca, ctx, *args, method="auto", **kw):
    """rms_avgcorr with the method set for this call only (the setting stays
    with the shared context otherwise)."""
    try:
        return ca.rms_avgcorr(*args, method=method, ctx=ctx, **kw)
    finally:
        ctx.check(ctx._L.rmsd_avgcorr_set_method(ctx.handle, 0))


@pytest.mark.parametrize("use_mass", [False, True])
@pytest.mark.parametrize("first,method", [(False, "running"), (False, "prefix"), (True, "running"),
                                          (True, "prefix")])
@pytest.mark.parametrize("stop_offset", [(-1, 1), (40, 3), (-1, 7)])
def test_avgcorr_matches_oracle(ctx, oracle, use_mass, first, method, stop_offset):
    import torch

    import cpptraj_amd as ca
    stop, offset = stop_offset
    rng = np.random.default_rng(41 + use_mass + 2 * first)
    F, n = 97, 150
    X = synth.noisy(9, F, n, 0.5).reshape(F, -1).astype(np.float32)
    sel = np.sort(rng.choice(n, 101, replace=False)).astype(np.int32)
    m = synth.masses(rng, n)
    Xd = torch.as_tensor(X).cuda()
    seld = torch.as_tensor(sel).cuda()
    md = torch.as_tensor(m[sel]).cuda()
    R = None
    rc = None
    if not first:
        ref = (X[3].reshape(-1, 3) + rng.normal(size=(n, 3)) * 0.3).astype(np.float32)
        R = torch.as_tensor(ref.reshape(1, -1)).cuda()
        rc, _ = oracle.center_on_origin(ref[sel].astype(np.float64), m[sel], use_mass)
    w, ct, sd = _avgcorr(ca, ctx, Xd, seld, md, ref_frames=R, use_mass=use_mass, maxwindow=stop,
                         offset=offset, method=method)
    w_o, ct_o, sd_o = oracle.avgcorr(X, sel, m[sel], rc, use_mass, stop, offset)
    assert np.array_equal(w, w_o)
    tol = 5e-7 if first else TOL
    assert np.abs(ct.cpu().numpy() - ct_o).max() <= tol
    assert np.abs(sd.cpu().numpy() - sd_o).max() <= tol


@pytest.mark.parametrize("method", ["running", "prefix"])
def test_avgcorr_soa_frames(ctx, oracle, method):
    import torch

    import cpptraj_amd as ca
    F, n, ld = 60, 77, 96
    X = synth.noisy(10, F, n, 0.5).reshape(F, n, 3).astype(np.float32)
    S = np.zeros((F, 3, ld), np.float32)
    S[:, :, :n] = X.transpose(0, 2, 1)
    Sd = torch.as_tensor(S).cuda()
    # reference: frame 2 of a separate SoA set (perturbed copies, so that no
    # window compares a frame with itself)
    rng = np.random.default_rng(10)
    RX = np.stack([X[k] + rng.normal(size=(n, 3)).astype(np.float32) * 0.4 for k in (1, 4, 7)])
    RS = np.zeros((3, 3, ld), np.float32)
    RS[:, :, :n] = RX.transpose(0, 2, 1)
    w, ct, sd = _avgcorr(ca, ctx, Sd, ref_frames=torch.as_tensor(RS).cuda(), ref_index=2,
                         soa=True, natom=n, offset=2, method=method)
    rc, _ = oracle.center_on_origin(RX[2].astype(np.float64))
    _, ct_o, sd_o = oracle.avgcorr(X.reshape(F, -1), ref_sel_centered=rc, offset=2)
    assert np.abs(ct.cpu().numpy() - ct_o).max() <= TOL
    assert np.abs(sd.cpu().numpy() - sd_o).max() <= TOL


@pytest.mark.parametrize("use_mass", [False, True])
def test_avgcorr_prefix_many_tiles_with_drift(ctx, oracle, use_mass):
    # 300 frames (5 x 5 row tiles, windows on every diagonal class) of a
    # trajectory that drifts 8 A, so that the prefix sums are large.
    import torch

    import cpptraj_amd as ca
    rng = np.random.default_rng(77)
    F, n = 300, 60
    X = synth.noisy(11, F, n, 0.4).reshape(F, n, 3).astype(np.float64)
    X += np.linspace(0.0, 8.0, F)[:, None, None] * rng.normal(size=(1, n, 3)) + 40.0
    X = X.reshape(F, -1).astype(np.float32)
    m = synth.masses(rng, n)
    ref = (X[5].reshape(n, 3) + rng.normal(size=(n, 3)) * 0.2).astype(np.float32)
    rc, _ = oracle.center_on_origin(ref.astype(np.float64), m, use_mass)
    for stop, offset in ((-1, 1), (200, 64), (130, 5)):
        w, ct, sd = _avgcorr(ca, ctx, torch.as_tensor(X).cuda(), mass=torch.as_tensor(m).cuda(),
                             ref_frames=torch.as_tensor(ref.reshape(1, -1)).cuda(),
                             use_mass=use_mass, maxwindow=stop, offset=offset, method="prefix")
        w_o, ct_o, sd_o = oracle.avgcorr(X, None, m, rc, use_mass, stop, offset)
        assert np.array_equal(w, w_o)
        assert np.abs(ct.cpu().numpy() - ct_o).max() <= TOL
        assert np.abs(sd.cpu().numpy() - sd_o).max() <= TOL


def test_avgcorr_prefix_beyond_running_atom_limit(ctx, oracle):
    # 7,000 selected atoms: over the running method's LDS limit; the default
    # (auto) method takes the prefix form.
    import torch

    import cpptraj_amd as ca
    rng = np.random.default_rng(78)
    F, n = 24, 7000
    X = synth.noisy(12, F, n, 0.5).reshape(F, -1).astype(np.float32)
    ref = (X[2].reshape(n, 3) + rng.normal(size=(n, 3)) * 0.3).astype(np.float32)
    rc, _ = oracle.center_on_origin(ref.astype(np.float64))
    w, ct, sd = _avgcorr(ca, ctx, torch.as_tensor(X).cuda(),
                         ref_frames=torch.as_tensor(ref.reshape(1, -1)).cuda())
    _, ct_o, sd_o = oracle.avgcorr(X, ref_sel_centered=rc)
    assert np.abs(ct.cpu().numpy() - ct_o).max() <= TOL
    assert np.abs(sd.cpu().numpy() - sd_o).max() <= TOL


def test_avgcorr_prefix_matches_running_3000_frames(ctx):
    # Every window of 3,000 frames x 200 atoms: the two methods agree.
    import torch

    import cpptraj_amd as ca
    rng = np.random.default_rng(79)
    F, n = 3000, 200
    X = synth.noisy(13, F, n, 0.6).reshape(F, -1).astype(np.float32)
    m = synth.masses(rng, n)
    Xd, md = torch.as_tensor(X).cuda(), torch.as_tensor(m).cuda()
    R = torch.as_tensor(X[7:8] + rng.normal(size=(1, 3 * n)).astype(np.float32) * 0.3).cuda()
    out = {}
    for method in ("running", "prefix"):
        w, ct, sd = _avgcorr(ca, ctx, Xd, mass=md, ref_frames=R, use_mass=True, method=method)
        out[method] = (ct.cpu().numpy(), sd.cpu().numpy())
    assert len(w) == F - 1
    assert np.abs(out["running"][0] - out["prefix"][0]).max() <= TOL
    assert np.abs(out["running"][1] - out["prefix"][1]).max() <= TOL


@pytest.mark.parametrize("use_mass", [False, True])
def test_avgcorr_first_prefix_matches_running_3000_frames(ctx, use_mass):
    # 'first': every window's reference is its own first averaged frame.
    import torch

    import cpptraj_amd as ca
    rng = np.random.default_rng(80)
    F, n = 3000, 150
    X = synth.noisy(14, F, n, 0.6).reshape(F, -1).astype(np.float32)
    m = synth.masses(rng, n)
    Xd, md = torch.as_tensor(X).cuda(), torch.as_tensor(m).cuda()
    out = {}
    for method in ("running", "prefix"):
        w, ct, sd = _avgcorr(ca, ctx, Xd, mass=md, use_mass=use_mass, method=method)
        out[method] = (ct.cpu().numpy(), sd.cpu().numpy())
    assert np.abs(out["running"][0] - out["prefix"][0]).max() <= 5e-7
    assert np.abs(out["running"][1] - out["prefix"][1]).max() <= 5e-7


def test_avgcorr_errors(ctx):
    import torch

    import cpptraj_amd as ca
    X = torch.zeros((1, 30), dtype=torch.float32, device="cuda")
    with pytest.raises(ca.RmsdError, match="Not enough frames"):
        ca.rms_avgcorr(X, ctx=ctx)
    Y = torch.zeros((4, 3 * 4000), dtype=torch.float32, device="cuda")
    with pytest.raises(ca.RmsdError, match="selected atoms with 'first'"):
        _avgcorr(ca, ctx, Y, method="running")
    Z = torch.zeros((4, 3 * 7000), dtype=torch.float32, device="cuda")
    with pytest.raises(ca.RmsdError, match="selected atoms"):
        _avgcorr(ca, ctx, Z, ref_frames=Z[:1], method="running")
    with pytest.raises(ca.RmsdError, match="unknown rmsavgcorr method"):
        ctx.check(ctx._L.rmsd_avgcorr_set_method(ctx.handle, 7))


@pytest.mark.parametrize("F", [126, 127, 128, 190, 191, 192, 256, 321])
@pytest.mark.parametrize("n,use_mass,offset", [(5, False, 1), (11, True, 1), (32, False, 70), (43, True, 2)])
def test_avgcorr_gram_tile_edges(ctx, F, n, use_mass, offset):
    """Tiles off the diagonal (distances as a product): frame counts at the
    edges of the 64-row tiles, coordinates that leave a stage of 32 unfilled and
    windows that cross only some tiles, against the running sum.  A drift of 8 A
    over the trajectory makes the prefix sums large against their differences."""
    import torch

    import cpptraj_amd as ca
    rng = np.random.default_rng(F + n)
    X3 = synth.noisy(F + n, 1, n, 0.0) + rng.normal(scale=0.5, size=(F, n, 3)) + np.linspace(0, 8, F)[:, None, None]
    X = torch.as_tensor(X3.reshape(F, -1).astype(np.float32)).cuda()
    R = X[3:4].clone()
    m = torch.as_tensor(synth.masses(rng, n)).cuda()
    kw = dict(ref_frames=R, mass=m, use_mass=use_mass, offset=offset)
    w, ct, sd = _avgcorr(ca, ctx, X, method="prefix", **kw)
    w2, ct2, sd2 = _avgcorr(ca, ctx, X, method="running", **kw)
    assert np.array_equal(w, w2)
    # The windows those tiles hold: 65 frames and more (window 1 also has the
    # reference fitted to itself, noise of sqrt(eps E0 / M) on either side).
    far = torch.as_tensor(w >= 65).cuda()
    assert float((ct - ct2)[far].abs().max()) <= TOL
    # SD = sqrt(mean(r^2) - mean(r)^2): rounding of the two means, ~1e-15 r^2,
    # under the root.
    assert float((sd ** 2 - sd2 ** 2)[far].abs().max()) <= 1e-12 * float(ct2.max()) ** 2


def _exact_windows(X, ref, windows):
    """Mean and SD of each window's RMSDs in extended precision, and the mean and
    the root mean square over its fits of 64 eps E0 / (W r) (64 roundings of E0 in
    the FP64 solve)."""
    L = np.longdouble
    F, n = X.shape[:2]
    X = X.astype(L)
    P = np.concatenate([np.zeros((1, n, 3), L), np.cumsum(X, 0)])
    y = ref.astype(L) - ref.astype(L).mean(0)
    gy = (y * y).sum()
    out = []
    for w in windows:
        a = (P[w:] - P[:-w]) / w
        a = a - a.mean(1, keepdims=True)
        S = np.stack([(a[:, :, c, None] * y[None]).sum(1) for c in range(3)], 1)
        C = np.stack([np.cross(S[:, 1], S[:, 2]), np.cross(S[:, 2], S[:, 0]), np.cross(S[:, 0], S[:, 1])], 1)
        T = (S * S).sum((1, 2))
        c2, c1, c0 = -2 * T, -8 * (S[:, 0] * C[:, 0]).sum(1), T * T - 4 * (C * C).sum((1, 2))
        E0 = ((a * a).sum((1, 2)) + gy) / 2
        lam = E0.copy()
        for _ in range(60):
            lam = lam - (((lam * lam + c2) * lam + c1) * lam + c0) / (4 * lam ** 3 + 2 * c2 * lam + c1)
        r = np.sqrt(2 * (E0 - lam) / n)
        tol = 64 * np.finfo(float).eps * E0 / (n * r)
        out.append([r.mean(), np.sqrt(((r - r.mean()) ** 2).mean()), tol.mean(),
                    np.sqrt((tol ** 2).mean())])
    return np.array(out, float).T


@pytest.mark.parametrize("motion", ["none", "still", "diffusing", "jumping", "breathing 3", "breathing 10"])
def test_avgcorr_large_motions(ctx, motion):
    """Trajectories whose prefix sums are large against their differences: common
    translations of 8,192 A, and internal motion of up to ten times the
    reference's size with a period of 65 frames (10: tiles that leave the product
    for the differences).  Coordinates are multiples of 2^-10 A, 256 frames and
    16 atoms: prefix sums, means and centroids are exact in FP64, what is left is
    the solve's rounding.  Neither the mean nor the SD of a window's RMSDs (also
    where two fits hardly differ) can be further off than the fits are."""
    import torch

    import cpptraj_amd as ca
    F, n = 256, 16
    rng = np.random.default_rng(17)
    u = rng.normal(size=(n, 3))
    chain = np.cumsum(3.8 * u / np.linalg.norm(u, axis=1)[:, None], 0)
    chain -= chain.mean(0)
    X = chain + rng.normal(scale=0.5, size=(F, n, 3))
    f = np.arange(F)[:, None, None]
    if motion == "diffusing":
        X += np.cumsum(np.round(rng.normal(scale=50.0, size=(F, 1, 3))), 0)
    elif motion == "jumping":
        X += np.where(f % 65 < 32, 8192.0, -8192.0)
    elif motion == "still":
        X = np.repeat(X[:1], F, 0)
    elif motion != "none":
        X *= 1 + float(motion.split()[1]) * np.sin(2 * np.pi * f / 65)
    X = (np.round(X * 1024) / 1024).astype(np.float32)
    assert np.array_equal(X.astype(np.float64) * 1024, np.round(X.astype(np.float64) * 1024))
    ref = (np.round((chain + rng.normal(scale=0.3, size=(n, 3))) * 1024) / 1024).astype(np.float32)
    w, ct, sd = _avgcorr(ca, ctx, torch.as_tensor(X.reshape(F, -1)).cuda(),
                         ref_frames=torch.as_tensor(ref.reshape(1, -1)).cuda(), method="prefix")
    mean, dev, tol, tol_rms = _exact_windows(X, ref, w)
    assert np.all(np.abs(ct.cpu().numpy() - mean) <= tol)
    assert np.all(np.abs(sd.cpu().numpy() - dev) <= tol_rms)
