"""GPU gradients (rmsd_fit_backward, rmsd_pairwise_backward) against the FP64
analytic gradient of the oracle and against central finite differences.

The reference has no RMSD derivative; the oracle's analytic gradient
(orc_rmsd_grad_target) is itself pinned by central differences in
tests/test_oracle.py.  Tolerances: analytic agreement 1e-9 relative to the
largest gradient component; finite differences (FP64, h = 1e-4 A) 1e-6.
"""
import numpy as np
import pytest

from cpptraj_amd import synth

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    a = np.ascontiguousarray(a)
    dt = {np.float32: torch.float32, np.float64: torch.float64, np.int32: torch.int32}[a.dtype.type]
    return torch.as_tensor(a, dtype=dt).cuda()


def oracle_target_grad(o, x, ref, m, um):
    rc, _ = o.center_on_origin(ref, m, um)
    return o.rmsd_grad_target(x, rc, m, um)


@pytest.mark.parametrize("use_mass", [False, True])
def test_fit_backward_matches_oracle(oracle, ctx, use_mass):
    from cpptraj_amd.autograd import fit_backward
    F, n = 64, 500
    X = synth.noisy(41, F, n, 1.0)
    m = synth.masses(np.random.default_rng(41), n)
    gr = np.random.default_rng(42).normal(size=F)
    g = fit_backward(dev(X), dev(X[:1]), dev(gr), dev(m), use_mass, ctx=ctx).cpu().numpy()
    ref = X[0].astype(np.float64)
    for f in range(F):
        r, ge = oracle_target_grad(oracle, X[f].astype(np.float64), ref, m, use_mass)
        ge = gr[f] * ge
        scale = max(np.abs(ge).max(), 1e-30)
        if f == 0:  # the reference itself: RMSD ~ 0, gradient only required finite
            assert np.isfinite(g[0]).all()
            continue
        assert np.abs(g[f] - ge).max() <= 1e-9 * scale, f


def test_fit_backward_finite_differences(oracle, ctx):
    from cpptraj_amd.autograd import fit_backward
    F, n = 4, 40
    X = synth.noisy(43, F, n, 1.0)
    m = synth.masses(np.random.default_rng(43), n)
    g = fit_backward(dev(X), dev(X[:1]), dev(np.ones(F)), dev(m), True, ctx=ctx).cpu().numpy()
    ref = X[0].astype(np.float64)
    rc, _ = oracle.center_on_origin(ref, m, True)
    h = 1e-4
    for f in (1, 3):
        x = X[f].astype(np.float64)
        fd = np.zeros_like(x)
        for a in range(n):
            for c in range(3):
                p = x.copy(); p[a, c] += h
                q = x.copy(); q[a, c] -= h
                fd[a, c] = (oracle.rmsd_centered_ref(p, rc, m, True)[0] -
                            oracle.rmsd_centered_ref(q, rc, m, True)[0]) / (2 * h)
        assert np.abs(g[f] - fd).max() <= 1e-6


@pytest.mark.parametrize("use_mass", [False, True])
def test_pairwise_block_backward_matches_oracle(oracle, ctx, use_mass):
    from cpptraj_amd.autograd import pairwise_backward
    FA, FB, n = 37, 29, 60
    X = synth.noisy(44, FA + FB, n, 0.8)  # one chain, independent noise: RMSD ~ 1 A
    A, B = X[:FA], X[FA:]
    m = synth.masses(np.random.default_rng(44), n)
    G = np.random.default_rng(46).normal(size=(FA, FB))
    ga, gb = pairwise_backward(dev(A), dev(B), dev(G), dev(m), use_mass, ctx=ctx)
    ga, gb = ga.cpu().numpy(), gb.cpu().numpy()
    ea = np.zeros_like(ga)
    eb = np.zeros_like(gb)
    for i in range(FA):
        for j in range(FB):
            _, gi = oracle_target_grad(oracle, A[i].astype(np.float64), B[j].astype(np.float64), m, use_mass)
            _, gj = oracle_target_grad(oracle, B[j].astype(np.float64), A[i].astype(np.float64), m, use_mass)
            ea[i] += G[i, j] * gi
            eb[j] += G[i, j] * gj
    sa = np.abs(ea).max()
    sb = np.abs(eb).max()
    assert np.abs(ga - ea).max() <= 1e-9 * sa
    assert np.abs(gb - eb).max() <= 1e-9 * sb


def test_autograd_function_matches_raw(ctx):
    import torch
    from cpptraj_amd.autograd import RmsdToReference, PairwiseRmsd, fit_backward
    X = synth.noisy(47, 16, 80, 1.0)
    Xt = dev(X).requires_grad_(True)
    ref = dev(X[:1])
    loss = RmsdToReference.apply(Xt, ref).sum()
    loss.backward()
    raw = fit_backward(dev(X), ref, torch.ones(16, dtype=torch.float64, device="cuda"), ctx=ctx)
    assert torch.allclose(Xt.grad.double(), raw.to(torch.float32).double())
    A = dev(X[:6]).requires_grad_(True)
    Bm = dev(X[6:]).requires_grad_(True)
    PairwiseRmsd.apply(A, Bm).sum().backward()
    assert A.grad.shape == (6, 80, 3) and Bm.grad.shape == (10, 80, 3)
    assert torch.isfinite(A.grad).all() and torch.isfinite(Bm.grad).all()


def test_differentiation_workload_sizes(oracle, ctx):
    """4096 frames x 2000 atoms mass-weighted fit backward, and a 512 x 512
    block backward at 2000 atoms; checked on sampled frames / rows."""
    import torch
    from cpptraj_amd.autograd import fit_backward, pairwise_backward
    F, n = 4096, 2000
    X = synth.noisy(48, F, n, 1.0)
    m = synth.masses(np.random.default_rng(48), n)
    Xd = dev(X)
    g = fit_backward(Xd, Xd[:1], torch.ones(F, dtype=torch.float64, device="cuda"), dev(m), True,
                     ctx=ctx)
    ref = X[0].astype(np.float64)
    for f in (1, 1000, 4095):
        _, ge = oracle_target_grad(oracle, X[f].astype(np.float64), ref, m, True)
        assert np.abs(g[f].cpu().numpy() - ge).max() <= 1e-9 * np.abs(ge).max()
    A, B = Xd[:512], Xd[512:1024]
    G = torch.ones((512, 512), dtype=torch.float64, device="cuda")
    ga, gb = pairwise_backward(A, B, G, dev(m), True, ctx=ctx)
    for i in (0, 311):
        e = np.zeros((n, 3))
        for j in range(512):
            _, gi = oracle_target_grad(oracle, X[i].astype(np.float64), X[512 + j].astype(np.float64), m, True)
            e += gi
        assert np.abs(ga[i].cpu().numpy() - e).max() <= 1e-9 * np.abs(e).max()


@pytest.mark.parametrize("F", [3, 700])
@pytest.mark.parametrize("n", [2, 5, 64, 65, 128, 129, 259, 513, 1027, 2051, 3075, 8192, 8193])
def test_fit_backward_in_registers(ctx, n, F):
    """The one-launch gradient (no selection) against the separate kernels (an
    identity selection takes them) at the edges of its sizes, FP64, and its FP32
    form against its FP64 one; a frame equal to the reference has no gradient."""
    import ctypes as C
    import torch
    import cpptraj_amd as ca
    X = dev(synth.noisy(n, F, n, 1.0)) if n * F < 3000000 else dev(synth.noisy(n, 9, n, 1.0))
    F = X.shape[0]
    m = dev(synth.masses(np.random.default_rng(n), n))
    gr = torch.linspace(-1.0, 2.0, F, dtype=torch.float64, device="cuda")
    sel = torch.arange(n, dtype=torch.int32, device="cuda")
    ref = X[1:2].clone()
    out = {}
    for key, s, fn, dt in (("new", None, ctx._L.rmsd_fit_backward, torch.float64),
                           ("f32", None, ctx._L.rmsd_fit_backward_f32, torch.float32),
                           ("old", sel, ctx._L.rmsd_fit_backward, torch.float64)):
        d, r = ca.frames_desc(X, s, m), ca.frames_desc(ref, s, m)
        out[key] = torch.full((F, n, 3), 9.0, dtype=dt, device="cuda")
        ctx.check(fn(ctx.handle, C.byref(d), C.byref(r), 0, 1, C.c_void_p(gr.data_ptr()),
                     C.c_void_p(out[key].data_ptr())))
    new, old = out["new"].cpu().numpy(), out["old"].cpu().numpy()
    assert torch.equal(out["f32"], out["new"].float())
    assert np.isfinite(new).all()
    if n > 2:  # two atoms: the rotation is not unique
        rest = [f for f in range(F) if f != 1]
        assert np.abs(new[rest] - old[rest]).max() <= 1e-9 * np.abs(old[rest]).max()


@pytest.mark.parametrize("FA,FB", [(1, 1), (1, 40), (16, 17), (33, 5), (20, 64)])
@pytest.mark.parametrize("n,use_mass", [(3, False), (31, True), (128, False), (133, True), (514, True)])
def test_pairwise_backward_edges(oracle, ctx, FA, FB, n, use_mass):
    """The block gradient at the edges of its 16-frame blocks, partner stages,
    atom tiles and weight stages against the oracle's gradient of one row and one
    column, and its FP32 form against its FP64 one."""
    import torch
    from cpptraj_amd.autograd import _pairwise_backward, pairwise_backward
    X = synth.noisy(n + FA, FA + FB, n, 0.8)
    A, B = X[:FA], X[FA:]
    m = synth.masses(np.random.default_rng(n), n)
    G = np.random.default_rng(FB).normal(size=(FA, FB)).astype(np.float32)
    ga, gb = pairwise_backward(dev(A), dev(B), dev(G).double(), dev(m), use_mass, ctx=ctx)
    fa, fb = _pairwise_backward(dev(A), dev(B), dev(G), dev(m), use_mass, torch.float32, ctx=ctx)
    assert torch.equal(fa, ga.float()) and torch.equal(fb, gb.float())
    assert torch.isfinite(ga).all() and torch.isfinite(gb).all()
    if n == 3:  # a plane: the two methods' rotations agree to ~1e-8 only
        return
    i, j = FA - 1, FB - 1
    ei, ej = np.zeros((n, 3)), np.zeros((n, 3))
    for q in range(FB):
        ei += G[i, q] * oracle_target_grad(oracle, A[i].astype(np.float64),
                                           B[q].astype(np.float64), m, use_mass)[1]
    for q in range(FA):
        ej += G[q, j] * oracle_target_grad(oracle, B[j].astype(np.float64),
                                           A[q].astype(np.float64), m, use_mass)[1]
    assert np.abs(ga[i].cpu().numpy() - ei).max() <= 1e-9 * np.abs(ei).max()
    assert np.abs(gb[j].cpu().numpy() - ej).max() <= 1e-9 * np.abs(ej).max()


@pytest.mark.parametrize("F,n", [(2359, 1000), (2360, 1000), (18431, 128), (18433, 128), (18433, 131)])
def test_fit_backward_either_side_of_the_fp64_line(ctx, F, n):
    """FP64 gradients of 9 * 2^18 atoms and more leave the one-launch form (beyond
    128 atoms a frame): both sides of that line against the selection's kernels."""
    import ctypes as C
    import torch
    import cpptraj_amd as ca
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    base = torch.randn((1, n, 3), generator=g, device="cuda") * 10
    X = base + torch.randn((F, n, 3), generator=g, device="cuda")
    m = dev(synth.masses(np.random.default_rng(n), n))
    gr = torch.linspace(-1.0, 2.0, F, dtype=torch.float64, device="cuda")
    out = []
    for sel in (None, torch.arange(n, dtype=torch.int32, device="cuda")):
        d, r = ca.frames_desc(X, sel, m), ca.frames_desc(base, sel, m)
        out.append(torch.full((F, n, 3), 9.0, dtype=torch.float64, device="cuda"))
        ctx.check(ctx._L.rmsd_fit_backward(ctx.handle, C.byref(d), C.byref(r), 0, 1,
                                           C.c_void_p(gr.data_ptr()),
                                           C.c_void_p(out[-1].data_ptr())))
    assert float((out[0] - out[1]).abs().max()) <= 1e-9 * float(out[1].abs().max())


@pytest.mark.parametrize("use_mass", [0, 1])
@pytest.mark.parametrize("n", [50, 64, 66, 128, 131, 200, 255, 256])
def test_fit_backward_several_frames_per_wave(ctx, n, use_mass):
    """From 16,384 frames on a wave takes 8, 4 or 2 small frames: the bits of the
    same frames in calls below that (FP64 as far as the larger call stays in the
    one-launch form)."""
    import ctypes as C
    import torch
    import cpptraj_amd as ca
    F = 16384 + 5
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    base = torch.randn((1, n, 3), generator=g, device="cuda") * 10
    X = base + torch.randn((F, n, 3), generator=g, device="cuda")
    m = dev(synth.masses(np.random.default_rng(n), n))
    gr = torch.linspace(-1.0, 2.0, F, dtype=torch.float64, device="cuda")
    for fn, dt in ((ctx._L.rmsd_fit_backward_f32, torch.float32),
                   (ctx._L.rmsd_fit_backward, torch.float64)):
        if dt == torch.float64 and n > 131:
            continue

        def grad(s):
            x, q = X[s], gr[s]
            d, r = ca.frames_desc(x, None, m), ca.frames_desc(base, None, m)
            out = torch.full((len(x), n, 3), 9.0, dtype=dt, device="cuda")
            ctx.check(fn(ctx.handle, C.byref(d), C.byref(r), 0, use_mass,
                         C.c_void_p(q.data_ptr()), C.c_void_p(out.data_ptr())))
            return out
        whole = grad(slice(0, F))
        for s in (slice(0, 9000), slice(9000, F)):
            assert torch.equal(whole[s], grad(s))
