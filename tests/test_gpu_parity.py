"""GPU parity: the HIP library (through the C ABI) against the CPU oracle on the same
seeded inputs.  Bar: relative L2 <= 1e-12 for FP64 fields and particle values, bit-exact
for remesh node indices and particle counts."""
import numpy as np
import pytest

from vpm_free_amd import cases

pytestmark = pytest.mark.gpu

TOL = 1e-12
BOUNDSUM = {"spectral": 2, "lattice": 0, "direct": 1}


def rel_l2(a, b):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    nb = np.linalg.norm(b.ravel())
    return np.linalg.norm((a - b).ravel()) / (nb if nb > 0 else 1.0)


def say(*a):
    print(*a, flush=True)


@pytest.fixture(scope="module")
def ctx(vpmlib):
    V = vpmlib
    p = V.Params.make(0.125)
    c = V.VPM(p)
    yield c
    c.close()


def test_solve_zero_bc(ctx, oracle):
    rng = np.random.default_rng(1)
    nn = np.array([21, 18, 25], np.int32)
    xb = np.array([-1.0, -0.5, -0.7, 0, 0, 0])
    dpm = np.array([0.1, 0.07, 0.09])
    rhs = rng.standard_normal((nn[2], nn[1], nn[0], 3))
    win = np.array([1, 1, 1, nn[0], nn[1], nn[2]], np.int32)
    say("case: solve zero-bc", nn.tolist())
    ref = oracle.solve_window(xb, dpm, nn, win, rhs, zero_bc=True)
    got = ctx.stage_solve(xb, dpm, nn, 3, win, rhs, zero_bc=True)
    assert rel_l2(got, ref) <= TOL


def test_solve_window_bc(ctx, oracle):
    rng = np.random.default_rng(2)
    nn = np.array([30, 27, 24], np.int32)
    xb = np.array([-1.0, -0.5, -0.7, 0, 0, 0])
    dpm = np.array([0.05, 0.06, 0.07])
    rhs = rng.standard_normal((nn[2], nn[1], nn[0], 3))
    sol = rng.standard_normal((nn[2], nn[1], nn[0], 3))
    win = np.array([4, 3, 5, 26, 25, 20], np.int32)
    say("case: solve window bc", win.tolist())
    ref = oracle.solve_window(xb, dpm, nn, win, rhs, sol=sol)
    got = ctx.stage_solve(xb, dpm, nn, 3, win, rhs, sol=sol)
    assert rel_l2(got, ref) <= TOL


def _blob_rhs(nn, xb, dpm, centre=(0.1, -0.05, 0.02), s=0.15):
    x = xb[0] + np.arange(nn[0]) * dpm[0]
    y = xb[1] + np.arange(nn[1]) * dpm[1]
    z = xb[2] + np.arange(nn[2]) * dpm[2]
    Z, Y, X = np.meshgrid(z, y, x, indexing="ij")
    r2 = (X - centre[0]) ** 2 + (Y - centre[1]) ** 2 + (Z - centre[2]) ** 2
    g = np.exp(-r2 / s ** 2)
    return np.stack([g, -0.5 * g * X, 0.3 * g * Y], axis=-1)


def test_pmesh_inf(ctx, oracle):
    nn = np.array([33, 29, 31], np.int32)
    dpm = np.array([1 / 16, 1 / 16, 1 / 16])
    xb = np.array([-1.0, -0.875, -0.9375, 0, 0, 0])
    rhs = _blob_rhs(nn, xb, dpm)
    sol = np.zeros_like(rhs)
    say("case: pmesh_inf", nn.tolist())
    ref = oracle.pmesh_inf(xb, dpm, nn, rhs, sol)
    got = ctx.stage_pmesh_inf(xb, dpm, nn, rhs, sol)
    assert rel_l2(got, ref) <= TOL


@pytest.mark.parametrize("itype", [4, 2, 3, 5, 6])
def test_project(ctx, oracle, itype):
    """project_particles_3D + project_vol3d with every projection function of
    projection_fun (pmproject.f90:391-431): itype 4 takes the node-tile kernel, the others
    the one-thread-per-node gather."""
    rng = np.random.default_rng(3)
    nn = np.array([24, 20, 22], np.int32)
    dpm = np.array([0.1, 0.1, 0.1])
    xb = np.array([-1.0, -1.0, -1.0, 0, 0, 0])
    n = 5000
    xp = np.stack([rng.uniform(-0.8, 1.2, n), rng.uniform(-0.8, 0.8, n), rng.uniform(-0.8, 1.0, n)], axis=1)
    qp = np.concatenate([rng.standard_normal((n, 3)), np.full((n, 1), 1e-3)], axis=1)
    nnb = np.array([1, 1, 1, nn[0], nn[1], nn[2]], np.int32)
    say("case: project", n, "itype", itype)
    ref = oracle.project(xb, dpm, nn, nnb, xp, qp, itype=itype)
    got = ctx.stage_project(xb, dpm, nn, nnb, xp, qp, itype=itype)
    assert np.linalg.norm(ref) > 0
    assert rel_l2(got, ref) <= TOL


def _ring_case(h, sigma):
    xp, qp = cases.single_ring(h=h, sigma=sigma)
    return xp, qp


@pytest.mark.parametrize("h,sigma", [(0.125, 0.2), (1 / 16, 0.1)])
def test_vpm_mode2_ring(vpmlib, oracle, h, sigma):
    V = vpmlib
    xp, qp = _ring_case(h, sigma)
    say("case: vpm mode 2 ring h=%g sigma=%g n=%d" % (h, sigma, xp.shape[0]))
    po = oracle.Params.make(h)
    go = oracle.define_sizes(po, xp)
    up_r, gp_r, f = oracle.vpm2(po, go, xp, qp, fields=True)
    with V.VPM(V.Params.make(h)) as c:
        up, gp = np.zeros_like(xp), np.zeros_like(xp)
        c.vpm(xp, qp, up, gp, xp.shape[0], 3, 0, 0)
        assert bytes(c.geometry)[: 8 * 9 + 4 * 9] == bytes(go)[: 8 * 9 + 4 * 9]
        c.vpm(xp, qp, up, gp, xp.shape[0], 3, 2, 1)
        errs = {
            "rhs": rel_l2(c.get_grid(0), f["rhs"]),
            "psi": rel_l2(c.get_grid(1), f["psi"]),
            "vel": rel_l2(c.get_grid(3), f["vel"]),
            "sol": rel_l2(c.get_grid(2), f["sol"]),
            "up": rel_l2(up, up_r),
            "gp": rel_l2(gp, gp_r),
        }
    say("  rel L2:", errs)
    for k, v in errs.items():
        assert v <= TOL, (k, v)


@pytest.mark.parametrize("h,sigma,tree", [(0.125, 0.2, 0), (1 / 16, 0.1, 0), (1 / 16, 0.1, 1)])
@pytest.mark.parametrize("prec", [0, 1])
def test_vpm_mode2_spectral_shortcuts(vpmlib, oracle, h, sigma, tree, prec):
    """vpm(2) with both spectral shortcuts of the fine solves forced on small blocks (they are
    taken by default from 150^3 nodes): the zero-BC solve's normal derivatives from its spectrum
    (face_derivs = 1), and the second solve evaluated only on the inner box's faces and at the
    coarse samples (fine_partial = 1) -- the nodes yaps reads.  Every grid, UP and GP against the
    oracle at 1e-12 in FP64, at the mixed form's 1e-5 in the mixed form."""
    V = vpmlib
    xp, qp = _ring_case(h, sigma)
    say("case: vpm mode 2 spectral shortcuts h=%g tree=%d precision %d n=%d" % (h, tree, prec, xp.shape[0]))
    po = oracle.Params.make(h, iyntree=tree, ilevmax=3)
    go = oracle.define_sizes(po, xp)
    up_r, gp_r, f = oracle.vpm2(po, go, xp, qp, fields=True)
    out = {}
    for on in (1, 0):
        with V.VPM(V.Params.make(h, iyntree=tree, ilevmax=3)) as c:
            c.set_option("face_derivs", on)
            c.set_option("fine_partial", on)
            c.set_precision(prec)
            up, gp = np.zeros_like(xp), np.zeros_like(xp)
            c.vpm(xp, qp, up, gp, xp.shape[0], 3, 0, 0)
            c.vpm(xp, qp, up, gp, xp.shape[0], 3, 2, 1)
            out[on] = {"psi": c.get_grid(1), "vel": c.get_grid(3), "sol": c.get_grid(2), "up": up.copy(),
                       "gp": gp.copy()}
    ref = {"psi": f["psi"], "vel": f["vel"], "sol": f["sol"], "up": up_r, "gp": gp_r}
    errs = {k: rel_l2(out[1][k], ref[k]) for k in ref}
    say("  rel L2 vs oracle:", errs)
    if prec == 0:
        for k, v in errs.items():
            assert v <= TOL, (k, v)
    else:
        say("  (without them:", {k: rel_l2(out[0][k], ref[k]) for k in ref}, ")")
        for k, v in errs.items():
            assert v <= 1e-5, (k, v)


def test_remesh_exact(vpmlib, oracle):
    V = vpmlib
    h = 0.125
    xp, qp = _ring_case(h, 0.2)
    rng = np.random.default_rng(5)
    xp = xp + rng.uniform(-0.3, 0.3, xp.shape) * h  # off-node positions
    say("case: remesh n=%d" % xp.shape[0])
    po = oracle.Params.make(h)
    go = oracle.define_sizes(po, xp)
    xr, qr = oracle.remesh(po, go, xp, qp)
    with V.VPM(V.Params.make(h)) as c:
        c.vpm(xp, qp, None, None, xp.shape[0], 3, 0, 0)
        xg, qg = c.remesh_particles_3d(xp, qp, mrem=1)
    assert xg.shape == xr.shape
    assert np.array_equal(xg, xr)  # node positions bit-exact, k->j->i order
    assert rel_l2(qg, qr) <= TOL


def test_rk2_step_and_diagnostics(vpmlib, oracle):
    V = vpmlib
    h = 0.125
    xp, qp = _ring_case(h, 0.2)
    say("case: rk2 step n=%d" % xp.shape[0])
    po = oracle.Params.make(h)
    go = oracle.define_sizes(po, xp)
    x1, q1 = oracle.step_rk2(po, go, xp, qp, 0.01, ntime=1)
    with V.VPM(V.Params.make(h)) as c:
        c.upload(xp, qp)
        c.vpm_resident(0, 0)
        c.step_rk2(0.01, ntime=1)
        xg, qg, _, _ = c.download()
        circ, imp = c.diagnostics()
    assert xg.shape == x1.shape
    assert np.array_equal(xg, x1)
    assert rel_l2(qg, q1) <= TOL
    circ_r, imp_r = oracle.diagnostics(x1, q1)
    assert np.allclose(circ, circ_r, rtol=0, atol=1e-13)
    assert rel_l2(imp, imp_r) <= 1e-12


@pytest.mark.parametrize("nn", [(35, 23, 27), (38, 12, 20), (47, 45, 13)])
def test_solve_all_radix_classes(ctx, oracle, nn):
    """Lengths m + 1 with prime factors 17, 11, 13, 37, 5, 23 and 3: matrix products over whole planes,
    which do not depend on them."""
    rng = np.random.default_rng(sum(nn))
    nn = np.array(nn, np.int32)
    xb = np.array([0.3, -0.2, 0.1, 0, 0, 0])
    dpm = np.array([0.05, 0.04, 0.06])
    rhs = rng.standard_normal((nn[2], nn[1], nn[0], 3))
    sol = rng.standard_normal((nn[2], nn[1], nn[0], 3))
    win = np.array([1, 1, 1, nn[0], nn[1], nn[2]], np.int32)
    say("case: solve radix classes", nn.tolist())
    ref = oracle.solve_window(xb, dpm, nn, win, rhs, sol=sol)
    got = ctx.stage_solve(xb, dpm, nn, 3, win, rhs, sol=sol)
    assert rel_l2(got, ref) <= TOL


# lines that still take an FFT, by their largest radix: FP64 lines above the products' 367 points
# (4: 384, 512; 7: 375, 392; 17: 374, 390; 37: 370, 391; above 37: 376, 410, 427), FP32 lines above 208
# points without larger factors (4: 243, 256; 7: 245, 280; 17: 242, 255, 264, 286, and the compile-time
# plans of 272 and 288)
FFT64 = [384, 512, 375, 392, 374, 390, 370, 391, 376, 410, 427]
FFT32 = [243, 256, 245, 280, 242, 255, 264, 286, 272, 288]


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("length,prec", [(n, 0) for n in FFT64] + [(n, 1) for n in FFT32])
def test_solve_fft_lines(ctx, oracle, length, prec, axis):
    """One long axis of m = length - 1 points, Dirichlet values on all faces: FP64 within 1e-12 of the
    oracle, the mixed form (five FP32 passes) within 1e-6."""
    rng = np.random.default_rng(length + axis)
    nn = np.array([9, 12, 10], np.int32)
    nn[axis] = length + 1
    xb = np.array([0.3, -0.2, 0.1, 0, 0, 0])
    dpm = np.array([0.05, 0.04, 0.06])
    rhs = rng.standard_normal((nn[2], nn[1], nn[0], 3))
    sol = rng.standard_normal((nn[2], nn[1], nn[0], 3))
    win = np.array([1, 1, 1, nn[0], nn[1], nn[2]], np.int32)
    say("case: solve FFT lines", nn.tolist(), "precision", prec)
    ref = oracle.solve_window(xb, dpm, nn, win, rhs, sol=sol)
    try:
        ctx.set_precision(prec)
        got = ctx.stage_solve(xb, dpm, nn, 3, win, rhs, sol=sol)
    finally:
        ctx.set_precision(0)
    assert rel_l2(got, ref) <= (TOL if prec == 0 else 1e-6)


def _lap7(u, h):
    """7-point Laplacian at the interior nodes of u (nz, ny, nx)."""
    c = u[1:-1, 1:-1, 1:-1]
    return ((u[1:-1, 1:-1, 2:] - 2 * c + u[1:-1, 1:-1, :-2]) / h[0] ** 2 +
            (u[1:-1, 2:, 1:-1] - 2 * c + u[1:-1, :-2, 1:-1]) / h[1] ** 2 +
            (u[2:, 1:-1, 1:-1] - 2 * c + u[:-2, 1:-1, 1:-1]) / h[2] ** 2)


@pytest.mark.parametrize("n", [289, 273, 161, 145])
def test_solve_full_size_plans(ctx, n):
    """The block sizes of the 256-cubed and 128-cubed workloads -- sizes the oracle is too slow for:
    289 with the compile-time FFT plans of both forms (FP64 288 = 4.4.2.9 or 8.4.9, FP32 576 =
    4.4.4.9, 8.8.9 or 16.4.9; padded LDS sequences, register-capped kernels, as the tuner picks
    them), 273 with FP64 products and the FP32 plans of 544 = 17.4.4.2 or 17.8.4, 161 and 145 with
    products in both forms.  The FP64 solution satisfies the 7-point equations to rounding, and the
    mixed form agrees with it to FP32 accuracy."""
    rng = np.random.default_rng(n)
    nn = np.array([n, n, n], np.int32)
    h = np.array([1 / 64] * 3)
    xb = np.array([-2.0, -2.0, -2.0, 0, 0, 0])
    rhs = rng.standard_normal((n, n, n, 3))
    sol = rng.standard_normal((n, n, n, 3))
    win = np.array([1, 1, 1, n, n, n], np.int32)
    say("case: full-size solve", n)
    try:
        ctx.set_precision(0)
        u = ctx.stage_solve(xb, h, nn, 3, win, rhs, sol=sol)
        ctx.set_precision(1)
        um = ctx.stage_solve(xb, h, nn, 3, win, rhs, sol=sol)
    finally:
        ctx.set_precision(0)
    for c in range(3):
        res = _lap7(u[..., c], h) - rhs[1:-1, 1:-1, 1:-1, c]
        assert np.abs(res).max() < 1e-8 * np.abs(rhs).max(), c
    assert rel_l2(um, u) < 1e-6


@pytest.mark.parametrize("mode", ["spectral", "lattice", "direct"])
def test_boundary_sum_forms(vpmlib, oracle, mode):
    """The three evaluations of the fine boundary sums (spectral convolution + batched
    products, lattice 1/r tables, direct LDS source tiles) against the oracle's direct sum,
    on a non-cubic block (every face pair has its own geometry)."""
    V = vpmlib
    nn = np.array([65, 57, 49], np.int32)
    dpm = np.array([1 / 32, 1 / 30, 1 / 28])
    xb = np.array([-1.0, -0.95, -0.85, 0, 0, 0])
    rhs = _blob_rhs(nn, xb, dpm, centre=(0.02, -0.03, 0.01), s=0.25)
    sol = np.zeros_like(rhs)
    say("case: boundary sums", mode, nn.tolist())
    ref = oracle.pmesh_inf(xb, dpm, nn, rhs, sol)
    with V.VPM(V.Params.make(0.125)) as c:
        c.set_option("boundsum", BOUNDSUM[mode])
        got = c.stage_pmesh_inf(xb, dpm, nn, rhs, sol)
    assert rel_l2(got, ref) <= TOL


@pytest.mark.parametrize("nn,levmax", [((65, 57, 49), 3), ((43, 43, 43), 2), ((33, 29, 31), 3)])
def test_boundary_sum_tree(vpmlib, oracle, nn, levmax):
    """Tree form of pmesh's boundary sums (pm.inp tree = 1) against the oracle's tree:
    faces of whole groups; dummy rows and columns with the corner cell the links leave
    out; faces whose finer rows hold two cells beyond the whole groups (shifted links)."""
    V = vpmlib
    nn = np.array(nn, np.int32)
    dpm = np.array([1 / 32, 1 / 30, 1 / 28])
    xb = np.array([-1.0, -0.95, -0.85, 0, 0, 0])
    rhs = _blob_rhs(nn, xb, dpm, centre=(0.02, -0.03, 0.01), s=0.25)
    sol = np.zeros_like(rhs)
    say("case: tree boundary sums", nn.tolist(), "levmax", levmax)
    try:
        oracle.set_tree(levmax)
        ref = oracle.pmesh_inf(xb, dpm, nn, rhs, sol)
    finally:
        oracle.set_tree(-1)
    direct = oracle.pmesh_inf(xb, dpm, nn, rhs, sol)
    with V.VPM(V.Params.make(0.125)) as c:
        got = c.stage_pmesh_inf(xb, dpm, nn, rhs, sol, itree=1, levmax=levmax)
    err = rel_l2(got, ref)
    say("  rel L2 vs oracle tree %.2e (tree vs direct %.2e)" % (err, rel_l2(ref, direct)))
    assert rel_l2(ref, direct) > 1e3 * TOL  # the tree's sums are not the direct ones
    assert err <= TOL


@pytest.mark.parametrize("nn,levmax,h", [((65, 57, 49), 3, 1 / 32), ((49, 65, 57), 2, 1 / 32), ((65, 57, 49), 3, 0.1),
                                         ((57, 49, 65), 2, 0.3), ((33, 33, 33), 4, 1 / 32), ((17, 25, 33), 3, 1 / 32)])
def test_boundary_sum_tree_ties(vpmlib, oracle, nn, levmax, h):
    """Equal spacings: many targets lie at r = 10 sqrt(DS) of a group, exactly where the spacing is a
    power of two and to rounding where it is not, and r < 10 sqrt(DS) decides which terms are taken (the
    other choice changes the sums by 5e-7 to 2e-6).  24 trees in the smallest two: parts of one and of two."""
    V = vpmlib
    nn = np.array(nn, np.int32)
    dpm = np.full(3, h)
    xb = np.array([*(-h * np.array([24.0, 17.0, 20.0])), 0, 0, 0])
    c0 = xb[:3] + (nn - 1) * h / 2
    rhs = _blob_rhs(nn, xb, dpm, centre=tuple(c0 + h), s=8 * h)
    sol = np.zeros_like(rhs)
    say("case: tree boundary sums on ties", nn.tolist(), "levmax", levmax, "h", h)
    try:
        oracle.set_tree(levmax)
        ref = oracle.pmesh_inf(xb, dpm, nn, rhs, sol)
    finally:
        oracle.set_tree(-1)
    with V.VPM(V.Params.make(0.125)) as c:
        got = c.stage_pmesh_inf(xb, dpm, nn, rhs, sol, itree=1, levmax=levmax)
    assert rel_l2(got, ref) <= TOL


@pytest.mark.parametrize("h,sigma", [(0.125, 0.2), (1 / 16, 0.1)])
def test_vpm_mode2_tree(vpmlib, oracle, h, sigma):
    """vpm(2) with the shipped pm.inp tree settings (tree = 1, 3 levels): the block solve
    takes ilevmax levels, the coarse solve ilevmax - 1 (yaps3d.f90:46-48, 286-292)."""
    V = vpmlib
    xp, qp = _ring_case(h, sigma)
    say("case: vpm mode 2 tree h=%g n=%d" % (h, xp.shape[0]))
    po = oracle.Params.make(h, iyntree=1, ilevmax=3)
    go = oracle.define_sizes(po, xp)
    up_r, gp_r, f = oracle.vpm2(po, go, xp, qp, fields=True)
    with V.VPM(V.Params.make(h, iyntree=1, ilevmax=3)) as c:
        up, gp = np.zeros_like(xp), np.zeros_like(xp)
        c.vpm(xp, qp, up, gp, xp.shape[0], 3, 0, 0)
        c.vpm(xp, qp, up, gp, xp.shape[0], 3, 2, 1)
        errs = {"sol": rel_l2(c.get_grid(2), f["sol"]), "up": rel_l2(up, up_r), "gp": rel_l2(gp, gp_r)}
    say("  rel L2:", errs)
    for k, v in errs.items():
        assert v <= TOL, (k, v)


@pytest.mark.parametrize("nn,itree,levmax,origin", [((33, 29, 31), 0, 1, False), ((65, 57, 49), 0, 1, False),
                                                     ((65, 57, 49), 1, 3, False), ((43, 43, 43), 1, 2, True),
                                                     ((33, 29, 31), 1, 3, False)])
def test_boundary_sum_panels(vpmlib, oracle, nn, itree, levmax, origin):
    """Constant-source panel sums (pm.inp ibctyp = 3, FSOUR_A4 in the target plane's frame)
    against the oracle: direct form (point-source sum + near-field panel corrections) and
    tree form (tree_calc_3d_s, with its top-level cells weighted by the first cell's source;
    with `origin` the box holds the origin, where the reference's top-level dummies sit)."""
    V = vpmlib
    nn = np.array(nn, np.int32)
    dpm = np.array([1 / 32, 1 / 30, 1 / 28])
    if origin:
        xb = np.array([-(nn[0] - 1) * dpm[0] / 2, -(nn[1] - 1) * dpm[1] / 2 + 0.01, -0.3, 0, 0, 0])
    else:
        xb = np.array([-1.0, -0.95, -0.85, 0, 0, 0])
    c0 = xb[:3] + (nn - 1) * dpm / 2
    rhs = _blob_rhs(nn, xb, dpm, centre=tuple(c0 + np.array([0.02, -0.03, 0.01])), s=0.25)
    sol = np.zeros_like(rhs)
    say("case: panel boundary sums", nn.tolist(), "itree", itree, "levmax", levmax, "origin", origin)
    try:
        oracle.set_ibctyp(3)
        oracle.set_tree(levmax if itree else -1)
        ref = oracle.pmesh_inf(xb, dpm, nn, rhs, sol)
    finally:
        oracle.set_ibctyp(2)
        oracle.set_tree(-1)
    point = oracle.pmesh_inf(xb, dpm, nn, rhs, sol)
    with V.VPM(V.Params.make(0.125)) as c:
        got = c.stage_pmesh_inf(xb, dpm, nn, rhs, sol, itree=itree, levmax=levmax, ibctyp=3)
    err = rel_l2(got, ref)
    say("  rel L2 vs oracle %.2e (panels vs points %.2e)" % (err, rel_l2(ref, point)))
    assert rel_l2(ref, point) > 1e3 * TOL
    assert err <= TOL


@pytest.mark.parametrize("h,sigma,tree", [(0.125, 0.2, 0), (0.125, 0.2, 1), (1 / 16, 0.1, 1)])
def test_vpm_mode2_panels(vpmlib, oracle, h, sigma, tree):
    """vpm(2) with pm.inp ibctyp = 3 (direct and tree forms) against the oracle."""
    V = vpmlib
    xp, qp = _ring_case(h, sigma)
    say("case: vpm mode 2 panels h=%g tree=%d n=%d" % (h, tree, xp.shape[0]))
    po = oracle.Params.make(h, ibctyp=3, iyntree=tree, ilevmax=3)
    go = oracle.define_sizes(po, xp)
    up_r, gp_r, f = oracle.vpm2(po, go, xp, qp, fields=True)
    with V.VPM(V.Params.make(h, ibctyp=3, iyntree=tree, ilevmax=3)) as c:
        up, gp = np.zeros_like(xp), np.zeros_like(xp)
        c.vpm(xp, qp, up, gp, xp.shape[0], 3, 0, 0)
        c.vpm(xp, qp, up, gp, xp.shape[0], 3, 2, 1)
        errs = {"sol": rel_l2(c.get_grid(2), f["sol"]), "up": rel_l2(up, up_r), "gp": rel_l2(gp, gp_r)}
    say("  rel L2:", errs)
    for k, v in errs.items():
        assert v <= TOL, (k, v)


@pytest.mark.parametrize("h,sigma,blocks,tree,ibctyp", [
    (0.125, 0.2, (2, 1, 1), 0, 2), (0.125, 0.2, (1, 2, 1), 0, 2), (0.125, 0.2, (2, 2, 2), 0, 2),
    (0.125, 0.2, (3, 2, 1), 1, 2), (0.125, 0.2, (2, 1, 2), 0, 3), (1 / 16, 0.1, (6, 1, 1), 1, 2)])
@pytest.mark.parametrize("shortcuts", [0, 1])
def test_vpm_mode2_blocks(vpmlib, oracle, h, sigma, blocks, tree, ibctyp, shortcuts):
    """vpm(2) with NBI x NBJ x NBK yaps blocks on one device (rhsscat_3d, every block's fine
    solve, the coarse problem from all blocks' samples, interp_stencil with the neighbours'
    fine solutions, solget_3d) against the oracle; (6, 1, 1) with tree = 1, 3 levels is the
    shipped pm.inp's combination.  `shortcuts`: the spectral normal derivatives and the
    selected-node second solve forced on (several blocks keep every node of the second solve,
    as the neighbours read it)."""
    V = vpmlib
    xp, qp = _ring_case(h, sigma)
    say("case: vpm mode 2 blocks %s h=%g tree=%d ibctyp=%d n=%d" % (blocks, h, tree, ibctyp, xp.shape[0]))
    kw = dict(blocks=blocks, iyntree=tree, ilevmax=3, ibctyp=ibctyp)
    po = oracle.Params.make(h, **kw)
    go = oracle.define_sizes(po, xp)
    up_r, gp_r, f = oracle.vpm2(po, go, xp, qp, fields=True)
    with V.VPM(V.Params.make(h, **kw)) as c:
        c.set_option("face_derivs", shortcuts)
        c.set_option("fine_partial", shortcuts)
        up, gp = np.zeros_like(xp), np.zeros_like(xp)
        c.vpm(xp, qp, up, gp, xp.shape[0], 3, 0, 0)
        assert bytes(c.geometry) == bytes(go)
        c.vpm(xp, qp, up, gp, xp.shape[0], 3, 2, 1)
        errs = {
            "rhs": rel_l2(c.get_grid(0), f["rhs"]),
            "psi": rel_l2(c.get_grid(1), f["psi"]),
            "vel": rel_l2(c.get_grid(3), f["vel"]),
            "sol": rel_l2(c.get_grid(2), f["sol"]),
            "up": rel_l2(up, up_r),
            "gp": rel_l2(gp, gp_r),
        }
    say("  rel L2:", errs)
    for k, v in errs.items():
        assert v <= TOL, (k, v)


@pytest.mark.parametrize("nn", [(145, 40, 44), (289, 21, 19)])
def test_solve_many_batches(ctx, oracle, nn):
    """Windows with more line batches than resident work-groups (every work-group loops
    over several batches) and x lines long enough that a thread pre-processes several
    slot pairs; Dirichlet values on all faces."""
    rng = np.random.default_rng(sum(nn) + 7)
    nn = np.array(nn, np.int32)
    xb = np.array([-0.4, 0.2, -0.1, 0, 0, 0])
    dpm = np.array([1 / 64, 1 / 50, 1 / 40])
    rhs = rng.standard_normal((nn[2], nn[1], nn[0], 3))
    sol = rng.standard_normal((nn[2], nn[1], nn[0], 3))
    win = np.array([1, 1, 1, nn[0], nn[1], nn[2]], np.int32)
    say("case: solve many batches", nn.tolist())
    ref = oracle.solve_window(xb, dpm, nn, win, rhs, sol=sol)
    got = ctx.stage_solve(xb, dpm, nn, 3, win, rhs, sol=sol)
    assert rel_l2(got, ref) <= TOL


MIXED_TOL = 1e-5


@pytest.mark.parametrize("h,sigma", [(1 / 16, 0.1)])
def test_vpm_mode2_mixed(vpmlib, oracle, h, sigma):
    """Mixed form (FP32 Poisson passes, FP64 boundary sums) against the FP64 oracle: every
    field and the particle velocities within relative L2 1e-5."""
    V = vpmlib
    xp, qp = _ring_case(h, sigma)
    say("case: vpm mode 2 mixed ring h=%g sigma=%g n=%d" % (h, sigma, xp.shape[0]))
    po = oracle.Params.make(h)
    go = oracle.define_sizes(po, xp)
    up_r, gp_r, f = oracle.vpm2(po, go, xp, qp, fields=True)
    with V.VPM(V.Params.make(h)) as c:
        c.set_precision(1)
        up, gp = np.zeros_like(xp), np.zeros_like(xp)
        c.vpm(xp, qp, up, gp, xp.shape[0], 3, 0, 0)
        c.vpm(xp, qp, up, gp, xp.shape[0], 3, 2, 1)
        errs = {
            "psi": rel_l2(c.get_grid(1), f["psi"]),
            "vel": rel_l2(c.get_grid(3), f["vel"]),
            "sol": rel_l2(c.get_grid(2), f["sol"]),
            "up": rel_l2(up, up_r),
            "gp": rel_l2(gp, gp_r),
        }
    say("  rel L2 vs FP64:", errs)
    for k, v in errs.items():
        assert v <= MIXED_TOL, (k, v)
    assert errs["up"] > 0.0  # the FP32 passes ran


def test_vpm_modes_4_and_5(vpmlib, oracle):
    """WhatToDo 4 (stretching from the velocity grids of a preceding mode-1 call, then
    interpolation) and 5 (diffusion -NI lap(w), UP = 0, GP interpolated) against the oracle."""
    V = vpmlib
    h = 0.125
    xp, qp = _ring_case(h, 0.2)
    rng = np.random.default_rng(11)
    xm = xp + rng.uniform(-0.2, 0.2, xp.shape) * h  # particles moved after the mode-1 call
    po = oracle.Params.make(h)
    go = oracle.define_sizes(po, xp)
    _, _, f = oracle.vpm2(po, go, xp, qp, fields=True)
    up4_r, gp4_r, _ = oracle.vpm45(po, go, xm, qp, 4, vel=f["vel"])
    up5_r, gp5_r, _ = oracle.vpm45(po, go, xm, qp, 5, ni=0.02)
    say("case: vpm modes 4 and 5, n=%d" % xp.shape[0])
    with V.VPM(V.Params.make(h)) as c:
        up, gp = np.zeros_like(xp), np.zeros_like(xp)
        c.vpm(xp, qp, up, gp, xp.shape[0], 3, 0, 0)
        c.vpm(xp, qp, up, gp, xp.shape[0], 3, 1, 1)
        up4, gp4 = np.full_like(xp, 7.0), np.full_like(xp, 7.0)
        c.vpm(xm, qp, up4, gp4, xm.shape[0], 3, 4, 1)
        up5, gp5 = np.full_like(xp, 7.0), np.full_like(xp, 7.0)
        c.vpm(xm, qp, up5, gp5, xm.shape[0], 3, 5, 1, NI=0.02)
    errs = {"up4": rel_l2(up4, up4_r), "gp4": rel_l2(gp4, gp4_r), "gp5": rel_l2(gp5, gp5_r)}
    say("  rel L2:", errs)
    for k, v in errs.items():
        assert v <= TOL, (k, v)
    assert np.all(up5 == 0.0)


def test_boundary_sums_spectral_long_axis(vpmlib):
    """Spectral boundary sums on a block with one 289-node axis, where the transforms along
    that axis run the 576-point compile-time plan (one wave per sequence) and the others the
    runtime wave plans, against the direct LDS-tile sums (pinned to the oracle on smaller
    blocks); the oracle's direct sum is too slow at this size."""
    V = vpmlib
    nn = np.array([289, 33, 41], np.int32)
    dpm = np.array([1 / 64, 1 / 60, 1 / 56])
    xb = np.array([-2.25, -0.27, -0.36, 0, 0, 0])
    rhs = _blob_rhs(nn, xb, dpm, centre=(0.1, -0.01, 0.02), s=0.08)
    sol = np.zeros_like(rhs)
    say("case: spectral boundary sums, 289-node axis", nn.tolist())
    out = {}
    for mode in ("spectral", "direct"):
        with V.VPM(V.Params.make(0.125)) as c:
            c.set_option("boundsum", BOUNDSUM[mode])
            out[mode] = c.stage_pmesh_inf(xb, dpm, nn, rhs, sol)
    assert rel_l2(out["spectral"], out["direct"]) <= TOL


@pytest.mark.parametrize("prec,tol", [(0, TOL), (1, 2e-6)])
def test_pmesh_inf_reuse_full_size(vpmlib, prec, tol):
    """The second fine solve of pmesh_inf starts from the first one's x/y forward transforms
    less those of the folded Dirichlet values; at the 289-node block (compile-time plans, the
    spectral boundary sums' 576-point path) it must agree with the two full solves.  In the
    mixed form the two orders differ by FP32 rounding (measured 6e-7..1.0e-6 depending on how
    the transforms form their twiddle powers); a wrong fold or transform shows as 1e-3 or more."""
    V = vpmlib
    nn = np.array([289, 289, 289], np.int32)
    dpm = np.array([1 / 64] * 3)
    xb = np.array([-2.25, -2.25, -2.25, 0, 0, 0])
    rhs = _blob_rhs(nn, xb, dpm, centre=(0.1, -0.05, 0.02), s=0.3)
    sol = np.zeros_like(rhs)
    say("case: pmesh_inf forward-pass reuse, 289^3, precision", prec)
    out = {}
    for reuse in ("1", "0"):
        with V.VPM(V.Params.make(0.125)) as c:
            c.set_option("dst_reuse", int(reuse))
            c.set_precision(prec)
            out[reuse] = c.stage_pmesh_inf(xb, dpm, nn, rhs, sol)
    assert rel_l2(out["1"], out["0"]) <= tol


@pytest.mark.parametrize("nn", [(251, 91, 161), (163, 251, 91), (95, 161, 243)])
@pytest.mark.parametrize("prec,tol", [(0, TOL), (1, 2e-6)])
def test_pmesh_inf_reuse_unequal(vpmlib, nn, prec, tol):
    """The same on boxes above the size from which the transforms are kept, with three extents and
    three spacings, short and long spans of rows in the correction, and, in the mixed form, FP32 lines
    of products beside FFT lines on each axis."""
    V = vpmlib
    nn = np.array(nn, np.int32)
    dpm = np.array([1 / 64, 1 / 51, 1 / 43])
    xb = np.array([-1.1, -0.9, -1.3, 0, 0, 0])
    c0 = xb[:3] + (nn - 1) * dpm / 2
    rhs = _blob_rhs(nn, xb, dpm, centre=tuple(c0 + 0.02), s=0.25 * float(np.min((nn - 1) * dpm)))
    sol = np.zeros_like(rhs)
    say("case: pmesh_inf forward-pass reuse", nn.tolist(), "precision", prec)
    out = {}
    for reuse in (1, 0):
        with V.VPM(V.Params.make(0.125)) as c:
            c.set_option("dst_reuse", reuse)
            c.set_precision(prec)
            out[reuse] = c.stage_pmesh_inf(xb, dpm, nn, rhs, sol)
    assert rel_l2(out[1], out[0]) <= tol
    assert not np.array_equal(out[1], out[0])  # the correction ran


@pytest.mark.parametrize("nn,levmax,ibctyp", [((33, 29, 31), -1, 2), ((65, 57, 49), -1, 2), ((43, 43, 43), 2, 2),
                                               ((33, 29, 31), -1, 3)])
@pytest.mark.parametrize("prec", [0, 1])
def test_pmesh_inf_spectral_face_derivs(vpmlib, oracle, nn, levmax, ibctyp, prec):
    """pmesh with the zero-BC solve's normal derivatives taken from its sine spectrum after the
    z pass (option face_derivs = 1: face sums of the work array, then products with the sine
    matrices; no y and x inverse passes) against the oracle, which differentiates the solved
    field (calc_normalderiv_3d); point and panel sources, direct and tree sums.  FP64 at 1e-12;
    the mixed form's FP32 passes within 2e-6 (the derivatives themselves are FP64 sums here)."""
    V = vpmlib
    nn = np.array(nn, np.int32)
    dpm = np.array([1 / 32, 1 / 30, 1 / 28])
    xb = np.array([-1.0, -0.95, -0.85, 0, 0, 0])
    rhs = _blob_rhs(nn, xb, dpm, centre=(0.02, -0.03, 0.01), s=0.25)
    sol = np.zeros_like(rhs)
    say("case: spectral face derivatives", nn.tolist(), "levmax", levmax, "ibctyp", ibctyp, "precision", prec)
    try:
        oracle.set_ibctyp(ibctyp)
        oracle.set_tree(levmax)
        ref = oracle.pmesh_inf(xb, dpm, nn, rhs, sol)
    finally:
        oracle.set_ibctyp(2)
        oracle.set_tree(-1)
    out = {}
    for fd in (1, 0):
        with V.VPM(V.Params.make(0.125)) as c:
            c.set_option("face_derivs", fd)
            c.set_precision(prec)
            out[fd] = c.stage_pmesh_inf(xb, dpm, nn, rhs, sol, itree=int(levmax >= 0), levmax=max(levmax, 1),
                                        ibctyp=ibctyp)
    err, err0 = rel_l2(out[1], ref), rel_l2(out[0], ref)
    say("  rel L2 vs oracle: spectral %.2e, from the field %.2e" % (err, err0))
    assert err <= (TOL if prec == 0 else 2e-6)


def test_pmesh_inf_spectral_face_derivs_full_size(vpmlib):
    """The spectral normal derivatives at the 289-node block (work-array rows of 287 points padded
    to 288; the compile-time sine-transform plans): in FP64 against the stencil on the solved
    field at 1e-12; in the mixed form both against the FP64 result, where the spectral ones
    (FP64 sums of the FP32 spectrum) must stay within the mixed form's 1e-5 and no further off
    than the stencil on the FP32-solved field."""
    V = vpmlib
    nn = np.array([289, 289, 289], np.int32)
    dpm = np.array([1 / 64] * 3)
    xb = np.array([-2.25, -2.25, -2.25, 0, 0, 0])
    rhs = _blob_rhs(nn, xb, dpm, centre=(0.1, -0.05, 0.02), s=0.3)
    sol = np.zeros_like(rhs)
    say("case: spectral face derivatives, 289^3")
    out = {}
    for prec in (0, 1):
        for fd in (1, 0):
            with V.VPM(V.Params.make(0.125)) as c:
                c.set_option("face_derivs", fd)
                c.set_precision(prec)
                out[prec, fd] = c.stage_pmesh_inf(xb, dpm, nn, rhs, sol)
    e64 = rel_l2(out[0, 1], out[0, 0])
    e1, e0 = rel_l2(out[1, 1], out[0, 0]), rel_l2(out[1, 0], out[0, 0])
    say("  FP64 spectral vs field %.2e; mixed vs FP64: spectral %.2e, field %.2e" % (e64, e1, e0))
    assert e64 <= TOL
    assert e1 <= 1e-5
    assert e1 <= 1.05 * e0


def test_vpm_mode2_call_sequence_kept_zeros(vpmlib, oracle):
    """One single-block context, several vpm(2) calls at the geometry of the first one
    (idefine = 1): ring + blob; the same again (the block RHS keeps its zeros between calls
    and only tiles emptied since the last call are cleared); the ring alone (the blob's tiles
    empty and must be cleared); a mixed-form call; the ring + blob in FP64 again; the ring
    alone twice.  RHS grid, UP and GP against the oracle after every call."""
    V = vpmlib
    h = 1 / 16
    xr, qr = cases.single_ring(h=h, sigma=0.1)
    rng = np.random.default_rng(21)
    nb = 1500
    xb = rng.uniform(-0.3, 0.3, (nb, 3)) + np.array([0.3, -0.2, 1.1])
    qb = np.concatenate([rng.standard_normal((nb, 3)) * h ** 3, np.full((nb, 1), h ** 3)], axis=1)
    xa, qa = np.concatenate([xr, xb]), np.concatenate([qr, qb])
    po = oracle.Params.make(h)
    go = oracle.define_sizes(po, xa)
    ref = {}
    for name, (x, q) in {"a": (xa, qa), "r": (xr, qr)}.items():
        up_r, gp_r, f = oracle.vpm2(po, go, x, q, fields=True)
        ref[name] = (up_r, gp_r, f["rhs"])
    say("case: vpm(2) call sequence, ring %d + blob %d particles" % (xr.shape[0], nb))

    def check(c, name, x, q, tol=TOL):
        up, gp = np.zeros_like(x), np.zeros_like(x)
        c.vpm(x, q, up, gp, x.shape[0], 3, 2, 1)
        up_r, gp_r, rhs_r = ref[name]
        errs = {"rhs": rel_l2(c.get_grid(0), rhs_r), "up": rel_l2(up, up_r), "gp": rel_l2(gp, gp_r)}
        say("  call", name, errs)
        for k, v in errs.items():
            assert v <= tol, (name, k, v)

    with V.VPM(V.Params.make(h)) as c:
        c.vpm(xa, qa, None, None, xa.shape[0], 3, 0, 0)
        check(c, "a", xa, qa)
        check(c, "a", xa, qa)
        check(c, "r", xr, qr)
        c.set_precision(1)
        check(c, "a", xa, qa, tol=1e-5)
        c.set_precision(0)
        check(c, "a", xa, qa)
        check(c, "r", xr, qr)
        check(c, "r", xr, qr)


def test_tuner_choices_keep_results(vpmlib):
    """The autotuner picks kernel variants and persistent grid sizes by timing them; at h=1/16
    (products of 16 or 32 lines, stencil and matrix tiles) the results are those of the fixed
    defaults bit for bit: every work item's sums do not depend on which work-group takes it.  FFT
    lines and tuned interpolation grids: test_kept_zeros_and_tuning (test_gpu_tiles.py).  (The
    plan variants of the 288-, 544- and 576-point lengths round differently; the full-size parity
    tests cover them.)"""
    V = vpmlib
    h = 1 / 16
    xp, qp = cases.single_ring(h=h, sigma=0.1)
    out = {}
    for tuning in (1, 0):
        with V.VPM(V.Params.make(h)) as c:
            c.set_option("tuning", tuning)
            for prec in (0, 1):
                c.set_precision(prec)
                up, gp = np.zeros_like(xp), np.zeros_like(xp)
                c.vpm(xp, qp, up, gp, xp.shape[0], 3, 0, 0)
                c.vpm(xp, qp, up, gp, xp.shape[0], 3, 2, 1)
                out[(tuning, prec)] = (up, gp)
            rep = c.tuning_report()
        say("tuning", tuning, "report:\n" + rep)
        assert "sine transforms" in rep
        if tuning:
            assert "ms)" in rep
    for prec in (0, 1):
        assert np.array_equal(out[(1, prec)][0], out[(0, prec)][0])
        assert np.array_equal(out[(1, prec)][1], out[(0, prec)][1])


def test_tuner_variants_same_bits(vpmlib):
    """Every launch forced to its variant v (option tune_variant) gives the same velocity and
    stretching grids, UP and GP bit for bit, for every v and both forms, at h=1/16, with the fine
    solves' spectral shortcuts on: the curl/stretch tile shapes, with the velocity ring alone or
    with the stream function kept in registers and one LDS plane, the FP64 matrix-product tile
    shapes, the face sums' rows in flight, the lines per work-group of the sine products."""
    V = vpmlib
    h = 1 / 16
    xp, qp = cases.single_ring(h=h, sigma=0.1)
    ref = {}
    for v in range(7):
        with V.VPM(V.Params.make(h)) as c:
            c.set_option("tune_variant", v)
            c.set_option("face_derivs", 1)
            c.set_option("fine_partial", 1)
            for prec in (0, 1):
                c.set_precision(prec)
                up, gp = np.zeros_like(xp), np.zeros_like(xp)
                c.vpm(xp, qp, up, gp, xp.shape[0], 3, 0, 0)
                c.vpm(xp, qp, up, gp, xp.shape[0], 3, 2, 1)
                got = (c.get_grid(3), c.get_grid(2), up, gp)
                say("case: tune_variant", v, "precision", prec)
                if v == 0:
                    ref[prec] = got
                    continue
                for name, a, b in zip(("vel", "sol", "up", "gp"), got, ref[prec]):
                    assert np.array_equal(a, b), (v, prec, name, float(np.max(np.abs(a - b))))
            rep = c.tuning_report()
        assert "forced" in rep


@pytest.mark.parametrize("nn,prec", [((244, 20, 21), 1), ((20, 244, 21), 1), ((21, 20, 244), 1), ((244, 226, 246), 1),
                                     ((130, 131, 141), 0), ((210, 130, 300), 0)])
def test_solve_variants_same_bits(vpmlib, nn, prec):
    """Solves with every launch forced to its variant v give the same bits: both batch orders of the
    FP32 FFT passes along each axis (runtime plans), 16 and 32 lines per work-group of the products."""
    V = vpmlib
    rng = np.random.default_rng(sum(nn))
    nn = np.array(nn, np.int32)
    rhs, sol = rng.standard_normal((2, nn[2], nn[1], nn[0], 3))
    win = np.array([1, 1, 1, *nn], np.int32)
    ref = None
    for v in (0, 1):
        with V.VPM(V.Params.make(0.125)) as c:
            c.set_option("tune_variant", v)
            c.set_precision(prec)
            say("case: solve variants", nn.tolist(), "precision", prec, "variant", v)
            got = c.stage_solve(np.zeros(6), np.array([0.05, 0.04, 0.06]), nn, 3, win, rhs, sol=sol)
            rep = c.tuning_report()
        assert "forced" in rep and ("matrix products" in rep if prec == 0 else "pass FP32 L=" in rep)
        assert ref is None or np.array_equal(got, ref)
        ref = got
