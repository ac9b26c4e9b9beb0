"""The projection's two tile forms at the line between them (SMALL_TILES tiles of 16 x 4 x 4
nodes): every tile its own work-group up to it, the list of occupied tiles above it
(pmproject.f90:43-153)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nn", [(128, 128, 128), (129, 128, 128), (17, 5, 6)])
def test_project_tile_forms(vpmlib, oracle, nn):
    """A blob away from most tiles, particles on the last nodes and a cell with more particles
    than a tile stages at once, twice with different clouds: FP64 within 1e-12 of the oracle and
    empty nodes exactly zero."""
    V = vpmlib
    rng = np.random.default_rng(nn[0])
    nn = np.array(nn, np.int32)
    h = 0.1
    xb = np.array([-1.0, -0.5, -0.7, 0, 0, 0])
    top = xb[:3] + h * (nn - 1)
    nnb = np.array([1, 1, 1, *nn], np.int32)
    with V.VPM(V.Params.make(0.125)) as c:
        for part in range(2):
            lo = xb[:3] + h * (1.0 + 0.2 * part)
            blob = rng.uniform(lo, np.minimum(lo + 2.0, top - h), size=(3000, 3))
            full = xb[:3] + h * (np.minimum(nn, 4) - 1.5) + rng.uniform(0, 0.3 * h, size=(700, 3))
            xp = np.concatenate([blob, full, top - h * rng.uniform(0, 1, size=(20, 3))])
            qp = np.concatenate([rng.standard_normal((len(xp), 3)), np.full((len(xp), 1), 1e-3)], axis=1)
            print("case: project tiles", nn.tolist(), "cloud", part, flush=True)
            ref = oracle.project(xb, np.full(3, h), nn, nnb, xp, qp)
            got = c.stage_project(xb, np.full(3, h), nn, nnb, xp, qp)
            assert np.linalg.norm(got - ref) <= 1e-12 * np.linalg.norm(ref)
            empty = np.all(ref[..., :3] == 0, axis=-1)
            assert np.all(got[..., :3][empty] == 0)


def test_kept_zeros_and_tuning(vpmlib, oracle):
    """vpm(2) calls of one context on a block above the line (17955 projection and 12393 interpolation
    tiles), where only the tiles emptied since the last call are cleared: cloud + blob, the same
    again, the cloud alone, a mixed-form call, cloud + blob in FP64, the cloud alone twice.  The RHS
    within 1e-12 of the oracle (mixed 1e-6) and zero where the oracle's is; UP and GP those of a
    fresh context bit for bit, and those of the tuner's choices too (FP32 FFT lines in two batch
    orders, interpolation grids, stencil and matrix tiles)."""
    V = vpmlib
    rng = np.random.default_rng(8)
    h = 1 / 16
    ext = np.array([12.0, 12.0, 3.0])
    xr = rng.uniform(0, 1, size=(3000, 3)) * ext
    xr[:2] = np.zeros(3), ext
    lo, hi = np.array([4.0, 5.0, 0.5]), np.array([6.0, 7.0, 2.5])
    xr = xr[~np.all((xr > lo - 4 * h) & (xr < hi + 4 * h), axis=1)]
    xa = np.concatenate([xr, rng.uniform(lo, hi, size=(1500, 3))])
    qa = np.concatenate([h**3 * rng.standard_normal((len(xa), 3)), np.full((len(xa), 1), h**3)], axis=1)
    clouds = {"a": (xa, qa), "r": (xr, qa[:len(xr)])}

    def context(tuning=0):
        c = V.VPM(V.Params.make(h))
        c.set_option("tuning", tuning)
        c.vpm(xa, qa, None, None, len(xa), 3, 0, 0)
        return c

    def call(c, name, prec):
        x, q = clouds[name]
        c.set_precision(prec)
        up, gp = np.zeros_like(x), np.zeros_like(x)
        print("case: kept zeros, cloud", name, "precision", prec, flush=True)
        c.vpm(x, q, up, gp, len(x), 3, 2, 1)
        return up, gp

    fresh = {}
    for name, prec in (("a", 0), ("r", 0), ("a", 1)):
        with context() as c:
            fresh[name, prec] = call(c, name, prec)
            g = c.geometry
    nn, nb = np.array(g.nn, np.int32), np.array(g.nnbl[:3])
    assert np.prod(-(-nb // [16, 4, 4])) > 8192 and np.prod(-(-(nn + 3) // [8, 8, 4])) > 8192
    box = np.array(g.xbound), np.array(g.dpm), nn, np.array([1, 1, 1, *nn], np.int32)
    rhs = {name: oracle.project(*box, x, q)[..., :3] for name, (x, q) in clouds.items()}
    with context() as c:
        for name, prec in (("a", 0), ("a", 0), ("r", 0), ("a", 1), ("a", 0), ("r", 0), ("r", 0)):
            got = call(c, name, prec)
            grid, ref = c.get_grid(0)[..., :3], rhs[name]
            assert np.linalg.norm(grid - ref) <= (1e-6 if prec else 1e-12) * np.linalg.norm(ref)
            assert np.all(grid[np.all(ref == 0, axis=-1)] == 0)
            for u, v in zip(got, fresh[name, prec]):
                assert np.array_equal(u, v), (name, prec)
    with context(tuning=1) as c:
        for name, prec in (("a", 0), ("a", 1)):
            for u, v in zip(call(c, name, prec), fresh[name, prec]):
                assert np.array_equal(u, v), ("tuned", prec)
        rep = c.tuning_report()
    assert "pass FP32 L=" in rep and "interpolation tiles" in rep and "ms)" in rep
