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
