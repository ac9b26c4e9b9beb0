"""Equal neighbouring yaps blocks solved together (vpmx_api.hip, same_blocks) against the same
blocks solved one by one (the spectral normal derivatives keep them apart)."""
import ctypes

import numpy as np
import pytest

import test_oracle_yaps as Y
from vpm_free_amd import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks,weights", [((4, 1, 1), ((1, 1, 2, 1), (1,), (1,))), ((2, 1, 2), None)])
def test_groups_of_equal_blocks(vpmlib, blocks, weights):
    """Groups of one and of several blocks, all of one size and not: FP64 within 1e-11 (two solves
    and the second differences of a field whose parts differ by rounding)."""
    V = vpmlib
    h = 0.125
    rng = np.random.default_rng(len(blocks) + blocks[0])
    xp = rng.uniform(-1, 1, size=(3000, 3)) * np.array([2.5, 1.0, 1.0])
    qp = np.concatenate([rng.standard_normal((len(xp), 3)), np.full((len(xp), 1), h**3)], axis=1)
    out = []
    for apart in (0, 1):
        with V.VPM(V.Params.make(h, blocks=blocks, ncoarse=Y.NCOARSE)) as c:
            if weights is not None:
                c.set_block_weights(*weights)
            c.set_option("face_derivs", apart)
            up, gp = np.zeros_like(xp), np.zeros_like(xp)
            print("case: block groups", blocks, weights, "apart", apart, flush=True)
            c.vpm(xp, qp, up, gp, len(xp), 3, 0, 0)
            c.vpm(xp, qp, up, gp, len(xp), 3, 2, 1)
            out.append((c.get_grid(1), up, gp))
    for a, b in zip(*out):
        assert np.linalg.norm(a - b) <= 1e-11 * np.linalg.norm(b)


def test_ncoarse_changed_after_mode_0(vpmlib):
    """One block whose geometry was defined with another ncoarse: its samples, every 16 nodes, fall on
    every second coarse node.  The call is taken, and the stream function solves the 7-point equations
    of the inner box for the projected strengths (parity unpinned: the oracle's footprint has holes
    there, the library's is the box around the samples)."""
    V = vpmlib
    h = 0.125
    xp, qp = cases.single_ring(h=h, sigma=0.2)
    print("case: ncoarse 8, then 16", flush=True)
    with V.VPM(V.Params.make(h)) as c:
        up, gp = np.zeros_like(xp), np.zeros_like(xp)
        c.vpm(xp, qp, up, gp, len(xp), 3, 0, 0)
        other = V.Params.make(h, ncoarse=16)
        c._check(c._lib.vpmx_set_params(c._h, ctypes.byref(other)))
        c.vpm(xp, qp, up, gp, len(xp), 3, 2, 1)
        psi, rhs = c.get_grid(1), c.get_grid(0)[..., :3]
    assert np.all(np.isfinite(up)) and np.all(np.isfinite(gp)) and np.linalg.norm(up) > 0
    mid = psi[1:-1, 1:-1, 1:-1]
    lap = sum(np.roll(psi, s, a)[1:-1, 1:-1, 1:-1] - mid for a in range(3) for s in (1, -1)) / h**2
    assert np.abs(lap - rhs[1:-1, 1:-1, 1:-1]).max() <= 1e-11 * np.abs(rhs).max()
