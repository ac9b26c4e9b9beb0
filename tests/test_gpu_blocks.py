"""Equal neighbouring yaps blocks solved together (vpmx_api.hip, same_blocks) against the same
blocks solved one by one (the spectral normal derivatives keep them apart)."""
import numpy as np
import pytest

import test_oracle_yaps as Y

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
