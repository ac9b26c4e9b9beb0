"""The cells that the projection's node tiles read (p2m_cells.h): every entry of the start table lies
in the table, for views that reach past the grid by ncoarse nodes on each side (CPU); projections
through the block layout with such views (pmproject.f90:43-153)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vpm_free_amd", "csrc")

# Per tile row that exists: the two entries of the test for particles and the staged ones, against
# the table's bounds, the row's own entries, and the cells that reach the tile's nodes in the grid.
PROBE = r"""
#include <cstdio>
#include <cstdlib>
#include "p2m_cells.h"
using namespace vpmx;
int main(int, char **v) {
    const int n0 = atoi(v[1]), n1 = atoi(v[2]), n2 = atoi(v[3]), pad = atoi(v[4]), cn = n0 + 3;
    const int64_t ncells = (int64_t)cn * (n1 + 3) * (n2 + 3);
    const int t0 = (n0 + 2 * pad + PT_X - 1) / PT_X, t1 = (n1 + 2 * pad + PT_Y - 1) / PT_Y, t2 = (n2 + 2 * pad + PT_Z - 1) / PT_Z;
    long rows = 0;
    for (int tz = 0; tz < t2; tz++)
        for (int ty = 0; ty < t1; ty++)
            for (int tx = 0; tx < t0; tx++)
                for (int r = 0; r < PT_ROWS; r++) {
                    const int I0 = tx * PT_X - pad + 1, J0 = ty * PT_Y - pad + 1, K0 = tz * PT_Z - pad + 1;
                    const int64_t row = p2m_row(J0, K0, r, n1, n2);
                    const int cj = J0 - 2 + r % 7, ck = K0 - 2 + r / 7;
                    if ((row >= 0) != (cj >= -1 && cj <= n1 + 1 && ck >= -1 && ck <= n2 + 1)) return 1;
                    if (row < 0) continue;
                    if (row != (cj + 1) + (int64_t)(n1 + 3) * (ck + 1)) return 2;
                    rows++;
                    int64_t was = -1;
                    for (int c = 0; c <= PC_X; c++) {
                        const int64_t e = p2m_entry(I0, c, row, n0);
                        if (e < 0 || e > ncells) return 3;
                        if (e < row * cn || e > (row + 1) * cn || e < was) return 4;
                        const int cx = I0 - 2 + c;  // a cell of the grid keeps its own entry
                        if (cx >= -1 && cx <= n0 + 1 && e != row * cn + cx + 1) return 5;
                        was = e;
                    }
                }
    printf("%ld\n", rows);
    return 0;
}
"""


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("cells")
    (d / "probe.cpp").write_text(PROBE)
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", CSRC, str(d / "probe.cpp"), "-o", str(d / "probe")], check=True)
    return str(d / "probe")


@pytest.mark.parametrize("pad", [0, 4, 8, 16, 24, 32, 50])
@pytest.mark.parametrize("n", [(33, 41, 25), (49, 33, 57), (41, 49, 33), (6, 7, 8), (32, 47, 40)])
def test_entries_in_the_table(probe, n, pad):
    r = subprocess.run([probe, *map(str, n), str(pad)], capture_output=True, text=True)
    assert r.returncode == 0 and int(r.stdout) > 0, r.returncode


@pytest.mark.gpu
@pytest.mark.parametrize("ncoarse", [4, 8, 16, 24, 32])
@pytest.mark.parametrize("prec", [0, 1])
def test_project_into_padded_block(vpmlib, oracle, ncoarse, prec):
    """vpm(5) projects into a block that is ncoarse nodes larger than the grid on each side; particles
    at the far ends of the box, two clouds in turn: FP64 within 1e-12 of the oracle, FP32 sums within
    1e-6."""
    V = vpmlib
    h = 0.125
    rng = np.random.default_rng(ncoarse)
    ext = h * np.array([20.0, 27.0, 13.0])
    with V.VPM(V.Params.make(h, ncoarse=ncoarse)) as c:
        c.set_precision(prec)
        for part in range(2):
            xp = rng.uniform(0.0, 1.0, size=(900, 3)) * ext * (1.0 if part == 0 else 0.4)
            xp[:2] = np.zeros(3), ext
            qp = np.concatenate([rng.standard_normal((len(xp), 3)), np.full((len(xp), 1), h**3)], axis=1)
            up, gp = np.zeros_like(xp), np.zeros_like(xp)
            print("case: padded projection, ncoarse", ncoarse, "precision", prec, "cloud", part, flush=True)
            c.vpm(xp, qp, up, gp, len(xp), 3, 0, 0)
            c.vpm(xp, qp, up, gp, len(xp), 3, 5, 1)
            g = c.geometry
            nn = np.array(g.nn, np.int32)
            ref = oracle.project(np.array(g.xbound), np.array(g.dpm), nn, np.array([1, 1, 1, *nn], np.int32), xp, qp)
            got = c.get_grid(0)
            err = np.linalg.norm(got[..., :3] - ref[..., :3]) / np.linalg.norm(ref[..., :3])
            assert err <= (1e-12 if prec == 0 else 1e-6), err
