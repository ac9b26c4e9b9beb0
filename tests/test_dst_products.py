"""DST-I passes as folded products with the sine matrix (k_dstm.hip): the folding identity in
numpy (CPU), and Dirichlet solves at the sizes where the kernels' tiles end, against the oracle
(pmsolve.f90:284-432)."""
import numpy as np
import pytest


def _folded(x):
    """The transform by the kernels' folding: sums and differences of mirrored points, the
    differences folded once more when m is odd, one product per part."""
    m = len(x)
    h = m // 2
    S = lambda k, j: np.sin(np.pi * ((k[:, None] * j[None]) % (2 * (m + 1))) / (m + 1))
    out = np.full(m, np.nan)
    j = np.arange(1, h + 1)
    e, o = x[:h] + x[::-1][:h], x[:h] - x[::-1][:h]
    if m % 2:
        e = np.append(e, x[h])
        k = 2 * np.arange(h + 1) + 1
        out[k - 1] = S(k, np.arange(1, h + 2)) @ e
        f = h // 2
        oe = np.append(o[:f] + o[::-1][:f], o[f:h - f])
        oo = o[:f] - o[::-1][:f]
        k = 4 * np.arange(h - f) + 2
        out[k - 1] = S(k, np.arange(1, h - f + 1)) @ oe
        k = 4 * np.arange(f) + 4
        out[k - 1] = S(k, np.arange(1, f + 1)) @ oo
    else:
        k = 2 * np.arange(h) + 1
        out[k - 1] = S(k, j) @ e
        out[k] = S(k + 1, j) @ o
    return out


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 7, 16, 31, 33, 40, 79, 95, 128, 223])
def test_folded_transform(m):
    x = np.random.default_rng(m).standard_normal(m)
    j = np.arange(1, m + 1)
    ref = np.sin(np.pi * (np.outer(j, j) % (2 * (m + 1))) / (m + 1)) @ x
    got = _folded(x)
    assert np.linalg.norm(got - ref) <= 1e-13 * np.linalg.norm(ref)


# interior points per axis: one point; the 16-output blocks' edges in every segment; the largest
# planes of k_dstm_plane and the first sizes past them; the longest lines of each axis
SIZES = [(1, 2, 3), (15, 17, 16), (31, 33, 32), (63, 64, 65), (95, 95, 7), (98, 95, 8), (129, 127, 9), (223, 9, 11),
         (10, 224, 9), (9, 10, 223), (175, 13, 24), (24, 176, 10), (11, 12, 175)]


# longer lines: lengths whose m + 1 has a large factor, the 288-point transform beside products,
# the longest products (odd and even) and the first length past them on each axis
LONG = [(231, 9, 10), (9, 271, 10), (10, 9, 303), (367, 10, 9), (9, 362, 7), (10, 9, 367), (287, 8, 287), (8, 287, 271),
        (368, 9, 10), (9, 368, 10), (9, 10, 368), (300, 31, 9)]
# the mixed form's: large factors, the last length of the FP32 rule
LONG32 = [(231, 9, 10), (9, 247, 8), (8, 10, 207), (208, 207, 9)]


@pytest.mark.gpu
@pytest.mark.parametrize("m", SIZES + [(*m, 0) for m in LONG] + [(*m, 1) for m in LONG32])
def test_solve_products(vpmlib, oracle, m):
    """Zero and given Dirichlet values; FP64 within 1e-12, and the mixed form (FP32 arrays between
    five passes of FP64 sums: five roundings of 6e-8) within 1e-6."""
    V = vpmlib
    form, m = m[3:], m[:3]  # a fourth entry: that precision only
    rng = np.random.default_rng(sum(m))
    nn = np.array(m, np.int32) + 2
    xb = np.array([-1.0, -0.5, -0.7, 0, 0, 0])
    dpm = np.array([0.02, 0.03, 0.025])
    win = np.array([1, 1, 1, nn[0], nn[1], nn[2]], np.int32)
    rhs = rng.standard_normal((nn[2], nn[1], nn[0], 3))
    sol = rng.standard_normal((nn[2], nn[1], nn[0], 3))
    zero = oracle.solve_window(xb, dpm, nn, win, rhs, zero_bc=True)
    given = oracle.solve_window(xb, dpm, nn, win, rhs, sol=sol)
    for prec, tol in ((0, 1e-12), (1, 1e-6)):
        if form and prec not in form:
            continue
        with V.VPM(V.Params.make(0.125)) as c:
            c.set_precision(prec)
            print("case: products solve", m, "precision", prec, flush=True)
            a = c.stage_solve(xb, dpm, nn, 3, win, rhs, zero_bc=True)
            b = c.stage_solve(xb, dpm, nn, 3, win, rhs, sol=sol)
        for got, ref in ((a, zero), (b, given)):
            assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref)
