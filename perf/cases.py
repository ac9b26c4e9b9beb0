"""Timed cases of the VPM core: what a program that links the library has it do.

Every case is one kind of call over a range of sizes:

  vpm2      vpm(WhatToDo=2) on the caller's host arrays, the reference's own call shape: one
            evaluation of velocity and stretching per pass.
  steps     a time loop with the particles resident on the GPU: upload, K RK2 steps, download.
  fields    the same with the remesh of every step, and the velocity field at its end read back.
  batch     many independent rings stepped together as one replayed graph, then read back.
  gradient  the probe energy of one evaluation and its gradient (adjoint), on host arrays.
  rollout   the probe energy after K RK2 steps with remesh and its gradient through them.

The particles are thin-core vortex rings on a lattice of spacing h, displaced from their nodes
by up to a quarter cell as they are between remeshes, with strengths that vary along the ring;
eight zero-strength particles pin the box.  A seed sets the displacements and the variation, so
all seeds of a case share one geometry and one particle count.  exact() is a plain torch FP64 evaluation of the
same equations.
"""
import math

import numpy as np
import torch

from vpm_free_amd import vpm as V

DT = 0.01
NCOARSE = 8
PROBES = 4096


# ------------------------------------------------------------------ cases
def _case(name, kind, cells, **kw):
    c = {"name": name, "kind": kind, "cells": cells, "half_z": 2.0, "rings": 1, "sigma": 0.1, "form": "fp64",
         "bi": 1, "bj": 1, "bk": 1, "tree": 0, "steps": 1, "clouds": 0}
    c.update(kw)
    return c


def listed():
    return [
        # a first look at a flow, a unit test, a coarse parameter study: the latency of one call
        _case("vpm2_32", "vpm2", 32, sigma=0.2),
        # the 64^3 thin-core ring, plain FP64 form (the library's default)
        _case("vpm2_64", "vpm2", 64),
        # flat box of an odd number of cells, mixed form: rings travel, so boxes are rarely cubes
        _case("vpm2_flat_151_mixed", "vpm2", 151, half_z=1.2, rings=2, form="mixed"),
        # the 256^3 leapfrogging rings through the host-array call of the Fortran interface
        _case("vpm2_256", "vpm2", 256, rings=2, sigma=0.08),
        # the shipped pm.inp's solver options: 6x1x1 yaps blocks, tree boundary sums, 3 levels
        _case("vpm2_tree_6x1x1", "vpm2", 96, bi=6, tree=1),
        # several yaps blocks, mixed form: how a domain too large for one block runs
        _case("vpm2_blocks_2x2x2_mixed", "vpm2", 128, rings=2, bi=2, bj=2, bk=2, form="mixed"),
        # a small simulation: many short steps between two looks at the particles
        _case("steps_64_mixed", "steps", 64, steps=10, form="mixed"),
        # the 256^3 time loop, mixed form, between two remeshes
        _case("steps_256_mixed", "steps", 256, rings=2, sigma=0.08, steps=4, form="mixed"),
        # a time loop with the remesh of every step, plain FP64 form, and the velocity field
        # (read by a plotting or coupling program) at its end
        _case("fields_128", "fields", 128, rings=2, steps=8),
        # independent clouds of 32^3..128^3 cells stepped together
        _case("batch_32", "batch", 128, clouds=32, steps=2, form="mixed"),
        # one gradient on the 128^3 ring
        _case("gradient_128", "gradient", 128, sigma=0.22),
        # gradient through two remeshed steps
        _case("rollout_64", "rollout", 64, sigma=0.2, steps=2),
    ]


def draw(rng):
    kind = rng.choice(["vpm2"] * 4 + ["steps"] * 2 + ["fields", "batch", "gradient", "rollout"])
    form = rng.choice(["fp64", "mixed"])

    def cells(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == "vpm2":
        n = cells(28, 250)
        kw = dict(rings=rng.choice([1, 2]), half_z=round(rng.uniform(1.2, 2.0), 2), form=form)
        if n < 130 and rng.random() < 0.35:
            kw.update(bi=rng.choice([1, 2, 3]), bj=rng.choice([1, 2]), bk=rng.choice([1, 2]))
        kw["sigma"] = _sigma(n, kw["rings"], rng.uniform(0.08, 0.12))
        c = _case("", kind, n, **kw)
    elif kind in ("steps", "fields"):
        n, rings = cells(28, 250 if kind == "steps" else 128), rng.choice([1, 2])
        c = _case("", kind, n, rings=rings, sigma=_sigma(n, rings, rng.uniform(0.08, 0.12)), form=form,
                  half_z=round(rng.uniform(1.2, 2.0), 2), steps=2 if n > 160 else rng.choice([3, 5, 8]))
    elif kind == "batch":
        c = _case("", kind, rng.choice([64, 96, 128]), clouds=rng.randint(3, 32), steps=rng.choice([1, 2, 3]), form=form)
    elif kind == "gradient":
        n = cells(30, 128)
        c = _case("", kind, n, sigma=_sigma(n, 1, rng.uniform(0.12, 0.22)), half_z=round(rng.uniform(1.4, 2.0), 2))
    else:
        n = cells(30, 64)
        c = _case("", kind, n, sigma=_sigma(n, 1, rng.uniform(0.12, 0.2)), steps=rng.choice([1, 2]))
    del c["name"]
    return c


def _sigma(n, rings, s):
    """A core at least 1.3 cells wide that stays inside the box."""
    return round(min(max(s, 1.3 * 4.0 / n), 0.1 if rings == 2 else 0.2), 4)


def _rings(case):
    """(radius, height) of the rings, and the half extents of the box."""
    half = (2.0, 2.0, case["half_z"])
    rings = [(1.0, 0.0)] if case["rings"] == 1 else [(1.0, -0.25), (1.2, 0.25)]
    return rings, half


# ------------------------------------------------------------------ inputs
def _cloud(h, half, rings, sigma, axis, seed):
    """Particles of Gaussian-core rings at lattice cell centres where |w| > 1e-6, displaced by
    up to h/4, with strengths QP(1:3) = -w h^3 and volume QP(4) = h^3."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    rng = np.random.default_rng(seed)
    n = [int(round(2 * e / h)) for e in half]
    c = [torch.arange(k, dtype=torch.float64, device=dev).add_(0.5).mul_(h).sub_(e) for k, e in zip(n, half)]
    z, y, x = torch.meshgrid(c[2], c[1], c[0], indexing="ij")
    pts = torch.stack([x.reshape(-1), y.reshape(-1), z.reshape(-1)], dim=1)
    a = torch.tensor(axis, dtype=torch.float64, device=dev)
    w = torch.zeros_like(pts)
    for radius, height in rings:
        d = pts - height * a
        s = (d * a).sum(dim=1)
        radial = d - s[:, None] * a
        r = radial.norm(dim=1)
        mag = 1.0 / (math.pi * sigma ** 2) * torch.exp(-((r - radius) ** 2 + s ** 2) / sigma ** 2)
        er = radial / r.clamp_min(1e-300)[:, None]
        w += mag[:, None] * torch.linalg.cross(a.expand_as(er), er)
    keep = w.norm(dim=1) > 1e-6
    xp, w = pts[keep].cpu().numpy(), w[keep].cpu().numpy()
    waves, phase, depth = rng.integers(1, 6), rng.uniform(0, 2 * math.pi), rng.uniform(0.02, 0.1)
    w *= 1.0 + depth * np.sin(waves * np.arctan2(xp[:, 1:2], xp[:, :1]) + phase)
    xp = xp + rng.uniform(-0.25 * h, 0.25 * h, size=xp.shape)
    qp = np.concatenate([-w * h ** 3, np.full((len(w), 1), h ** 3)], axis=1)
    corners = np.array([[i, j, k] for k in (-half[2], half[2]) for j in (-half[1], half[1]) for i in (-half[0], half[0])])
    cq = np.zeros((8, 4))
    cq[:, 3] = h ** 3
    return np.concatenate([corners, xp]), np.concatenate([cq, qp])


def _particles(case, seed):
    rings, half = _rings(case)
    h = 4.0 / case["cells"]
    half = tuple(h * round(2 * e / h) / 2 for e in half)
    axis = np.array([0.03, -0.02, 1.0])
    return h, *_cloud(h, half, rings, case["sigma"], axis / np.linalg.norm(axis), 1000 + seed)


def _batch_rings(case):
    """(radius, core, cells, axis) of the batch's rings."""
    rng = np.random.default_rng(3)
    grids = np.array([g for g in (32, 48, 64, 96, 128) if g <= case["cells"]])
    prob = 1.0 / grids.astype(float) ** 3
    out = []
    for _ in range(case["clouds"]):
        axis = rng.standard_normal(3)
        out.append((rng.uniform(0.5, 1.5), rng.uniform(0.05, 0.15), int(rng.choice(grids, p=prob / prob.sum())),
                    axis / np.linalg.norm(axis)))
    return out


def _batch_particles(case, seed):
    out = []
    for i, (radius, sigma, n, axis) in enumerate(_batch_rings(case)):
        half = radius + 4.0 * sigma
        h = 2.0 * half / n
        out.append((h, *_cloud(h, (half,) * 3, [(radius, 0.0)], sigma, axis, 2000 + 64 * seed + i)))
    return out


def _probes(seed):
    return np.random.default_rng(3000 + seed).uniform(-1.2, 1.2, size=(PROBES, 3))


def _params(case, h):
    return V.Params.make(h, blocks=(case["bi"], case["bj"], case["bk"]), iyntree=case["tree"], ilevmax=3 if case["tree"] else 1,
                         ncoarse=NCOARSE)


_kept = {}  # the context of the case in hand: a program makes one and feeds it its particles


def _context(case, h):
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _kept:
        _kept.clear()
        c = V.VPM(_params(case, h))
        c.set_precision(1 if case["form"] == "mixed" else 0)
        _kept[key] = c
    return _kept[key]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        clouds = _batch_particles(case, seed)
        _kept.clear()
        b = V.Batch(len(clouds))
        for i, (h, xp, qp) in enumerate(clouds):
            c = b.cloud(i, V.Params.make(h))
            c.set_precision(1 if case["form"] == "mixed" else 0)
            c.upload(xp, qp)
            c.vpm_resident(0, 0)
        return {"case": case, "batch": b}
    h, xp, qp = _particles(case, seed)
    c = _context(case, h)
    c.upload(xp, qp)
    c.vpm_resident(0, 0)  # define_sizes: the box
    return {"case": case, "ctx": c, "xp": xp, "qp": qp, "up": np.zeros_like(xp), "gp": np.zeros_like(xp),
            "probes": _probes(seed) if kind in ("gradient", "rollout") else None}


# ------------------------------------------------------------------ one pass
def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "batch":
        b = state["batch"]
        for _ in range(case["steps"]):
            b.step_rk2(0.1 * DT, remesh=False, graph=True)
        return [b.cloud(i).download()[:2] for i in range(case["clouds"])]
    c, xp, qp = state["ctx"], state["xp"], state["qp"]
    if kind == "vpm2":
        c.vpm(xp, qp, state["up"], state["gp"], len(xp), 3, 2, 1)
        return {"up": state["up"], "gp": state["gp"]}
    if kind in ("steps", "fields"):
        c.upload(xp, qp)
        for k in range(case["steps"]):
            c.step_rk2(DT, ntime=k + 1, remesh=kind == "fields")
        if kind == "steps":
            return dict(zip(("xp", "qp", "up", "gp"), c.download()))
        c.vpm_resident(1, case["steps"] + 1)
        return {"vel": c.get_grid(3)}
    if kind == "gradient":
        j, dq, dx = c.adjoint_probe_energy(xp, qp, state["probes"])
    else:
        j, dq, dx = c.adjoint_rollout(xp, qp, state["probes"], case["steps"], DT)
    return {"J": j, "dq": dq, "dx": dx}


def work(case):
    """Particles in and out; the flops of the sine transforms by 2.5 N log2 N per line and of the
    64-node stencils (the boundary sums count as their transforms)."""
    def tube(radius, sigma, gain_area, h):
        rho2 = sigma ** 2 * math.log(1.0 / (math.pi * gain_area) / 1e-6)
        return 2 * math.pi ** 2 * radius * rho2 / h ** 3

    def one(h, half, rings, sigma):
        n = sum(tube(r, sigma, sigma ** 2, h) for r, _ in rings)
        nodes = [2 * e / h + 9 for e in half]
        vol = nodes[0] * nodes[1] * nodes[2]
        line = 2.5 * sum(math.log2(2 * m) for m in nodes)
        # three solves (two of the block, one of the box) of three components, forward and back
        return n, n * 64 * 20 + 3 * 3 * 2 * vol * line

    if case["kind"] == "batch":
        per = []
        for r, s, n, _ in _batch_rings(case):
            half = r + 4 * s
            per.append(one(2 * half / n, (half,) * 3, [(r, 0.0)], s))
        n, fl = sum(p[0] for p in per), 2 * case["steps"] * sum(p[1] for p in per)
        return {"bytes": n * 2 * 56.0, "flops": fl}
    rings, half = _rings(case)
    n, fl = one(4.0 / case["cells"], half, rings, case["sigma"])
    if case["kind"] == "vpm2":
        return {"bytes": n * (56.0 + 48.0), "flops": fl}
    if case["kind"] == "steps":
        return {"bytes": n * (56.0 + 104.0), "flops": 2 * case["steps"] * fl}
    if case["kind"] == "fields":
        nodes = [2 * e * case["cells"] / 4.0 + 9 for e in half]
        return {"bytes": n * 56.0 + nodes[0] * nodes[1] * nodes[2] * 24.0, "flops": (2 * case["steps"] + 1) * fl}
    evals = 1 if case["kind"] == "gradient" else 2 * case["steps"] + 1
    return {"bytes": n * (56.0 + 48.0), "flops": 2 * evals * fl}


# ------------------------------------------------------------------ the same in plain torch, 64 bits
def _m4(x):
    a = x.abs()
    return torch.where(a < 1, 1 - 2.5 * a ** 2 + 1.5 * a ** 3, torch.where(a < 2, 0.5 * (2 - a) ** 2 * (1 - a), torch.zeros_like(a)))


def _tsc(a):
    a = abs(a)
    return 0.0 if a > 1.5 else 0.5 * (1.5 - a) ** 2 if a >= 0.5 else 0.5 * (a + 1.5) ** 2 - 1.5 * (a + 0.5) ** 2


def _lround(v):
    return int(math.floor(v + 0.5))


def _geometry(case, h, xp):
    """The grids of define_sizes: global box, yaps blocks, coarse grid (x, y, z order)."""
    nb = (case["bi"], case["bj"], case["bk"])
    x0, n, blocks = [], [], []
    cuts = []
    for d in range(3):
        lo, hi = float(xp[:, d].min()) - 4.0 * h, float(xp[:, d].max()) + 4.0 * h
        size = nb[d] * NCOARSE
        m = _lround(abs(hi - lo) / h) + 1
        extra = size - (m - 1) % size
        if extra % 2 == 0:
            lo, hi = lo - (extra // 2) * h, hi + (extra // 2) * h
        else:
            lo, hi = lo - (1 + extra // 2) * h, hi + (extra // 2) * h
        m = _lround(abs(hi - lo) / h) + 1
        x0.append(lo)
        n.append(m)
        units = _lround((hi - lo) / h) // NCOARSE
        cuts.append([NCOARSE * (units * i // nb[d]) for i in range(nb[d] + 1)])
    for k in range(nb[2]):
        for j in range(nb[1]):
            for i in range(nb[0]):
                at = (i, j, k)
                lo = [cuts[d][at[d]] for d in range(3)]
                size = [cuts[d][at[d] + 1] - cuts[d][at[d]] + 1 for d in range(3)]
                blocks.append({"at": at, "lo": lo, "inner": size, "n": [s + 2 * NCOARSE for s in size],
                               "x0": [(x0[d] + lo[d] * h) - NCOARSE * h for d in range(3)]})
    hc = NCOARSE * h
    coarse = {"x0": [v - 4 * hc for v in x0], "n": [(m - 1) // NCOARSE + 9 for m in n], "h": hc}
    return {"h": h, "x0": x0, "n": n, "blocks": blocks, "coarse": coarse}


def _stencil(g, x):
    """Flat node, weight of each of a particle's 64 nodes, with nodes outside the grid masked."""
    n, h = g["n"], g["h"]
    node, wt, ok = [], [], []
    for d in range(3):
        cell = torch.trunc((x[:, d].detach() - g["x0"][d]) / h).long()
        i = [cell + s for s in (-1, 0, 1, 2)]
        wt.append([_m4((x[:, d] - g["x0"][d] - v.double() * h) / h) for v in i])
        ok.append([(v >= 0) & (v < n[d]) for v in i])
        node.append([v.clamp(0, n[d] - 1) for v in i])
    for c in range(4):
        for b in range(4):
            for a in range(4):
                yield (node[2][c] * n[1] + node[1][b]) * n[0] + node[0][a], \
                    wt[0][a] * wt[1][b] * wt[2][c] * (ok[0][a] & ok[1][b] & ok[2][c])


def _project(g, x, q):
    out = torch.zeros(g["n"][0] * g["n"][1] * g["n"][2], 3, dtype=torch.float64, device=x.device)
    for at, w in _stencil(g, x):
        out = out.index_add_(0, at, w[:, None] * q[:, :3]) if not out.requires_grad else out.index_add(0, at, w[:, None] * q[:, :3])
    return (out / g["h"] ** 3).t().reshape(3, g["n"][2], g["n"][1], g["n"][0])


def _gather(g, x, *fields):
    flat = [f.reshape(3, -1).t() for f in fields]
    out = [torch.zeros(len(x), 3, dtype=torch.float64, device=x.device) for _ in fields]
    for at, w in _stencil(g, x):
        out = [o + w[:, None] * f[at] for o, f in zip(out, flat)]
    return out


def _sine(m, dev):
    k = torch.arange(1, m + 1, device=dev)
    return torch.sin(math.pi / (m + 1) * ((k[:, None] * k[None]) % (2 * (m + 1))).double())


def _along(f, s, axis):
    """Every line of f along the axis (of 1 z, 2 y, 3 x) times the symmetric matrix s."""
    t = f.transpose(axis, 3)
    return (t.reshape(-1, t.shape[3]).contiguous() @ s).reshape(t.shape).transpose(axis, 3)


def _solve(rhs, h, face=None):
    """Seven-point Dirichlet solve of a whole window (3, z, y, x); face: {axis: (low, high)}."""
    f = rhs[:, 1:-1, 1:-1, 1:-1].clone()
    if face is not None:
        lo, hi = face[3]
        f[..., 0] -= lo[:, 1:-1, 1:-1] / h ** 2
        f[..., -1] -= hi[:, 1:-1, 1:-1] / h ** 2
        lo, hi = face[2]
        f[:, :, 0] -= lo[:, 1:-1, 1:-1] / h ** 2
        f[:, :, -1] -= hi[:, 1:-1, 1:-1] / h ** 2
        lo, hi = face[1]
        f[:, 0] -= lo[:, 1:-1, 1:-1] / h ** 2
        f[:, -1] -= hi[:, 1:-1, 1:-1] / h ** 2
    m = f.shape[1:]
    s = [_sine(k, f.device) for k in m]
    lam = [4 / h ** 2 * torch.sin(math.pi / (2 * (k + 1)) * torch.arange(1, k + 1, dtype=torch.float64, device=f.device)) ** 2 for k in m]
    for a in range(3):
        f = _along(f, s[a], a + 1)
    f = f / -(lam[0][:, None, None] + lam[1][:, None] + lam[2])
    for a in range(3):
        f = _along(f, s[a], a + 1) * (2.0 / (m[a] + 1))
    out = torch.nn.functional.pad(f, (1, 1, 1, 1, 1, 1))
    if face is not None:
        out = _with_faces(out, face)
    return out


def _with_faces(f, face):
    out = f.clone()
    out[:, 0], out[:, -1] = face[1]
    out[:, :, 0], out[:, :, -1] = face[2]
    out[..., 0], out[..., -1] = face[3]
    return out


def _face_sources(s0, h):
    """-(outward normal derivative) * area / 4 pi at the centres of the face cells."""
    a = (25.0 / 12.0, -4.0, 3.0, -4.0 / 3.0, 0.25)
    out = {}
    for axis in (1, 2, 3):
        for side in (0, 1):
            n = s0.shape[axis]
            d = sum(w * s0.select(axis, i if side == 0 else n - 1 - i) for i, w in enumerate(a)) / h
            d = 0.25 * (d[:, :-1, :-1] + d[:, :-1, 1:] + d[:, 1:, 1:] + d[:, 1:, :-1])
            out[axis, side] = -d * h * h / (4 * math.pi)
    return out


def _boundary(src, n, h):
    """Potential of the face sources at the nodes of every face; n: nodes along z, y, x.
    Along an axis that target and source face share the kernel depends on the offset alone: a
    zero-padded convolution by FFT."""
    dev = src[1, 0].device
    n = {1: n[0], 2: n[1], 3: n[2]}

    def arange(k):
        return torch.arange(k, dtype=torch.float64, device=dev)

    def offsets(k):  # target node - source cell centre, in the order of a circular convolution
        e = arange(2 * k)
        return torch.where(e < k, e, e - 2 * k) - 0.5

    out = {}
    for ta in (1, 2, 3):
        u, v = [a for a in (1, 2, 3) if a != ta]
        both = {0: 0.0, 1: 0.0}
        for sa in (1, 2, 3):
            if sa == ta:
                su, sv = 2 * n[u], 2 * n[v]
                r2 = offsets(n[u])[:, None] ** 2 + offsets(n[v])[None] ** 2
                sf = [torch.fft.rfft2(src[sa, s], s=(su, sv)) for s in (0, 1)]
                for gap in (0, n[ta] - 1):
                    kf = torch.fft.rfft2(1.0 / (h * torch.sqrt(r2 + float(gap) ** 2)))
                    for t in (0, 1):
                        s = t if gap == 0 else 1 - t
                        both[t] = both[t] + torch.fft.irfft2(kf * sf[s], s=(su, sv))[:, :n[u], :n[v]]
                continue
            c = u if sa == v else v  # the axis both faces hold; sa runs on the target, ta on the source
            size = 2 * n[c]
            q = arange(n[ta] - 1) + 0.5
            p = arange(n[sa])
            for s in (0, 1):
                # sources as (component, cell along ta, cell along c)
                f = src[sa, s]
                f = f if (ta < c) else f.transpose(1, 2)
                sf = torch.fft.rfft(f, n=size, dim=2).permute(2, 1, 0).contiguous()
                dp = p - (0 if s == 0 else n[sa] - 1)
                for t in (0, 1):
                    dq = q - (0 if t == 0 else n[ta] - 1)
                    r2 = dp[:, None, None] ** 2 + dq[:, None] ** 2 + offsets(n[c]) ** 2
                    kf = torch.fft.rfft(1.0 / (h * torch.sqrt(r2)), dim=2).permute(2, 0, 1).contiguous()
                    w = torch.fft.irfft(torch.matmul(kf, sf).permute(2, 1, 0), n=size, dim=2)[..., :n[c]]
                    both[t] = both[t] + (w if sa < c else w.transpose(1, 2))
                    del kf, r2
        out[ta] = (both[0], both[1])
    return out


def _free_space(rhs, h):
    """Infinite-domain solve of a grid: zero-boundary solve, its surface sources' potential on
    the faces, Dirichlet solve."""
    src = _face_sources(_solve(rhs, h), h)
    return _solve(rhs, h, _boundary(src, rhs.shape[1:], h))


def _psi(g, rhs):
    """The yaps composition: block solves, coarse solve, corrected inner faces, inner solves."""
    h, coarse, dev = g["h"], g["coarse"], rhs.device
    B, cn, hc = g["blocks"], coarse["n"], coarse["h"]
    fine, inner, samp, rc = [], [], [], torch.zeros(3, cn[2], cn[1], cn[0], dtype=torch.float64, device=dev)
    for b in B:
        lo, m = b["lo"], b["inner"]
        w = rhs[:, lo[2]:lo[2] + m[2], lo[1]:lo[1] + m[1], lo[0]:lo[0] + m[0]].clone()
        for d in range(3):
            if b["at"][d] > 0:
                w.select(3 - d, 0).zero_()
        inner.append(w)
        fine.append(_free_space(torch.nn.functional.pad(w, (NCOARSE,) * 6), h))
        b["c0"] = [_lround((b["x0"][d] - coarse["x0"][d]) / hc) for d in range(3)]
        b["cn"] = [(b["n"][d] - 1) // NCOARSE + 1 for d in range(3)]
        s = fine[-1][:, ::NCOARSE, ::NCOARSE, ::NCOARSE]
        c0, cm = b["c0"], b["cn"]
        pad = (c0[0], cn[0] - c0[0] - cm[0], c0[1], cn[1] - c0[1] - cm[1], c0[2], cn[2] - c0[2] - cm[2])
        samp.append(torch.nn.functional.pad(s, pad))
        mid = s[:, 1:-1, 1:-1, 1:-1]
        lap = (s[:, 2:, 1:-1, 1:-1] + s[:, :-2, 1:-1, 1:-1] + s[:, 1:-1, 2:, 1:-1] + s[:, 1:-1, :-2, 1:-1]
               + s[:, 1:-1, 1:-1, 2:] + s[:, 1:-1, 1:-1, :-2] - 6 * mid) / hc ** 2
        rc = rc + torch.nn.functional.pad(lap, tuple(p + 1 for p in pad))
    solc = _free_space(rc, hc)
    out = torch.zeros_like(rhs)
    for b, w in zip(B, inner):
        m = b["inner"]
        face = {}
        for axis in (1, 2, 3):
            d = 3 - axis
            pair = []
            for side in (0, m[d] - 1):
                rng = [[NCOARSE + side] if e == d else list(range(NCOARSE, NCOARSE + m[e])) for e in range(3)]
                pair.append(_corrected(g, b, rng, fine, samp, solc).select(axis, 0))
            face[axis] = tuple(pair)
        f = _solve(w, h, face)
        lo = b["lo"]
        if len(B) == 1:
            return f
        out = out.clone()
        out[:, lo[2]:lo[2] + m[2], lo[1]:lo[1] + m[1], lo[0]:lo[0] + m[0]] = f
    return out


def _corrected(g, b, rng, fine, samp, solc):
    """Face values of block b at its nodes rng (per axis, 0-based): its own fine solution, plus the
    quadratic-spline interpolation of the coarse solution less the samples of the blocks whose
    footprint holds the stencil, plus those neighbours' fine solutions."""
    h, coarse, dev, B = g["h"], g["coarse"], solc.device, g["blocks"]
    hc = coarse["h"]
    near, wt = [], []
    for d in range(3):
        x = [b["x0"][d] + i * h for i in rng[d]]
        near.append([_lround((v - coarse["x0"][d]) / hc) for v in x])
        wt.append(torch.tensor([[_tsc((v - coarse["x0"][d] - (c + s) * hc) / hc) for s in (-1, 0, 1)] for v, c in zip(x, near[d])],
                               dtype=torch.float64, device=dev))
    idx = [torch.tensor(v, device=dev) for v in near]

    def interp(f):
        for axis, d in ((1, 2), (2, 1), (3, 0)):
            sh = [1, 1, 1, 1]
            sh[axis] = -1
            f = sum(wt[d][:, s].reshape(sh) * f.index_select(axis, idx[d] + s - 1) for s in range(3))
        return f

    def grid3(ok):
        return (ok[2][:, None, None] & ok[1][:, None] & ok[0]).double()

    def pick(f, at):
        return f.index_select(1, at[2]).index_select(2, at[1]).index_select(3, at[0])

    i = [torch.tensor(r, device=dev) for r in rng]
    own = fine[B.index(b)]
    val = pick(own, i) + interp(solc)
    for o, f, s in zip(B, fine, samp):
        inside = grid3([(idx[d] - 1 >= o["c0"][d]) & (idx[d] + 1 < o["c0"][d] + o["cn"][d]) for d in range(3)])
        val = val - inside * interp(s)
        if o is b or any(abs(o["at"][d] - b["at"][d]) > 1 for d in range(3)):
            continue
        at = [i[d] + _lround((b["x0"][d] - o["x0"][d]) / h) for d in range(3)]
        ok = grid3([(at[d] >= 0) & (at[d] < o["n"][d]) for d in range(3)])
        val = val + inside * ok * pick(f, [at[d].clamp(0, o["n"][d] - 1) for d in range(3)])
    return val


def _curl(psi, h):
    def d(c, axis):
        f = psi[c]
        lo = [slice(1, -1)] * 3
        hi = [slice(1, -1)] * 3
        lo[axis], hi[axis] = slice(0, -2), slice(2, None)
        return (f[tuple(hi)] - f[tuple(lo)]) / (2 * h)

    u = torch.stack([d(2, 1) - d(1, 0), d(0, 0) - d(2, 2), d(1, 2) - d(0, 1)])
    return torch.nn.functional.pad(u, (1,) * 6)


def _stretch(rhs, u, h):
    out = 0.0
    for j, axis in ((0, 2), (1, 1), (2, 0)):
        f = rhs[j][None] * u
        lo = [slice(None)] + [slice(2, -2)] * 3
        hi = [slice(None)] + [slice(2, -2)] * 3
        lo[axis + 1], hi[axis + 1] = slice(1, -3), slice(3, -1)
        out = out - (f[tuple(hi)] - f[tuple(lo)]) / (2 * h)
    return torch.nn.functional.pad(out, (2,) * 6)


def _vpm2(g, x, q):
    rhs = _project(g, x, q)
    u = _curl(_psi(g, rhs), g["h"])
    s = _stretch(rhs, u, g["h"])
    up, gl = _gather(g, x, u, s)
    return up, gl * q[:, 3:4]


def _remesh(g, x, q):
    n, h = g["n"], g["h"]
    f = _project(g, x, q)
    f = f[:, 2:-2, 2:-2, 2:-2].reshape(3, -1).t()
    keep = f.detach().norm(dim=1) >= float(np.float32(1e-9))
    c = [g["x0"][d] + h * torch.arange(2, n[d] - 2, dtype=torch.float64, device=x.device) for d in range(3)]
    z, y, xx = torch.meshgrid(c[2], c[1], c[0], indexing="ij")
    pts = torch.stack([xx.reshape(-1), y.reshape(-1), z.reshape(-1)], dim=1)[keep]
    return pts, torch.cat([f[keep] * h ** 3, torch.full((len(pts), 1), h ** 3, dtype=torch.float64, device=x.device)], dim=1)


def _step(g, x, q, dt, remesh):
    def move(u, s, t):
        return x + t * u, torch.cat([q[:, :3] - t * s, q[:, 3:]], dim=1)

    u, s = _vpm2(g, x, q)
    xm, qm = move(u, s, 0.5 * dt)
    u, s = _vpm2(g, xm, qm)
    x, q = move(u, s, dt)
    if remesh:
        x, q = _remesh(g, x, q)
    return x, q, u, s


def _host(*t):
    return [v.detach().cpu().numpy() for v in t]


def exact(case, seed):
    if case["tree"]:
        return None  # the tree's sums are an approximation of their own: no 64-bit value but its own
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def on(a):
        return torch.from_numpy(a).to(dev)

    kind = case["kind"]
    if kind == "batch":
        out = []
        one = _case("", "steps", 0)
        for h, xp, qp in _batch_particles(case, seed):
            g, x, q = _geometry(one, h, xp), on(xp), on(qp)
            for _ in range(case["steps"]):
                x, q, _, _ = _step(g, x, q, 0.1 * DT, False)
            out.append(_host(x, q))
        return out
    h, xp, qp = _particles(case, seed)
    g, x, q = _geometry(case, h, xp), on(xp), on(qp)
    if kind == "vpm2":
        up, gp = _host(*_vpm2(g, x, q))
        return {"up": up, "gp": gp}
    if kind in ("steps", "fields"):
        for _ in range(case["steps"]):
            x, q, u, s = _step(g, x, q, DT, kind == "fields")
        if kind == "steps":
            return dict(zip(("xp", "qp", "up", "gp"), _host(x, q, u, s)))
        return {"vel": _host(_curl(_psi(g, _project(g, x, q)), h))[0]}
    x.requires_grad_(True)
    q.requires_grad_(True)
    y, p = x, q
    for _ in range(case["steps"] if kind == "rollout" else 0):
        y, p, _, _ = _step(g, y, p, DT, True)
    u = _curl(_psi(g, _project(g, y, p)), g["h"])
    (v,) = _gather(g, on(_probes(seed)), u)
    J = 0.5 * (v ** 2).sum()
    gx, gq = torch.autograd.grad(J, (x, q))
    return {"J": float(J.detach()), "dq": _host(gq[:, :3])[0], "dx": _host(gx)[0]}
