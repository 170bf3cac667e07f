"""Performance cases of the DG-SWEM step: what a user of the framework has it do.

Every case goes through the Python host's public entry points (`dgswem_amd.gpu.GpuSolver`,
`Ensemble`, `dgswem_amd.adjoint.gauge_misfit`); the handle they keep is the one a program keeps.

kinds
* tide      a tidal basin with a wetting/drying shelf, slope limiter and Manning friction advanced
            `steps` steps between two outputs of its state (the plain method);
* forecast  the same, reading the nodal fields (what fort.63/fort.64 hold) instead of the modes;
* coupled   a small basin advanced one step per call with the nodal values and the running maximum
            elevation updated after every step, as the Fortran time loop does;
* river     a channel with a specified normal flux, no limiter (wetting/drying in the stage), linear
            friction and the three-stage scheme;
* ocean     a spherical basin under the tidal potential with Coriolis, all wet;
* ensemble  uneven spherical storm basins under their own hurricanes, batched, replaying graphs;
* gradient  loss and gradient of a gauge misfit with respect to Manning's n and the depth by the
            checkpointed adjoint, through the torch front end, on an all-wet basin;
* storm_gradient  the batched adjoint of storm members with limiter and wetting/drying.

Runs go on from pass to pass and start again from their initial state after `HORIZON` steps.
The bathymetry, Manning field, tides, tracks and initial state come from the seed; the
triangulations are the repository's seeded Delaunay and structured meshes.
"""
from __future__ import annotations

import dataclasses
import functools
import math

import numpy as np
import torch

from dgswem_amd import adjoint, gpu, mesh

HORIZON = 2000
# tidal potential: amplitude (m), frequency (rad/s), elasticity factor, nodal factor, argument (deg)
POTENTIAL = [(0.242334, 1.405189e-4, 0.693, 1.02, 11.0), (0.112841, 1.454441e-4, 0.693, 1.0, 0.0),
             (0.046398, 1.378797e-4, 0.693, 1.02, 42.0), (0.141565, 7.292117e-5, 0.736, 0.93, 7.0),
             (0.100514, 6.759774e-5, 0.695, 0.9, 355.0)]


def listed():
    return [
        # the drop-in's time loop on a small basin: launch and call latency
        {"name": "coupled_1600", "kind": "coupled", "p": 1, "nx": 40, "ny": 20, "steps": 40},
        # small regional runs, between two outputs, at both orders
        {"name": "tide_5k_p1", "kind": "tide", "p": 1, "elements": 5003, "steps": 100},
        {"name": "tide_20k_p2", "kind": "tide", "p": 2, "elements": 20011, "steps": 60},
        # river reach with an inflow hydrograph, wetting/drying without limiter
        {"name": "river_30k_p1", "kind": "river", "p": 1, "nx": 201, "ny": 75, "steps": 60},
        # ordinary coastal run
        {"name": "tide_120k_p1", "kind": "tide", "p": 1, "elements": 120013, "steps": 80},
        # spherical ocean basin under the tidal potential
        {"name": "ocean_60k_p2", "kind": "ocean", "p": 2, "elements": 60007, "steps": 30},
        # large runs at both orders
        {"name": "tide_300k_p2", "kind": "tide", "p": 2, "elements": 300007, "steps": 40},
        {"name": "forecast_1m_p1", "kind": "forecast", "p": 1, "elements": 1000000, "steps": 150},
        # storm-surge ensembles at both orders
        {"name": "ensemble_16_p1", "kind": "ensemble", "p": 1, "members": 16, "low": 8000, "high": 60000,
         "steps": 60},
        {"name": "ensemble_6_p2", "kind": "ensemble", "p": 2, "members": 6, "low": 10000, "high": 50000,
         "steps": 30},
        # calibration: gradients on an all-wet basin, and of a batch of storms with a dry coast
        {"name": "gradient_50k_p1", "kind": "gradient", "p": 1, "elements": 50021, "steps": 80},
        {"name": "storm_gradient_4x25k_p2", "kind": "storm_gradient", "p": 2, "members": 4, "low": 20000,
         "high": 30000, "steps": 30},
    ]


def _between(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi], odd ones included."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["coupled", "tide", "tide", "tide", "river", "ocean", "forecast", "ensemble", "gradient",
                       "storm_gradient"])
    p = rng.choice([1, 1, 2])
    if kind == "coupled":
        return {"kind": kind, "p": p, "nx": _between(rng, 10, 90), "ny": _between(rng, 8, 40),
                "steps": rng.randint(20, 50)}
    if kind == "river":
        return {"kind": kind, "p": p, "nx": _between(rng, 40, 260), "ny": _between(rng, 20, 80),
                "steps": rng.randint(20, 60)}
    if kind == "ensemble":
        low = _between(rng, 3000, 15000)
        return {"kind": kind, "p": p, "members": rng.randint(2, 12 if p == 1 else 6), "low": low,
                "high": low * rng.randint(2, 4), "steps": rng.randint(15, 40)}
    if kind == "storm_gradient":
        low = _between(rng, 3000, 15000)
        return {"kind": kind, "p": p, "members": rng.randint(1, 4), "low": low, "high": 2 * low,
                "steps": rng.randint(10, 30)}
    if kind == "gradient":
        return {"kind": kind, "p": p, "elements": _between(rng, 3000, 60000), "steps": rng.randint(20, 80)}
    if kind == "forecast":
        return {"kind": kind, "p": 1, "elements": _between(rng, 100000, 600000), "steps": rng.randint(40, 120)}
    if kind == "ocean":
        return {"kind": kind, "p": p, "elements": _between(rng, 3000, 100000), "steps": rng.randint(20, 60)}
    return {"kind": kind, "p": p, "elements": _between(rng, 1500, 400000 if p == 1 else 200000),
            "steps": rng.randint(20, 80)}


# ------------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=48)
def _delaunay(elements, p, wet, spherical):
    kw = dict(n_elem=elements, seed=7, p=p, cfl=0.27 if p == 1 else 0.13, nsteps=HORIZON)
    if wet:
        kw.update(depth_range=(10.0, 3000.0), shelf=False, wetdry=False, slopeflag=0, cf=1e-4)
    if spherical:
        kw.update(ics=2)
    return mesh.delaunay_basin(**kw)


@functools.lru_cache(maxsize=64)
def _storm(elements, p, k):
    return mesh.storm_basin(elements, seed=70 + k, p=p, cfl=0.27 if p == 1 else 0.13, nsteps=HORIZON,
                            depth_range=(10.0, 300.0) if p == 2 else (5.0, 4000.0), cf=1e-4 if p == 2 else 0.0025)


@functools.lru_cache(maxsize=32)
def _structured(nx, ny, p, river):
    if river:
        c = mesh.structured_basin(nx=nx, ny=ny, dx=500.0, dy=500.0, depth=6.0, amp=0.4, manning=None, p=p,
                                  dt=8.0 if p == 1 else 4.0, rk_stage=3, slopeflag=0, nolifa=2, nolibf=0,
                                  cori=1.0e-4, flow_side=True, flow_amp=1.0)
    else:
        c = mesh.structured_basin(nx=nx, ny=ny, p=p, dt=10.0 if p == 1 else 6.0)
    return c


def _waves(rng, x, y, n=4):
    """Smooth field in [-1, 1] on points of the unit square: a few random plane waves."""
    f = np.zeros_like(x)
    for _ in range(n):
        f += np.cos(rng.uniform(1.0, 14.0) * x + rng.uniform(1.0, 14.0) * y + rng.uniform(0.0, 6.28)) / n
    return f


def _unit(c):
    return (c.x - c.x.min()) / np.ptp(c.x), (c.y - c.y.min()) / np.ptp(c.y)


def _seeded(c, seed, k=0):
    """The case with bathymetry, friction and boundary forcing of the seed."""
    rng = np.random.default_rng([seed, k])
    x, y = _unit(c)
    p = dataclasses.replace(c.params)
    p.emo = p.emo * rng.uniform(0.7, 1.3, (p.emo.shape[0], 1))
    p.efa = p.efa + rng.uniform(0.0, 6.0, (p.efa.shape[0], 1))
    if p.nffr:
        p.qnam = p.qnam * rng.uniform(0.7, 1.3, (p.nffr, 1))
    man = None if c.manning is None else rng.uniform(0.02, 0.03, c.np_)
    return dataclasses.replace(c, params=p, dp=c.dp * (1.0 + 0.05 * _waves(rng, x, y)), manning=man)


def _sizes(case):
    r = np.random.default_rng(case["members"])
    return [int(v) for v in np.exp(r.uniform(math.log(case["low"]), math.log(case["high"]), case["members"]))]


def _cases(case, seed):
    """The run (or the members) of a case."""
    kind, p = case["kind"], case["p"]
    if kind in ("ensemble", "storm_gradient"):
        return [_seeded(_storm(n, p, k), seed, k) for k, n in enumerate(_sizes(case))]
    if kind in ("coupled", "river"):
        c = _seeded(_structured(case["nx"], case["ny"], p, kind == "river"), seed)
        if kind == "river":                        # a bank that rises above the datum
            _, y = _unit(c)
            c = dataclasses.replace(c, dp=c.dp * (1.0 - 1.15 * y ** 4))
        return [c]
    c = _seeded(_delaunay(case["elements"], p, kind in ("ocean", "gradient"), kind == "ocean"), seed)
    if kind == "ocean":
        q = c.params
        t = np.array(POTENTIAL).T
        q.ntip, q.ntif, q.tpk, q.amigt, q.etrf, q.fft = 1, len(POTENTIAL), t[0], t[1], t[2], t[3]
        q.facet, q.pert = t[4] * math.pi / 180.0, 2.0 * math.pi / t[1]
    return [c]


def _cold(c):
    """Cold start: at rest, elements whose bottom rises above H0 dry with the surface at H0."""
    ze = np.zeros((c.ne, c.dofh))
    wd = np.ones(c.ne, np.int32)
    if c.params.nolifa >= 2:
        d = c.dp[c.nm - 1]
        z = np.maximum(c.params.h0 - d, 0.0)
        dry = z.sum(axis=1) > 0.0
        ze[dry, 0] = z[dry].mean(axis=1)
        ze[dry, 1] = -(z[dry, 0] + z[dry, 1]) / 6.0 + z[dry, 2] / 3.0
        ze[dry, 2] = 0.5 * (z[dry, 1] - z[dry, 0])
        wd[dry] = 0
    return ze, wd


def _moving(c, seed, k=0):
    """A basin in motion: smooth elevation and currents, fading out toward the dry coast."""
    rng = np.random.default_rng([seed, 100 + k])
    x, y = _unit(c)
    ze, wd = _cold(c)
    out = [ze, np.zeros_like(ze), np.zeros_like(ze)]
    fade = np.clip((c.dp - 1.0) / 10.0, 0.0, 1.0)
    speed = 0.3 * np.sqrt(10.0 / (c.dp.clip(0.0) + 10.0)) * c.dp.clip(0.0)
    for f, a in enumerate((0.4, speed, speed)):
        v = (a * fade * _waves(rng, x, y))[c.nm - 1]
        wet = wd == 1
        out[f][wet, 0] = v[wet].mean(axis=1)
        out[f][wet, 1] = -(v[wet, 0] + v[wet, 1]) / 6.0 + v[wet, 2] / 3.0
        out[f][wet, 2] = 0.5 * (v[wet, 1] - v[wet, 0])
    return out[0], out[1], out[2], wd


def _observations(case, seed, ng):
    """Observed gauge series: a slow oscillation of each gauge."""
    rng = np.random.default_rng([seed, 200])
    t = np.arange(1, case["steps"] + 1)[:, None] / case["steps"]
    return 0.3 * np.sin(6.28 * (t * rng.uniform(0.2, 1.0, (1, ng)) + rng.uniform(0.0, 1.0, (1, ng))))


def prepare(case, seed):
    kind = case["kind"]
    cs = _cases(case, seed)
    starts = [_moving(c, seed, k) for k, c in enumerate(cs)]
    solvers = [gpu.GpuSolver(c) for c in cs]
    s = solvers[0]
    if kind in ("ensemble", "storm_gradient"):
        s = gpu.Ensemble(solvers)
        for m in solvers:
            m.close()
        s.use_graph(kind == "ensemble")
    start = tuple(np.concatenate([a[j] for a in starts]) for j in range(4))
    s.set_state(*start)
    st = {"kind": kind, "steps": case["steps"], "solver": s, "start": start}
    if kind == "coupled":
        st["etamax"] = np.full(s.np_, -99999.0)
        s.set_etamax(st["etamax"])
    if kind in ("gradient", "storm_gradient"):
        ng = 20
        g = [adjoint.seeded_gauges(c, ng, seed + k) for k, c in enumerate(cs)]
        off = np.cumsum([0] + [c.ne for c in cs])
        s.set_gauges(*(np.concatenate([a[j] + (off[k] if j == 0 else 0) for k, a in enumerate(g)]) for j in range(3)))
        data = _observations(case, seed, ng * len(cs))
        st["problem"] = adjoint.MisfitProblem(solver=s, nsteps=case["steps"], data=data, weight=1.0 / data.size,
                                              state0=start, it0=0)
        st["manning"] = torch.from_numpy(np.concatenate([c.manning for c in cs])).requires_grad_()
        st["dp"] = torch.from_numpy(np.concatenate([c.dp for c in cs])).requires_grad_()
    return st


def run(state):
    s, n, kind = state["solver"], state["steps"], state["kind"]
    if kind in ("gradient", "storm_gradient"):
        state["manning"].grad = state["dp"].grad = None
        loss = adjoint.gauge_misfit(state["manning"], state["dp"], state["problem"])
        loss.backward()
        return {"loss": loss.detach(), "manning": state["manning"].grad, "dp": state["dp"].grad}
    if s.it + n > HORIZON:                         # the run ends: the next one starts
        s.set_state(*state["start"])
        s.it = 0
        if kind == "coupled":
            s.set_etamax(state["etamax"])
    if kind == "coupled":
        for _ in range(n):
            s.step(1, sync=False)
            s.nodal_update()
        eta, u, v, code, etamax = s.get_nodal()
        return {"eta": eta, "u": u, "v": v, "nodecode": code, "etamax": etamax}
    s.step(n, sync=False)
    if kind == "forecast":
        eta, u, v, code = s.nodal()
        return {"eta": eta, "u": u, "v": v, "nodecode": code}
    ze, qx, qy, wd = s.state()
    return {"ze": ze, "qx": qx, "qy": qy, "wdflg": wd}


def _elements(case):
    if case["kind"] in ("ensemble", "storm_gradient"):
        return sum(_sizes(case))
    return case.get("elements") or 2 * case["nx"] * case["ny"]


def work(case):
    """Per element and stage: the state read and written, half the scheme's base state, the element's
    geometry, depth, friction and connectivity (300 bytes at p=1, 480 at p=2), and the operations of
    the flux at each edge's points once, the quadrature, the update and the limiter.  The
    gradient's reverse sweep reads the state, the cotangents and the mesh and writes the cotangents,
    with about twice the forward's operations, after one forward sweep."""
    p, kind = case["p"], case["kind"]
    stages = 3 if kind == "river" else 2
    n = _elements(case) * stages * case["steps"]
    b, f = (300.0, 1100.0) if p == 1 else (480.0, 3400.0)
    if kind in ("gradient", "storm_gradient"):
        b, f = b + (9 if p == 1 else 18) * 8 * 3 + 84, 3.0 * f
    return {"bytes": b * n, "flops": f * n}


# ------------------------------------------------------------------------------------------------
# the same step in plain torch, 64 bits
# ------------------------------------------------------------------------------------------------
G = 9.81
# Shu-Osher coefficients [stage][earlier state] of SSP(2,2) and SSP(3,2)
RK = {2: ([[1.0], [0.5, 0.5]], [[1.0], [0.0, 0.5]]),
      3: ([[1.0], [0.087353119859156, 0.912646880140844], [0.344956917166841, 0.0, 0.655043082833159]],
          [[0.528005024856522], [0.0, 0.481882138633993], [0.022826837460491, 0.0, 0.345866039233415]])}


def _basis(p, r, s):
    """Values and derivatives of the Dubiner modes, by degree: 1, P01, P10, P02, P11, P20."""
    r, s = np.asarray(r, float), np.asarray(s, float)
    a, o = (1.0 + 2.0 * r + s) / 2.0, np.ones_like(r)
    v = [o, (1.0 + 3.0 * s) / 2.0, a]
    dr = [0 * o, 0 * o, o]
    ds = [0 * o, 1.5 * o, 0.5 * o]
    if p == 2:
        h = (1.0 - s) / 2.0
        v += [(5.0 * s * s + 2.0 * s - 1.0) / 2.0, a * (3.0 + 5.0 * s) / 2.0, 1.5 * a * a - 0.5 * h * h]
        dr += [0 * o, (3.0 + 5.0 * s) / 2.0, 3.0 * a]
        ds += [5.0 * s + 1.0, (3.0 + 5.0 * s) / 4.0 + 2.5 * a, 1.5 * a + 0.5 * h]
    return np.stack(v, -1), np.stack(dr, -1), np.stack(ds, -1)


class _Model:
    """One run of the explicit DG step on whole arrays."""

    def __init__(self, c, dev):
        self.c, q = c, c.params
        T = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)
        I = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.int64, device=dev)
        self.T, self.p, self.dof, self.dt = T, c.dg.ph, c.dofh, q.dtdp
        p, nm = self.p, c.nm.astype(np.int64) - 1
        ne, npt = len(nm), len(c.x)
        self.ne, self.np, self.nm = ne, npt, I(nm)
        X, Y = c.x[nm], c.y[nm]
        areas = (X[:, 0] - X[:, 2]) * (Y[:, 1] - Y[:, 2]) + (X[:, 2] - X[:, 1]) * (Y[:, 0] - Y[:, 2])
        # quadrature
        if p == 1:
            orb = [(1.0 / 6.0, 1.0 / 3.0)]
            self.xg, wg = np.array([-1.0, 0.0, 1.0]), np.array([1.0, 4.0, 1.0]) / 3.0
        else:
            orb = [(0.4459484909159648863, 0.2233815896780114657), (0.0915762135097707435, 0.1099517436553218676)]
            self.xg, wg = np.array([-1.0, -5.0 ** -0.5, 5.0 ** -0.5, 1.0]), np.array([1.0, 5.0, 5.0, 1.0]) / 6.0
        bc = np.array([b for a, _ in orb for b in ((a, a, 1 - 2 * a), (a, 1 - 2 * a, a), (1 - 2 * a, a, a))])
        wa = np.array([2.0 * w for _, w in orb for _ in range(3)])
        ra, sa = -bc[:, 0] + bc[:, 1] - bc[:, 2], -bc[:, 0] - bc[:, 1] + bc[:, 2]
        va, dra, dsa = _basis(p, ra, sa)
        mi = np.array([0.5, 1.0, 3.0, 1.5, 4.5, 7.5])[: self.dof]
        x = self.xg
        ve = np.stack([_basis(p, *rs)[0] for rs in ((-x, x), (-1 + 0 * x, -x), (x, -1 + 0 * x))])
        self.corner = T(_basis(1, [-1.0, 1.0, -1.0], [-1.0, -1.0, 1.0])[0])
        self.vc = T(_basis(p, [-1.0, 1.0, -1.0], [-1.0, -1.0, 1.0])[0])
        self.va, self.dra, self.dsa, self.ve = T(va), T(dra), T(dsa), T(ve)
        self.mw, self.sr = T(mi * wa[:, None]), T(mi * wa[:, None] * va)
        self.eq = T(2.0 * mi * ve * wg[:, None])
        self.psi = T(bc)
        # geometry
        A = 0.5 * areas
        self.areas = T(areas)
        self.drdx, self.dsdx = T((Y[:, 2] - Y[:, 0]) / A), T((Y[:, 0] - Y[:, 1]) / A)
        self.drdy, self.dsdy = T((X[:, 0] - X[:, 2]) / A), T((X[:, 1] - X[:, 0]) / A)
        # edges: local edge L runs from vertex L+1 to L+2; the two halves of an internal edge
        a, b = nm[:, [1, 2, 0]].ravel(), nm[:, [2, 0, 1]].ravel()
        key = np.minimum(a, b) * npt + np.maximum(a, b)
        order = np.argsort(key, kind="stable")
        same = np.flatnonzero(key[order][1:] == key[order][:-1])
        h1, h2 = order[same], order[same + 1]
        rest = np.ones(len(key), bool)
        rest[h1] = rest[h2] = False
        out = np.flatnonzero(rest)
        kind, pos = {}, {}
        n = 0
        for seg in c.open_segs:
            for i in range(len(seg) - 1):
                k = (int(min(seg[i], seg[i + 1])) - 1) * npt + int(max(seg[i], seg[i + 1])) - 1
                kind[k], pos[k] = 1, (n, int(seg[i]) - 1)
                n += 1
            n += 1
        n = 0
        for t, seg in c.land_segs:
            if t == 2:
                for i in range(len(seg) - 1):
                    k = (int(min(seg[i], seg[i + 1])) - 1) * npt + int(max(seg[i], seg[i + 1])) - 1
                    kind[k], pos[k] = 3, (n, int(seg[i]) - 1)
                    n += 1
                n += 1
        kd = np.array([kind.get(k, 2) for k in key[out]], int)

        def side(h):
            e, L = h // 3, h % 3
            va_, vb_ = nm[e, (L + 1) % 3], nm[e, (L + 2) % 3]
            dx, dy = c.x[vb_] - c.x[va_], c.y[vb_] - c.y[va_]
            ln = np.hypot(dx, dy)
            return I(e), I(L), T(dy / ln)[:, None], T(-dx / ln)[:, None], ln

        e1, L1, nx, ny, ln = side(h1)
        self.int = (e1, L1, I(h2 // 3), I(h2 % 3), nx, ny, T(ln / areas[h1 // 3])[:, None], T(ln / areas[h2 // 3])[:, None])
        self.bnd = {}
        for k in (1, 2, 3):
            h = out[kd == k]
            if len(h):
                e, L, nx, ny, ln = side(h)
                more = {}
                if k != 2:
                    pp = [pos[v] for v in key[h]]
                    at, first = np.array([v[0] for v in pp]), np.array([v[1] for v in pp])
                    flip = first != nm[h // 3, (h % 3 + 1) % 3]  # listed against the element's own direction
                    lo, hi = at + flip, at + 1 - flip
                    am, ph = (q.emo, q.efa) if k == 1 else (q.qnam, q.qnph)
                    xx = x[None, None, :]
                    if k == 1:
                        more = {"a": (T(am[:, lo]), T(am[:, hi])), "p": (T(ph[:, lo]), T(ph[:, hi]))}
                    else:
                        mid = lambda f: 0.5 * (f[:, lo] + f[:, hi])[..., None] + 0.5 * (f[:, hi] - f[:, lo])[..., None] * xx
                        more = {"a": T(mid(am)), "p": T(mid(ph))}
                self.bnd[k] = (e, L, nx, ny, T(ln / areas[h // 3])[:, None], more)
        # spherical factors at the area and edge points
        self.sph = q.ics == 2
        if self.sph:
            yv = np.stack([Y.mean(axis=1), -(Y[:, 0] + Y[:, 1]) / 6.0 + Y[:, 2] / 3.0, 0.5 * (Y[:, 1] - Y[:, 0])], 1)
            f = lambda ph: math.cos(q.sfea0) / np.cos(np.einsum("ek,...k->e...", yv, ph[..., :3]) / 6378206.4)
            self.sfq, self.sfe = T(f(va)), T(f(ve))
        self.cori = T((c.corif[nm]).mean(axis=1))[:, None]
        self.set(T(c.dp), None if c.manning is None else T(c.manning))
        rk_a, rk_b = RK[c.dg.rk_stage]
        self.rk_a, self.rk_b, s = rk_a, rk_b, c.dg.rk_stage
        C = np.zeros((s, s))
        for j in range(s):
            for i in range(j, s):
                C[i, j] = (rk_b[i][j] if j < len(rk_b[i]) else 0.0) + sum(C[l - 1, j] * rk_a[i][l] for l in range(j + 1, i + 1))
        self.ct = [0.0] + [C[k - 1].sum() for k in range(1, s)]
        if q.ntip:
            self.lon, self.cc, self.s2 = T(c.slam), T(np.cos(c.sfea) ** 2), T(np.sin(2.0 * c.sfea))
        if q.nws == 8:
            self._track()

    def set(self, dp, manning):
        d = dp[self.nm]
        self.d = d
        self.hb = torch.stack([d.mean(1), -(d[:, 0] + d[:, 1]) / 6.0 + d[:, 2] / 3.0, 0.5 * (d[:, 1] - d[:, 0])], 1)
        self.nbar = None if manning is None else manning[self.nm].mean(1)[:, None]

    # ---- hurricane
    def _track(self):
        st, rec = self.c.storm, np.asarray(self.c.storm.records, float)
        days = np.array([0, 31, 60, 91, 121, 152, 182, 213, 244, 274, 305, 335]) if st.irefyr % 4 == 0 else \
            np.array([0, 31, 59, 90, 120, 151, 181, 212, 243, 273, 304, 334])
        sec = lambda mo, dy, hr: (days[np.asarray(mo, int) - 1] + np.asarray(dy) - 1) * 86400.0 + np.asarray(hr) * 3600.0
        t = sec(rec[:, 1], rec[:, 2], rec[:, 3]) - sec(st.irefmo, st.irefday, st.irefhr)
        lat, lon, spd = rec[:, 6] / 10.0, -rec[:, 7] / 10.0, rec[:, 8] * 0.51444444
        cp, rmw, re, d2 = rec[:, 9] * 100.0, rec[:, 11] * 1.852000003180799, 6378206.4, math.pi / 180.0
        dt = np.diff(t)
        s = np.sin(np.diff(lon) * d2 / 2.0)
        tx = np.copysign(re * 2.0 * np.arcsin(np.sqrt(np.cos(lat[1:] * d2) * np.cos(lat[:-1] * d2) * s * s)) / dt, np.diff(lon))
        ty = re * np.diff(lat) * d2 / dt
        self.track = (t, np.stack([lat, lon, spd, cp, rmw, np.r_[tx[0], tx], np.r_[ty[0], ty]]))
        self.nlon, self.nlat = self.T(self.c.slam / d2), self.T(self.c.sfea / d2)

    def _met(self, time):
        t, v = self.track
        lat, lon, spd, cp, rmw, tx, ty = (float(np.interp(time, t, r)) for r in v)
        st, d2 = self.c.storm, math.pi / 180.0
        deficit = max(101300.0 - cp, 100.0)
        spd = (spd - math.hypot(tx, ty)) / st.bladj
        B = min(max(1.15 * 2.718281828459045 * spd * spd / deficit, 1.0), 2.5)
        dx, dy = (self.nlon - lon) * d2, (self.nlat - lat) * d2
        th = torch.atan2(dy, dx)
        rad = 6378206.4 * 2.0 * torch.asin(torch.sqrt(torch.sin(dy / 2) ** 2 + math.cos(lat * d2) * torch.cos(self.nlat * d2) * torch.sin(dx / 2) ** 2))
        cor = 2.0 * 2.0 * math.pi / 86164.2 * torch.sin(self.nlat * d2)
        rb = (rmw * 1000.0 / rad) ** B
        press = (cp + deficit * torch.exp(-rb)) / (1000.0 * G)
        vr = torch.sqrt(rb * torch.exp(1.0 - rb) * spd * spd + (rad * cor) ** 2 / 4.0) - rad * cor / 2.0
        f = vr.abs() / spd
        vr = vr * (1.2 if st.storm_number == 2 else 1.0)
        wx = -vr * torch.sin(th) * st.bladj * 0.88 + f * tx
        wy = vr * torch.cos(th) * st.bladj * 0.88 + f * ty
        wm = torch.sqrt(wx * wx + wy * wy)
        cd = (0.001 * (0.75 + 0.067 * wm)).clamp(max=0.0035)
        return 0.001293 * cd * wx * wm, 0.001293 * cd * wy * wm, press

    # ---- flux
    def _llf(self, zi, ze, xi, xe, yi, ye, hi, he, sfi, sfe, nx, ny, g):
        def one(z, x, y, h, sf):
            d = z + h
            u, v, gh = x / d, y / d, g * z * (0.5 * z + h)
            c2 = g * d * (ny * ny + (nx * sf) ** 2)
            c = torch.where(c2 > 0, c2, torch.ones_like(c2)).sqrt() * (c2 > 0)
            un = u * nx + v * ny
            return (x * sf * nx + y * ny, (x * u + gh) * sf * nx + x * v * ny, x * v * sf * nx + (y * v + gh) * ny, un.abs() + c)

        a, b = one(zi, xi, yi, hi, sfi), one(ze, xe, ye, he, sfe)
        em = torch.maximum(a[3], b[3])
        return [0.5 * (p + q) - 0.5 * em * j for p, q, j in zip(a, b, (ze - zi, xe - xi, ye - yi))]

    def _at(self, u, e, L, flip=False):
        ph = self.ve[L]
        ph = ph.flip(1) if flip else ph
        tr = [torch.einsum("ek,eik->ei", w[e], ph) for w in u] + [torch.einsum("ek,eik->ei", self.hb[e], ph[..., :3])]
        sf = self.sfe[e, L] if self.sph else torch.ones_like(tr[0])
        return ph, tr + [sf.flip(1) if flip and self.sph else sf]

    def rhs(self, u, wd, it, stage, met, tip, ramp, timedg):
        q = self.c.params
        wet = wd[:, None] == 1
        R = [torch.zeros_like(w) for w in u]

        def add(f, e, w):
            for i in range(3):
                R[i] = R[i].index_add(0, e, torch.einsum("ei,eik->ek", f[i], w))

        # internal edges
        e1, L1, e2, L2, nx, ny, f1, f2 = self.int
        _, a = self._at(u, e1, L1)
        _, b = self._at(u, e2, L2, True)
        F = self._llf(a[0], b[0], a[1], b[1], a[2], b[2], a[3], b[3], a[4], b[4], nx, ny, G)
        in_, ex = list(F), list(F)
        w1, w2 = wd[e1][:, None] == 1, wd[e2][:, None] == 1
        if bool((~(w1 & w2)).any()):
            big = F[0].abs() > 1e-8
            di, de = big & ~w1, big & w1 & ~w2
            mirror = lambda t: (t[1] - 2.0 * (t[1] * nx + t[2] * ny) * nx, t[2] - 2.0 * (t[1] * nx + t[2] * ny) * ny)
            mb, ma = mirror(b), mirror(a)
            r1 = self._llf(b[0], b[0], mb[0], b[1], mb[1], b[2], b[3], b[3], b[4], b[4], nx, ny, G)
            r3 = self._llf(a[0], a[0], a[1], ma[0], a[2], ma[1], a[3], a[3], a[4], a[4], nx, ny, G)
            z = self._llf(a[0], b[0], a[1], b[1], a[2], b[2], a[3], b[3], a[4], b[4], nx, ny, 0.0)
            m1, m2, m3, m4 = di & (F[0] > 0), di & (F[0] < 0), de & (F[0] < 0), de & (F[0] > 0)
            f0 = torch.where(m1, r1[0], torch.where(m3, r3[0], F[0]))
            zero = torch.zeros_like(f0)
            in_ = [f0] + [torch.where(m1, zero, torch.where(m2, z[i], torch.where(m3, r3[i], F[i]))) for i in (1, 2)]
            ex = [f0] + [torch.where(m1, r1[i], torch.where(m3, zero, torch.where(m4, z[i], F[i]))) for i in (1, 2)]
            on = (w1 | w2).expand_as(f0)
            in_, ex = ([torch.where(on, v, zero) for v in s] for s in (in_, ex))
        add(in_, e1, -f1[..., None] * self.eq[L1])
        add(ex, e2, f2[..., None] * self.eq[L2].flip(1))
        # boundary edges of wet elements
        for k, (e, L, nx, ny, fac, more) in self.bnd.items():
            _, t = self._at(u, e, L)
            z, x, y, h, sf = t
            ze, xe, ye = z, x, y
            if k == 2:
                qn = x * nx + y * ny
                xe, ye = x - 2.0 * qn * nx, y - 2.0 * qn * ny
            else:
                w, per, ff, face = (q.amig, q.per, q.ff, q.face) if k == 1 else (q.famig, q.fper, q.fff, q.fface)
                col = lambda v: self.T(v).reshape(-1, *([1] * (more["a"][0].dim() - 1 if k == 1 else 2)))
                arg = col(w * (timedg - np.floor(timedg / per) * per) + face)
                if k == 1:
                    t1, t2 = (col(ff) * ramp * A * torch.cos(arg - P) for A, P in zip(more["a"], more["p"]))
                    xg = self.T(self.xg)[None, :]
                    t1, t2 = t1.sum(0)[:, None], t2.sum(0)[:, None]
                    ze = 0.5 * (t1 + t2) + 0.5 * (t2 - t1) * xg
                    ze = torch.where(ze + h <= 0, h.abs() + q.h0, ze)
                else:
                    qn = (col(ff) * ramp * more["a"] * torch.cos(arg - more["p"])).sum(0)
                    xe, ye = -nx * qn, -ny * qn
            F = self._llf(z, ze, x, xe, y, ye, h, h, sf, sf, nx, ny, G)
            on = wet[e].expand_as(z)
            add([torch.where(on, v, torch.zeros_like(v)) for v in F], e, -fac[..., None] * self.eq[L])
        # volume quadrature
        ze, qx, qy = (w @ self.va.T for w in u)
        hq = self.hb @ self.va[:, :3].T
        d = ze + hq
        d = torch.where(wet, d, torch.ones_like(d))
        sf = self.sfq if self.sph else torch.ones_like(d)
        U, V, gh = qx / d, qy / d, G * ze * (0.5 * ze + hq)
        fric = self.T(q.tau if q.nolibf == 0 else q.cf)
        if self.nbar is not None:
            fric = (G * self.nbar ** 2 / d.clamp(min=1e-300) ** (1.0 / 3.0)).clamp(min=q.cf)
        tau = fric * torch.ones_like(d)
        if q.nolibf == 0:
            tau = q.cf * torch.ones_like(d)
        else:
            m2 = U * U + V * V
            tau = (tau * torch.where(m2 > 0, m2, torch.ones_like(m2)).sqrt() * (m2 > 0) / d).clamp(max=0.9 / self.dt)
        bx = self.hb[:, 1] * 1.5 * self.dsdx + self.hb[:, 2] * (self.drdx + 0.5 * self.dsdx)
        by = self.hb[:, 1] * 1.5 * self.dsdy + self.hb[:, 2] * (self.drdy + 0.5 * self.dsdy)
        sx = -tau * qx + G * ze * bx[:, None] * sf + self.cori * qy
        sy = -tau * qy + G * ze * by[:, None] - self.cori * qx
        px = torch.stack([-0.5 * (self.drdx + self.dsdx), 0.5 * self.drdx, 0.5 * self.dsdx], 1)
        py = torch.stack([-0.5 * (self.drdy + self.dsdy), 0.5 * self.drdy, 0.5 * self.dsdy], 1)
        if met is not None:
            wx, wy, pr = (ramp * v[self.nm] for v in met)
            sx = sx + wx @ self.psi.T - G * sf * d * (px * pr).sum(1)[:, None]
            sy = sy + wy @ self.psi.T - G * d * (py * pr).sum(1)[:, None]
        if tip is not None:
            sx = sx + ramp * G * d * sf * (px * tip[self.nm]).sum(1)[:, None]
            sy = sy + ramp * G * d * (py * tip[self.nm]).sum(1)[:, None]
        flux = ((qx * sf, qy, None), ((qx * U + gh) * sf, qx * V, sx), (qx * V * sf, qy * V + gh, sy))
        for i, (fx, fy, s) in enumerate(flux):
            v = torch.einsum("ei,ik->ek", fx, self.mw * self.dra) * self.drdx[:, None] + \
                torch.einsum("ei,ik->ek", fx, self.mw * self.dsa) * self.dsdx[:, None] + \
                torch.einsum("ei,ik->ek", fy, self.mw * self.dra) * self.drdy[:, None] + \
                torch.einsum("ei,ik->ek", fy, self.mw * self.dsa) * self.dsdy[:, None]
            if s is not None:
                v = v + s @ self.sr
            R[i] = R[i] + torch.where(wet, v, torch.zeros_like(v))
        return R

    # ---- limiter and wetting/drying
    def limit(self, u):
        out = []
        flat = self.nm.T.reshape(-1)
        for w in u:
            m = w[:, 0].detach().repeat(3)
            lo = torch.full((self.np,), 99999.0, dtype=w.dtype, device=w.device).scatter_reduce(0, flat, m, "amin")[self.nm]
            hi = torch.full((self.np,), -99999.0, dtype=w.dtype, device=w.device).scatter_reduce(0, flat, m, "amax")[self.nm]
            c = w[:, 0]
            v = torch.maximum(torch.minimum(w[:, :3] @ self.corner.T, hi), lo)
            v = list(v.T)
            for _ in range(3):
                sd = ((v[0] + v[1] + v[2]) / 3.0 - c) * 3.0
                sg = torch.copysign(torch.ones_like(sd), sd)
                dif = [(t - c) * sg > 0 for t in v]
                k = sum(t.to(c) for t in dif)
                for i in range(3):
                    red = torch.where(dif[i], sd * sg / k.clamp(min=1.0), torch.zeros_like(c))
                    k = k - dif[i].to(c)
                    red = torch.minimum(red, torch.where(sg > 0, v[i] - lo[:, i], hi[:, i] - v[i]))
                    sd = sd - red * sg
                    v[i] = v[i] - red * sg
            n = w.clone()
            n[:, 1] = -(v[0] + v[1]) / 6.0 + v[2] / 3.0
            n[:, 2] = 0.5 * (v[1] - v[0])
            out.append(n)
        return out

    def wetdry(self, u, wd):
        H0, zero, d = self.c.params.h0, 1e-6, self.d
        z = u[0][:, :3] @ self.corner.T
        h = d + z
        nd = (h <= H0 + zero).sum(1)
        avg = u[0][:, 0] + self.hb[:, 0]
        keep = (nd == 0) & (wd == 1)
        flat = (nd == 3) | ((nd > 0) & (avg <= H0 + zero))
        part = (nd > 0) & ~flat
        # redistribution: from the shallowest vertex to the deepest
        o = torch.sort(h, dim=1, stable=True)[1]
        hs = h.gather(1, o)
        d0 = hs[:, 0].clamp(min=H0) - hs[:, 0]
        d1 = (hs[:, 1] - 0.5 * d0).clamp(min=H0) - hs[:, 1]
        dh = torch.zeros_like(h).scatter(1, o, torch.stack([d0, d1, -d0 - d1], 1))
        hh = h + dh
        dry = hh <= H0 + 1e-10
        n2 = dry.sum(1)
        new = [w.clone() for w in u]
        for f in (1, 2):
            v = u[f][:, :3] @ self.corner.T
            s = (v * dry).sum(1) / (3.0 - n2).clamp(min=1.0)
            v = torch.where(dry, torch.zeros_like(v), v + s[:, None])
            v[n2 == 3] = 0.0
            m = torch.stack([v.mean(1), -(v[:, 0] + v[:, 1]) / 6.0 + v[:, 2] / 3.0, 0.5 * (v[:, 1] - v[:, 0])], 1)
            new[f][part, :3] = m[part]
        zh = hh - d
        new[0][part, 1] = (-(zh[:, 0] + zh[:, 1]) / 6.0 + zh[:, 2] / 3.0)[part]
        new[0][part, 2] = (0.5 * (zh[:, 1] - zh[:, 0]))[part]
        for f in range(3):
            new[f][part, 3:] = 0.0
            new[f][flat] = 0.0
        new[0][flat, 0] = torch.where(avg < zero, zero - self.hb[:, 0], u[0][:, 0])[flat]
        new[0][flat, 1:3] = -self.hb[flat, 1:3]
        some = (nd == 0) & ~keep
        top = torch.where(part, zh.gather(1, hh.argmax(1)[:, None])[:, 0],
                          torch.where(nd == 0, z.gather(1, h.argmax(1)[:, None])[:, 0], new[0][:, 0]))
        ok = top > -d.min(1)[0] + H0
        ok = torch.where(nd == 3, torch.zeros_like(ok), ok)
        lose = (part | some | flat) & ~ok
        for f in (1, 2):
            new[f][lose] = 0.0
        wd = torch.where(keep, wd, ok.to(wd))
        return new, wd

    def step(self, u, wd, it):
        q, dt = self.c.params, self.dt
        time = it * dt
        met = self._met(time) if q.nws == 8 else None
        us, rs = [u], []
        for k in range(len(self.rk_a)):
            ramp = math.tanh(2.0 * ((it - 1) + self.ct[k]) * dt / 86400.0 / q.dramp) if q.nramp else 1.0
            timedg = time - dt + self.ct[k] * dt
            tip = None
            if q.ntip:
                tip = 0.0
                for j in range(q.ntif):
                    n = math.floor(timedg / q.pert[j])
                    arg = q.amigt[j] * (timedg - n * q.pert[j]) + q.facet[j]
                    half = round(0.00014 / q.amigt[j]) == 1
                    am = ramp * q.etrf[j] * q.tpk[j] * q.fft[j]
                    tip = tip + am * ((self.cc if half else self.s2) * torch.cos(arg + (2.0 if half else 1.0) * self.lon))
            rs.append(self.rhs(us[-1], wd, it, k, met, tip, ramp, timedg))
            w = [sum(self.rk_a[k][j] * us[j][f] + self.rk_b[k][j] * dt * rs[j][f] for j in range(k + 1)) for f in range(3)]
            if self.c.dg.slopeflag:
                w = self.limit(w)
            if q.nolifa >= 2:
                w, wd = self.wetdry(w, wd)
            us.append(w)
        return us[-1], wd

    def nodal(self, u, wd):
        h = torch.zeros_like(u[0])
        h[:, :3] = self.hb
        z, x, y, b = (w @ self.vc.T for w in (*u, h))
        on = (wd[:, None] == 1).expand(-1, 3)
        w = torch.where(on, self.areas[:, None].expand(-1, 3), torch.zeros_like(z))
        tot = torch.zeros(self.np, dtype=z.dtype, device=z.device).index_add(0, self.nm.reshape(-1), w.reshape(-1))
        d = torch.where(on, z + b, torch.ones_like(z))
        f = lambda v: torch.zeros_like(tot).index_add(0, self.nm.reshape(-1), (w * v).reshape(-1)) / tot.clamp(min=1e-300)
        return f(z), f(x / d), f(y / d)


def exact(case, seed):
    """What `run` returns from a new state.  None where it would take too long
    and for the storm gradients, whose map has kinks at ties that no other program need break alike;
    the wet/dry flags, node codes and the maximum elevation, raised after every partial sum, have no
    64-bit value of their own."""
    kind, n = case["kind"], case["steps"]
    if kind == "storm_gradient" or _elements(case) * n * case["p"] > 200e6:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    cs = _cases(case, seed)
    got = []
    for k, c in enumerate(cs):
        m = _Model(c, dev)
        ze, qx, qy, wd = _moving(c, seed, k)
        u, w = [m.T(ze), m.T(qx), m.T(qy)], torch.as_tensor(wd, device=dev)
        if kind == "gradient":
            return _exact_gradient(case, seed, c, m, u, w)
        for it in range(1, n + 1):
            u, w = m.step(u, w, it)
        got.append([v.cpu().numpy() for v in (m.nodal(u, w) if kind in ("forecast", "coupled") else u)])
    out = [np.concatenate(v) for v in zip(*got)]
    if kind in ("forecast", "coupled"):
        more = {"etamax": None} if kind == "coupled" else {}
        return {"eta": out[0], "u": out[1], "v": out[2], "nodecode": None, **more}
    return {"ze": out[0], "qx": out[1], "qy": out[2], "wdflg": None}


def _exact_gradient(case, seed, c, m, u, w):
    from torch.utils.checkpoint import checkpoint
    el, r, s = adjoint.seeded_gauges(c, 20, seed)
    data = m.T(_observations(case, seed, 20))
    ph, el = m.T(_basis(c.dofh // 3, r, s)[0]), torch.as_tensor(el.astype(np.int64) - 1, device=u[0].device)
    mn, dp = m.T(c.manning).requires_grad_(), m.T(c.dp).requires_grad_()

    def one(z, x, y, mn, dp, it):
        m.set(dp, mn)
        v, _ = m.step([z, x, y], w, it)
        return tuple(v)

    loss = 0.0
    for it in range(1, case["steps"] + 1):
        u = checkpoint(one, *u, mn, dp, it, use_reentrant=False)
        loss = loss + ((u[0][el] * ph).sum(1) - data[it - 1]).square().sum()
    loss = loss / data.numel()
    loss.backward()
    return {"loss": loss.detach().cpu(), "manning": mn.grad.cpu(), "dp": dp.grad.cpu()}
