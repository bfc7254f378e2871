"""Timed cases of the framework's public entry points.

Each case is a pass that a user's program makes over and over: an initial
state goes in, a number of time steps (or a gradient, or a diagnostic) is
taken on the GPU, and what the program reads comes back.  The kinds:

* steps      -- SpaceDisc.SetVolField, run, GetVolField: a run between two
                snapshots
* driver     -- the reference drivers' loop: TimeDisc.CFLdt on the host, one
                Solvers call per step
* ensemble   -- independent meshes of several sizes advanced together
* gradient   -- forward and backward of adjoint.ShallowWaterRun
* tangent    -- SpaceDisc.tangent_run
* diagnostics -- Integrals and Stats of a resident state, per cell and total

Meshes, bathymetries and states are those of swe_fvm_amd.workloads (circular
wet/dry dam break, lake at rest over islands, Thacker's bowl, smooth humps
over submerged bumps), over the sizes of the tests and of bench.py, from a
few hundred cells to 4M.  Beyond 4M nothing changes but the length of a pass:
a step's data is several times the 256 MB Infinity Cache there already.
"""
import math

import numpy as np
import torch

import swe_fvm_amd as swe
from swe_fvm_amd import adjoint as AD
from swe_fvm_amd.ensemble import Ensemble

SCHEMES = {"Euler": [(0., 0., 1.)],
           "SSPRK2": [(0., 0., 1.), (.5, .5, .5)],
           "SSPRK3": [(0., 0., 1.), (.75, .25, .25), (1. / 3., 2. / 3., 2. / 3.)]}


# ------------------------------------------------------------------- cases --

def listed():
    return [
        # the reference's own driver on a small bowl: the host asks for the
        # CFL step and makes one solver call per step (latency is all)
        {"name": "driver_bowl_1k6", "kind": "driver", "field": "bowl", "n": 20, "flux": "HLL", "wave": "Einfeldt",
         "scheme": "SSPRK2", "steps": 10, "cfl": 0.15, "drain_length": False},
        # the smallest meshes stepped on the device, forward Euler in CFL mode
        {"name": "euler_lake_5k", "kind": "steps", "field": "lake", "n": 50, "flux": "HLL", "wave": "Rusanov",
         "scheme": "Euler", "steps": 100, "cfl": 0.15, "drain_length": False},
        # the Thacker comparison on its 100 x 100 grid with the convergent
        # draining option
        {"name": "bowl_40k", "kind": "steps", "field": "bowl", "n": 100, "flux": "HLLC", "wave": "Einfeldt",
         "scheme": "SSPRK2", "steps": 100, "cfl": 0.15, "drain_length": True},
        # an open channel with friction and rotation, fixed step, the third
        # order scheme, free-flow sides (a ragged size)
        {"name": "channel_62k", "kind": "steps", "field": "humps", "n": 177, "flux": "HLL", "wave": "Davis",
         "scheme": "SSPRK3", "steps": 60, "cfl": 0., "drain_length": False, "open": True},
        # the dam break at three sizes: one that lives in the caches, the
        # size of the lake test, and one that streams from HBM
        {"name": "dam_break_250k", "kind": "steps", "field": "dam", "n": 354, "flux": "HLLC", "wave": "Einfeldt",
         "scheme": "SSPRK2", "steps": 100, "cfl": 0.15, "drain_length": False},
        {"name": "dam_break_1m", "kind": "steps", "field": "dam", "n": 707, "flux": "HLLC", "wave": "Einfeldt",
         "scheme": "SSPRK2", "steps": 100, "cfl": 0.15, "drain_length": False},
        {"name": "dam_break_4m", "kind": "steps", "field": "dam", "n": 1414, "flux": "HLLC", "wave": "Einfeldt",
         "scheme": "SSPRK2", "steps": 100, "cfl": 0.15, "drain_length": False},
        # a batch of scenario runs of mixed sizes, each with its own step
        {"name": "ensemble_24x700k", "kind": "ensemble", "field": "humps", "n": 60, "n_max": 200, "members": 24,
         "flux": "HLLC", "wave": "Einfeldt", "scheme": "SSPRK2", "steps": 64, "cfl": 0.15, "drain_length": False},
        # the bathymetry inversion: one member with every intermediate kept,
        # and a batch that recomputes its segments from checkpoints
        {"name": "gradient_250k", "kind": "gradient", "field": "humps", "n": 354, "members": 1, "flux": "HLLC",
         "wave": "Einfeldt", "scheme": "SSPRK2", "steps": 20, "checkpoint": 50, "drain_length": False},
        {"name": "gradient_batch_1m", "kind": "gradient", "field": "humps", "n": 370, "members": 4, "flux": "HLLC",
         "wave": "Einfeldt", "scheme": "SSPRK2", "steps": 20, "checkpoint": 10, "drain_length": False},
        # the tangent-linear run that sensitivity studies take
        {"name": "tangent_60k", "kind": "tangent", "field": "humps", "n": 173, "members": 1, "flux": "HLLC",
         "wave": "Einfeldt", "scheme": "SSPRK2", "steps": 20, "drain_length": False},
        # monitoring of a resident run: mass, energies and health
        {"name": "diagnostics_500k", "kind": "diagnostics", "field": "lake", "n": 500, "flux": "HLLC",
         "wave": "Einfeldt", "scheme": "SSPRK2", "steps": 0, "drain_length": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps"] * 6 + ["driver", "ensemble", "gradient", "gradient", "tangent", "diagnostics"])
    c = {"kind": kind, "flux": rng.choice(["HLL", "HLLC"]), "wave": rng.choice(["Rusanov", "Davis", "Einfeldt"]),
         "scheme": rng.choice(["Euler", "SSPRK2", "SSPRK2", "SSPRK3"]), "drain_length": rng.random() < 0.3}
    if kind == "steps":
        c["field"] = rng.choice(["lake", "dam", "dam", "humps", "bowl"])
        c["n"] = _log_int(rng, 12, 300 if c["field"] == "bowl" else 1000)
        c["cfl"] = rng.choice([0.15, 0.15, 0.1, 0.])
        c["steps"] = rng.randint(40, 100)
        c["open"] = c["field"] == "humps" and rng.random() < 0.5
    elif kind == "driver":
        c.update(field=rng.choice(["bowl", "lake", "humps"]), n=_log_int(rng, 8, 150), cfl=0.15, steps=rng.randint(5, 30))
    elif kind == "ensemble":
        n = rng.randint(30, 100)
        c.update(field="humps", n=n, n_max=rng.randint(n + 1, 200), members=rng.randint(2, 24), cfl=0.15,
                 steps=rng.randint(16, 64))
    elif kind == "gradient":
        c.update(field="humps", n=_log_int(rng, 20, 370), members=rng.randint(1, 4), steps=rng.randint(5, 20),
                 checkpoint=rng.choice([4, 10, 50]))
    elif kind == "tangent":
        c.update(field="humps", n=_log_int(rng, 20, 250), members=1, steps=rng.randint(5, 20))
    else:
        c.update(field=rng.choice(["lake", "dam"]), n=_log_int(rng, 20, 700), steps=0)
    return c


# ------------------------------------------------------------------ inputs --

_MESHES = {}  # (kind, size) -> (nodes, topology, vertex ids): a mesh is read once by a program that uses it again


def _mesh(kind, n):
    if (kind, n) not in _MESHES:
        if kind == "struct":
            xyz, topo = swe.StructTriangMesh(n, n, 4. / n, -2., -2.)
        elif kind == "open":
            xyz, topo = swe.jittered_mesh(n, 0.25, n)
            t = topo.tables()
            b = np.nonzero(t["et"][:, 1] < 0)[0]
            x = 0.5 * (xyz[t["ep"][b, 0], 0] + xyz[t["ep"][b, 1], 0])
            topo = topo.with_boundary_tag(b[(x < x.min() + 1e-9) | (x > x.max() - 1e-9)], swe.FREE_FLOW)
        else:
            xyz, topo = swe.jittered_mesh(n, 0.25, n)
        _MESHES[kind, n] = xyz, topo, topo.tables()["tp"]
    return _MESHES[kind, n]


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _field(case, n, seed):
    """(Domain, T x 3 primitive state) of the case's field on a mesh of size n."""
    field = case["field"]
    kind = "struct" if field == "bowl" else "open" if case.get("open") else "jittered"
    xyz, topo, tp = _mesh(kind, n)
    xyz = xyz.copy()
    rng = np.random.default_rng(seed)
    dev = _device()
    x, y = (torch.as_tensor(xyz[:, k].copy(), device=dev) for k in (0, 1))
    tri = torch.as_tensor(tp, device=dev)
    cx, cy = (q[tri].mean(1) for q in (x, y))
    speed = torch.zeros((tri.shape[0], 2), dtype=torch.float64, device=dev)

    def bumps(q, r, amp, pos, width):
        z = torch.zeros_like(q)
        for a, (px, py), s in zip(amp, pos, width):
            z += float(a) * torch.exp(-((q - float(px)) ** 2 + (r - float(py)) ** 2) / (2 * float(s) ** 2))
        return z

    def taper(t):  # zero within 0.05 of the walls of [0, 1], one beyond 0.1
        u = torch.clamp((torch.minimum(t, 1 - t) - 0.05) / 0.05, 0, 1)
        return u * u * (3 - 2 * u)

    if field == "dam":  # h = 1 inside r < 0.2, 0.1 outside, dry pockets, Fourier bottom
        z = torch.zeros_like(x)
        for _ in range(24):
            m, k = rng.integers(-8, 9, 2)
            z += rng.uniform(-1, 1) * torch.cos(2 * math.pi * (int(m) * x + int(k) * y) + rng.uniform(0, 2 * math.pi))
        z *= 0.1 / z.abs().max()
        h = torch.where(torch.hypot(cx - 0.5, cy - 0.5) < 0.2, 1.0, 0.1).to(x)
        for _ in range(30):  # about 5 % of the cells
            ang, rad = rng.uniform(0, 2 * math.pi), rng.uniform(0.01, 0.04)
            px, py = 0.5 + 0.38 * math.cos(ang), 0.5 + 0.38 * math.sin(ang)
            h[torch.hypot(cx - px, cy - py) < rad] = 0.
        w = z[tri].mean(1) + h
    elif field == "lake":  # level 1 over bumps, two of them islands, the surface slightly disturbed
        z = bumps(x, y, np.concatenate([rng.uniform(1.05, 1.2, 2), rng.uniform(0.2, 0.95, 6)]),
                  rng.uniform(0.15, 0.85, (8, 2)), rng.uniform(0.04, 0.1, 8)) * taper(x) * taper(y)
        zc = z[tri]
        bc = zc.mean(1)
        level = 1. + bumps(cx, cy, [rng.uniform(0.01, 0.05)], rng.uniform(0.2, 0.8, (1, 2)), [0.1])
        w = torch.where(zc.amax(1) < 1., level, bc + torch.clamp(1. - bc, min=0.))
    elif field == "bowl":  # Thacker's paraboloid with a planar surface, dry rim
        z = 0.1 * (x * x + y * y)
        a, th = rng.uniform(0.2, 0.4), rng.uniform(0, 2 * math.pi)
        bc = z[tri].mean(1)
        h = torch.clamp(0.1 + 0.2 * a * (math.cos(th) * cx + math.sin(th) * cy) - 0.1 * a * a - bc, min=0.)
        om = math.sqrt(0.2)
        speed[:, 0] = torch.where(h > 0, -a * om * math.sin(th), 0.)
        speed[:, 1] = torch.where(h > 0, a * om * math.cos(th), 0.)
        w = bc + h
    else:  # humps: deep water over submerged bumps, a hump and a swell, released from a slow stream
        z = bumps(x, y, rng.uniform(0.1, 0.4, 6), rng.uniform(0.15, 0.85, (6, 2)),
                  rng.uniform(0.05, 0.15, 6)) * taper(x) * taper(y)
        w = 1. + bumps(cx, cy, [0.1], rng.uniform(0.3, 0.7, (1, 2)), [0.08])
        for _ in range(4):
            m, k = rng.integers(1, 4, 2)
            w += 1e-3 * torch.cos(2 * math.pi * (int(m) * cx + int(k) * cy) + rng.uniform(0, 2 * math.pi))
        if case.get("open"):
            speed[:, 0] = 0.1
    xyz[:, 2] = z.cpu().numpy()
    return swe.Domain(xyz, topo), torch.cat([w[:, None], speed], 1).cpu().numpy()


def _members(case, seed):
    """The case's members: one mesh, several of different sizes (ensemble) or several inversions of one mesh."""
    m = case.get("members", 1)
    if case["kind"] == "ensemble":
        sizes = np.round(np.exp(np.linspace(math.log(case["n"]), math.log(case["n_max"]), m))).astype(int)
    else:
        sizes = [case["n"]] * m
    return [_field(case, int(n), 1000 * seed + k) for k, n in enumerate(sizes)]


def _physics(case):
    opts = swe.OPT_DRAIN_LENGTH if case["drain_length"] else 0
    cor, tau = 0., 0.
    if case.get("open"):
        opts, cor, tau = opts | swe.OPT_FRICTION, 0.1, 0.05
    return opts, cor, tau


def _fixed_dt(case):
    return (4. if case["field"] == "bowl" else 1.) * 0.05 / case["n"]


class _State:
    pass


def _inputs(case, seed):
    s = _State()
    s.case = case
    mem = _members(case, seed)
    rng = np.random.default_rng([seed, 77])
    s.options, s.cor, s.tau = _physics(case)
    if case["kind"] == "ensemble":
        s.doms, s.prims = [d for d, _ in mem], [p for _, p in mem]
        return s
    s.dom = mem[0][0] if len(mem) == 1 else swe.stack_domains([d for d, _ in mem])[0]
    s.prim = np.concatenate([p for _, p in mem])
    s.z = s.dom.geometry[:, 2].copy()
    if case["kind"] == "gradient":
        s.bar = np.zeros_like(s.prim)  # the adjoint of a misfit: gauges, and a weak pull on every cell
        s.bar[:, :] = 1e-3 * rng.standard_normal(s.prim.shape)
        g = rng.choice(s.prim.shape[0], min(256, s.prim.shape[0]), replace=False)
        s.bar[g, 0] += rng.standard_normal(g.shape[0])
    elif case["kind"] == "tangent":
        s.dir, s.zdir = rng.standard_normal(s.prim.shape), 1e-2 * rng.standard_normal(s.z.shape)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    flux = getattr(swe.Fluxes, case["flux"])[getattr(swe.Wavespeeds, case["wave"])]
    if case["kind"] == "ensemble":
        s.ens = Ensemble(flux, s.doms, s.prims, cor=s.cor, tau=s.tau, options=s.options)
        return s
    s.sd = swe.SpaceDisc(flux, s.dom, s.prim, cor=s.cor, tau=s.tau, options=s.options)
    return s


# -------------------------------------------------------------------- pass --

def run(s):
    c = s.case
    if c["kind"] == "steps":
        s.sd.SetVolField(s.prim)
        s.sd.run(c["scheme"], c["steps"], dt=0. if c["cfl"] > 0 else _fixed_dt(c), cfl=c["cfl"])
        return s.sd.GetVolField()
    if c["kind"] == "driver":
        s.sd.SetVolField(s.prim)
        td = swe.TimeDisc(s.sd)
        s.sd.ComputeInterfaceValues()
        s.sd.ComputeFluxes()
        step, dts = getattr(swe.Solvers, c["scheme"]), []
        for _ in range(c["steps"]):
            dts.append(td.CFLdt())
            step(td, dts[-1])
        return {"state": s.sd.GetVolField(), "dts": np.array(dts)}
    if c["kind"] == "ensemble":
        s.ens.reset()
        s.ens.set_states(s.prims)
        s.ens.run(c["scheme"], cfl=c["cfl"], t_end=10., max_steps=c["steps"])
        t, n = s.ens.times()
        return {"state": np.concatenate(s.ens.states()), "t": t, "steps": n}
    if c["kind"] == "gradient":
        prim = torch.tensor(s.prim, requires_grad=True)
        z = torch.tensor(s.z, requires_grad=True)
        out = AD.ShallowWaterRun.apply(prim, z, s.sd, c["steps"], c["scheme"], _fixed_dt(c), c["checkpoint"])
        gp, gz = torch.autograd.grad(out, (prim, z), torch.from_numpy(s.bar))
        return {"state": out.detach(), "state_grad": gp, "z_grad": gz}
    if c["kind"] == "tangent":
        s.sd.SetVolField(s.prim)
        dot, _ = s.sd.tangent_run(s.dir, c["steps"], z_dot=s.zdir, scheme=c["scheme"], dt=_fixed_dt(c))
        return {"state": s.sd.GetVolField(), "tangent": dot}
    total, cells = s.sd.Integrals(per_cell=True)
    st = s.sd.Stats()
    return {"total": total, "cells": cells, "nonfinite": st["nonfinite"],
            "extremes": np.array([st["hmin"], st["hmax"], st["umax"], st["cmax"]])}


def _cells(case):
    if case["kind"] == "ensemble":
        m = case["members"]
        return int(sum(2 * round(n) ** 2 for n in np.exp(np.linspace(math.log(case["n"]), math.log(case["n_max"]), m))))
    return (4 if case["field"] == "bowl" else 2) * case["n"] ** 2 * case.get("members", 1)


def work(case):
    """Per stage and cell: the state in and out (24 B each), 3 neighbours and
    3 nodes by index (24 B), half a node (12 B), from the second stage on the
    step's first state (24 B); a host state crosses once each way (24 B)."""
    T = _cells(case)
    ns = len(SCHEMES[case["scheme"]])
    step = 84. * ns + 24. * (ns - 1)
    flops = 430. * ns
    if case["kind"] == "diagnostics":
        return {"bytes": T * (24. + 24. + 12. + 24.), "flops": 200. * T}
    if case["kind"] == "gradient":  # the state, its adjoint and the corner heights' once more backwards
        return {"bytes": T * (case["steps"] * (2 * step + 72. * ns) + 120.), "flops": 4 * flops * T * case["steps"]}
    if case["kind"] == "tangent":
        return {"bytes": T * (case["steps"] * 2 * step + 96.), "flops": 3 * flops * T * case["steps"]}
    return {"bytes": T * (case["steps"] * step + 48.), "flops": flops * T * case["steps"]}


# --------------------------------------------------------- 64-bit reference --

def _sel(c, a, b):
    return torch.where(c, a, b)


def _min(a, b):
    return _sel(b < a, b, a)


def _max(a, b):
    return _sel(a < b, b, a)


def _wet(h):
    return h > 1e-12


def _plane(p0, p1, p2):
    """Gradient of the plane through three points (x, y, z), 2x2 with partial pivoting."""
    a, b = [q - o for q, o in zip(p1, p0)], [q - o for q, o in zip(p2, p0)]
    swap = b[0].abs() > a[0].abs()
    a, b = [_sel(swap, v, u) for u, v in zip(a, b)], [_sel(swap, u, v) for u, v in zip(a, b)]
    m = b[0] / a[0]
    gy = (b[2] - m * a[2]) / (b[1] - m * a[1])
    return (a[2] - a[1] * gy) / a[0], gy


def _cubic_root(b, c, d, lo, hi):
    """Root of x^3 + b x^2 + c x + d between lo and hi by halving; the nearer end where the signs agree."""
    f = lambda x: ((x + b) * x + c) * x + d  # noqa: E731
    flo, fhi = f(lo), f(hi)
    end = _sel(flo.abs() < fhi.abs(), lo, hi)
    none = torch.signbit(flo) == torch.signbit(fhi)
    for _ in range(60):
        x = 0.5 * (lo + hi)
        up = torch.signbit(flo) != torch.signbit(f(x))
        lo, hi = _sel(up, lo, x), _sel(up, x, hi)
    return _sel(none, end, 0.5 * (lo + hi))


class _Plain:
    """One mesh (or several side by side) stepped with torch operations in 64 bits."""

    def __init__(self, geometry, tables, case, options, cor, tau, member=None):
        dev = _device()
        t = {k: torch.as_tensor(np.ascontiguousarray(v), device=dev) for k, v in tables.items()}
        self.x, self.y = (torch.as_tensor(geometry[:, k].copy(), device=dev) for k in (0, 1))
        self.ep, self.et, self.tp, self.te, self.tt = (t[k] for k in ("ep", "et", "tp", "te", "tt"))
        self.hllc, self.wave, self.cor = case["flux"] == "HLLC", case["wave"], cor
        self.fric = tau if options & swe.OPT_FRICTION else 0.
        self.by_len = bool(options & swe.OPT_DRAIN_LENGTH)
        self.member = None if member is None else torch.as_tensor(member, device=dev)
        X, Y, tp, ep = self.x[self.tp], self.y[self.tp], self.tp, self.ep
        self.cx, self.cy = ((q[:, 0] * (1 / 3) + q[:, 1] * (1 / 3)) + q[:, 2] * (1 / 3) for q in (X, Y))
        self.area = 0.5 * ((X[:, 1] - X[:, 0]) * (Y[:, 2] - Y[:, 0]) - (X[:, 2] - X[:, 0]) * (Y[:, 1] - Y[:, 0])).abs()
        dx, dy = self.x[ep[:, 1]] - self.x[ep[:, 0]], self.y[ep[:, 1]] - self.y[ep[:, 0]]
        self.len = torch.sqrt(dx * dx + dy * dy)
        self.mx, self.my = (0.5 * (q[ep[:, 0]] + q[ep[:, 1]]) for q in (self.x, self.y))
        tx, ty = dx / self.len, dy / self.len
        f = self.et[:, 0]
        flip = (self.cx[f] - self.x[ep[:, 0]]) * ty - tx * (self.cy[f] - self.y[ep[:, 0]]) > 0
        self.tx, self.ty = _sel(flip, -tx, tx), _sel(flip, -ty, ty)  # the outward normal of et0 is (ty, -tx)
        self.inner = torch.nonzero(self.et[:, 1] != swe.SOLID_WALL)[:, 0]
        self.wall = torch.nonzero(self.et[:, 1] == swe.SOLID_WALL)[:, 0]
        right = _sel(self.et[:, 1] < 0, f, self.et[:, 1])
        self.left, self.right = f[self.inner], right[self.inner]
        self.dmin = _min(2 * self.area[self.left] / self.len[self.inner], 2 * self.area[self.right] / self.len[self.inner])
        self.bnd = (self.tt < 0).any(1)
        self.sign = _sel(self.et[self.te, 0] == torch.arange(tp.shape[0], device=dev)[:, None], 1., -1.).to(self.x)

    def level(self, zmin, zmax, bc, w):
        """The constant level that holds the cell's water (partially wet cells)."""
        mid = 3 * bc - zmin - zmax
        lim = mid + (zmax - mid) * (zmax - mid) / (zmax - zmin) / 3
        h = w - bc
        y = 3 * h * (zmax - zmin) * (mid - zmin)
        low = zmin + torch.sign(y) * y.abs().pow(1 / 3)
        k = zmax - zmin
        high = _cubic_root(-3 * zmax, 3 * (mid * zmax + zmax * zmin - mid * zmin),
                           k * (3 * h * (zmax - mid) - mid * (mid + zmin)) - zmin * zmin * zmax, mid, zmax)
        return _sel(w >= zmax, w, _sel(w <= lim, low, high))

    def reconstruct(self, w, z):
        """Level at the centroid, gradient and class (0 dry, 1 partially, 2 fully wet) of every cell."""
        zc = z[self.tp]
        bc = (zc[:, 0] * (1 / 3) + zc[:, 1] * (1 / 3)) + zc[:, 2] * (1 / 3)
        zmin, zmax = _min(_min(zc[:, 0], zc[:, 1]), zc[:, 2]), _max(_max(zc[:, 0], zc[:, 1]), zc[:, 2])
        dry = ~_wet(w - bc)
        cls = _sel(dry, 0, _sel(~self.bnd & (zmax < w), 2, 1))
        X, Y = self.x[self.tp], self.y[self.tp]
        w0, gx, gy = w, torch.zeros_like(w), torch.zeros_like(w)
        d = torch.nonzero(dry)[:, 0]
        if d.numel():
            g = _plane(*[(X[d, k], Y[d, k], zc[d, k]) for k in range(3)])
            w0, gx, gy = (a.index_put((d,), v) for a, v in ((w0, bc[d]), (gx, g[0]), (gy, g[1])))
        part = torch.nonzero((cls == 1) & ~(w >= zmax))[:, 0]
        if part.numel():
            w0 = w0.index_put((part,), self.level(zmin[part], zmax[part], bc[part], w[part]))
        first = w0  # the level of partially wet cells after the first pass
        i = torch.nonzero(cls == 2)[:, 0]
        nb = self.tt[i]
        i = i[~(dry[nb]).any(1)]
        nb, e = self.tt[i], self.te[i]
        full = ~self.bnd[nb] & (zmax[nb] < w[nb])
        ze = 0.5 * (z[self.ep[e, 0]] + z[self.ep[e, 1]])
        a = _sel(first[nb] - ze >= 0, first[nb], ze)
        px, py = _sel(full, self.cx[nb], self.mx[e]), _sel(full, self.cy[nb], self.my[e])
        pz = _sel(full, w[nb], 0.5 * (w[i][:, None] + a))
        g0, g1 = _plane(*[(px[:, k], py[:, k], pz[:, k]) for k in range(3)])
        ok = torch.ones_like(i, dtype=torch.bool)
        for k in range(3):
            at = g0 * (X[i, k] - self.cx[i]) + g1 * (Y[i, k] - self.cy[i]) + w[i]
            ok = ok & _wet(at - zc[i, k])
            v = w[i] + (g0 * (self.mx[e[:, k]] - self.cx[i]) + g1 * (self.my[e[:, k]] - self.cy[i]))
            lo, hi = _min(w[i], w[nb[:, k]]), _max(w[i], w[nb[:, k]])
            ok = ok & (lo <= v) & (v <= hi)
        gx = gx.index_put((i,), _sel(ok, g0, torch.zeros_like(g0)))
        gy = gy.index_put((i,), _sel(ok, g1, torch.zeros_like(g1)))
        q = torch.nonzero((cls == 1) & ~(w > zmax) & ~(zmax - zmin < 1e-13))[:, 0]
        if q.numel():
            w0, gx, gy = self.shore(q, z, zc, bc, w, first, gx, gy, w0)
        return w0, gx, gy, cls, bc

    def shore(self, q, z, zc, bc, w, first, gx, gy, w0):
        """Second pass: the plane of partially wet cells from the highest level around their lowest vertex."""
        X, Y = self.x[self.tp], self.y[self.tp]
        at = first[:, None] + (gx[:, None] * (X - self.cx[:, None]) + gy[:, None] * (Y - self.cy[:, None]))
        at = _sel(at - zc >= 0, at, zc)
        top = z.scatter_reduce(0, self.tp.reshape(-1), at.reshape(-1), "amax")
        o = torch.argsort(zc[q], dim=1, stable=True)
        pick = lambda a: [torch.gather(a[q], 1, o)[:, k] for k in range(3)]  # noqa: E731
        Qx, Qy, Qz = pick(X), pick(Y), pick(zc)
        w23 = top[torch.gather(self.tp[q], 1, o)[:, 0]]
        b23, b12, b13 = Qz
        h23, hi = w23 - b23, w[q] - bc[q]
        rb, rh = (b12 - b23) / (b13 - b23), hi / h23
        d1, d2 = h23 * rb / 3, h23 * (2 * b13 - b12 - b23) / (b13 - b23) / 3
        k2, k3 = torch.sqrt(3 * rh / rb), torch.sqrt(3 * rh * rb)
        mix = lambda t, m, n: [t * Qx[m] + (1 - t) * Qx[n], t * Qy[m] + (1 - t) * Qy[n], t * Qz[m] + (1 - t) * Qz[n]]  # noqa: E731
        p1a, p2a = mix(k2, 1, 0), mix(k3, 2, 0)
        dw = 1.5 * (hi - d2)
        p1b, p2b = [Qx[1], Qy[1], Qz[1] + dw + (1 - rb) * h23], [Qx[2], Qy[2], Qz[2] + dw]
        al, be = 3 * rh, (b13 - b12) / (b13 - b23)
        k1 = 1 - _cubic_root(torch.zeros_like(be), (al - 3) / be, (1 + be - al) / (be * be), torch.zeros_like(be), torch.ones_like(be))
        p1c = [Qx[1], Qy[1], b12 + k1 / (1 - be * (1 - k1)) * be * h23]
        p2c = mix(k1, 2, 1)
        low, high = hi <= d1, hi >= d2
        p1 = [_sel(low, a, _sel(high, b, c)) for a, b, c in zip(p1a, p1b, p1c)]
        p2 = [_sel(low, a, _sel(high, b, c)) for a, b, c in zip(p2a, p2b, p2c)]
        g0, g1 = _plane([Qx[0], Qy[0], w23], p1, p2)
        keep = low | high | ~(k1 < 1e-13)
        q, g0, g1 = q[keep], g0[keep], g1[keep]
        lev = w23[keep] + (g0 * (self.cx[q] - Qx[0][keep]) + g1 * (self.cy[q] - Qy[0][keep]))
        return w0.index_put((q,), lev), gx.index_put((q,), g0), gy.index_put((q,), g1)

    def slot(self, m, c, e, ze):
        """Value of cell c's reconstruction at the midpoint of edge e."""
        w0, gx, gy, u, v = m
        a = w0[c] + (gx[c] * (self.mx[e] - self.cx[c]) + gy[c] * (self.my[e] - self.cy[c]))
        h = a - ze
        on = (h >= 0) & _wet(h)
        fac = _sel(h < 1e-3, math.sqrt(2.) * h / torch.sqrt(h * h + 1e-6), torch.ones_like(h))
        zero = torch.zeros_like(h)
        return _sel(on, a, ze), _sel(on, u[c] * fac, zero), _sel(on, v[c] * fac, zero)

    def fluxes(self, m, w, bc, z):
        """Numerical flux of every edge, outward of its first cell, and the length-to-wavespeed of the inner ones."""
        zero = torch.zeros_like(self.len)
        F = [zero, zero, zero]
        k = self.wall
        h = (w - bc)[self.et[k, 0]]
        p = _sel(_wet(h), 0.5 * h * h, torch.zeros_like(h))
        F[1], F[2] = F[1].index_put((k,), p * self.ty[k]), F[2].index_put((k,), p * -self.tx[k])
        k = self.inner
        ze = 0.5 * (z[self.ep[k, 0]] + z[self.ep[k, 1]])
        L, R = self.slot(m, self.left, k, ze), self.slot(m, self.right, k, ze)
        on = torch.nonzero((L[0] - ze) + (R[0] - ze) > 1e-10)[:, 0]
        k, ze, L, R = k[on], ze[on], [q[on] for q in L], [q[on] for q in R]
        tx, ty = self.tx[k], self.ty[k]
        nx, ny = ty, -tx
        hl, hr = L[0] - ze, R[0] - ze
        ul, vl, ur, vr = L[1] * nx + L[2] * ny, L[1] * tx + L[2] * ty, R[1] * nx + R[2] * ny, R[1] * tx + R[2] * ty
        cl, cr = torch.sqrt(hl), torch.sqrt(hr)
        if self.wave == "Rusanov":
            al = -_max(ul.abs() + cl, ur.abs() + cr)
            ar = -al
        elif self.wave == "Davis":
            al, ar = _min(ul - cl, ur - cr), _max(ul + cl, ur + cr)
        else:
            ro, co = (cl * ul + cl * ur) / (cl + cr), torch.sqrt(0.5 * (hl + hr))
            al, ar = _min(ul - cl, ro - co), _max(ur + cr, ro + co)

        def flux(h, u, v):
            s = _sel(_wet(h), h, torch.ones_like(h))
            hn = h * u * nx + h * v * ny
            f = hn, hn / s * (h * u) + 0.5 * h * h * nx, hn / s * (h * v) + 0.5 * h * h * ny
            return [_sel(_wet(h), q, torch.zeros_like(q)) for q in f]

        Fl, Fr = flux(hl, L[1], L[2]), flux(hr, R[1], R[2])
        Ul, Ur = (hl, hl * L[1], hl * L[2]), (hr, hr * R[1], hr * R[2])
        nil = torch.zeros_like(hl)
        if self.hllc:
            us = ((ar - ur) * hr * ur - (al - ul) * hl * ul + 0.5 * (hl * hl - hr * hr)) / (hr * (ar - ur) - hl * (al - ul))
            right = us <= 0
            h, u, vt, s = _sel(right, hr, hl), _sel(right, ur, ul), _sel(right, vr, vl), _sel(right, ar, al)
            star = h * (s - u) / (s - us)
            s = _sel(right, _max(nil, ar), _min(nil, al))
            Us = star, star * (vt * tx + us * ty), star * (vt * nx + us * ny)
            G = [_sel(right, fr, fl) + s * (a - _sel(right, b, c)) for fr, fl, a, b, c in zip(Fr, Fl, Us, Ur, Ul)]
            speed = _max(torch.full_like(al, 1e-13), _max(al, ar))
            live = torch.ones_like(right)
        else:
            al, ar = _min(nil, al), _max(nil, ar)
            live = ar - al > 1e-10
            den = _sel(live, ar - al, torch.ones_like(al))
            G = [_sel(live, (ar * fl - al * fr + al * ar * (b - a)) / den, nil) for fl, fr, a, b in zip(Fl, Fr, Ul, Ur)]
            speed = _max(-al, ar)
        F = [f.index_put((k,), g) for f, g in zip(F, G)]
        lw = _sel(live, self.dmin[on] / (abs(self.cor) + speed), torch.ones_like(speed)).detach()
        return F, lw, self.left[on]

    def limits(self, lw, cell):
        """The smallest length-to-wavespeed (of each member)."""
        if self.member is None:
            return torch.clamp(lw.min(), max=1.) if lw.numel() else torch.ones((), device=lw.device, dtype=lw.dtype)
        r = torch.ones(int(self.member.max()) + 1, dtype=lw.dtype, device=lw.device)
        return r.scatter_reduce(0, self.member[cell], lw, "amin")

    def stage(self, S, U0, z, coef, dt, cfl):
        a0, a1, cc = coef
        w, u, v = S
        w0, gx, gy, cls, bc = self.reconstruct(w, z)
        nil = torch.zeros_like(w)
        m = w0, gx, gy, _sel(cls == 0, nil, u), _sel(cls == 0, nil, v)
        F, lw, cell = self.fluxes(m, w, bc, z)
        if dt is None:
            dt = cfl * self.limits(lw, cell)
        step = dt if self.member is None else dt[self.member]
        d = cc * step
        h = w - bc
        out = self.sign * F[0][self.te]
        if self.by_len:
            out = out * self.len[self.te]
        out = _max(torch.zeros_like(out), out)
        out = out[:, 0] + out[:, 1] + out[:, 2]
        drain = _sel(_wet(h), _sel(out > 1e-13, self.area * h / _sel(out > 1e-13, out, torch.ones_like(out)),
                                   torch.full_like(h, math.inf)), nil)
        r = [nil, nil, nil]
        for k in range(3):
            e, sg, nb = self.te[:, k], self.sign[:, k], self.tt[:, k]
            other = _sel(nb < 0, torch.full_like(drain, math.inf), drain[_sel(nb < 0, torch.zeros_like(nb), nb)])
            dk = _min(d + nil, _sel(sg * F[0][e] > 0, drain, other))
            ze = 0.5 * (z[self.ep[e, 0]] + z[self.ep[e, 1]])
            sw, su, sv = self.slot(m, slice(None), e, ze)
            he, ce = sw - ze, self.len[e] / self.area
            p = 0.5 * he * he
            nx, ny = sg * self.ty[e], -sg * self.tx[e]
            s1, s2 = gx - self.cor * sv, gy + self.cor * su
            r[0] = r[0] - dk * sg * ce * F[0][e]
            r[1] = r[1] - dk * sg * ce * F[1][e] - d / 3 * s1 * he + dk * (nx * ce * p)
            r[2] = r[2] - dk * sg * ce * F[2][e] - d / 3 * s2 * he + dk * (ny * ce * p)
        if self.fric:
            r[1], r[2] = r[1] - d * self.fric * h * m[3], r[2] - d * self.fric * h * m[4]
        U = h, h * u, h * v
        if a0:
            h0 = U0[0] - bc
            U = [a0 * a + a1 * b for a, b in zip((h0, h0 * U0[1], h0 * U0[2]), U)]
        H = [a + b for a, b in zip(U, r)]
        wet = _wet(H[0])
        safe = _sel(wet, H[0], torch.ones_like(H[0]))
        inv = _sel(safe < 1e-3, math.sqrt(2.) * safe / torch.sqrt(safe ** 4 + 1e-12), 1. / safe)
        new = _sel(wet, H[0] + bc, bc), _sel(wet, H[1] * inv, nil), _sel(wet, H[2] * inv, nil)
        return new, dt, lw, cell

    def step(self, S, z, scheme, dt=None, cfl=0.15, clip=None):
        U0, cur, last = S, S, None
        for n, coef in enumerate(SCHEMES[scheme]):
            if n == 0 and dt is None and clip is not None:  # members end at their last time
                full = self.stage(cur, U0, z, coef, None, cfl)[1]
                dt = torch.minimum(full, clip)
            cur, dt, *last = self.stage(cur, U0, z, coef, dt, cfl)
        return cur, dt, last


def _integrals(P, S, z):
    """Mass, kinetic and potential energy of every cell; partially wet cells by quadrature over 100 sub-triangles."""
    w, u, v = S
    w0, gx, gy, cls, bc = P.reconstruct(w, z)
    h = w - bc
    out = torch.stack([h, 0.5 * h * (u * u + v * v), 0.5 * h * h + h * bc], 1) * P.area[:, None]
    out[cls == 0] = 0.
    q = torch.nonzero(cls == 1)[:, 0]
    X, Y, Z = P.x[P.tp[q]], P.y[P.tp[q]], z[P.tp[q]]
    pts = [torch.stack([a[:, k] for a in (X, Y, Z)], 1) for k in range(3)]
    n = 10
    di, dj = (pts[1] - pts[0]) / n, (pts[2] - pts[0]) / n
    acc = torch.zeros((q.shape[0], 2), dtype=w.dtype, device=w.device)

    def add(p):
        a = w0[q] + (gx[q] * (p[:, 0] - P.cx[q]) + gy[q] * (p[:, 1] - P.cy[q]))
        d = a - p[:, 2]
        on = d >= 0
        d = _sel(on, d, torch.zeros_like(d))
        acc[:, 0] += 0.5 * d * _sel(on, u[q] * u[q] + v[q] * v[q], torch.zeros_like(d)) / n
        acc[:, 1] += (0.5 * d * d + d * p[:, 2]) / n

    for a in range(n):
        for b in range(n - a):
            c = pts[0] + a * di + b * dj + (di + dj) / 3
            add(c)
            if b < n - a - 1:
                add(c + (di + dj) / 3)
    out[q, 1:] = P.area[q][:, None] * acc / n
    return out


def exact(case, seed):
    s = _inputs(case, seed)
    ensemble = case["kind"] == "ensemble"
    dom = swe.stack_domains(s.doms)[0] if ensemble else s.dom
    prim = np.concatenate(s.prims) if ensemble else s.prim
    dev = _device()
    member = np.repeat(np.arange(len(s.prims)), [p.shape[0] for p in s.prims]) if ensemble else None
    P = _Plain(dom.geometry, dom.topology.tables(), case, s.options, s.cor, s.tau, member)
    z = torch.as_tensor(dom.geometry[:, 2].copy(), device=dev)
    S = tuple(torch.as_tensor(prim[:, k].copy(), device=dev) for k in range(3))
    host = lambda q: torch.stack(tuple(q), 1).cpu()  # noqa: E731
    dt = None if case.get("cfl") else torch.tensor(_fixed_dt(case), dtype=torch.float64, device=dev)
    if case["kind"] in ("steps", "driver") or ensemble:
        dts, t = [], torch.zeros(len(s.prims) if ensemble else 1, dtype=torch.float64, device=dev)
        with torch.no_grad():
            if case["kind"] == "driver":
                w0, gx, gy, cls, bc = P.reconstruct(S[0], z)
                nil = torch.zeros_like(w0)
                m = w0, gx, gy, _sel(cls == 0, nil, S[1]), _sel(cls == 0, nil, S[2])
                last = P.fluxes(m, S[0], bc, z)[1:]
            for _ in range(case["steps"]):
                if case["kind"] == "driver":
                    dts.append(case["cfl"] * P.limits(*last))
                    S, _, last = P.step(S, z, case["scheme"], dt=dts[-1])
                else:
                    S, d, _ = P.step(S, z, case["scheme"], dt=dt, cfl=case["cfl"], clip=10. - t if ensemble else None)
                    t = t + d
        if case["kind"] == "driver":
            return {"state": host(S), "dts": torch.stack(dts).cpu()}
        if ensemble:
            return {"state": host(S), "t": t.cpu(), "steps": torch.full((len(s.prims),), case["steps"])}
        return host(S)
    if case["kind"] == "diagnostics":
        with torch.no_grad():
            cells = _integrals(P, S, z)
            w0, gx, gy, cls, bc = P.reconstruct(S[0], z)
            h, sp = S[0] - bc, torch.hypot(S[1], S[2])
            on = _wet(h)
            ext = torch.stack([h.min(), h.max(), sp[on].max(), (sp + torch.sqrt(torch.clamp(h, min=0.)))[on].max()])
        return {"total": cells.sum(0).cpu(), "cells": cells.cpu(), "nonfinite": 0, "extremes": ext.cpu()}
    if case["kind"] == "tangent":  # forward mode, step by step
        dot = tuple(torch.as_tensor(s.dir[:, k].copy(), device=dev) for k in range(3))
        zd = torch.as_tensor(s.zdir, device=dev)
        for _ in range(case["steps"]):
            # J d by two reverse sweeps: the gradient of y . (J^T y) at a dummy y
            X = [q.detach().requires_grad_() for q in S + (z,)]
            out, _, _ = P.step(tuple(X[:3]), X[3], case["scheme"], dt=dt)
            y = [torch.ones_like(o).requires_grad_() for o in out]
            g = torch.autograd.grad(out, X, y, create_graph=True)
            dot = torch.autograd.grad(g, y, list(dot) + [zd], allow_unused=True)
            S = tuple(o.detach() for o in out)
        return {"state": host(S), "tangent": host(dot)}
    states = [S]
    with torch.no_grad():
        for _ in range(case["steps"]):
            states.append(P.step(states[-1], z, case["scheme"], dt=dt)[0])
    bar = [torch.as_tensor(s.bar[:, k].copy(), device=dev) for k in range(3)]
    zbar = torch.zeros_like(z)
    for S in reversed(states[:-1]):
        X = [q.detach().requires_grad_() for q in S + (z,)]
        *bar, zb = torch.autograd.grad(P.step(tuple(X[:3]), X[3], case["scheme"], dt=dt)[0], X, bar)
        zbar += zb
    return {"state": host(states[-1]), "state_grad": host(bar), "z_grad": zbar.cpu()}
