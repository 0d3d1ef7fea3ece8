"""Timed cases: what a user of the lattice-Boltzmann engine has it do.

A pass of a stepping case is one output interval of a simulation: a number of
steps and the fields that a program then writes (density, velocity, colour,
viscosity).  A pass of a solve is the call that returns the permeability, and
a pass of a batch is a set of requests from their admission to their results.
Contexts, node lists and initial states are made once, before the first pass;
each pass goes on from the state that the last one left.

listed() and draw() give the cases, prepare() the state, run() one pass,
work() the bytes and operations of a pass, exact() the results of the first
pass in plain torch, in 64 bits, on the dense box.
"""
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "badchimp-cpp_amd"))

import lbamd  # noqa: E402
from lbamd.halo import exchange, exchange_lists  # noqa: E402

LATTICE = {"D2Q9": lbamd.D2Q9, "D3Q19": lbamd.D3Q19}
PRECISION = {"f64": lbamd.FP64, "f32s": lbamd.FP32S, "f16s": lbamd.FP16S}
BYTES = {"f64": 8, "f32s": 4, "f16s": 2}

FORCE = 1e-6  # body force along x, as in the permeability and channel workloads
TAU = {"bgk": 1.0, "trt_sym": 1.0, "trt_anti": 0.875}
TWO_PHASE = {"tau0": 1.0, "tau1": 1.0, "sigma": 0.01, "beta": 0.7}
MOMX = 1e-4  # mean momentum along x that the flux controller holds
TOL = 1e-12  # relative change of k at which a solve stops; the step limits here come first
POOL = 8 << 30


# ------------------------------------------------------------------- cases
def _case(name, kind, lattice, precision, shape, steps, periodic="x", porosity=0.40, radius=8.0, **more):
    nx, ny, nz = tuple(shape) + (1,) * (3 - len(shape))
    c = {"kind": kind, "lattice": lattice, "precision": precision, "nx": nx, "ny": ny, "nz": nz,
         "periodic": periodic, "porosity": porosity, "radius": radius, "steps": steps, "sample": 1}
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the plain channel of the reference's std_case: a small node list, where
        # the latency of a step counts
        _case("channel", "step", "D2Q9", "f64", (256, 128), 1000, op="bgk", porosity=1.0, radius=0.0),
        # one step at a time with the halo exchanged between two ranks: the
        # smallest calls
        _case("ranks", "ranks", "D3Q19", "f64", (48, 25, 23), 20, op="bgk", porosity=0.45, radius=4.0),
        # a large two-dimensional porous medium in float storage
        _case("porous2d", "step", "D2Q9", "f32s", (1021, 509), 1000, op="bgk", porosity=0.6, radius=12.0),
        # the headline workload: 256^3 sphere pack, double precision
        _case("pack256", "step", "D3Q19", "f64", (256, 256, 256), 400, op="bgk"),
        # a ragged pack with the two-relaxation-time operator in float storage
        _case("trt", "step", "D3Q19", "f32s", (201, 173, 149), 400, op="trt", porosity=0.35, radius=6.0),
        # a permeability solve of a small sample (one request of an ensemble)
        _case("perm48", "perm", "D3Q19", "f32s", (48, 48, 48), 1000, radius=4.0),
        # a permeability solve of a large ragged sample in half storage
        _case("perm_half", "perm", "D3Q19", "f16s", (161, 143, 150), 400, porosity=0.38),
        # a representative volume, periodic along every axis
        _case("periodic", "step", "D3Q19", "f64", (127, 120, 117), 300, op="bgk", periodic="xyz", radius=7.0),
        # a generalized-Newtonian fluid in a pack (viscosity from a table)
        _case("rheology", "step", "D3Q19", "f64", (101, 96, 90), 300, op="rheology", porosity=0.45, radius=5.0),
        # the colour-gradient two-phase loop with its flux controller
        _case("twophase192", "twophase", "D3Q19", "f64", (192, 192, 192), 200, porosity=0.38, saturation=0.5,
              op="momx"),
        # a relative-permeability solve of a ragged sample in float storage
        _case("relperm", "relperm", "D3Q19", "f32s", (130, 111, 97), 400, porosity=0.42, radius=6.0,
              saturation=0.6),
        # a mix of requests resident together: 24 samples of uneven size, three
        # in ten of them two-phase
        _case("batch", "batch", "D3Q19", "f32s", (32, 128, 0), 300, solves=24, two_phase=0.3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    return dict(_draw(rng), sample=rng.randint(2, 10**6))


def _draw(rng):
    kind = rng.choice(["channel", "ranks", "porous2d", "step", "step", "periodic", "perm", "perm", "twophase",
                       "relperm", "batch"])
    phi = round(rng.uniform(0.30, 0.50), 3)
    rad = round(rng.uniform(3.0, 8.0), 2)
    prec = rng.choice(["f64", "f32s", "f16s"])

    def box(lo, hi):
        return tuple(max(lo, min(hi, int(_log_int(rng, lo, hi)))) for _ in range(3))

    if kind == "channel":
        return _case("", "step", "D2Q9", rng.choice(["f64", "f32s"]),
                     (_log_int(rng, 48, 512), _log_int(rng, 24, 256)), rng.randint(300, 1500), op="bgk",
                     porosity=1.0, radius=0.0)
    if kind == "ranks":
        return _case("", "ranks", "D3Q19", rng.choice(["f64", "f32s"]), box(16, 64), rng.randint(5, 30), op="bgk",
                     porosity=phi, radius=3.0)
    if kind == "porous2d":
        return _case("", "step", "D2Q9", prec, (_log_int(rng, 200, 1500), _log_int(rng, 100, 1000)),
                     rng.randint(200, 1200), op="bgk", porosity=round(rng.uniform(0.5, 0.8), 3), radius=10.0)
    if kind == "step":
        return _case("", "step", "D3Q19", prec, box(32, 200), rng.randint(50, 400),
                     op=rng.choice(["bgk", "trt", "rheology"]), porosity=phi, radius=rad)
    if kind == "periodic":
        return _case("", "step", "D3Q19", prec, box(32, 150), rng.randint(50, 300), op=rng.choice(["bgk", "trt"]),
                     periodic=rng.choice(["xyz", "xz"]), porosity=phi, radius=rad)
    if kind == "perm":
        return _case("", "perm", "D3Q19", prec, box(32, 180), 100 * rng.randint(2, 6), porosity=phi, radius=rad)
    if kind == "twophase":
        return _case("", "twophase", "D3Q19", prec, box(32, 150), rng.randint(40, 200), porosity=phi, radius=rad,
                     periodic=rng.choice(["x", "x", "xyz"]), saturation=round(rng.uniform(0.2, 0.8), 3),
                     op=rng.choice(["momx", "fixed"]))
    if kind == "relperm":
        return _case("", "relperm", "D3Q19", rng.choice(["f64", "f32s"]), box(48, 130), 100 * rng.randint(2, 4),
                     porosity=phi, radius=rad, saturation=round(rng.uniform(0.2, 0.8), 3))
    return _case("", "batch", "D3Q19", prec, (32, _log_int(rng, 64, 128), 0), 100 * rng.randint(2, 3),
                 solves=rng.randint(6, 24), two_phase=0.3 if prec == "f32s" else 0.0)


# ------------------------------------------------------------------- inputs
def _shape(c):
    return (c["nx"], c["ny"]) if c["lattice"] == "D2Q9" else (c["nx"], c["ny"], c["nz"])


def _geometry(c):
    """The sample: positive for fluid, 0 for solid, closed on the axes that are not periodic."""
    shape = _shape(c)
    if c["radius"] == 0.0:
        geo = np.ones(shape, dtype=np.int32)
        geo[:, 0] = geo[:, -1] = 0
        return geo
    return lbamd.sphere_pack(shape, c["radius"], c["porosity"], c["sample"], periodic=c["periodic"], walls=True)[0]


def _cells(c, seed):
    """Density of the start per cell (two densities for two phases); the fluid is at rest."""
    rng = np.random.default_rng(seed)
    shape = _shape(c)
    if c["kind"] in ("twophase", "relperm"):
        r0 = (rng.random(shape) < c["saturation"]).astype(np.float64)
        return np.stack([r0, 1.0 - r0], axis=-1)
    return 1.0 + 1e-4 * rng.standard_normal(shape)


def _table():
    """A shear-thinning viscosity against the square of the strain rate (Carreau)."""
    sr = np.logspace(-16, -4, 40)
    return sr, 0.02 + 0.15 * (1.0 + sr / 1e-11) ** -0.2


def _requests(c, seed):
    """The samples of a batch: (geometry, initial phase-0 density or None) of uneven cubes."""
    rng = np.random.default_rng(seed)
    out = []
    n = c["solves"]
    # one size from each of n equal shares of the range's logarithm, so that the
    # work of a batch depends little on the seed
    share = (np.arange(n) + rng.uniform(0.0, 1.0, n)) / n
    sizes = np.rint(np.exp(np.log(c["nx"]) + share * np.log(c["ny"] / c["nx"]))).astype(int)
    two = np.zeros(n, dtype=bool)
    if c["two_phase"] > 0:
        two[:: max(1, int(round(1.0 / c["two_phase"])))] = True
    for k in range(n):
        geo = lbamd.sphere_pack((int(sizes[k]),) * 3, float(rng.uniform(3.0, 8.0)), float(rng.uniform(0.30, 0.50)),
                                int(rng.integers(1, 2**31)), periodic="x", walls=True)[0]
        sw = float(rng.uniform(0.2, 0.8))
        rho0 = np.where(geo > 0, (rng.random(geo.shape) < sw).astype(np.float64), 0.0) if two[k] else None
        out.append((geo, rho0))
    return out


def _at(topo, per_cell):
    """Values of the nodes of a node list from those of the box's cells (node 0, the ghost, gets zeros)."""
    pos = topo.positions()
    out = np.zeros((topo.n_nodes,) + per_cell.shape[topo.nD:])
    inside = np.all(pos >= 0, axis=1)
    out[inside] = per_cell[tuple(np.mod(pos[inside], per_cell.shape[: topo.nD]).T)]
    return out


def _context(c, topo, cells):
    ctx = lbamd.Context(LATTICE[c["lattice"]], PRECISION[c["precision"]])
    ctx.set_topology_from(topo)
    rho = _at(topo, cells)
    rest = np.zeros((topo.n_nodes, topo.nD))
    if rho.ndim == 2:
        wall = topo.node_types() == 1
        rho[wall] = (1.0, 0.0)  # wetted by phase 0
        ctx.set_wall_densities(rho)
        for k in range(2):
            ctx.init_equilibrium(2, k, rho, rest, rho_field=k)
    else:
        ctx.init_equilibrium(1, 0, rho, rest)
    return ctx


def prepare(case, seed):
    c = dict(case)
    if c["kind"] == "batch":
        b = lbamd.Batch(LATTICE[c["lattice"]], PRECISION[c["precision"]], POOL, 100)
        return {"case": c, "batch": b, "requests": _requests(c, seed)}
    geo = _geometry(c)
    cells = _cells(c, seed)
    lat = LATTICE[c["lattice"]]
    state = {"case": c, "n_box": float(geo.size)}
    if c["kind"] == "ranks":
        split = geo.copy()
        split[c["nx"] // 2:] *= 2
        topos = [lbamd.Topology.from_geometry(split, lat, c["periodic"], rank=r + 1) for r in range(2)]
        lists = exchange_lists(topos)
        state["contexts"] = [_context(c, t, cells) for t in topos]
        state["exchanges"] = [{x[0]: ctx.halo_add(*x) for x in lists[r]} for r, ctx in enumerate(state["contexts"])]
        return state
    topo = lbamd.Topology.from_geometry(geo, lat, c["periodic"])
    state["context"] = _context(c, topo, cells)
    topo.close()
    if c.get("op") == "rheology":
        state["context"].set_viscosity_table(*_table())
    return state


# ---------------------------------------------------------------------- run
def run(state):
    c = state["case"]
    force = (FORCE, 0.0, 0.0)
    n = c["steps"]
    if c["kind"] == "batch":
        return _run_batch(state, force)
    if c["kind"] == "ranks":
        ctxs = state["contexts"]
        for _ in range(n):
            for ctx in ctxs:
                ctx.step_bgk(1, TAU["bgk"], force)
            exchange(ctxs, state["exchanges"])
        return [{"rho": ctx.download_scalar(lbamd.RHO), "vel": ctx.download_vel()} for ctx in ctxs]
    ctx = state["context"]
    tp = TWO_PHASE
    # two checks in a solve: it runs to its step limit also near the steady
    # state, which the passes come to after some time
    if c["kind"] == "perm":
        k, steps = ctx.solve_permeability(TAU["bgk"], force, n // 2, TOL, n, state["n_box"])
        return {"k": k, "steps": steps, "vel": ctx.download_vel()}
    if c["kind"] == "relperm":
        k, steps = ctx.solve_relperm(tp["tau0"], tp["tau1"], tp["sigma"], tp["beta"], force, n // 2, TOL, n,
                                     state["n_box"])
        return {"k0": k[0], "k1": k[1], "steps": steps, "phi": ctx.download_scalar(lbamd.PHI)}
    if c["kind"] == "twophase":
        if c["op"] == "momx":
            ctx.step_cg(n, tp["tau0"], tp["tau1"], tp["sigma"], tp["beta"], lbamd.FORCE_MOMX, (MOMX, 0.0, 0.0))
        else:
            ctx.step_cg(n, tp["tau0"], tp["tau1"], tp["sigma"], tp["beta"], lbamd.FORCE_FIXED, force)
        return {"rho": ctx.download_scalar(lbamd.RHO, 2), "phi": ctx.download_scalar(lbamd.PHI),
                "vel": ctx.download_vel(), "force": ctx.last_force()}
    if c["op"] == "rheology":
        ctx.step_rheology(n, force)
        return {"rho": ctx.download_scalar(lbamd.RHO), "vel": ctx.download_vel(),
                "visc": ctx.download_scalar(lbamd.VISC)}
    if c["op"] == "trt":
        ctx.step_trt(n, TAU["trt_sym"], TAU["trt_anti"], force)
    else:
        ctx.step_bgk(n, TAU["bgk"], force)
    return {"rho": ctx.download_scalar(lbamd.RHO), "vel": ctx.download_vel()}


def _run_batch(state, force):
    """Requests admitted to an empty pool, advanced until all have their results."""
    c, b, reqs = state["case"], state["batch"], state["requests"]
    tp = TWO_PHASE
    single = [k for k, r in enumerate(reqs) if r[1] is None]
    waiting = [k for k, r in enumerate(reqs) if r[1] is not None]
    todo = list(single)
    got = {}
    while len(got) < len(reqs):
        if todo:
            m = b.add_many([reqs[k][0] for k in todo], "x", TAU["bgk"], force, TOL, c["steps"], todo)
            todo = todo[m:]
        while waiting:
            geo, rho0 = reqs[waiting[0]]
            if not b.add_twophase(geo, "x", rho0, 1.0, tp["tau0"], tp["tau1"], tp["sigma"], tp["beta"], force,
                                  TOL, c["steps"], waiting[0]):
                break
            waiting.pop(0)
        b.advance(c["steps"] // 100)
        for r in b.collect():
            got[r["tag"]] = r
    order = range(len(reqs))
    return {"k": np.array([got[k]["k"] for k in order]), "steps": np.array([got[k]["steps"] for k in order]),
            "k_phase": np.array([got[k]["k_phase"] if reqs[k][1] is not None else (0.0, 0.0) for k in order])}


# --------------------------------------------------------------------- work
def work(case):
    """Each step reads every population once and writes it once; the fields are written once."""
    c = dict(case)
    q, d = (9, 2) if c["lattice"] == "D2Q9" else (19, 3)
    s = BYTES[c["precision"]]
    if c["kind"] == "batch":
        # mean of the cells of a size drawn with a uniform logarithm; porosity 0.4 on average
        a, b = c["nx"], c["ny"]
        cells = (b**3 - a**3) / (3.0 * math.log(b / a)) if b > a else a**3
        nodes = 0.4 * cells * c["solves"]
        fields = 1.0 + c["two_phase"]
        return {"bytes": nodes * c["steps"] * 2.0 * q * s * fields, "flops": nodes * c["steps"] * 20.0 * q * fields}
    nodes = c["porosity"] * c["nx"] * c["ny"] * c["nz"]
    two = c["kind"] in ("twophase", "relperm")
    out = {"twophase": 8.0 * (d + 3), "relperm": 8.0, "perm": 8.0 * d}.get(c["kind"], 8.0 * (d + 1))
    return {"bytes": nodes * (c["steps"] * 2.0 * q * s * (2 if two else 1) + out),
            "flops": nodes * c["steps"] * (40.0 * q if two else 15.0 * q)}


# -------------------------------------------------------------------- exact
_E2 = [(1, 0), (1, 1), (0, 1), (-1, 1), (-1, 0), (-1, -1), (0, -1), (1, -1), (0, 0)]
_H3 = [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (1, -1, 0), (1, 0, 1), (1, 0, -1), (0, 1, 1), (0, 1, -1)]
_E3 = _H3 + [tuple(-v for v in e) for e in _H3] + [(0, 0, 0)]


class _Dense:
    """The scheme on the whole box in 64 bits: pull streaming, half-way bounce-back at the solid cells."""

    def __init__(self, lattice, geo):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.e = _E2 if lattice == "D2Q9" else _E3
        rest = {"D2Q9": 16 / 36, "D3Q19": 12 / 36}[lattice]
        axis = {"D2Q9": 4 / 36, "D3Q19": 2 / 36}[lattice]
        self.w = [rest if not any(e) else axis if sum(map(abs, e)) == 1 else 1 / 36 for e in self.e]
        self.rev = [self.e.index(tuple(-v for v in e)) for e in self.e]
        self.nd = geo.ndim
        self.dims = tuple(range(geo.ndim))
        self.fluid = torch.as_tensor(np.asarray(geo) > 0, device=self.dev)
        self.from_fluid = [torch.roll(self.fluid, e, self.dims) for e in self.e]

    def tensor(self, a):
        return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=self.dev)

    def stream(self, f):
        return [torch.where(self.from_fluid[q], torch.roll(f[q], self.e[q], self.dims), f[self.rev[q]])
                for q in range(len(self.e))]

    def along(self, q, v):
        """e_q . v for a list of components (None for the rest direction)."""
        r = None
        for x, y in zip(self.e[q], v):
            if x:
                t = y if x > 0 else -y
                r = t if r is None else r + t
        return r if r is not None else 0.0 * v[0]

    def moment(self, f, d):
        r = None
        for q, e in enumerate(self.e):
            if e[d]:
                r = (f[q] if r is None else r + f[q]) if e[d] > 0 else (-f[q] if r is None else r - f[q])
        return r

    def single(self, f, op, force):
        """One step: (post-collision populations, rho, u, viscosity, first moment with half the force)."""
        rho = sum(f)
        F = [torch.full((), v, dtype=torch.float64, device=self.dev) for v in force[: self.nd]]
        j = [self.moment(f, d) + 0.5 * F[d] for d in range(self.nd)]
        u = [x / rho for x in j]
        uu, uF = sum(x * x for x in u), sum(x * y for x, y in zip(u, F))
        eu = [self.along(q, u) for q in range(len(self.e))]
        eF = [self.along(q, F) for q in range(len(self.e))]
        feq = [w * rho * (1 + 3 * a + 4.5 * (a * a - uu / 3)) for w, a in zip(self.w, eu)]
        visc = None
        if op == "trt":
            ts, ta = TAU["trt_sym"], TAU["trt_anti"]
            out = []
            for q, r in enumerate(self.rev):
                even = 0.5 * (f[q] + f[r]) - 0.5 * (feq[q] + feq[r])
                odd = 0.5 * (f[q] - f[r]) - 0.5 * (feq[q] - feq[r])
                guo = self.w[q] * ((1 - 0.5 / ta) * 3 * eF[q] + (1 - 0.5 / ts) * 9 * (eF[q] * eu[q] - uF / 3))
                out.append(f[q] - even / ts - odd / ta + guo)
            return out, rho, u, visc, j[0]
        tau = TAU["bgk"]
        if op == "rheology":
            sq = 0.0
            for a in range(self.nd):
                for b in range(self.nd):
                    s = sum((x - y) * (e[a] * e[b] - (1 / 3 if a == b else 0.0)) for x, y, e in zip(f, feq, self.e))
                    sq = sq + (s + 0.5 * (u[a] * F[b] + u[b] * F[a])) ** 2
            sr, nu = (self.tensor(v) for v in _table())
            i = torch.clamp(torch.searchsorted(sr, sq, right=True) - 1, 0, sr.numel() - 2)
            t = torch.clamp((sq - sr[i]) / (sr[i + 1] - sr[i]), 0.0, 1.0)
            visc = nu[i] + t * (nu[i + 1] - nu[i])
            tau = 3 * visc / rho + 0.5
        out = [x - (x - y) / tau + w * (1 - 0.5 / tau) * (3 * b + 9 * (b * a - uF / 3))
               for x, y, w, a, b in zip(f, feq, self.w, eu, eF)]
        return out, rho, u, visc, j[0]

    def two_phase(self, f0, f1, force, momx, wall):
        """One colour-gradient step: (f0, f1 after collision, rho0, rho1, phi, u, force along x)."""
        r0, r1 = sum(f0), sum(f1)
        rho = r0 + r1
        phi = torch.where(self.fluid, (r0 - r1) / rho, self.tensor(wall))
        ft = [a + b for a, b in zip(f0, f1)]
        j = [self.moment(ft, d) for d in range(self.nd)]
        F = [torch.full((), v, dtype=torch.float64, device=self.dev) for v in force[: self.nd]]
        if momx is not None:
            F[0] = 2 * (momx - j[0][self.fluid].sum() / self.fluid.sum())
        u = [(x + 0.5 * y) / rho for x, y in zip(j, F)]
        tp = TWO_PHASE
        nu = [(tp["tau0"] - 0.5) / 3, (tp["tau1"] - 0.5) / 3]
        tau = 3 * rho / (r0 / nu[0] + r1 / nu[1]) + 0.5
        g = [sum(3 * w * e[d] * torch.roll(phi, tuple(-v for v in e), self.dims)
                 for w, e in zip(self.w, self.e) if e[d]) for d in range(self.nd)]
        norm = torch.sqrt(sum(x * x for x in g))
        g = [x / (norm + (norm < 2.220446049250313e-16)) for x in g]
        uu, uF = sum(x * x for x in u), sum(x * y for x, y in zip(u, F))
        n0, n1 = [], []
        three = self.nd == 3
        for q, e in enumerate(self.e):
            w, size = self.w[q], sum(map(abs, e))
            B = {0: -12 / 54 if three else -16 / 108, 1: 1 / 54 if three else 8 / 108, 2: 2 / 54 if three else 5 / 108}[size]
            a, b, cg = self.along(q, u), self.along(q, F), self.along(q, g)
            feq = w * rho * (1 + 3 * a + 4.5 * (a * a - uu / 3))
            t = ft[q] - (ft[q] - feq) / tau + w * (1 - 0.5 / tau) * (3 * b + 9 * (b * a - uF / 3))
            t = t + 1.125 * norm * tp["sigma"] / tau * (w * cg * cg - B)
            rc = tp["beta"] * r0 * r1 / rho * w * cg / math.sqrt(size) if size else 0.0
            n0.append(r0 / rho * t + rc)
            n1.append(r1 / rho * t - rc)
        return n0, n1, r0, r1, phi, u, F[0], ft


def _exact_single(lattice, geo, cells, op, steps, check=0):
    """(rho, u, viscosity of the last step, k averaged over the last `check` steps)."""
    D = _Dense(lattice, geo)
    rho = torch.where(D.fluid, D.tensor(cells), 1.0)
    f = [w * rho for w in D.w]
    jx = 0.0
    for s in range(steps):
        f, rho, u, visc, j0 = D.single(f, op, (FORCE, 0.0, 0.0))
        if check and s >= steps - check:
            jx += float(j0[D.fluid].sum())
        f = D.stream(f)
    k = (TAU["bgk"] - 0.5) / 3 * (jx / check / geo.size) / FORCE if check else None
    return rho, u, visc, k


def _exact_two(lattice, geo, cells, steps, momx):
    """(rho0, rho1, phi, u, force, [k0, k1] of the state before the last step)."""
    D = _Dense(lattice, geo)
    r = D.tensor(cells)
    f0 = [torch.where(D.fluid, w * r[..., 0], w) for w in D.w]
    f1 = [torch.where(D.fluid, w * r[..., 1], 0.0) for w in D.w]
    wall = np.ones(geo.shape)
    for s in range(steps):
        f0, f1, r0, r1, phi, u, Fx, ft = D.two_phase(f0, f1, (FORCE, 0.0, 0.0), MOMX if momx else None, wall)
        if s == steps - 1:
            j = D.moment(ft, 0)
            k = [float(((x / (r0 + r1)) * j)[D.fluid].sum()) / geo.size / FORCE * (t - 0.5) / 3
                 for x, t in ((r0, TWO_PHASE["tau0"]), (r1, TWO_PHASE["tau1"]))]
        f0, f1 = D.stream(f0), D.stream(f1)
    return r0, r1, phi, u, float(Fx), k


def _nodes(topo, *fields):
    """Values per node from dense fields (several become the components); nodes that are not advanced hold 0."""
    v = torch.stack([f.cpu() for f in fields], dim=-1).numpy() if len(fields) > 1 else fields[0].cpu().numpy()
    out = np.zeros((topo.n_nodes,) + v.shape[topo.nD:])
    b = topo.bulk()
    pos = topo.positions()[b]
    out[b] = v[tuple(np.mod(pos, v.shape[: topo.nD]).T)]
    return out


def _cost(c):
    """Rough seconds of the dense box on a GPU."""
    two = c["kind"] in ("twophase", "relperm")
    cells = float(c["nx"]) * c["ny"] * max(1, c["nz"])
    return c["steps"] * (6e-3 + cells * (9e-9 if two or c.get("op") == "rheology" else 2.4e-9))


def exact(case, seed):
    c = dict(case)
    if c["kind"] == "batch":
        k, kp = [], []
        for geo, rho0 in _requests(c, seed):
            if rho0 is None:
                cells = np.ones(geo.shape)
                k.append(_exact_single(c["lattice"], geo, cells, "bgk", c["steps"], 100)[3])
                kp.append((0.0, 0.0))
            else:
                two = _exact_two(c["lattice"], geo, np.stack([rho0, 1.0 - rho0], axis=-1), c["steps"], False)[5]
                k.append(two[0] + two[1])
                kp.append(two)
        return {"k": np.array(k), "steps": None, "k_phase": np.array(kp)}
    if _cost(c) > 20.0:
        return None
    geo, cells = _geometry(c), _cells(c, seed)
    lat = LATTICE[c["lattice"]]
    topo = lbamd.Topology.from_geometry(geo, lat, c["periodic"])
    if c["kind"] in ("twophase", "relperm"):
        momx = c.get("op") == "momx"
        r0, r1, phi, u, fx, k = _exact_two(c["lattice"], geo, cells, c["steps"], momx)
        if c["kind"] == "relperm":
            return {"k0": k[0], "k1": k[1], "steps": None, "phi": _nodes(topo, phi)}
        return {"rho": _nodes(topo, r0, r1), "phi": _nodes(topo, phi), "vel": _nodes(topo, *u),
                "force": np.array([fx, 0.0, 0.0])}
    op = c.get("op", "bgk")
    rho, u, visc, k = _exact_single(c["lattice"], geo, cells, op, c["steps"], c["steps"] // 2 if c["kind"] == "perm" else 0)
    if c["kind"] == "perm":
        return {"k": k, "steps": None, "vel": _nodes(topo, *u)}
    if c["kind"] == "ranks":
        split = geo.copy()
        split[c["nx"] // 2:] *= 2
        topos = [lbamd.Topology.from_geometry(split, lat, c["periodic"], rank=r + 1) for r in range(2)]
        return [{"rho": _nodes(t, rho), "vel": _nodes(t, *u)} for t in topos]
    out = {"rho": _nodes(topo, rho), "vel": _nodes(topo, *u)}
    if op == "rheology":
        out["visc"] = _nodes(topo, visc)
    return out
