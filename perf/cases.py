"""What the performance of this library is measured on: coupled time steps
(and the pressure solve alone) over the range of its use.

``listed()`` gives the named cases, ``draw(rng)`` one more of the same ranges.
``prepare`` builds a case's contexts with their state on the GPU and pinned
host buffers for the results; ``run`` advances it by one output interval and
downloads the whole state, as a program that writes snapshots does. Cells,
markers and bodies are in lattice units (spacing 1) except where ``si`` is set.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ibm-dem_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ctypes  # noqa: E402

import ibmdem  # noqa: E402
from ibmdem import cases as gen  # noqa: E402
from ibmdem.abi import (BC_INFLOW, BC_OUTFLOW, BC_PERIODIC, BC_WALL, FP64, MIXED,  # noqa: E402
                        SCHEME_RK3, SolveInfo)

P, W = BC_PERIODIC, BC_WALL
SIDES = {
    "periodic": [P] * 6,
    "walls": [W] * 6,
    "channel": [P, P, W, W, P, P],
    "bed": [W, W, W, W, BC_INFLOW, BC_OUTFLOW],
    "crossflow": [BC_INFLOW, BC_OUTFLOW, P, P, P, P],
}


def _case(name, kind, n, sides, spheres=0, diameter=12.0, mixed=False, steps=5, members=1, si=False,
          packed=False):
    c = {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "sides": sides, "spheres": spheres,
         "diameter": diameter, "mixed": mixed, "steps": steps, "members": members, "si": si,
         "packed": packed}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest coupled step: a few spheres in contact in a small
        # periodic box, advanced one step at a time under a host program's
        # control; launches and waits decide
        _case("cluster-32", "step", (32, 24, 28), "periodic", 6, 8.0, steps=1, packed=True),
        # one sphere settling in a tall closed box, the validation run
        _case("settling-64x256", "step", (64, 64, 256), "walls", 1, 16.0, steps=10),
        # spheres settling in a box whose extents were set by its physical
        # size: halving ends early, at odd extents
        _case("ragged-100x76x130", "step", (100, 76, 130), "walls", 24, 12.0, steps=2),
        # the channel of the original program: water in SI units between two
        # walls, driven to a mean velocity; the spacing is no power of two
        _case("channel-si-240x32", "step", (240, 32, 240), "channel", 86, 12.0, steps=8, si=True),
        # the periodic suspension, in FP64 and with the mixed-precision solver
        _case("suspension-256", "step", (256, 256, 256), "periodic", 2000, 12.0, steps=8),
        _case("suspension-256-mixed", "step", (256, 256, 256), "periodic", 2000, 12.0, mixed=True, steps=8),
        # the largest: a fluidized bed with inflow below and outflow on top
        _case("bed-192x768-mixed", "step", (192, 192, 768), "bed", 10000, 10.0, mixed=True, steps=5),
        # flow past free spheres between an inflow and an outflow side, with
        # the force on a held sphere recorded every step
        _case("crossflow-512x256", "step", (512, 256, 64), "crossflow", 200, 8.0, steps=8),
        # many uneven settling cases advanced together
        _case("batch-64-mixed", "batch", (64, 64, 128), "walls", 20, 12.0, mixed=True, steps=5, members=64),
        # the fluid alone with the three-stage Runge-Kutta scheme
        _case("rk3-128", "rk3", (128, 128, 128), "periodic", steps=2),
        # the pressure solve alone, as a host program with its own advection calls it
        _case("poisson-128x96x160", "poisson", (128, 96, 160), "walls", steps=1),
        # a sediment: spheres packed in contact on the floor of a box
        _case("sediment-128", "step", (128, 128, 128), "walls", 700, 10.0, steps=4, packed=True),
    ]


def _extent(rng, lo, hi, multiple):
    """An extent, even over its logarithm."""
    return multiple * max(1, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / multiple))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "batch", "rk3", "poisson"])
    # halving reaches small levels for multiples of 16, ends early otherwise
    mult = rng.choice([16, 16, 16, 8, 2])
    top = 128 if mult == 2 else 224
    n = tuple(_extent(rng, 24, top, mult) for _ in range(3))
    diameter = round(rng.uniform(7.0, 14.0), 3)
    vol = n[0] * n[1] * n[2]
    most = max(1, int(0.11 * vol / (math.pi * (diameter + 2) ** 3 / 6)))
    spheres = max(1, round(math.exp(rng.uniform(0, math.log(most)))))
    mixed = rng.random() < 0.4
    steps = max(1, min(8, int(4e7 / vol)))
    if kind == "step":
        sides = rng.choice(["periodic", "walls", "channel", "bed", "crossflow"])
        return _case("", kind, n, sides, spheres, diameter, mixed, steps, si=sides == "channel" and rng.random() < 0.5,
                     packed=sides in ("periodic", "walls") and rng.random() < 0.3)
    if kind == "batch":
        n = tuple(_extent(rng, 32, 96, 16) for _ in range(3))
        return _case("", kind, n, "walls", rng.randint(1, 20), diameter, mixed, 4, rng.randint(2, 48))
    if kind == "rk3":
        return _case("", kind, n, rng.choice(["periodic", "walls", "channel"]), 0, diameter, mixed,
                     max(1, min(2, steps)))
    return _case("", kind, n, rng.choice(["periodic", "walls", "channel"]), 0, diameter, mixed, 1)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _pinned(shape):
    return torch.empty(shape, dtype=torch.float64, pin_memory=True).numpy()


def _ptr(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double if a.dtype == np.float64 else ctypes.c_int32))


def _centres(rng, n, box, pitch, spread, margin, packed=False):
    """n sites of a lattice of the given pitch inside the box, each moved by
    up to `spread` per dimension; fewer where the box holds fewer. The lattice
    is stretched to the box and its sites are taken at random, or it is
    packed: at the pitch itself, from the bottom up."""
    count = [max(1, int((b - 2 * margin) // pitch)) for b in box]
    step = [pitch if packed else (b - 2 * margin) / c for b, c in zip(box, count)]
    sites = np.arange(count[0] * count[1] * count[2])
    sites = (sites if packed else rng.permutation(sites))[:n]
    at = np.stack([sites % count[0], sites // count[0] % count[1], sites // (count[0] * count[1])], axis=1)
    c = margin + (at + 0.5) * np.asarray(step)
    return c + rng.uniform(-spread, spread, size=c.shape)


def _smooth(rng, shape, amplitude, out):
    """A smooth velocity component: a product of one-dimensional modes."""
    def mode(m):
        x = 2 * np.pi * np.arange(m) / m
        a, b, c = rng.uniform(0, 2 * np.pi, size=3)
        return np.sin(x + a) + 0.4 * np.sin(2 * x + b) + 0.2 * np.sin(5 * x + c)
    z, y, x = (mode(m) for m in shape)
    np.multiply((amplitude * z)[:, None, None], y[:, None] * x[None, :], out=out)


def _setup(case, rng, n):
    """(ibmdem case, markers, bodies, (velocity scale, mean flow)) of one context."""
    sides = SIDES[case["sides"]]
    kind, D, nu, u = case["kind"], case["diameter"], 0.04, 0.1
    kw = dict(precision=MIXED if case["mixed"] else FP64)
    h, rho, mean = 1.0, 2.0, 0.0
    if kind == "rk3":
        cs = gen.build_case(*n, sides, visc=0.05, dt=0.4, time_scheme=SCHEME_RK3, **kw)
        return cs, None, None, (u, 0.0)
    if case["sides"] == "crossflow":
        mean = 0.5
        cs = gen.build_case(*n, sides, visc=mean * 32 / 200, kn_coeff=1e5, restitution=0.9, u_max=2 * mean,
                            inflow=(mean, 0.0, 0.0), **kw)
        u = 0.05
    elif case["sides"] == "bed":
        g = (40 * nu) ** 2 / (1.5 * 1000.0)
        mean, rho = math.sqrt(1.5 * g * 10.0), 2.5
        cs = gen.build_case(*n, sides, visc=nu, gravity=(0, 0, -g), kn_coeff=1e5, restitution=0.9,
                            u_max=2 * mean, inflow=(0.0, 0.0, mean), **kw)
        u = 0.02
    elif case["si"]:
        h, rho, u, mean = 9e-3 / 240, 2650.0, 0.02, 0.1
        cs = gen.build_case(*n, sides, h=h, visc=1e-6, rhof=1e3, dt=5e-5, gravity=(0, 0, -9.81),
                            bulk_switch=(1, 0, 1), bulk_target=(mean, 0, 0), **kw)
        cs.kn_coeff = 4e4
    else:
        g = u * u / ((rho - 1) * D)
        periodic = case["sides"] == "periodic"
        cs = gen.build_case(*n, sides, visc=u * D / 40, gravity=(0, 0, -g), kn_coeff=1e5, restitution=0.9,
                            bulk_switch=(1, 1, 1) if periodic else (0, 0, 0), u_max=2 * u, **kw)
    if kind == "poisson":
        return cs, None, None, (u, 0.0)
    # a packing's shells lie closer than the contact candidate distance, a
    # suspension's surfaces at least two spacings apart
    margin = 0.0 if case["sides"] == "periodic" else 1.0
    c = _centres(rng, case["spheres"], n, D + (0.93 if case["packed"] else 2.4),
                 0.01 if case["packed"] else 0.08, margin, case["packed"])
    if case["sides"] == "bed":
        # the sizes belong to the case, not to the seed
        dia = np.clip(np.exp(np.random.default_rng(len(c)).normal(math.log(0.8 * D), 0.15, size=len(c))), 0.6 * D, D)
    else:
        dia = np.full(len(c), D)
    held = len(c) - 1 if case["sides"] == "crossflow" else -1
    mk, bd = gen.place_spheres(cs, [gen.Sphere(tuple(x * h), d * h, rho, gen.markers_for_diameter(d), b == held)
                                    for b, (x, d) in enumerate(zip(c, dia))], h)
    v = rng.normal(0.0, 0.1 * u, size=bd.v.shape)
    if case["sides"] != "periodic":
        v *= 0.1
    if held >= 0:
        v[:, held] = 0.0
    bd.v[:] = bd.vold[:] = v
    mk.v[:] = v[:, mk.body]
    return cs, mk, bd, (u, mean)


class _Member:
    """One context with its result buffers; the fields' buffers carry the
    initial state up first."""

    def __init__(self, sim, case, rng, mk, bd, flow, fields):
        self.sim = sim
        self.fields = fields
        shape = sim.shape
        u, mean = flow
        for f in fields[:3]:
            _smooth(rng, shape, 0.2 * u, f)
        fields[3][...] = 0.0
        if mean:
            fields[2 if case["sides"] == "bed" else 0][...] += mean
        self.mk = self.bd = None
        if mk is not None:
            sim.upload_bodies(bd)
            sim.upload_markers(mk)
            self.mk, self.bd = mk, bd
            for a in ("x", "v", "fdrag", "fcol"):
                setattr(mk, a, _pinned(mk.x.shape))
            # what does not change is not downloaded
            self.mks, self.bds = mk.struct(), bd.struct()
            for a in ("vol", "mass", "radeff", "body"):
                setattr(self.mks, a, None)
            for a in ("inertia", "mass", "rho", "fixed"):
                setattr(self.bds, a, None)
        sim.call("ibmdem_upload_fields", *[_ptr(f) for f in fields])

    def download(self):
        sim = self.sim
        sim.call("ibmdem_download_fields", *[_ptr(f) for f in self.fields])
        if self.mk is not None:
            sim.call("ibmdem_download_markers", ctypes.byref(self.mks))
            sim.call("ibmdem_download_bodies", ctypes.byref(self.bds))


def prepare(case, seed):
    case = dict(case)
    rng = np.random.default_rng(seed)
    n = (case["nx"], case["ny"], case["nz"])
    state = {"case": case}
    if case["kind"] == "batch":
        sets, cells = [], []
        uneven = np.random.default_rng(case["members"])   # the sizes belong to the case
        for _ in range(case["members"]):
            m = tuple(16 * max(2, int(uneven.integers(v // 32, 3 * v // 32 + 1))) for v in n)
            one = dict(case, spheres=int(uneven.integers(1, 2 * case["spheres"] + 1)))
            sets.append(_setup(one, rng, m))
            cells.append(m[0] * m[1] * m[2])
        batch = ibmdem.batch([s[0] for s in sets])
        flat = [_pinned((sum(cells),)) for _ in range(4)]
        state["members"], at = [], 0
        for (cs, mk, bd, flow), sim, c in zip(sets, batch.sims, cells):
            fields = [f[at:at + c].reshape(sim.shape) for f in flat]
            at += c
            state["members"].append(_Member(sim, case, rng, mk, bd, flow, fields))
        state.update(batch=batch, flat=flat)
        return state
    cs, mk, bd, flow = _setup(case, rng, n)
    sim = ibmdem.simulation(cs)
    shape = sim.shape
    state["sim"] = sim
    if case["kind"] == "poisson":
        b = _rhs(case, seed)
        sim.upload_poisson_rhs(b)
        state["pcorr"] = _pinned(shape)
        return state
    state["member"] = _Member(sim, case, rng, mk, bd, flow, [_pinned(shape) for _ in range(4)])
    if case["sides"] == "crossflow" and mk is not None:
        held = bd.mass.size - 1
        sim.probe_bodies([held], case["steps"])
    return state


def _rhs(case, seed):
    """A divergence: smooth modes and noise, of zero mean."""
    rng = np.random.default_rng(seed)
    b = np.empty((case["nz"], case["ny"], case["nx"]))
    _smooth(rng, b.shape, 0.05, b)
    b += 0.01 * rng.standard_normal(b.shape, dtype=np.float32)
    return b - b.mean()


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _body_arrays(bd):
    return {"x": bd.x, "v": bd.v, "omega": bd.omega, "rot": bd.rot_glo, "fdrag": bd.fdrag}


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        infos = state["batch"].run(case["steps"])
        for m in state["members"]:
            m.download()
        mem = state["members"]
        return {"fields": state["flat"], "iterations": np.array([i.iterations for i in infos]),
                "markers": np.concatenate([m.mk.x.ravel() for m in mem]),
                "bodies": np.concatenate([np.concatenate([m.bd.x, m.bd.v, m.bd.omega]).ravel() for m in mem])}
    sim = state["sim"]
    if case["kind"] == "poisson":
        info = SolveInfo()
        sim.call("ibmdem_poisson_solve", ctypes.byref(info))
        sim.call("ibmdem_download_poisson", _ptr(state["pcorr"]), None)
        return {"pcorr": state["pcorr"], "iterations": int(info.iterations)}
    m = state["member"]
    info = sim.run(case["steps"])
    m.download()
    out = {"fields": m.fields, "iterations": int(info.iterations)}
    if m.mk is not None:
        out.update(x=m.mk.x, v=m.mk.v, fdrag=m.mk.fdrag, bodies=_body_arrays(m.bd))
        if case["sides"] == "crossflow":
            out["probe"] = sim.probe_read()[1]
    return out


def work(case):
    """Per step: the four fields read and written, the markers' positions,
    velocities and forces read and written; arithmetic of the stencils, the
    projection's solve (a few hundred operations a cell for ten digits) and
    the two 108-tap kernels of every forcing iteration."""
    cells = case["nx"] * case["ny"] * case["nz"] * case["members"]
    markers = case["spheres"] * math.pi * case["diameter"] ** 2 * case["members"]
    s = case["steps"]
    if case["kind"] == "poisson":
        return {"bytes": 16.0 * cells, "flops": 400.0 * cells}
    if case["kind"] == "rk3":
        return {"bytes": 3.0 * s * 64.0 * cells, "flops": 3.0 * s * 650.0 * cells}
    return {"bytes": s * (64.0 * cells + 168.0 * markers), "flops": s * (650.0 * cells + 5 * 700.0 * markers)}


def exact(case, seed):
    """The pressure solve's solution by a spectral transform of the operator
    (walls: its even extension); None for the other kinds, whose values come
    from many coupled operators."""
    if case["kind"] != "poisson":
        return None
    b = torch.from_numpy(_rhs(case, seed))
    walls = [SIDES[case["sides"]][2 * d] == W for d in (2, 1, 0)]
    shape = b.shape
    for d in range(3):
        if walls[d]:
            b = torch.cat([b, b.flip(d)], dim=d)
    lam = torch.zeros(1, 1, 1, dtype=torch.float64)
    for d in range(3):
        m = b.shape[d]
        e = 2 - 2 * torch.cos(2 * math.pi * torch.arange(m, dtype=torch.float64) / m)
        lam = lam + e.reshape([-1 if q == d else 1 for q in range(3)])
    lam[0, 0, 0] = 1.0
    xh = torch.fft.fftn(b) / lam
    xh[0, 0, 0] = 0.0
    x = torch.fft.ifftn(xh).real[:shape[0], :shape[1], :shape[2]].contiguous()
    return {"pcorr": x - x[0, 0, 0], "iterations": None}
