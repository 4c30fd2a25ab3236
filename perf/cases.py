"""Timing cases of the public entry points, with a float64 reference of each.

A case is a dict of plain values:

* ``op``      ``step`` (one ``Simulator.step(dt)``), ``simulate`` (one
              ``Simulator.simulate(t)`` with the CFL dt policy), ``mpi`` (one
              step of the one-rank ``MPISimulator`` with its halo exchange) or
              ``ensemble`` (one ``Ensemble.advance()``, 8 steps of every
              instance);
* ``scheme``  a key of ``SCHEMES``;
* ``math``    ``default`` (what the scheme runs with when the caller says
              nothing), ``fast`` or ``exact``;
* ``nx, ny``  interior cells; ``bc`` a key of ``BOUNDARIES``; ``steps`` the
              steps a ``simulate`` pass covers; ``count``, ``side_min``,
              ``side_max`` the instances of an ensemble.

The states are developed flows (depth or density jumps, Gaussian bumps, a
smooth velocity field and noise), drawn on the device from the seed alone.
"""

import math

import numpy as np
import torch

from finitevolumegpu_amd.EE2D_KP07_dimsplit import EE2D_KP07_dimsplit
from finitevolumegpu_amd.Ensemble import Ensemble
from finitevolumegpu_amd.FORCE import FORCE
from finitevolumegpu_amd.HLL import HLL
from finitevolumegpu_amd.HLL2 import HLL2
from finitevolumegpu_amd.HipContext import HipContext
from finitevolumegpu_amd.KP07 import KP07
from finitevolumegpu_amd.KP07_dimsplit import KP07_dimsplit
from finitevolumegpu_amd.LxF import LxF
from finitevolumegpu_amd.MPISimulator import MPISimulator
from finitevolumegpu_amd.Simulator import BoundaryCondition
from finitevolumegpu_amd.WAF import WAF

# the simulators hold their parameters in float32
G, THETA, THETA_HLL2, EULER_G, GAMMA = (float(np.float32(v)) for v in (9.81, 1.3, 1.8, 0.1, 1.4))

# scheme -> (class, variables, floating-point operations per cell and step as
# the scheme's formulas count them)
SCHEMES = {
    "kp07_dimsplit": (KP07_dimsplit, 3, 420),
    "hll2": (HLL2, 3, 480),
    "waf": (WAF, 3, 680),
    "ee2d_kp07_dimsplit": (EE2D_KP07_dimsplit, 4, 720),
    "lxf": (LxF, 3, 70),
    "hll": (HLL, 3, 130),
    "force": (FORCE, 3, 110),
    "kp07": (KP07, 3, 320),
}

# edges as (north, south, east, west)
_T = BoundaryCondition.Type
BOUNDARIES = {
    "reflective": (_T.Reflective,) * 4,
    "periodic": (_T.Periodic,) * 4,
    "outflow": (_T.Outflow,) * 4,
    "channel": (_T.Reflective, _T.Reflective, _T.Periodic, _T.Periodic),
}


def _case(name, op, scheme, nx, ny, bc, math="default", **more):
    return dict({"name": name, "op": op, "scheme": scheme, "nx": nx, "ny": ny, "bc": bc, "math": math}, **more)


def listed():
    return [
        # the smallest call: one step of a test-sized basin, where launches and latency are all there is
        _case("kp07_128", "step", "kp07_dimsplit", 128, 128, "reflective"),
        # the small dam break of the regression runs: 200 steps to a save time under the CFL policy
        _case("kp07_256_simulate", "simulate", "kp07_dimsplit", 256, 256, "reflective", steps=200),
        # the headline grid
        _case("kp07_4096", "step", "kp07_dimsplit", 4096, 4096, "reflective"),
        # a size of the published autotuning runs, odd and so ragged in every split
        _case("hll2_2047", "step", "hll2", 2047, 2047, "periodic"),
        # WAF in its default (bitwise) arithmetic: an ordinary ragged grid and the headline one
        _case("waf_1023x777", "step", "waf", 1023, 777, "reflective"),
        _case("waf_4096", "step", "waf", 4096, 4096, "reflective"),
        # Euler in its default (bitwise) arithmetic: an ordinary column, and one rank's share of the large run
        _case("ee2d_512", "step", "ee2d_kp07_dimsplit", 512, 512, "channel"),
        _case("ee2d_8192_mpi", "mpi", "ee2d_kp07_dimsplit", 8192, 8192, "channel"),
        # Euler in the arithmetic a user chooses for speed, odd width
        _case("ee2d_fast_3001x4032", "step", "ee2d_kp07_dimsplit", 3001, 4032, "channel", math="fast"),
        # a first-order scheme (one ghost cell, one launch a step) at the headline size
        _case("hll_4096", "step", "hll", 4096, 4096, "reflective"),
        # the unsplit second-order scheme with its two Runge-Kutta stages
        _case("kp07u_2048x1500", "step", "kp07", 2048, 1500, "outflow"),
        # a batch of independent basins of uneven size
        _case("ensemble_48", "ensemble", "kp07_dimsplit", 0, 0, "reflective", count=48, side_min=64, side_max=1024),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.random()
    if kind < 0.12:
        lo = rng.randint(64, 128)
        return {"op": "ensemble", "scheme": rng.choice(("kp07_dimsplit", "kp07_dimsplit", "hll2", "ee2d_kp07_dimsplit")),
                "nx": 0, "ny": 0, "bc": rng.choice(("reflective", "outflow")), "math": "default",
                "count": rng.randint(8, 48), "side_min": lo, "side_max": _log_uniform(rng, lo + 64, 900)}
    if kind < 0.24:
        return {"op": "simulate", "scheme": rng.choice(("kp07_dimsplit", "hll2", "kp07")),
                "nx": _log_uniform(rng, 64, 512), "ny": _log_uniform(rng, 64, 512),
                "bc": rng.choice(("reflective", "outflow", "periodic")), "math": "default",
                "steps": rng.randint(60, 120)}
    scheme = rng.choice(("kp07_dimsplit", "kp07_dimsplit", "hll2", "waf", "ee2d_kp07_dimsplit", "ee2d_kp07_dimsplit",
                         "lxf", "hll", "force", "kp07"))
    arithmetic = "default"
    if rng.random() < 0.25:
        arithmetic = {"waf": "fast", "ee2d_kp07_dimsplit": "fast"}.get(scheme, "exact")
    if scheme == "ee2d_kp07_dimsplit" and rng.random() < 0.4:
        return {"op": "mpi", "scheme": scheme, "nx": _log_uniform(rng, 128, 6000), "ny": _log_uniform(rng, 128, 6000),
                "bc": rng.choice(("channel", "periodic")), "math": arithmetic}
    return {"op": "step", "scheme": scheme, "nx": _log_uniform(rng, 64, 4096), "ny": _log_uniform(rng, 64, 4096),
            "bc": rng.choice(tuple(BOUNDARIES)), "math": arithmetic}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _sides(case):
    """Sides of an ensemble's instances, spread evenly over the logarithm."""
    k, lo, hi = case["count"], math.log(case["side_min"]), math.log(case["side_max"])
    return [int(round(math.exp(lo + (hi - lo) * (i + 0.5) / k))) for i in range(k)]


def _flow(gen, nx, ny):
    """x and y cell centres in [0, 1), a smooth velocity field and noise."""
    dev = _device()
    draw01 = lambda *shape: torch.rand(shape, generator=gen, device=dev)  # noqa: E731
    x = ((torch.arange(nx, device=dev) + 0.5) / nx)[None, :]
    y = ((torch.arange(ny, device=dev) + 0.5) / ny)[:, None]
    c = draw01(2, 4)
    tau = 2.0 * math.pi
    u = 0.35 * torch.sin(tau * (y + c[0, 0])) + 0.2 * torch.cos(tau * (2 * x + c[0, 1])) * torch.sin(tau * (y + c[0, 2]))
    v = 0.35 * torch.sin(tau * (x + c[1, 0])) + 0.2 * torch.cos(tau * (2 * y + c[1, 1])) * torch.sin(tau * (x + c[1, 2]))
    return x, y, u, v, draw01


def _swe_state(gen, nx, ny):
    x, y, u, v, draw01 = _flow(gen, nx, ny)
    p = draw01(17, 4)
    h = 1.0 + 0.5 * ((x - 0.3 - 0.4 * p[0, 0]) ** 2 + (y - 0.3 - 0.4 * p[0, 1]) ** 2 < 0.02)
    for a, w, cx, cy in p[1:9].tolist():
        w = 0.01 + 0.04 * w
        h = h + (0.05 + 0.25 * a) * torch.exp(-((x - cx) / w) ** 2 / 2) * torch.exp(-((y - cy) / w) ** 2 / 2)
    h = h + 1e-3 * (2.0 * draw01(ny, nx) - 1.0)
    return [h, h * u, h * v]


def _euler_state(gen, nx, ny):
    """Heavy over light fluid in a sheared flow, near-hydrostatic pressure."""
    x, y, u, v, draw01 = _flow(gen, nx, ny)
    above = y > 0.5 + 0.02 * torch.cos(2.0 * math.pi * (2 * x + draw01(1)))
    rho = torch.where(above, 2.0, 1.0) + 1e-3 * draw01(ny, nx)
    p = 2.5 - 0.5 * EULER_G * rho * (y - 0.5) + 1e-3 * draw01(ny, nx)
    return [rho, rho * u, rho * v, p / (GAMMA - 1.0) + 0.5 * rho * (u * u + v * v)]


def _fields(case, seed):
    """One list of float32 host fields per grid of the case."""
    gen = torch.Generator(device=_device()).manual_seed(int(seed))
    make = _euler_state if SCHEMES[case["scheme"]][1] == 4 else _swe_state
    sizes = [(s, s) for s in _sides(case)] if case["op"] == "ensemble" else [(case["nx"], case["ny"])]
    return [[f.float().contiguous().cpu().numpy() for f in make(gen, nx, ny)] for nx, ny in sizes]


def _dx(case, nx):
    return 0.5 / nx if case["scheme"] == "ee2d_kp07_dimsplit" else 1.0


def _dt(case, nx, ny):
    """A fixed step at a Courant number below one half of the scheme's limit
    for these states (wave speeds up to about 5 and 3)."""
    if case["scheme"] == "ee2d_kp07_dimsplit":
        return float(np.float32(0.4 / 3.0 * _dx(case, nx)))
    return float(np.float32(0.08))


# ---------------------------------------------------------------------------
# Preparation and one pass
# ---------------------------------------------------------------------------

_CONTEXT = []


def _context():
    if not _CONTEXT:
        _CONTEXT.append(HipContext(device=0, autotuning=False))
    return _CONTEXT[0]


class _DeviceArray:
    """A pitched float32 device region for ``torch.as_tensor``."""

    def __init__(self, owner, address, shape, strides):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "strides": strides, "typestr": "<f4",
                                         "data": (address, False), "version": 2}


def _view(array):
    address = array.data_ptr + array.y_halo * array.pitch + 4 * array.x_halo
    return torch.as_tensor(_DeviceArray(array, address, (array.ny, array.nx), (array.pitch, 4)), device="cuda")


def _boundary(case):
    return BoundaryCondition(dict(zip(("north", "south", "east", "west"), BOUNDARIES[case["bc"]])))


def prepare(case, seed):
    ctx = _context()
    arithmetic = None if case["math"] == "default" else case["math"]
    fields = _fields(case, seed)
    if case["op"] == "ensemble":
        euler = case["scheme"] == "ee2d_kp07_dimsplit"
        specs = []
        for f in fields:
            ny, nx = f[0].shape
            d = _dx(case, nx)
            specs.append({"fields": f, "nx": nx, "ny": ny, "dx": d, "dy": d, "g": EULER_G if euler else G,
                          "t_end": 1e9, "bc": _boundary(case), "gamma": GAMMA if euler else None})
        ens = Ensemble(ctx, case["scheme"], specs, math=arithmetic, steps_per_graph=8)
        # after an even number of steps an instance's state is in its first buffer
        views = []
        for i, f in enumerate(fields):
            I = ens.host_table[i]
            ny, nx = f[0].shape
            views.append(torch.as_tensor(_DeviceArray(
                ens, I.field[0][0] + 2 * I.pitch + 8, (ens.nvars, ny, nx),
                (I.field[0][1] - I.field[0][0], I.pitch, 4)), device="cuda"))
        return {"op": "ensemble", "ensemble": ens, "views": views}
    cls, nvars, _ = SCHEMES[case["scheme"]]
    nx, ny = case["nx"], case["ny"]
    d = _dx(case, nx)
    args = (EULER_G, GAMMA) if nvars == 4 else (G,)
    sim = cls(ctx, *fields[0], nx, ny, d, d, *args, boundary_conditions=_boundary(case), math=arithmetic)
    if case["op"] == "mpi":
        sim = MPISimulator(sim)
    return {"op": case["op"], "sim": sim, "dt": np.float32(_dt(case, nx, ny)), "t": case.get("steps", 0) * 0.1,
            "views": {}}


def run(state):
    if state["op"] == "ensemble":
        state["ensemble"].advance()
        return state["views"]
    sim = state["sim"]
    if state["op"] == "simulate":
        sim.simulate(state["t"])
    else:
        sim.step(state["dt"])
    views, out = state["views"], []
    for array in sim.getOutput().gpu_variables:
        v = views.get(array.data_ptr)
        if v is None:
            v = views[array.data_ptr] = _view(array)
        out.append(v)
    return out


def work(case):
    _, nvars, flops = SCHEMES[case["scheme"]]
    if case["op"] == "ensemble":
        cells, steps = sum(s * s for s in _sides(case)), 8
    else:
        cells, steps = case["nx"] * case["ny"], case.get("steps", 1)
    return {"bytes": 2 * 4 * nvars * cells, "flops": flops * cells * steps}


# ---------------------------------------------------------------------------
# Float64 reference: each scheme in global form on padded arrays
# ---------------------------------------------------------------------------

def _ghosts(n, gc, low, high):
    """Source cell of each padded cell of an axis, and which are mirrored."""
    idx, mirrored = [], []
    for k in range(-gc, n + gc):
        kind = low if k < 0 else high
        if 0 <= k < n:
            idx.append(k)
        elif kind == _T.Periodic:
            idx.append(k % n)
        elif kind == _T.Reflective:
            idx.append(-1 - k if k < 0 else 2 * n - 1 - k)
        else:
            idx.append(0 if k < 0 else n - 1)
        mirrored.append(kind == _T.Reflective and not 0 <= k < n)
    return idx, mirrored


def _pad(q, gc, bc):
    """Fields (list of (ny, nx)) with ``gc`` ghost cells a side."""
    north, south, east, west = BOUNDARIES[bc]
    ny, nx = q[0].shape
    dev = q[0].device
    ix, mx = _ghosts(nx, gc, west, east)
    iy, my = _ghosts(ny, gc, south, north)
    out = [f[torch.tensor(iy, device=dev)][:, torch.tensor(ix, device=dev)] for f in q]
    sign = lambda m: torch.tensor([-1.0 if v else 1.0 for v in m], dtype=torch.float64, device=dev)  # noqa: E731
    out[1] = out[1] * sign(mx)[None, :]
    out[2] = out[2] * sign(my)[:, None]
    return out


def _turn(q):
    """The fields seen by the other direction: axes and momenta swapped."""
    return [q[0].T, q[2].T, q[1].T] + [f.T for f in q[3:]]


class _Swe:
    """Shallow-water fluxes; the state is (h, normal momentum, tangential momentum)."""

    def F(self, q):
        u = q[1] / q[0]
        return [q[1], q[1] * u + 0.5 * G * q[0] * q[0], q[2] * u]

    predictor = F

    def speed(self, q):
        return q[1] / q[0], torch.sqrt(G * q[0])


class _Euler:
    """Euler fluxes; the state is (rho, normal, tangential momentum, E)."""

    def pressure(self, q):
        return (GAMMA - 1.0) * (q[3] - 0.5 * (q[1] * q[1] + q[2] * q[2]) / q[0])

    def F(self, q, p=None):
        p = self.pressure(q) if p is None else p
        u = q[1] / q[0]
        return [q[1], q[1] * u + p, q[2] * u, u * (q[3] + p)]

    def predictor(self, q):
        return self.F(q, GAMMA)  # the scheme's half step takes gamma for the pressure

    def speed(self, q):
        return q[1] / q[0], torch.sqrt(GAMMA * self.pressure(q) / q[0])


def _central_upwind(eq, l, r):
    (ul, cl), (ur, cr) = eq.speed(l), eq.speed(r)
    am = torch.clamp(torch.minimum(ul - cl, ur - cr), max=0.0)
    ap = torch.clamp(torch.maximum(ul + cl, ur + cr), min=0.0)
    return [((ap * a - am * b) + ap * am * (y - x)) / (ap - am) for a, b, x, y in zip(eq.F(l), eq.F(r), l, r)]


def _hll_flux(eq, l, r):
    (ul, cl), (ur, cr) = eq.speed(l), eq.speed(r)
    hl, hr = l[0], r[0]
    star = 0.5 * (hl + hr) - 0.25 * (ur - ul) * (hl + hr) / (cl + cr)
    one = torch.ones_like(star)
    sl = ul - cl * torch.where(star > hl, torch.sqrt(0.5 * ((star + hl) * star / (hl * hl))), one)
    sr = ur + cr * torch.where(star > hr, torch.sqrt(0.5 * ((star + hr) * star / (hr * hr))), one)
    out = []
    for a, b, x, y in zip(eq.F(l), eq.F(r), l, r):
        mid = (sr * a - sl * b + sr * sl * (y - x)) / (sr - sl)
        out.append(torch.where(sl >= 0, a, torch.where(sr <= 0, b, mid)))
    return out


def _minmod(b, c, f):
    same = (torch.sign(b) == torch.sign(f)) & (b != 0)
    return torch.where(same, torch.sign(b) * torch.minimum(torch.minimum(b.abs(), c.abs()), f.abs()), 0.0 * b)


def _slopes(q, theta):
    """Limited slopes of every cell but the first and last of each row."""
    out = []
    for f in q:
        d = f[:, 1:] - f[:, :-1]
        out.append(_minmod(theta * d[:, :-1], 0.5 * (f[:, 2:] - f[:, :-2]), theta * d[:, 1:]))
    return out


def _muscl_sweep(q, d, dt, theta, eq, flux):
    """Limited faces, half-step predictor, flux, update; two cells lost a side."""
    s = _slopes(q, theta)
    left = [f[:, 1:-1] - 0.5 * k for f, k in zip(q, s)]
    right = [f[:, 1:-1] + 0.5 * k for f, k in zip(q, s)]
    k = dt / (2.0 * d)
    gain = [k * (a - b) for a, b in zip(eq.predictor(left), eq.predictor(right))]
    f = flux(eq, [(a + e)[:, :-1] for a, e in zip(right, gain)], [(a + e)[:, 1:] for a, e in zip(left, gain)])
    return [a[:, 2:-2] + dt / d * (b[:, :-1] - b[:, 1:]) for a, b in zip(q, f)]


def _waf_sweep(q, d, dt):
    h, hu, hv = q
    u, v, c = hu / h, hv / h, torch.sqrt(G * h)
    at = lambda f, k: f[:, k:f.shape[1] - 3 + k]  # noqa: E731  cells i-1, i, i+1, i+2 of interface (i, i+1): k = 0..3
    star = (0.5 * (c[:, :-1] + c[:, 1:]) + 0.25 * (u[:, :-1] - u[:, 1:])) ** 2 / G
    eps = 1e-6
    desing = lambda x: torch.copysign(torch.maximum(  # noqa: E731
        x.abs(), torch.clamp(x * x / (2 * eps) + 0.5 * eps, max=eps)), x)
    d1, d2, d3 = desing(star - h[:, :-1]), desing(v[:, 1:] - v[:, :-1]), desing(h[:, 1:] - star)
    hl, hr, ul, ur, vl, vr, cl, cr = (at(f, k) for f in (h, u, v, c) for k in (1, 2))
    mid = star[:, 1:-1]
    one = torch.ones_like(mid)
    sl = ul - cl * torch.where(mid > hl, torch.sqrt(0.5 * (mid + hl) * mid) / hl, one)
    sr = ur + cr * torch.where(mid > hr, torch.sqrt(0.5 * (mid + hr) * mid) / hr, one)
    sm = (sl * hr * (ur - sr) - sr * hl * (ul - sl)) / (hr * (ur - sr) - hl * (ul - sl))
    al, ar = hl * (sl - ul) / (sl - sm), hr * (sr - ur) / (sr - sm)
    ql, qr = [at(f, 1) for f in q], [at(f, 2) for f in q]
    f1, f4 = _Swe().F(ql), _Swe().F(qr)
    f2 = [a + sl * (b - x) for a, b, x in zip(f1, (al, al * sm, al * vl), ql)]
    f3 = [a + sr * (b - x) for a, b, x in zip(f4, (ar, ar * sm, ar * vr), qr)]
    weights = []
    for speed, den in ((sl, d1), (sm, d2), (sr, d3)):
        cour = speed * dt / d
        r = torch.where(cour > 0, den[:, :-2], den[:, 2:]) / den[:, 1:-1]
        lim = torch.clamp(torch.minimum(torch.minimum(1.9 * r, 0.5 * (1.0 + r)), 1.9 * one), min=0.0)
        weights.append(torch.copysign(one, cour) * (1.0 - (1.0 - cour.abs()) * lim))
    flux = [0.5 * (a + e) - 0.5 * (weights[0] * (b - a) + weights[1] * (k - b) + weights[2] * (e - k))
            for a, b, k, e in zip(f1, f2, f3, f4)]
    return [a[:, 2:-2] + dt / d * (b[:, :-1] - b[:, 1:]) for a, b in zip(q, flux)]


def _split_substep(scheme, q, order, d, dt, bc):
    euler = scheme == "ee2d_kp07_dimsplit"
    eq = _Euler() if euler else _Swe()
    if scheme == "waf":
        sweep = {0: lambda p: _waf_sweep(p, d, dt), 1: lambda p: _waf_sweep(p, d, dt)}
    else:
        theta = THETA_HLL2 if scheme == "hll2" else THETA
        fx = _hll_flux if euler or scheme == "hll2" else _central_upwind
        fy = _hll_flux if scheme == "hll2" else _central_upwind
        sweep = {0: lambda p: _muscl_sweep(p, d, dt, theta, eq, fx), 1: lambda p: _muscl_sweep(p, d, dt, theta, eq, fy)}
    p = _pad(q, 2, bc)
    for axis in ((0, 1) if order == 0 else (1, 0)):
        p = sweep[0](p) if axis == 0 else _turn(sweep[1](_turn(p)))
    if euler:
        mv = p[2]
        p[2] = mv - EULER_G * p[0] * dt
        p[3] = p[3] - EULER_G * mv * dt
    return [f.contiguous() for f in p]


def _first_order_flux(scheme, l, r, d, dt):
    eq = _Swe()
    if scheme == "hll":
        return _hll_flux(eq, l, r)
    fl, fr = eq.F(l), eq.F(r)
    if scheme == "lxf":
        return [0.5 * (a + b) + d / (4.0 * dt) * (x - y) for a, b, x, y in zip(fl, fr, l, r)]
    mid = eq.F([0.5 * (x + y) + dt / (2.0 * d) * (a - b) for a, b, x, y in zip(fl, fr, l, r)])
    return [0.5 * (0.5 * (a + b) + d / (2.0 * dt) * (x - y) + m) for a, b, x, y, m in zip(fl, fr, l, r, mid)]


def _edge_fluxes(scheme, q, d, dt):
    return _first_order_flux(scheme, [f[:, :-1] for f in q], [f[:, 1:] for f in q], d, dt)


def _first_order_step(scheme, q, d, dt, bc):
    p = _pad(q, 1, bc)
    if scheme == "lxf":
        fx = _edge_fluxes(scheme, [f[1:-1] for f in p], d, dt)
        fy = _turn(_edge_fluxes(scheme, _turn([f[:, 1:-1] for f in p]), d, dt))
        return [a + dt / d * (b[:, :-1] - b[:, 1:]) + dt / d * (e[:-1] - e[1:]) for a, b, e in zip(q, fx, fy)]
    for axis in (0, 1):
        f = _edge_fluxes(scheme, p if axis == 0 else _turn(p), d, dt)
        s = p if axis == 0 else _turn(p)
        s = [a[:, 1:-1] + dt / d * (b[:, :-1] - b[:, 1:]) for a, b in zip(s, f)]
        p = s if axis == 0 else _turn(s)
    return [f.contiguous() for f in p]


def _unsplit_flux(q):
    s = _slopes(q, THETA)
    return _central_upwind(_Swe(), [(f[:, 1:-1] + 0.5 * k)[:, :-1] for f, k in zip(q, s)],
                           [(f[:, 1:-1] - 0.5 * k)[:, 1:] for f, k in zip(q, s)])


def _unsplit_stage(q, d, dt, bc):
    p = _pad(q, 2, bc)
    fx = _unsplit_flux([f[2:-2] for f in p])
    fy = _turn(_unsplit_flux(_turn([f[:, 2:-2] for f in p])))
    return [a + dt / d * (b[:, :-1] - b[:, 1:]) + dt / d * (e[:-1] - e[1:]) for a, b, e in zip(q, fx, fy)]


def _reference_step(case, q, d, dt):
    scheme, bc = case["scheme"], case["bc"]
    dt = float(np.float32(dt))
    if scheme in ("kp07_dimsplit", "hll2", "waf", "ee2d_kp07_dimsplit"):
        half = float(np.float32(0.5 * dt))
        return _split_substep(scheme, _split_substep(scheme, q, 0, d, half, bc), 1, d, half, bc)
    if scheme == "kp07":
        one = _unsplit_stage(q, d, dt, bc)
        return [0.5 * (a + b) for a, b in zip(q, _unsplit_stage(one, d, dt, bc))]
    return _first_order_step(scheme, q, d, dt, bc)


def _cfl_dt(case, q, d):
    """The step of the CFL policy for the state q (the Euler scheme's limit
    takes sqrt(gamma rho) for the sound speed)."""
    c = torch.sqrt((G if len(q) == 3 else GAMMA) * q[0])
    limit = min(float((d / ((q[k] / q[0]).abs() + c)).min()) for k in (1, 2))
    return 0.5 * 0.9 * limit


def _grid(case, fields):
    ny, nx = fields[0].shape
    d = float(np.float32(_dx(case, nx)))
    q = [torch.from_numpy(f).to(_device()).double() for f in fields]
    if case["op"] != "simulate":
        ensemble = case["op"] == "ensemble"
        dt = _cfl_dt(case, q, d) if ensemble else _dt(case, nx, ny)
        for _ in range(8 if ensemble else 1):
            q = _reference_step(case, q, d, dt)
        return q
    t, t_end, n = 0.0, case["steps"] * 0.1, 0
    last = q
    while t < t_end:
        if n % 100 == 0:
            # the unsplit scheme reports the limit of its last stage before the average
            dt = _cfl_dt(case, last, d)
        cur = float(np.float32(min(dt, t_end - t)))
        if not cur > 0.0:
            break
        if case["scheme"] == "kp07":
            one = _unsplit_stage(q, d, cur, case["bc"])
            last = _unsplit_stage(one, d, cur, case["bc"])
            q = [0.5 * (a + b) for a, b in zip(q, last)]
        else:
            q = last = _reference_step(case, q, d, cur)
        t += cur
        n += 1
    return q


def exact(case, seed):
    grids = [_grid(case, f) for f in _fields(case, seed)]
    if case["op"] == "ensemble":
        return [torch.stack(q) for q in grids]
    return grids[0]
