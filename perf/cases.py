"""The work this framework is timed on: resident grids in 1D, 2D and 3D that
advance a few steps, a batch of uneven blasts, a mixed stream of served
requests, and the one-step call on host arrays, each through the public entry
points and with the schemes, sizes and precisions of the benchmarks and tests.

A case is a dict of plain values:
  kind   "grid"    one resident mlau_amd.Solver; a pass is `steps` steps
         "batch"   an Ensemble: add every member, run, download, remove
         "served"  a Server: submit every request, wait, take the results
         "call"    one step of the reference-named entry on host arrays
  problem, nx, ny, nz, odr, flux, rk, ctw, precision, steps   (grid, call)
  cfl    dt from the device's signal-speed check after every step, or fixed
  members, nmin, nmax, steps, precision                        (batch)
  mix    requests as "dim:interior size", precision            (served)

`exact` restates the scheme in plain torch at 64 bits.
"""
import ctypes
import math

import numpy as np
import torch

import mlau_amd as M
from mlau_amd import problems as P
from mlau_amd.ensemble import Ensemble, member
from mlau_amd.server import Server

OFF = 4  # ghost cells per side
CFL = 0.4
PERIODIC = (0,) * 8
# y walls of the Kelvin-Helmholtz set-up: mirrored, normal momentum and field odd
KHI_Y = (1, 1, -1, 1, 1, 1, -1, 1)


def _grid(name, problem, nx, ny=1, nz=1, odr=4, flux="lhlld", precision="fp64", steps=8, cfl=True, rk=3, ctw=1,
          kind="grid"):
    return dict(name=name, kind=kind, problem=problem, nx=nx, ny=ny, nz=nz, odr=odr, flux=flux, precision=precision,
                steps=steps, cfl=cfl, rk=rk, ctw=ctw)


def listed():
    return [
        # the Brio-Wu shock tube at its benchmark size: open boundary, one dt, nothing but latency
        _grid("tube_1024", "tube", 1024, odr=2, flux="mlau", steps=32, cfl=False),
        # a long periodic wave train at fourth order, an odd length near the largest served tube
        _grid("wave_8191", "wave", 8191, steps=16, cfl=False),
        # the vortex at the size of a quick look: few cells, every launch counts
        _grid("vortex_64", "vortex", 64, 64, steps=8),
        # the headline: the vortex at 2048^2 with the dt check on the device
        _grid("vortex_2048", "vortex", 2048, 2048, steps=8),
        # a rectangular vortex in mixed precision, neither side a multiple of a wavefront
        _grid("vortex_mixed_1300x810", "vortex", 1300, 810, precision="mixed", steps=8),
        # Kelvin-Helmholtz between walls: mirrored ghosts, MUSCL with MLAU, odd sizes
        _grid("khi_walls_515x391", "khi", 515, 391, odr=2, flux="mlau", steps=8),
        # a small 3D shear layer with unequal odd sides
        _grid("shear_45x36x51", "shear", 45, 36, 51, flux="mlau", steps=8),
        # the 3D benchmark: the low-Mach shear layer at 256^3
        _grid("shear_256", "shear", 256, 256, 256, flux="mlau", steps=1),
        # the same layer at a served size in mixed precision
        _grid("shear_mixed_128", "shear", 128, 128, 128, flux="mlau", precision="mixed", steps=4),
        # a batch of uneven MUSCL blasts (half MLAU, half HLLD), host to host
        dict(name="blasts_32", kind="batch", members=32, nmin=64, nmax=512, steps=64, precision="fp64"),
        # a burst of served requests of every dimension, each run to its end time
        dict(name="served_7", kind="served", mix="1:300,1:2048,1:5000,2:96,2:496,3:48,3:96", precision="mixed"),
        # the reference driver's own way in: one step per call on host arrays
        _grid("call_512", "vortex", 512, 512, steps=1, cfl=False, kind="call"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["tube", "wave", "vortex", "vortex", "khi", "shear", "shear", "batch", "served", "call"])
    odr = rng.choice([2, 3, 4, 4])
    flux = rng.choice(["mlau", "hlld", "lhlld"])
    precision = rng.choice(["fp64", "fp64", "mixed", "mixed_recon"])
    rk = rng.choice([3, 3, 2])
    steps = rng.choice([1, 3, 8, 16, 21])
    if what in ("tube", "wave"):
        c = _grid("", what, _log_int(rng, 100, 16384), odr=odr, flux=flux, precision=precision, steps=steps,
                  cfl=False, rk=rk)
    elif what in ("vortex", "khi"):
        nx, ny = _log_int(rng, 40, 2048), _log_int(rng, 40, 2048)
        steps = max(1, min(steps, 2048 * 2048 * 8 // (nx * ny)))
        c = _grid("", what, nx, ny, odr=odr, flux=flux, precision=precision, steps=steps, rk=rk,
                  ctw=rng.choice([1, 1, 0]))
    elif what == "shear":
        nx, ny, nz = (_log_int(rng, 18, 200) for _ in range(3))
        steps = max(1, min(steps, 256 ** 3 // (nx * ny * nz)))
        c = _grid("", what, nx, ny, nz, odr=odr, flux=flux, precision=precision, steps=steps, rk=rk)
    elif what == "call":
        dim = rng.choice([1, 2, 2, 3])
        if dim == 1:
            c = _grid("", "tube", _log_int(rng, 100, 16384), odr=odr, flux=flux, steps=1, cfl=False, kind="call")
        elif dim == 2:
            c = _grid("", "vortex", _log_int(rng, 40, 1024), _log_int(rng, 40, 1024), odr=odr, flux=flux, steps=1,
                      cfl=False, kind="call")
        else:
            c = _grid("", "shear", *(_log_int(rng, 18, 96) for _ in range(3)), odr=odr, flux=flux, steps=1, cfl=False,
                      kind="call")
    elif what == "batch":
        n = _log_int(rng, 3, 40)
        c = dict(kind="batch", members=n, nmin=64, nmax=rng.choice([128, 256, 512]), steps=rng.choice([4, 20, 50]),
                 precision=rng.choice(["fp64", "mixed_recon"]))
    else:
        sizes = ["1:%d" % _log_int(rng, 256, 6000), "2:%d" % (16 * _log_int(rng, 4, 40)),
                 "3:%d" % (16 * _log_int(rng, 2, 6))]
        sizes += [rng.choice(sizes).split(":")[0] + ":%d" % (16 * rng.randint(2, 6)) for _ in range(rng.randint(0, 4))]
        c = dict(kind="served", mix=",".join(sizes), precision=rng.choice(["mixed", "fp64"]))
    c.pop("name", None)
    return c


# --------------------------------------------------------------------- inputs
def _dims(case):
    return {"tube": 1, "wave": 1, "vortex": 2, "khi": 2, "shear": 3}[case["problem"]]


def _bounds(case):
    """Boundary flags (x, y, z) per field; 0 is periodic."""
    return PERIODIC, (KHI_Y if case["problem"] == "khi" else PERIODIC), PERIODIC


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _centres(n, device):
    return (torch.arange(n + 2 * OFF, dtype=torch.float64, device=device) - OFF + 0.5) / n


def _state(case, seed):
    """Initial fields (float64, ghosts filled, the framework's layout) on the
    device and what the grid needs to know: spacing, gamma, bx, vfloor."""
    rng = np.random.default_rng(seed)
    u = rng.random(8)
    what, nx, ny, nz = case["problem"], case["nx"], case["ny"], case["nz"]
    dev = _device()
    g = dict(dx=1.0 / nx, dy=1.0 / ny, dz=1.0 / nz, gamma=5.0 / 3.0, bx=0.0, vfloor=0.0)
    if what == "tube":  # Brio-Wu states scaled by 0.8..1.2, as the served tubes
        s = 0.8 + 0.4 * u
        f, _ = P.riemann_1d(nx, (s[0], s[1], 0, 0, 0, 1.0, 0), (0.125 * s[2], 0.1 * s[3], 0, 0, 0, -1.0, 0), 0.75, 2.0)
        g.update(gamma=2.0, bx=0.75, vfloor=1.0)
        return torch.from_numpy(f).to(dev), g
    if what == "wave":  # a transverse wave train on a sheared, compressed background
        x = 2 * math.pi * _centres(nx, dev)
        a, ph = 0.1 + 0.1 * u[0], 2 * math.pi * u[1:4]
        ro = 1.0 + 0.2 * torch.sin(x + ph[0])
        v = [0.3 * torch.sin(2 * x + ph[1]), a * torch.cos(3 * x + ph[2]), a * torch.sin(3 * x + ph[2])]
        by, bz = a * torch.cos(3 * x + ph[2]), a * torch.sin(3 * x + ph[2])
        g.update(bx=1.0, vfloor=1.0)
        en = 0.6 / (g["gamma"] - 1) + 0.5 * (ro * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2) + 1.0 + by * by + bz * bz)
        f = torch.stack([ro, ro * v[0], ro * v[1], ro * v[2], en, by, bz])
        return _fill(f, (PERIODIC,), 1), g
    X, Y = _centres(nx, dev), _centres(ny, dev)
    if what == "vortex":  # Orszag-Tang, shifted by a phase per axis
        px, py, amp = 2 * math.pi * u[0], 2 * math.pi * u[1], (0.9 + 0.2 * u[2]) / math.sqrt(4 * math.pi)
        X, Y = X[None, :], Y[:, None]
        xf, yf = X - 0.5 / nx, Y - 0.5 / ny
        one = torch.ones_like(X * Y)
        vx, vy = -torch.sin(2 * math.pi * Y + py) * one, torch.sin(2 * math.pi * X + px) * one
        pot = lambda x, y: amp * (torch.cos(2 * math.pi * y + py) / (2 * math.pi) + torch.cos(4 * math.pi * x + px) / (4 * math.pi))
        bx = _slope([pot(xf, yf + k / ny) for k in (-1, 0, 1, 2)], case["odr"]) * ny * one
        by = -_slope([pot(xf + k / nx, yf) for k in (-1, 0, 1, 2)], case["odr"]) * nx * one
        ro, pr = 25.0 / (36.0 * math.pi), 5.0 / (12.0 * math.pi)
        bxc, byc = _centre(bx, 0, case["odr"]), _centre(by, 1, case["odr"])
        en = pr / (g["gamma"] - 1) + 0.5 * (ro * (vx * vx + vy * vy) + bxc * bxc + byc * byc)
        zero = torch.zeros_like(one)
        f = torch.stack([ro * one, ro * vx, ro * vy, zero, en, bx, by, zero])
        g.update(vfloor=1.0)
        return _fill(f, _bounds(case), 2), g
    if what == "khi":  # two streams along x between walls in y, a weak field along them
        X, Y = X[None, :], Y[:, None] - 0.5
        one = torch.ones_like(X * Y)
        sh = torch.tanh(Y / 0.05) * one
        ro, vx = 1.0 + 0.25 * sh, 0.5 * sh
        vy = sum(0.01 * torch.sin(2 * math.pi * (m * X + float(u[m]))) for m in (1, 2, 3)) * torch.exp(-(Y / 0.1) ** 2)
        b0 = 0.1 + 0.1 * u[0]
        zero = torch.zeros_like(one)
        en = 1.0 / (g["gamma"] - 1) + 0.5 * (ro * (vx * vx + vy * vy) + b0 * b0)
        f = torch.stack([ro, ro * vx, ro * vy, zero, en, b0 * one, zero, zero])
        return _fill(f, _bounds(case), 2), g
    mach = 0.01 * 4.0 ** (u[0] - 0.5)  # the low-Mach double shear layer with seeded noise across it
    pr = 1.0 / (g["gamma"] * mach * mach)
    shape = (nz + 2 * OFF, ny + 2 * OFF, nx + 2 * OFF)
    f = torch.zeros((8,) + shape, dtype=torch.float64, device=dev)
    f[0] = 1.0
    f[1] = (mach * (torch.tanh((Y - 0.25) / 0.05) - torch.tanh((Y - 0.75) / 0.05) - 1.0))[None, :, None]
    # in mixed precision a layer under way: noise below 1e-3 of the flow is lost in its rounding
    noise = 1e-3 if case["precision"] == "fp64" else 0.1
    for n in (2, 3):
        f[n] = noise * mach * (2.0 * torch.from_numpy(rng.random(shape)).to(dev) - 1.0)
    f[5] = b0 = math.sqrt(2.0 * pr / 100.0)
    f[4] = pr / (g["gamma"] - 1) + 0.5 * (f[1] ** 2 + f[2] ** 2 + f[3] ** 2 + b0 * b0)
    return _fill(f, _bounds(case), 3), g


def _served(case, seed):
    """The requests of a mix: (fields, member) each, physical parameters from the seed."""
    u = np.random.default_rng(seed).random((len(case["mix"].split(",")), 5))
    out = []
    for r, item in enumerate(case["mix"].split(",")):
        dim, n = (int(v) for v in item.split(":"))
        if dim == 1:
            s = 0.8 + 0.4 * u[r]
            d = dict(kind=1, nx=n, rho_l=s[0], p_l=s[1], rho_r=0.125 * s[2], p_r=0.1 * s[3], flux="mlau")
        elif dim == 2:
            d = dict(kind=2, n=n, pratio=10.0 ** (1.0 + 2.0 * u[r, 0]), bmag=0.1 + 0.9 * u[r, 1],
                     bang=2 * math.pi * u[r, 2], flux="mlau" if r % 2 else "hlld")
        else:
            d = dict(kind=3, n=n, mach=10.0 ** (-2.0 + u[r, 0]), flux="mlau")
        f, p, sc = P.serve_request(d)
        # strong blasts keep 64-bit Riemann solvers in the mixed stream
        prec = "mixed_recon" if dim == 2 and case["precision"] == "mixed" else case["precision"]
        out.append((f, _member(f, p, M.scheme(sc["odr"], sc["rk"], sc["flux"], sc["ctw"], bc1d=sc.get("bc1d", "open"),
                                              precision=prec), P.SERVE_TEND[dim])))
    return out


def _member(f, p, sch, tend, max_steps=0):
    return member(f, sch, p["dx"], p.get("dy"), p.get("dz"), tend=tend, cfl=CFL, vfloor=p["vfloor"], gamma=p["gamma"],
                  bx=p.get("bx", 0.0), max_steps=max_steps)


def _blasts(case, seed):
    """Sizes and solvers of the batch benchmark's draws; strengths and fields from the seed."""
    u = np.random.default_rng(seed).random((case["members"], 3))
    out = []
    for k, d in enumerate(P.blast_ensemble_draws(case["members"], 3, case["nmin"], case["nmax"])):
        f, p = P.blast_2d(d["n"], 10.0 ** (1.0 + 2.0 * u[k, 0]), 0.1 + 0.9 * u[k, 1], 2 * math.pi * u[k, 2])
        out.append((f, p, d["flux"]))
    return out


class _Device:
    """One field of a Solver's device-resident state, seen by torch in place;
    keeps the Solver (and so the memory) alive."""

    def __init__(self, solver, ptr, shape):
        self.solver = solver
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f8", data=(ptr, False), version=2)


def prepare(case, seed):
    if case["kind"] == "served":
        return dict(case=case, server=Server(budget_bytes=24 << 30, steps_per_round=4), requests=_served(case, seed))
    if case["kind"] == "batch":
        sch = {fl: M.scheme(2, 3, fl, 1, precision=case["precision"]) for fl in ("mlau", "hlld")}
        mem = [(f, _member(f, p, sch[fl], 10.0, case["steps"])) for f, p, fl in _blasts(case, seed)]
        return dict(case=case, engine=Ensemble(budget_bytes=16 << 30), members=mem)
    f, g = _state(case, seed)
    dim = _dims(case)
    bounds = _bounds(case)
    sch = M.scheme(case["odr"], case["rk"], case["flux"], case["ctw"], dnxs=bounds[0], dnys=bounds[1], dnzs=bounds[2],
                   bc1d="open" if case["problem"] == "tube" else "periodic", precision=case["precision"])
    if case["kind"] == "call":
        dt = _dt(f, g, dim)
        return dict(case=case, fields=f.cpu().numpy(), grid=g, scheme=sch, dt=dt, dim=dim)
    s = M.Solver(f.cpu().numpy(), sch, g["dx"], g["dy"] if dim > 1 else None, g["dz"] if dim > 2 else None,
                 gamma=g["gamma"], bx=g["bx"])
    s.cfl(CFL, g["vfloor"])
    ptr = (ctypes.POINTER(ctypes.c_double) * 8)()
    if M.lib().mlau_device_fields(s._h, ptr) != 0:
        raise RuntimeError("mlau_device_fields failed")
    out = None
    if torch.cuda.is_available():
        out = [torch.as_tensor(_Device(s, ctypes.cast(ptr[n], ctypes.c_void_p).value, tuple(f.shape[1:])), device="cuda")
               for n in range(f.shape[0])]
    return dict(case=case, solver=s, grid=g, out=out)


def run(state):
    case = state["case"]
    if case["kind"] == "served":
        srv = state["server"]
        tickets = [srv.submit(f, m) for f, m in state["requests"]]
        out = []
        for t in tickets:
            srv.wait(t)
            out.append(srv.result(t)[0])
        return out
    if case["kind"] == "batch":
        eng = state["engine"]
        ids = [eng.add(f, m) for f, m in state["members"]]
        eng.run_all(chunk=32)
        out = [eng.download(i) for i in ids]
        for i in ids:
            eng.remove(i)
        return out
    g = state["grid"]
    if case["kind"] == "call":
        f = [a for a in state["fields"]]
        if state["dim"] == 1:
            M.mhd_fd4c_1d(*f, g["bx"], state["dt"], g["dx"], f[0].shape[-1], OFF, g["gamma"], state["scheme"])
        elif state["dim"] == 2:
            M.mhd_fd_ct_2d(*f, state["dt"], g["dx"], g["dy"], f[0].shape[-1], f[0].shape[-2], OFF, OFF, g["gamma"],
                           state["scheme"])
        else:
            M.mhd_fd_ct_3d(*f, state["dt"], g["dx"], g["dy"], g["dz"], f[0].shape[-1], f[0].shape[-2], f[0].shape[-3],
                           OFF, OFF, OFF, g["gamma"], state["scheme"])
        return f
    if case["cfl"]:
        state["solver"].step_cfl(case["steps"], CFL, g["vfloor"])
    else:
        state["solver"].step(case["steps"])
    return state["out"]


def work(case):
    """Per step the state is read and written once (the next step's dt needs
    all of it); operations per cell, stage and direction: projections,
    interpolation, Riemann solver and update as the formulas count them."""
    def need(cells, dim, odr, rk, steps):
        per = {1: 420, 2: 560, 3: 850, 4: 1150}[odr]
        return cells * steps * (7 if dim == 1 else 8) * 16.0, cells * steps * rk * dim * float(per)

    if case["kind"] == "served":
        parts = []
        for item in case["mix"].split(","):
            dim, n = (int(v) for v in item.split(":"))
            speed = {1: 2.7, 2: 4.0, 3: 60.0}[dim]  # a typical signal speed of the drawn states
            parts.append(need(n ** dim, dim, 4 if dim == 3 else 2, 3, math.ceil(P.SERVE_TEND[dim] * speed * n / CFL)))
    elif case["kind"] == "batch":
        parts = [need(d["n"] ** 2, 2, 2, 3, case["steps"])
                 for d in P.blast_ensemble_draws(case["members"], 3, case["nmin"], case["nmax"])]
    else:
        parts = [need(case["nx"] * case["ny"] * case["nz"], _dims(case), case["odr"], case["rk"], case["steps"])]
    return dict(bytes=sum(p[0] for p in parts), flops=sum(p[1] for p in parts))


# ---------------------------------------------------- the scheme at 64 bits
# Arrays [nz, ny, nx] (fewer axes in 2D and 1D), ghosts included; axis 0 is x.
def _at(f, ax, k):
    """f at index + k along an axis."""
    return torch.roll(f, -k, -1 - ax) if k else f


def _fill(f, bounds, dim):
    """Ghosts of a stack of fields under per-field flags, one axis after the other."""
    for ax in range(dim):
        for n in range(f.shape[0]):
            f[n] = _fill1(f[n], ax, bounds[ax][n], 1 if n == 5 + ax and f.shape[0] == 8 else 0)
    return f


def _fill1(f, ax, flag, stagger=0):
    n = f.shape[-1 - ax]
    at = torch.arange(n)
    sign = torch.ones(n, dtype=torch.float64)
    lo, hi = at < OFF, at >= n - OFF + (stagger if flag else 0)
    src = at.clone()
    if flag == 0:
        src[lo], src[hi] = at[lo] + n - 2 * OFF, at[hi] - n + 2 * OFF
    else:
        src[lo], src[hi] = 2 * OFF - 1 + stagger - at[lo], 2 * n - 2 * OFF + stagger - 1 - at[hi]
        sign[lo | hi] = float(flag)
    shape = [1] * f.dim()
    shape[-1 - ax] = n
    return f.index_select(f.dim() - 1 - ax, src.to(f.device)) * sign.to(f.device).view(shape)


def _slope(f, odr):
    return f[2] - f[1] if odr <= 2 else (27.0 * (f[2] - f[1]) - (f[3] - f[0])) / 24.0


def _diff(f, ax, odr):
    return _slope([_at(f, ax, k) for k in (-1, 0, 1, 2)], odr)


def _centre(f, ax, odr):
    if odr <= 2:
        return 0.5 * (f + _at(f, ax, 1))
    return 0.0625 * (9.0 * (f + _at(f, ax, 1)) - (_at(f, ax, -1) + _at(f, ax, 2)))


def _linear(f, ax, odr):
    """Linear face values of each cell: at its upper face and at its lower face."""
    a, b, c, d, e = (_at(f, ax, k) for k in (-2, -1, 0, 1, 2))
    if odr == 1:
        return c, c
    if odr == 2:
        return 0.25 * (-b + 4 * c + d), 0.25 * (-d + 4 * c + b)
    if odr == 3:
        return 0.125 * (-b + 6 * c + 3 * d), 0.125 * (-d + 6 * c + 3 * b)
    return (0.003125 * (9 * a - 56 * b + 234 * c + 144 * d - 11 * e),
            0.003125 * (9 * e - 56 * d + 234 * c + 144 * b - 11 * a))


def _limited(f, odr):
    """Limited face values (upper, lower) from five neighbouring values."""
    a, b, c, d, e = f
    if odr == 1:
        return c, c
    if odr == 2:
        p, q = c - b, d - c
        s = 0.5 * (torch.clamp(torch.maximum(p, q), max=0.0) + torch.clamp(torch.minimum(p, q), min=0.0))
        return c + s, c - s
    if odr == 3:
        t = (d - 2 * c + b) ** 2
        s0, s1 = 1 + t / ((b - c) ** 2 + 1e-40), 1 + t / ((d - c) ** 2 + 1e-40)
        w = 0.25 * s0 / (0.25 * s0 + 0.75 * s1)
        up = 0.5 * (w * (3 * c - b) + (1 - w) * (c + d))
        w = 0.75 * s0 / (0.75 * s0 + 0.25 * s1)
        return up, 0.5 * ((1 - w) * (3 * c - d) + w * (c + b))
    rough = lambda first, second: 1.0 / (((13.0 / 12.0) * second ** 2 + 0.25 * first ** 2) ** 2 + 1e-40)
    s0, s1, s2 = rough(a - 4 * b + 3 * c, a - 2 * b + c), rough(b - d, b - 2 * c + d), rough(e - 4 * d + 3 * c, e - 2 * d + c)

    def side(s0, s2, a, b, d, e):
        n = 1.0 / (0.075 * s0 + 0.65 * s1 + 0.275 * s2)
        w0, w1 = 0.075 * s0 * n, 0.65 * s1 * n
        return 0.125 * (w0 * (3 * a - 10 * b + 15 * c) + w1 * (-b + 6 * c + 3 * d) + (1 - w0 - w1) * (3 * c + 6 * d - e))

    return side(s0, s2, a, b, d, e), side(s2, s0, e, d, b, a)


def _athena(ro, by, bz, pr, bx, gamma):
    """Rows of left eigenvectors l1..l3, columns of right ones r1..r3 and the
    squared sound speed (primitive variables ro,vn,vt,vu,bt,bu,pr)."""
    tiny = 1e-12
    sro = torch.sqrt(ro)
    a2 = torch.abs(gamma * pr / ro)
    bt2 = by * by + bz * bz
    b2 = (bx * bx + bt2) / ro
    root = torch.sqrt(torch.abs((a2 + b2) ** 2 - 4 * a2 * bx * bx / ro))
    cf2, cs2 = torch.abs(0.5 * (a2 + b2 + root)), torch.abs(0.5 * (a2 + b2 - root))
    cf, cs, aa = torch.sqrt(cf2), torch.sqrt(cs2), torch.sqrt(a2)
    some = bt2 > tiny * (bx * bx + bt2)
    half = math.sqrt(0.5)
    norm = torch.sqrt(bt2)
    ty, tz = torch.where(some, by / norm, half), torch.where(some, bz / norm, half)
    some = some | (torch.abs(gamma * pr - bx * bx) > tiny * gamma * pr)
    norm = torch.sqrt(torch.abs(cf2 - cs2))
    af = torch.where(some, torch.sqrt(torch.abs(a2 - cs2)) / norm, 1.0)
    as_ = torch.where(some, torch.sqrt(torch.abs(cf2 - a2)) / norm, 0.0)
    sg = torch.where(bx > 0, 1.0, -1.0)
    d = 0.5 / a2
    left = [[None, -cf * af * d, cs * as_ * d * sg * ty, cs * as_ * d * sg * tz, aa * as_ * d * ty / sro,
             aa * as_ * d * tz / sro, af * d / ro],
            [None, None, -0.5 * tz, 0.5 * ty, -0.5 * tz * sg / sro, 0.5 * ty * sg / sro, None],
            [None, -cs * as_ * d, -cf * af * d * sg * ty, -cf * af * d * sg * tz, -aa * af * d * ty / sro,
             -aa * af * d * tz / sro, as_ * d / ro]]
    right = [[ro * af, -cf * af, cs * as_ * sg * ty, cs * as_ * sg * tz, aa * as_ * sro * ty, aa * as_ * sro * tz,
              af * gamma * pr],
             [None, None, -tz, ty, -sro * tz * sg, sro * ty * sg, None],
             [ro * as_, -cs * as_, -cf * af * sg * ty, -cf * af * sg * tz, -aa * af * sro * ty, -aa * af * sro * tz,
              as_ * gamma * pr]]
    mirror = [1, -1, -1, -1, 1, 1, 1]
    turn = lambda row: [None if v is None else (v if s > 0 else -v) for v, s in zip(row, mirror)]
    one = torch.ones_like(ro)
    left = left + [[one, None, None, None, None, None, -1.0 / a2]] + [turn(left[n]) for n in (2, 1, 0)]
    right = right + [[one, None, None, None, None, None, None]] + [turn(right[n]) for n in (2, 1, 0)]
    return left, right, (cf, torch.sqrt(bx * bx / ro), cs)


def _alfven(ro, by, bz, pr, bx, gamma):
    """Left rows and right columns of the Alfven/entropy projection."""
    c2, ca2 = gamma * pr / ro, bx * bx / ro
    cb2 = c2 + ca2 + (by * by + bz * bz) / ro
    cf2 = 0.5 * (cb2 + torch.sqrt(torch.abs(cb2 * cb2 - 4 * c2 * ca2)))
    sro, one, N = torch.sqrt(ro), torch.ones_like(ro), None
    left = [[N, one, N, N, N, N, N], [cf2, N, N, N, -by, -bz, -one], [N, N, N, N, by, bz, one],
            [N, N, sro, N, one, N, N], [N, N, sro, N, -one, N, N], [N, N, N, sro, N, one, N], [N, N, N, sro, N, -one, N]]
    i, h = 1.0 / cf2, 0.5 / sro
    right = [[N, one, N, N, N, N, N], [i, N, N, N, N, N, N], [i, N, N, N, N, N, one],
             [N, N, h, N, 0.5 * one, N, -0.5 * by], [N, N, h, N, -0.5 * one, N, 0.5 * by],
             [N, N, N, h, N, 0.5 * one, -0.5 * bz], [N, N, N, h, N, -0.5 * one, 0.5 * bz]]
    return left, right


def _faces(q, bn, mach2, gamma, ax, odr):
    """Face states of every cell (at its upper face, at its lower face) from
    primitives q = ro,vn,vt,vu,bt,bu,pr, in the characteristic fields."""
    near = [[_at(v, ax, k) for k in (-2, -1, 0, 1, 2)] for v in q]
    got = []
    for left, right in (_athena(q[0], q[4], q[5], q[6], bn, gamma)[:2], _alfven(q[0], q[4], q[5], q[6], bn, gamma)):
        up, low = [0.0] * 7, [0.0] * 7
        for lrow, rcol in zip(left, right):
            w = [sum(c * near[v][m] for v, c in enumerate(lrow) if c is not None) for m in range(5)]
            wu, wl = _limited(w, odr)
            for v, c in enumerate(rcol):
                if c is not None:
                    up[v], low[v] = up[v] + c * wu, low[v] + c * wl
        got.append((up, low))
    fast = torch.maximum(_at(mach2, ax, -1), torch.maximum(mach2, _at(mach2, ax, 1))) >= 1.0
    out = []
    for a, b in zip(*got):
        side = [torch.where(fast, x, y) for x, y in zip(a, b)]
        for v in range(1, 6):  # a variable that is zero over the stencil stays zero
            none = near[v][0] == 0
            for m in range(1, 5):
                none = none & (near[v][m] == 0)
            side[v] = torch.where(none, 0.0, side[v])
        out.append(side)
    return out


def _fastest(ro, pr, pm, bn2, gamma, v2=None):
    """Squared fast speed (with v2: the speed squared in place of the sound speed's)."""
    c2, ca2 = (gamma * pr / ro if v2 is None else v2), bn2 / ro
    cb2 = c2 + ca2 + 2 * pm / ro
    return 0.5 * (cb2 + torch.sqrt(torch.abs(cb2 * cb2 - 4 * c2 * ca2)))


def _sides(L, R, gamma):
    for ro, vn, vt, vu, bt, bu, pr in (L, R):
        v2, pm = vn * vn + vt * vt + vu * vu, 0.5 * (bt * bt + bu * bu)
        yield v2, pm, pr + pm, pr / (gamma - 1) + pm + 0.5 * ro * v2


def _flux_hlld(L, R, bn, gamma, dv0, dv1, low):
    rol, vnl, vtl, vul, btl, bul, prl = L
    ror, vnr, vtr, vur, btr, bur, prr = R
    tiny, b2, sg = 1e-8, bn * bn, torch.where(bn > 0, 1.0, -1.0)
    (v2l, pml, ptl, enl), (v2r, pmr, ptr, enr) = _sides(L, R, gamma)
    cm = torch.sqrt(torch.maximum(_fastest(rol, prl, pml, b2, gamma), _fastest(ror, prr, pmr, b2, gamma)))
    sl = torch.clamp(torch.minimum(vnl, vnr) - cm, max=0.0)
    sr = torch.clamp(torch.maximum(vnl, vnr) + cm, min=0.0)
    dl, dr = sl - vnl, sr - vnr
    rl, rr = rol * dl, ror * dr
    inv = 1.0 / (rr - rl)
    if low:
        slow = torch.sqrt(torch.maximum(_fastest(rol, prl, pml, b2, gamma, v2l), _fastest(ror, prr, pmr, b2, gamma, v2r)))
        theta = torch.clamp((cm - torch.clamp(dv0, max=0.0)) / (cm - torch.clamp(dv1, max=0.0)), max=1.0) ** 4
        m = torch.clamp(slow / cm, max=1.0)
        vc = (rr * vnr - rl * vnl - theta * (ptr - ptl)) * inv
        pc = (rr * ptl - rl * ptr + m * (2 - m) * rr * rl * (vnr - vnl)) * inv
    else:
        vc = (rr * vnr - rl * vnl - ptr + ptl) * inv
        pc = (rr * ptl - rl * ptr + rr * rl * (vnr - vnl)) * inv

    def star(ro, vn, vt, vu, bt, bu, pt, en, s, d, r):
        c = s - vc
        h = r * c - b2
        some = torch.abs(h) > tiny
        k, m = (vn - vc) * bn / h, (r * d - b2) / h
        vt2, vu2 = torch.where(some, vt + k * bt, vt), torch.where(some, vu + k * bu, vu)
        bt2, bu2 = torch.where(some, m * bt, bt), torch.where(some, m * bu, bu)
        vb2 = vt2 * bt2 + vu2 * bu2
        en2 = (d * en - pt * vn + pc * vc + bn * (vt * bt + vu * bu - vb2)) / c
        return r / c, vt2, vu2, bt2, bu2, vb2, en2

    ro2l, vt2l, vu2l, bt2l, bu2l, vb2l, en2l = star(rol, vnl, vtl, vul, btl, bul, ptl, enl, sl, dl, rl)
    ro2r, vt2r, vu2r, bt2r, bu2r, vb2r, en2r = star(ror, vnr, vtr, vur, btr, bur, ptr, enr, sr, dr, rr)
    ql, qr = torch.sqrt(ro2l), torch.sqrt(ro2r)
    i = 1.0 / (qr + ql)
    vt3, vu3 = (qr * vt2r + ql * vt2l + (bt2r - bt2l) * sg) * i, (qr * vu2r + ql * vu2l + (bu2r - bu2l) * sg) * i
    bt3 = (ql * bt2r + qr * bt2l + qr * ql * (vt2r - vt2l) * sg) * i
    bu3 = (ql * bu2r + qr * bu2l + qr * ql * (vu2r - vu2l) * sg) * i
    vb3 = vt3 * bt3 + vu3 * bu3
    en3l, en3r = en2l - ql * (vb2l - vb3) * sg, en2r + qr * (vb2r - vb3) * sg
    hl = vc > 0
    h2l, h2r = vc - torch.abs(bn) / ql > 0, ~(vc + torch.abs(bn) / qr > 0)
    pick = lambda l2, l3, r3, r2: torch.where(h2l, l2, torch.where(hl, l3, torch.where(h2r, r2, r3)))
    ro = torch.where(hl, ro2l, ro2r)
    vt, vu = pick(vt2l, vt3, vt3, vt2r), pick(vu2l, vu3, vu3, vu2r)
    bt, bu = pick(bt2l, bt3, bt3, bt2r), pick(bu2l, bu3, bu3, bu2r)
    en = pick(en2l, en3l, en3r, en2r)
    return [ro * vc, ro * vc * vc + pc - 0.5 * b2, ro * vt * vc - bn * bt, ro * vu * vc - bn * bu, bt * vc - bn * vt,
            bu * vc - bn * vu, (en + pc) * vc - bn * (vt * bt + vu * bu)]


def _flux_mlau(L, R, bn, gamma, dv0, dv1):
    rol, vnl, vtl, vul, btl, bul, prl = L
    ror, vnr, vtr, vur, btr, bur, prr = R
    tiny, b2, sg = 1e-8, bn * bn, torch.where(bn > 0, 1.0, -1.0)
    ba = sg * bn
    (v2l, pml, ptl, enl), (v2r, pmr, ptr, enr) = _sides(L, R, gamma)
    c = torch.sqrt(torch.maximum(_fastest(rol, prl, pml, b2, gamma), _fastest(ror, prr, pmr, b2, gamma)))
    slow = torch.sqrt(torch.maximum(_fastest(rol, prl, pml, b2, gamma, v2l), _fastest(ror, prr, pmr, b2, gamma, v2r)))
    sl = torch.clamp(torch.minimum(vnl, vnr) - c, max=0.0)
    sr = torch.clamp(torch.maximum(vnl, vnr) + c, min=0.0)
    theta = torch.clamp((c - torch.clamp(dv0, max=0.0)) / (c - torch.clamp(dv1, max=0.0)), max=1.0) ** 4

    def split(m, way):
        up = torch.where(m > 0, 1.0, -1.0)
        edge = 0.5 * (1 + way * up)
        k = m * m - 1
        b = torch.where(up * m > 1, edge, 0.25 * (m + way) ** 2 * (2 - way * m) + way * 0.1875 * m * k * k)
        return b, torch.where(up * m > 1, edge * m, way * (0.25 * (m + way) ** 2 + 0.125 * k * k))

    bl, fl = split(vnl / c, 1.0)
    br, fr = split(vnr / c, -1.0)
    mn = fl + fr
    mf = mn * c - torch.clamp(1 - torch.abs(mn), min=0.0) * theta / c * (ptr - ptl) / (rol + ror)
    left = mf > 0
    way = torch.where(left, 1.0, -1.0)
    up = lambda a, b: torch.where(left, a, b)
    mf = mf * up(rol, ror)
    ml, mr = torch.where(left, mf, 0.0), torch.where(left, 0.0, mf)
    pt = bl * ptl + br * ptr - 0.25 * bl * br * (rol + ror) * slow * (vnr - vnl) \
        - 0.5 * (1 - slow / c) * (bl + br - 1) * (ptl + ptr)
    dl, dr, sn = sl - vnl, sr - vnr, up(sl, sr)
    den = mf + up(rol * dl, ror * dr)
    vc = torch.where((torch.abs(den) > tiny) & (sn != 0), mf * sn / den, up(vnl, vnr))

    def star(ro, vn, vt, vu, bt, bu, s, d):
        e = s - vc
        h = ro * d * e - b2
        some = torch.abs(h) > tiny
        k = torch.where(some, (vc - vn) / h, 0.0)
        dvt, dvu, dbt, dbu = -bn * bt * k, -bn * bu * k, b2 * bt * k / e, b2 * bu * k / e
        m = d / e
        return torch.sqrt(ro * m), dvt, dvu, dbt, dbu, vt + dvt, vu + dvu, dbt + bt * m, dbu + bu * m, 1.0 / e

    ql, dvtl, dvul, dbtl, dbul, vt2l, vu2l, bt2l, bu2l, el = star(rol, vnl, vtl, vul, btl, bul, sl, dl)
    qr, dvtr, dvur, dbtr, dbur, vt2r, vu2r, bt2r, bu2r, er = star(ror, vnr, vtr, vur, btr, bur, sr, dr)
    i = 1.0 / (ql + qr)
    hold = lambda v: sg * torch.minimum(torch.clamp(v, min=0.0), ba)
    blb, brb = hold(ql * i * (ba + qr * vc)), hold(qr * i * (ba - ql * vc))
    blv, brv = hold(qr * i * (ba + mf / qr)), hold(ql * i * (ba - mf / ql))
    res = torch.clamp(ba - way * vc * up(ql, qr), min=0.0)
    cb, cv = i * res, ql * qr * i * res
    nvt = blb * vt2l + brb * vt2r + cb * (bt2r - bt2l) - vc * up(dbtl, dbtr)
    nvu = blb * vu2l + brb * vu2r + cb * (bu2r - bu2l) - vc * up(dbul, dbur)
    nbt = blv * bt2l + brv * bt2r + cv * (vt2r - vt2l) - mf * up(dvtl, dvtr)
    nbu = blv * bu2l + brv * bu2r + cv * (vu2r - vu2l) - mf * up(dvul, dvur)
    fmt, fmu = ml * vtl + mr * vtr - nbt, ml * vul + mr * vur - nbu
    fbt, fbu = ml * btl / rol + mr * btr / ror - nvt, ml * bul / rol + mr * bur / ror - nvu
    vb1 = up(vtl * btl + vul * bul, vtr * btr + vur * bur)
    vb2 = up(vt2l * bt2l + vu2l * bu2l, vt2r * bt2r + vu2r * bu2r)
    w = (mf * vc - b2) ** 2
    vb3 = torch.where(w > tiny * tiny, ((fmt * vc + fbt * bn) * (fmt * bn + fbt * mf) +
                                        (fmu * vc + fbu * bn) * (fmu * bn + fbu * mf)) / w, 0.0)
    nvb = sg * (ba * (sn * vb2 - vc * vb1) * up(el, er) + res * (vb3 - vb2))
    return [mf, ml * vnl + mr * vnr + pt - 0.5 * b2, fmt, fmu, fbt, fbu,
            ml * (enl + ptl) / rol + mr * (enr + ptr) / ror - nvb]


def _flux(name, L, R, bn, gamma, dv0, dv1):
    if name == "mlau":
        return _flux_mlau(L, R, bn, gamma, dv0, dv1)
    return _flux_hlld(L, R, bn, gamma, dv0, dv1, name == "lhlld")


def _dt(f, g, dim):
    """Largest stable time step of a state."""
    inner = (Ellipsis,) + ((slice(OFF, -OFF),) * dim if dim > 1 else (slice(None),))
    v = f[1:4] / f[0]
    if dim == 1:
        b2 = g["bx"] ** 2 + f[5] ** 2 + f[6] ** 2
        pr = (g["gamma"] - 1) * (f[4] - 0.5 * (f[0] * (v ** 2).sum(0) + b2))
        speed = torch.abs(v[0]) + torch.sqrt((g["gamma"] * pr + b2) / f[0])
    else:
        b = [0.5 * (f[5 + a] + _at(f[5 + a], a, 1)) if a < dim else f[5 + a] for a in range(3)]
        b2 = b[0] ** 2 + b[1] ** 2 + b[2] ** 2
        pr = (g["gamma"] - 1) * (f[4] - 0.5 * (f[0] * (v ** 2).sum(0) + b2))
        speed = torch.sqrt((v[:dim] ** 2).sum(0)) + torch.sqrt((g["gamma"] * pr + b2) / f[0])
    speed = speed[inner]
    top = max(float(speed[~torch.isnan(speed)].max()), g["vfloor"])
    return CFL * min(g["dx"], g["dy"] if dim > 1 else 1.0 / 0.1 ** 9, g["dz"] if dim > 2 else 1.0 / 0.1 ** 9) / top


def _weights(rk):
    return [(0.0, 1.0), (0.5 + (rk - 2) * 0.25, 0.5 - (rk - 2) * 0.25), (1.0 / 3.0, 2.0 / 3.0)][:rk]


def _open_ends(f, g, dt):
    """Characteristic open boundary of a tube: the ghosts next to each end."""
    out = f.clone()
    n, k = f.shape[1], dt / g["dx"]
    for side, sgn, inner in ((0, 1, OFF), (1, -1, n - OFF - 1)):
        ends = f[:, [inner, inner - sgn]].cpu()
        v = ends[1:4] / ends[0]
        pr = (g["gamma"] - 1) * (ends[4] - 0.5 * (ends[0] * (v ** 2).sum(0) + g["bx"] ** 2 + ends[5] ** 2 + ends[6] ** 2))
        prim = torch.stack([ends[0], v[0], v[1], v[2], ends[5], ends[6], pr])
        m = prim.mean(1)
        left, right, (cf, ca, cs) = _athena(m[0], m[4], m[5], m[6], torch.tensor(g["bx"], dtype=torch.float64), g["gamma"])
        speed = [m[1] - cf, m[1] - ca, m[1] - cs, m[1], m[1] + cs, m[1] + ca, m[1] + cf]
        q = torch.zeros(7, dtype=torch.float64)
        for row, col, s in zip(left, right, speed):
            w = sum(c * prim[a] for a, c in enumerate(row) if c is not None)
            s = float(s) * sgn
            w = w[1] if s > 0 else (1 + s * k) * w[1] - s * k * w[0]
            for a, c in enumerate(col):
                if c is not None:
                    q[a] += c * w
        en = q[6] / (g["gamma"] - 1) + 0.5 * (q[0] * (q[1:4] ** 2).sum() + g["bx"] ** 2 + q[4] ** 2 + q[5] ** 2)
        cell = torch.stack([q[0], q[0] * q[1], q[0] * q[2], q[0] * q[3], en, q[4], q[5]]).to(f.device)
        ghosts = list(range(OFF)) if side == 0 else list(range(n - OFF, n))
        out[:, ghosts] = cell[:, None]
    return out


def _step_1d(f, g, dt, odr, rk, flux, open_ends):
    u0, gamma, u = f, g["gamma"], f
    bn = torch.full_like(f[0], g["bx"])
    for n, (a, b) in enumerate(_weights(rk)):
        ro, v = u[0], u[1:4] / u[0]
        v2 = (v ** 2).sum(0)
        pr = (gamma - 1) * (u[4] - 0.5 * (ro * v2 + g["bx"] ** 2 + u[5] ** 2 + u[6] ** 2))
        up, low = _faces([ro, v[0], v[1], v[2], u[5], u[6], pr], bn, v2 * ro / (gamma * pr), gamma, 0, odr)
        fl = _flux(flux, [_at(x, 0, -1) for x in up], low, bn, gamma, v[0] - _at(v[0], 0, -1), torch.zeros_like(ro))
        base = _open_ends(u, g, dt) if n == 0 and open_ends else u
        new = base.clone()
        for k, c in enumerate((0, 1, 2, 3, 6, 4, 5)):
            new[k] = a * u0[k] + b * (u[k] - dt / g["dx"] * _diff(fl[c], 0, odr))
        new[:, :OFF], new[:, -OFF:] = base[:, :OFF], base[:, -OFF:]
        u = new if open_ends else _fill(new, (PERIODIC,), 1)
    return u


def _step(f, g, dt, dim, odr, rk, flux, ctw, bounds):
    """One Runge-Kutta step of the constrained-transport scheme in 2D or 3D."""
    u0, gamma, u = f, g["gamma"], f
    h = (g["dx"], g["dy"], g["dz"])
    inner = tuple(slice(OFF, -OFF) for _ in range(dim))
    for ra, rb in _weights(rk):
        ro, v = u[0], [u[1] / u[0], u[2] / u[0], u[3] / u[0]]
        c = [u[5 + a] for a in range(3)]
        for a in range(dim):
            c[a] = _centre(u[5 + a], a, odr)
            for b in range(dim):
                c[a] = _fill1(c[a], b, bounds[b][5 + a])
        v2 = v[0] ** 2 + v[1] ** 2 + v[2] ** 2
        pr = (gamma - 1) * (u[4] - 0.5 * (ro * v2 + c[0] ** 2 + c[1] ** 2 + c[2] ** 2))
        mach2 = v2 * ro / (gamma * pr)
        dv = []
        for a in range(dim):
            d = torch.minimum(_at(v[a], a, 1) - v[a], v[a] - _at(v[a], a, -1))
            for b in range(dim):
                d = _fill1(d, b, -bounds[b][1 + a] if a == b else bounds[b][1 + a])
            dv.append(d)
        flx, central = [], []
        for n in range(dim):
            t, w = (n + 1) % 3, (n + 2) % 3
            up, low = _faces([ro, v[n], v[t], v[w], c[t], c[w], pr], c[n], mach2, gamma, n, odr)
            bn = u[5 + n]
            sens = [torch.minimum(_at(dv[k], n, -1), dv[k]) for k in (t, w) if k < dim]
            fl = _flux(flux, [_at(x, n, -1) for x in up], low, bn, gamma, v[n] - _at(v[n], n, -1),
                       sens[0] if len(sens) == 1 else torch.minimum(*sens))
            del up, low
            cen = {}
            for k, slot in ((t, 4), (w, 5)):
                if k < dim:
                    a, b = _linear(c[k] * v[n], n, odr)
                    p, q = _linear(v[k], n, odr)
                    ql, qr = a - _at(bn, n, 1) * p, b - bn * q
                    cen[k] = 0.5 * (_at(ql, n, -1) + qr)
                    fl[slot] = fl[slot] - cen[k]
            flx.append(fl)
            central.append(cen)
        new = u.clone()
        for k in (0, 1, 2, 3, 4) + ((7,) if dim == 2 else ()):
            out = u[k][inner]
            for n in range(dim):
                slot = {0: 0, 4: 6, 7: 4 if n == 1 else 5}.get(k, 1 + (k - 1 - n) % 3)
                out = out - dt / h[n] * _diff(flx[n][slot], n, odr)[inner]
            new[k][inner] = ra * u0[k][inner] + rb * out
        efield = {}
        for a, b in ((0, 1), (1, 2), (2, 0)):
            if a >= dim or b >= dim:
                continue
            wt = torch.full_like(ro, 0.5)
            if ctw:
                four = lambda x: 0.25 * (x + _at(x, a, -1) + _at(x, b, -1) + _at(_at(x, a, -1), b, -1))
                i = 1.0 / torch.sqrt(four(ro))
                pa = torch.abs(four(v[a])) + torch.abs(0.5 * (u[5 + a] + _at(u[5 + a], b, -1)) * i)
                pb = torch.abs(four(v[b])) + torch.abs(0.5 * (u[5 + b] + _at(u[5 + b], a, -1)) * i)
                wt = (pa + 0.5e-6) / (pa + pb + 1e-6)
            corner = lambda x, ax: (lambda p: _at(p[0], ax, -1) + p[1])(_linear(x, ax, odr))
            efield[3 - a - b] = (-0.5 * (corner(flx[a][4], b) + (1 - wt) * corner(central[a][b], b)) +
                                 0.5 * (corner(flx[b][5], a) + wt * corner(central[b][a], a)))
        for a in range(dim):
            t, w = (a + 1) % 3, (a + 2) % 3
            out = u[5 + a]
            if t < dim:
                out = out - dt / h[t] * _diff(efield[w], t, odr)
            if w < dim:
                out = out + dt / h[w] * _diff(efield[t], w, odr)
            where = list(inner)
            if bounds[a][5 + a]:  # the scheme also moves the face at a wall
                where[-1 - a] = slice(OFF, -OFF + 1)
            where = tuple(where)
            new[5 + a][where] = ra * u0[5 + a][where] + rb * out[where]
        u = _fill(new, bounds, dim)
    return u


def _cost(case):
    """Rough seconds of exact() on the card."""
    cells = case["nx"] * case["ny"] * case["nz"]
    dim = _dims(case)
    return case["steps"] * case["rk"] * dim * (0.035 + cells * 1.2e-8)


def exact(case, seed):
    if case["kind"] in ("served", "batch") or _cost(case) > 18.0:
        return None  # hundreds of steps each: minutes in plain torch
    f, g = _state(case, seed)
    dim = _dims(case)
    dt = _dt(f, g, dim)
    for n in range(case["steps"]):
        if dim == 1:
            f = _step_1d(f, g, dt, case["odr"], case["rk"], case["flux"], case["problem"] == "tube")
        else:
            f = _step(f, g, dt, dim, case["odr"], case["rk"], case["flux"], case["ctw"], _bounds(case))
        if case["cfl"] and n + 1 < case["steps"]:
            dt = _dt(f, g, dim)
    return [x for x in f]
