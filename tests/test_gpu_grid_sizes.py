"""Launch shapes chosen from the grid's size: each range of sizes gives the
oracle's values, with remainders in every direction."""
import numpy as np
import pytest

import mlau_amd as M
from mlau_amd import ensemble as E
from mlau_amd import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

KHI_Y = (1, 1, -1, 1, 1, 1, -1, 1)


def assert_same(a, b, what):
    assert np.all(np.isfinite(b)), what
    assert np.array_equal(a, b), "%s: max |diff| %g" % (what, np.abs(a - b).max())


@pytest.mark.parametrize("walls", [False, True])
@pytest.mark.parametrize("ny,nx", [(4, 5), (9, 63), (66, 130), (300, 301), (770, 1025)])
def test_2d_march_lengths(gpu, ny, nx, walls):
    """y-sweep marches of 1, 2, 4 and 8 faces per lane, the last one cut short."""
    g, p = P.vortex_2d(max(nx, ny, 16), 4)
    f0 = np.ascontiguousarray(g[:, :ny + 8, :nx + 8])
    dny = KHI_Y if walls else (0,) * 8
    for n in range(8):
        O.lib().oc_bc2d(O._p(f0[n]), nx + 8, ny + 8, 4, 4, int(n == 5), 0, int(n == 6), dny[n])
    dt = 0.2 * p["dx"] / O.cfl_vmax_2d(f0, 4, p["gamma"], 1.0)
    f_o = f0.copy()
    for _ in range(2):
        O.step_2d(f_o, dt, p["dx"], p["dy"], 4, p["gamma"], O.scheme(4, 3, "lhlld", 1), dn=(0,) * 8, dny=dny)
    s = M.Solver(f0, M.scheme(4, 3, "lhlld", 1, dnys=dny), p["dx"], p["dy"], gamma=p["gamma"])
    s.set_dt(dt)
    s.step(2)
    assert_same(s.download(), f_o, "2D %dx%d" % (nx, ny))
    s.close()


# walls: primitives and weights in one pass below 1310720 cells with ghosts, two
# from there on
@pytest.mark.parametrize("ctw", [0, 1])
@pytest.mark.parametrize("ny,nx", [(5, 4), (31, 70), (1272, 1015), (1272, 1016)])
def test_2d_wall_primitive_passes(gpu, ny, nx, ctw):
    g, p = P.vortex_2d(max(nx, ny, 16), 4)
    f0 = np.ascontiguousarray(g[:, :ny + 8, :nx + 8])
    for n in range(8):
        O.lib().oc_bc2d(O._p(f0[n]), nx + 8, ny + 8, 4, 4, int(n == 5), 0, int(n == 6), KHI_Y[n])
    dt = 0.2 * p["dx"] / O.cfl_vmax_2d(f0, 4, p["gamma"], 1.0)
    f_o = f0.copy()
    O.step_2d(f_o, dt, p["dx"], p["dy"], 4, p["gamma"], O.scheme(2, 3, "mlau", ctw), dn=(0,) * 8, dny=KHI_Y)
    s = M.Solver(f0, M.scheme(2, 3, "mlau", ctw, dnys=KHI_Y), p["dx"], p["dy"], gamma=p["gamma"])
    s.set_dt(dt)
    s.step(1)
    assert_same(s.download(), f_o, "2D walls %dx%d" % (nx, ny))
    s.close()


# y- and z-sweep marches of 1 to 8 faces per lane; 1, 2 and 4 planes per thread
# in the aux, edge and update kernels; the last of each cut short
@pytest.mark.parametrize("nz,ny,nx", [(4, 5, 6), (30, 21, 25), (7, 120, 125), (63, 50, 70), (85, 96, 97),
                                      (131, 96, 127)])
def test_3d_marches(gpu, nz, ny, nx):
    g, p = P.ot_vortex_3d(max(nx, ny, nz, 16))
    f0 = np.ascontiguousarray(g[:, :nz + 8, :ny + 8, :nx + 8])
    P.periodic_fill(f0)
    dt = 5e-4
    f_o = f0.copy()
    O.step_3d(f_o, dt, p["dx"], p["dy"], p["dz"], 4, p["gamma"], O.scheme(4, 3, "mlau", 1))
    s = M.Solver(f0, M.scheme(4, 3, "mlau", 1), p["dx"], p["dy"], p["dz"], gamma=p["gamma"])
    s.set_dt(dt)
    s.step(1)
    assert_same(s.download(), f_o, "3D %dx%dx%d" % (nx, ny, nz))
    s.close()


# whole steps per launch in 1D: windows of 256 cells that own 256 - 2*halo, so
# one, two and more windows, a last one of a single cell, grids smaller than the
# halo, odd and even launch counts, and each number of steps per launch
@pytest.mark.parametrize("bc", ["open", "periodic", "periodic, other ghosts"])
@pytest.mark.parametrize("n,odr,rk,flux,steps", [
    (4, 2, 3, "mlau", 3), (5, 4, 3, "lhlld", 2), (9, 1, 1, "hlld", 1), (160, 4, 3, "lhlld", 8),
    (161, 4, 3, "mlau", 9), (184, 2, 3, "mlau", 12), (369, 2, 3, "lhlld", 7), (238, 2, 3, "roe", 1),
    (239, 3, 2, "hlld", 5), (500, 4, 1, "lhlld", 6), (140001, 2, 3, "mlau", 3), (400003, 4, 3, "lhlld", 1)])
def test_1d_windows(gpu, bc, n, odr, rk, flux, steps):
    f0, p = P.brio_wu(max(n, 16))
    f0 = np.ascontiguousarray(f0[:, (max(n, 16) - n) // 2:][:, :n + 8])
    x = np.arange(n + 8) / n
    f0[2] += 0.1 * f0[0] * np.sin(7 * x)
    f0[4] += 0.5 * f0[2] ** 2 / f0[0]
    if bc == "periodic":
        f0[:, :4], f0[:, -4:] = f0[:, n:n + 4].copy(), f0[:, 4:8].copy()
    dt = 0.2 / n / 4.0
    f_o = f0.copy()
    for _ in range(steps):
        O.step_1d(f_o, p["bx"], dt, 1.0 / n, 4, p["gamma"], O.scheme(odr, rk, flux, 1), periodic=bc != "open")
    s = M.Solver(f0, M.scheme(odr, rk, flux, 1, bc1d=bc.split(",")[0]), 1.0 / n, gamma=p["gamma"], bx=p["bx"])
    s.set_dt(dt)
    s.step(steps)
    assert_same(s.download(), f_o, "1D %s n=%d" % (bc, n))
    t, _, k = s.time()
    assert k == steps and abs(t - steps * dt) < 1e-12
    s.close()


@pytest.mark.parametrize("bc", ["open", "periodic"])
@pytest.mark.parametrize("steps", [1, 2, 9])
def test_1d_cfl_loop(gpu, bc, steps):
    """dt from the whole grid after every step: one step per launch."""
    f0, p = P.brio_wu(301)
    f_o = f0.copy()
    dt = 0.4 * p["dx"] / O.vmax_1d(f_o, p["bx"], p["gamma"])
    for _ in range(steps):
        O.step_1d(f_o, p["bx"], dt, p["dx"], 4, p["gamma"], O.scheme(2, 3, "mlau", 1), periodic=bc != "open")
        dt = 0.4 * p["dx"] / O.vmax_1d(f_o, p["bx"], p["gamma"])
    s = M.Solver(f0, M.scheme(2, 3, "mlau", 1, bc1d=bc), p["dx"], gamma=p["gamma"], bx=p["bx"])
    s.cfl(0.4, 1.0)
    s.step_cfl(steps, 0.4, 1.0)
    assert s.time()[1] == dt
    assert_same(s.download(), f_o, "1D cfl loop " + bc)
    s.close()


# members with an open boundary: windows of 256 cells that own 182 (rk 3) or 206
# (rk 2), one, two and more of them, a last one of a single cell, members smaller
# than a window or of exactly one; ended by tend and by max_steps at each place in
# a launch of up to four steps; with 800 more members, which end after two
# steps, in stages before and in windows from then on
@pytest.mark.parametrize("chunk,more", [(1, 0), (3, 0), (8, 0), (21, 0), (1, 800), (3, 800)])
def test_1d_member_windows(gpu, chunk, more):
    cases = [(5, 2, 3, "mlau", 0), (6, 1, 2, "roe", 1), (182, 2, 3, "mlau", 2), (183, 2, 3, "lhlld", 3),
             (206, 2, 2, "hlld", 4), (207, 1, 2, "mlau", 5), (248, 2, 3, "mlau", 6), (249, 2, 3, "hlld", 7),
             (365, 2, 3, "lhlld", 8), (413, 2, 2, "mlau", 9), (1093, 2, 3, "mlau", 0), (547, 2, 3, "mlau", 11)]
    cases += [(16, 2, 3, "mlau", 2)] * more
    ens = E.Ensemble(budget_bytes=1 << 28)
    ids, ref = [], []
    for k, (n, odr, rk, flux, most) in enumerate(cases):
        f0, p = P.brio_wu(max(n, 16))
        f0 = np.ascontiguousarray(f0[:, (max(n, 16) - n) // 2:][:, :n + 8])
        f0[2] += 0.1 * f0[0] * np.sin(7 * np.arange(n + 8) / n)
        f0[4] += 0.5 * f0[2] ** 2 / f0[0]
        tend = 3.0 / n
        m = E.member(f0, M.scheme(odr, rk, flux, 1), 1.0 / n, tend=tend, cfl=0.4, vfloor=1.0, gamma=p["gamma"],
                     bx=p["bx"], max_steps=most)
        ids.append(ens.add(f0, m))
        if k and cases[k] == cases[k - 1]:
            ref.append(ref[-1])
            continue
        g = f0.copy()
        t, ns, _ = O.run_to_1d(g, p["bx"], 1.0 / n, 4, p["gamma"], O.scheme(odr, rk, flux, 1), tend, 0.4, 1.0,
                              max_steps=most)
        ref.append((g, t, ns))
    ens.run_all(chunk=chunk)
    for k, i in enumerate(ids):
        _, t, _, ns = ens.status(i)
        assert (t, ns) == ref[k][1:], (cases[k], t, ns, ref[k][1:])
        assert_same(ens.download(i), ref[k][0], "1D member %s" % (cases[k],))
    ens.close()
