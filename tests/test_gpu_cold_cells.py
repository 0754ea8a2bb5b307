"""Cells of exactly zero pressure at rest (a cold medium held by its field): their
squared Mach number is 0 / 0, and the reference's max(m2[-1], max(m2[0], m2[+1]))
>= 1 is false wherever the last of the three is such a cell, whatever the others
are (mhd_fd4c_1d.c:155-166).  A supersonic stream that runs into one takes the
oracle's reconstruction, value for value."""
import numpy as np
import pytest

import mlau_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu

GAMMA, BX = 5.0 / 3.0, 0.75


def stream_1d(n):
    """Warm gas at rest, a supersonic warm stream along +x, cold gas at rest,
    warm gas at rest, a quarter each (+ 4 ghosts; both ends are alike)."""
    q = n // 4
    v, pr = np.zeros(n + 8), np.ones(n + 8)
    v[q:2 * q], pr[2 * q:3 * q] = 2.0, 0.0
    f = np.zeros((7, n + 8))
    f[0], f[1], f[5], f[6] = 1.0, v, 1.0, 0.5
    f[4] = pr / (GAMMA - 1.0) + 0.5 * (f[0] * (v * v) + (BX * BX + f[5] ** 2 + f[6] ** 2))
    p = (GAMMA - 1.0) * (f[4] - 0.5 * (f[0] * (v * v) + (BX * BX + f[5] ** 2 + f[6] ** 2)))
    assert np.all(p[2 * q:3 * q] == 0.0)
    return f


def assert_same(a, b, what):
    assert np.all(np.isfinite(b)), what
    assert np.array_equal(a, b), "%s: max |diff| %g" % (what, np.nanmax(np.abs(a - b)))


@pytest.mark.parametrize("odr,rk,flux", [(1, 1, "hlld"), (2, 1, "mlau"), (2, 2, "lhlld"), (4, 1, "lhlld")])
@pytest.mark.parametrize("bc", ["open", "periodic"])
@pytest.mark.parametrize("n", [40, 700])
def test_1d(gpu, n, bc, odr, rk, flux):
    f0 = stream_1d(n)
    dt = 0.02 / n
    f_o = f0.copy()
    O.step_1d(f_o, BX, dt, 1.0 / n, 4, GAMMA, O.scheme(odr, rk, flux, 1), periodic=bc == "periodic")
    s = M.Solver(f0, M.scheme(odr, rk, flux, 1, bc1d=bc), 1.0 / n, gamma=GAMMA, bx=BX)
    s.set_dt(dt)
    s.step(1)
    assert_same(s.download(), f_o, "1D %s" % bc)
    s.close()


@pytest.mark.parametrize("odr,rk,flux", [(1, 1, "hlld"), (2, 1, "mlau"), (2, 2, "lhlld"), (4, 1, "lhlld")])
def test_2d_along_x(gpu, odr, rk, flux):
    n = 40
    f1 = stream_1d(n)
    f0 = np.zeros((8, n + 8, n + 8))
    f0[:5] = f1[:5, None, :]
    f0[5], f0[6], f0[7] = BX, f1[5], f1[6]
    dt = 0.02 / n
    f_o = f0.copy()
    O.step_2d(f_o, dt, 1.0 / n, 1.0 / n, 4, GAMMA, O.scheme(odr, rk, flux, 1))
    s = M.Solver(f0, M.scheme(odr, rk, flux, 1), 1.0 / n, 1.0 / n, gamma=GAMMA)
    s.set_dt(dt)
    s.step(1)
    assert_same(s.download(), f_o, "2D")
    s.close()
