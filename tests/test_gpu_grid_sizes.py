"""Launch shapes chosen from the grid's size: each range of sizes gives the
oracle's values, with remainders in every direction."""
import numpy as np
import pytest

import mlau_amd as M
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
