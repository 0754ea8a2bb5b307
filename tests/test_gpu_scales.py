"""States in other units: densities, velocities and fields scaled over many orders of
magnitude give the oracle's values (FP64 division and square root without operand
scaling are exact while no operand is extreme)."""
import numpy as np
import pytest

import mlau_amd as M
from mlau_amd import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ro", [1e-200, 1e-100, 1e-24, 1e24, 1e60])
@pytest.mark.parametrize("vel", [1e-8, 1e8])
@pytest.mark.parametrize("odr,flux", [(2, "mlau"), (2, "hlld"), (4, "lhlld")])
def test_1d(gpu, ro, vel, odr, flux):
    n = 200
    f0, p = P.brio_wu(n)
    f0[2] += 0.1 * f0[0] * np.sin(7 * np.arange(n + 8) / n)
    f0[4] += 0.5 * f0[2] ** 2 / f0[0]
    f0[0] *= ro
    f0[1:4] *= ro * vel
    f0[4] *= ro * vel * vel
    f0[5:] *= np.sqrt(ro) * vel
    bx, dt = p["bx"] * np.sqrt(ro) * vel, 0.05 / n / vel
    f_o = f0.copy()
    for _ in range(3):
        O.step_1d(f_o, bx, dt, 1.0 / n, 4, p["gamma"], O.scheme(odr, 3, flux, 1))
    s = M.Solver(f0, M.scheme(odr, 3, flux, 1), 1.0 / n, gamma=p["gamma"], bx=bx)
    s.set_dt(dt)
    s.step(3)
    assert np.array_equal(s.download(), f_o, equal_nan=True)
    s.close()
