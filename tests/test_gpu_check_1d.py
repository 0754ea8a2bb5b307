"""The 1D signal-speed check (dt of mlau_cfl and of mlau_step_cfl)."""
import numpy as np
import pytest

import mlau_amd as M
from mlau_amd import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 249, 504, 505, 131063, 1000003, 2500001])
def test_maximum_over_all_cells(gpu, n):
    """The oracle's speed and dt wherever the fastest cell lies, ghosts included;
    NaN speeds do not count."""
    f0, p = P.brio_wu(max(n, 16))
    f0 = np.ascontiguousarray(f0[:, :n + 8])
    s = M.Solver(f0, M.scheme(2, 3, "mlau", 1, bc1d="open"), 1.0 / n, gamma=p["gamma"], bx=p["bx"])
    for k, at in enumerate([0, 3, n // 3, n + 3, n + 7]):
        f = f0.copy()
        f[1, at] += (5.0 + k) * f[0, at]
        f[4, at] += 0.5 * (f[1, at] ** 2 - f0[1, at] ** 2) / f[0, at]
        f[4, (at + 1) % (n + 8)] = np.nan
        s.upload(f)
        want = O.vmax_1d(f, p["bx"], p["gamma"], 1.0)
        assert want > 5.0
        assert s.cfl(0.4, 1.0) == (0.4 * (1.0 / n) / want, want)
    s.close()


def test_long_grid_is_not_held_up_by_its_blocks(gpu):
    """Every block adds to the same two words, one after the other: a check of 4M
    cells in 1D takes at most twice as long as in 2D, where the number of blocks has its limit."""
    us = {}
    for dim in (1, 2):
        if dim == 1:
            f, p = P.brio_wu(2048 * 2048)
            s = M.Solver(f, M.scheme(2, 3, "mlau", 1), p["dx"], gamma=p["gamma"], bx=p["bx"])
        else:
            f, p = P.vortex_2d(2048, 4)
            s = M.Solver(f, M.scheme(2, 3, "mlau", 1), p["dx"], p["dy"], gamma=p["gamma"])
        s.cfl(0.4, 1.0)
        s.kernel_timing(True)
        for _ in range(10):
            s.cfl(0.4, 1.0)
        ms, cnt = s.kernel_stats()["cfl%dd" % dim]
        us[dim] = 1e3 * ms / cnt
        s.close()
    print("check of 4M cells: 1D %.1f us, 2D %.1f us" % (us[1], us[2]))
    assert us[1] <= 2.0 * us[2], us
