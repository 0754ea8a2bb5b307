"""Large grids that run a stage's x sweep beside the others on a second stream: the launches
of both sides of the line, the values of the same sweeps one by one (tune bit 6), through
graph replays, per-kernel timing and several handles at once."""
import numpy as np
import pytest

import mlau_amd as M
from mlau_amd import problems as P

pytestmark = pytest.mark.gpu


def grid(dim, n):
    if dim == 2:
        f, p = P.vortex_2d(n, 4)
        return f, p, (p["dx"], p["dy"])
    f, p = P.ot_vortex_3d(n)
    return f, p, (p["dx"], p["dy"], p["dz"])


def solver(f, p, d, odr, flux, precision):
    s = M.Solver(f, M.scheme(odr, 3, flux, 1, precision=precision), *d, gamma=p["gamma"])
    s.set_dt(1e-4 * p["dx"])
    return s


@pytest.mark.parametrize("dim,n,odr,flux,precision,beside", [
    (2, 940, 2, "hlld", "mixed", False), (2, 941, 2, "hlld", "mixed", True), (2, 1441, 2, "lhlld", "mixed", False),
    (2, 1442, 2, "lhlld", "mixed", True), (2, 1442, 1, "lhlld", "fp64", True),
    (2, 1500, 2, "hlld", "fp64", False), (2, 1500, 4, "lhlld", "mixed", False), (2, 1725, 4, "lhlld", "mixed", True),
    (2, 1725, 3, "mlau", "mixed", True), (2, 1725, 3, "mlau", "mixed_recon", False), (2, 1725, 2, "roe", "mixed_recon", True),
    (3, 173, 2, "hlld", "mixed_recon", False), (3, 174, 2, "hlld", "mixed_recon", True), (3, 174, 1, "mlau", "fp64", True),
    (3, 174, 4, "lhlld", "mixed", True), (3, 174, 4, "mlau", "mixed_recon", False)])
def test_values_and_launches(gpu, monkeypatch, dim, n, odr, flux, precision, beside):
    f, p, d = grid(dim, n)
    monkeypatch.setenv("MLAU_TUNE", "64")
    s = solver(f, p, d, odr, flux, precision)
    s.step(1)
    want = s.download()
    s.close()
    monkeypatch.setenv("MLAU_TUNE", "0")
    s = solver(f, p, d, odr, flux, precision)
    s.step(1)
    assert np.array_equal(s.download(), want)
    s.upload(f)
    s.kernel_timing(True)
    s.step(1)
    st = {k: v[1] for k, v in s.kernel_stats().items() if "sweep" in k}
    x, y = ("xsweep2d_inl", "ysweep2d_inl") if dim == 2 else ("xsweep3d", "sweeps3d")
    assert st == ({x: 3, y: 3} if beside else {"sweeps%dd" % dim: 3})
    assert np.array_equal(s.download(), want)
    s.close()


def test_graphs_and_handles(gpu):
    """Replays of captured steps against steps one at a time, on two handles in turn."""
    f, p, d = grid(2, 1450)
    a, b, c = (solver(f, p, d, 2, "hlld", "mixed") for _ in range(3))
    for _ in range(3):
        a.step(8)
        b.step(8)
    for _ in range(24):
        c.step(1)
    want = c.download()
    assert np.array_equal(a.download(), want) and np.array_equal(b.download(), want)
    for s in (a, b, c):
        s.close()
