"""Per-kernel timing measures the launches that the steps make: the sweeps of a stage in
one launch, and one by one only where MLAU_TUNE bit 6 has the steps run so."""
import numpy as np
import pytest

import mlau_amd as M
from mlau_amd import problems as P

pytestmark = pytest.mark.gpu
KHI_Y = (1, 1, -1, 1, 1, 1, -1, 1)


def stats(monkeypatch, tune, dim, walls, precision):
    monkeypatch.setenv("MLAU_TUNE", str(tune))
    f, p = P.vortex_2d(70, 4) if dim == 2 else P.ot_vortex_3d(20)
    kw = dict(dnys=KHI_Y) if walls else {}
    s = M.Solver(f, M.scheme(4, 3, "lhlld", 1, precision=precision, **kw), *[p[k] for k in ("dx", "dy", "dz")[:dim]],
                 gamma=p["gamma"])
    s.set_dt(1e-4)
    s.kernel_timing(True)
    s.step(2)
    s.sync()
    st, out = {k: v[1] for k, v in s.kernel_stats().items()}, s.download()
    s.close()
    return {k: n for k, n in st.items() if "sweep" in k}, out


@pytest.mark.parametrize("precision", ["fp64", "mixed", "mixed_recon"])
@pytest.mark.parametrize("dim,walls", [(2, False), (2, True), (3, False)])
def test_sweeps(gpu, monkeypatch, dim, walls, precision):
    joint, a = stats(monkeypatch, 0, dim, walls, precision)
    single, b = stats(monkeypatch, 64, dim, walls, precision)
    assert joint == {"sweeps%dd" % dim: 6}
    tail = "" if dim == 3 or walls else "_inl"
    assert single == {"%ssweep%dd%s" % (x, dim, tail): 6 for x in "xyz"[:dim]}
    assert np.array_equal(a, b)
