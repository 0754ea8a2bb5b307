"""When open 1D members run in windows of whole steps: a group's launch of several steps
while the windows fill the 256 CUs at most three times, of one step while they fill them
once; stage launches otherwise. Same values either way."""
import numpy as np
import pytest

import mlau_amd as M
from mlau_amd import ensemble as E
from mlau_amd import problems as P

pytestmark = pytest.mark.gpu


def run(members, n, chunk, steps):
    ens = E.Ensemble(budget_bytes=1 << 30)
    ens.kernel_timing(True)
    f, p = P.brio_wu(n)
    m = E.member(f, M.scheme(2, 3, "mlau", 1), 1.0 / n, tend=1.0, cfl=0.4, vfloor=1.0, gamma=p["gamma"], bx=p["bx"])
    ids = [ens.add(f, m) for _ in range(members)]
    for _ in range(steps // chunk):
        ens.run(chunk)
    out = [ens.download(i) for i in ids], [ens.status(i) for i in ids]
    sweeps = ens.kernel_stats().get("ens_xsweep", (0.0, 0))[1]
    ens.close()
    return sweeps, out


# members of 200 cells: two windows each
@pytest.mark.parametrize("members,one,two", [(2, False, False), (128, False, False), (129, True, False),
                                             (384, True, False), (385, True, True)])
def test_path(gpu, members, one, two):
    s1, a = run(members, 200, 1, 6)
    s2, b = run(members, 200, 2, 6)
    assert (s1, s2) == (6 * one, 6 * two)
    assert a[1] == b[1]
    for x, y in zip(a[0], b[0]):
        assert np.array_equal(x, y)
