"""How many whole steps a 1D launch takes: 4 or 2 where their windows of 256 cells (own 256 less
two halos of 3 or 4 cells for each stage) fill no more rounds of the 256 CUs than one step's; periodic
grids at ODR 2, which take a stage in one launch, keep to that from 280,000 cells on and for single
steps of more than one round.  The values do not depend on it."""
import numpy as np
import pytest

import mlau_amd as M

pytestmark = pytest.mark.gpu
OWN = lambda odr, steps: 256 - 2 * 3 * steps * (3 if odr <= 2 else 4)


@pytest.mark.parametrize("n,odr,bc,steps,whole", [
    (256 * OWN(2, 4), 2, "open", 8, 2), (256 * OWN(2, 4) + 1, 2, "open", 8, 4), (256 * OWN(2, 2) + 1, 2, "open", 8, 8),
    (512 * OWN(4, 2), 4, "periodic", 8, 4), (512 * OWN(4, 2) + 1, 4, "periodic", 8, 8), (100000, 2, "periodic", 8, 4),
    (280000, 2, "periodic", 8, 4), (280001, 2, "periodic", 8, 0), (280001, 2, "open", 8, 4),
    (256 * OWN(2, 1), 2, "periodic", 1, 2), (256 * OWN(2, 1) + 1, 2, "periodic", 1, 0), (100000, 4, "periodic", 1, 2)])
def test_launches(gpu, n, odr, bc, steps, whole):
    """whole: launches of k_step1d, with the copy after an odd number of them."""
    x = np.arange(n + 8) / n
    ro, v, by = 1.0 + 0.2 * np.sin(9 * x), 0.3 * np.cos(7 * x), 0.5 + 0.2 * np.sin(5 * x)
    f = np.array([ro, ro * v, 0 * x, 0 * x, 1.5 + 0.5 * (ro * v * v + 1.0 + by * by), by, 0 * x])
    out = []
    for timing in (True, False):
        s = M.Solver(f, M.scheme(odr, 3, "mlau", 1, bc1d=bc), 1.0 / n, gamma=5.0 / 3.0, bx=1.0)
        s.set_dt(0.1 / n)
        if timing:
            s.kernel_timing(True)
            s.step(steps)
            st = {k: v[1] for k, v in s.kernel_stats().items()}
        else:  # one by one: another number of steps per launch
            for _ in range(steps):
                s.step(1)
        out.append(s.download())
        s.close()
    assert st.get("step1d", 0) == whole, st
    assert np.array_equal(out[0], out[1])
