"""Bits of the mixed forms: their results do not depend on how the work is cut.
The compiler fuses their multiply-adds as each kernel's code allows, so that two
kernels of the same formulas may round differently: every choice among kernels
is compared value for value here, for all solvers."""
import os
import re
import subprocess

import numpy as np
import pytest

import mlau_amd as M
from mlau_amd import ensemble as E
from mlau_amd import problems as P

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KHI_Y = (1, 1, -1, 1, 1, 1, -1, 1)
FLUXES = ["mlau", "roe", "hlld", "lhlld"]
MIXED = ["mixed", "mixed_recon"]

# interiors and the marches of their mixed sweeps: y (2D); y and z (3D)
SIZES_2D = {(66, 130): (1,), (300, 301): (2,), (700, 600): (4,), (1000, 900): (8,)}
SIZES_3D = {(21, 30, 25): (1, 1), (40, 41, 39): (2, 2), (63, 50, 70): (4, 4), (80, 81, 79): (8, 8),
            (128, 128, 128): (16, 16)}


def assert_same(a, b, what):
    """Equal, NaN for NaN: WCNS3 with the Roe solver leaves some corner cells of a cut vortex NaN on every path."""
    assert np.isfinite(b).mean() > 0.5, what
    assert np.array_equal(a, b, equal_nan=True), "%s: max |diff| %g" % (what, np.nanmax(np.abs(a - b)))


def test_sizes_take_each_march(tmp_path):
    """march_chunk, compiled for the host from its source text, gives the marches named above."""
    text = open(os.path.join(ROOT, "mlau_amd", "csrc", "mlau_common.h")).read()
    src = "\n".join(re.search(r, text, flags=re.S).group(0) for r in (
        r"__host__ __device__ __forceinline__ long xsweep_waves\(.*?\n", r"inline int march_chunk\(.*?\n\}"))
    c, exe = tmp_path / "m.cpp", tmp_path / "m"
    c.write_text("#include <cstdio>\n#include <cstdlib>\n#define __host__\n#define __device__\n#define __forceinline__ inline\n"
                 + src + r"""
int main(int, char **v)
{
  const int nz = atoi(v[1]), ny = atoi(v[2]), nx = atoi(v[3]);
  if (nz == 1) {  // mlau_2d.hip ychunk
    printf("%d\n", march_chunk((nx + 63) / 64, ny - 5, xsweep_waves(ny, nx), 0.5, 8, true));
    return 0;
  }
  const long xw = xsweep_waves((long)ny * nz, nx), yw = ((long)nx * nz + 63) / 64, zw = ((long)nx * ny + 63) / 64;
  printf("%d %d\n", march_chunk(yw, ny - 5, xw + zw * nz, 0.2, 16, true),
         march_chunk(zw, nz - 5, xw + yw * ny, 0.2, 16, true));  // mlau_3d.hip stage3d
}
""")
    subprocess.run(["g++", "-O1", "-std=c++17", str(c), "-o", str(exe)], check=True)
    run = lambda *n: tuple(int(x) for x in subprocess.run([str(exe)] + [str(k) for k in n], capture_output=True,
                                                          text=True, check=True).stdout.split())
    for (ny, nx), want in SIZES_2D.items():
        assert run(1, ny + 8, nx + 8) == want, (ny, nx)
    for (nz, ny, nx), want in SIZES_3D.items():
        assert run(nz + 8, ny + 8, nx + 8) == want, (nz, ny, nx)


def one_way(monkeypatch, tune, f0, sch, d, gamma, dt):
    monkeypatch.setenv("MLAU_TUNE", str(tune))
    s = M.Solver(f0, sch, *d, gamma=gamma)
    s.set_dt(dt)
    s.step(1)
    out = s.download()
    s.close()
    return out


# tune bit 6: the sweeps one by one in the longest marches
@pytest.mark.gpu
@pytest.mark.parametrize("precision", MIXED)
@pytest.mark.parametrize("flux", FLUXES)
@pytest.mark.parametrize("ny,nx", sorted(SIZES_2D))
def test_2d_any_march(gpu, monkeypatch, ny, nx, flux, precision):
    g, p = P.vortex_2d(max(nx, ny), 4)
    f0 = np.ascontiguousarray(g[:, :ny + 8, :nx + 8])
    P.periodic_fill(f0)
    for odr in (1, 2, 3, 4):
        for walls in (False, True):
            sch = M.scheme(odr, 3, flux, odr & 1, precision=precision, dnys=KHI_Y if walls else (0,) * 8)
            a, b = [one_way(monkeypatch, t, f0, sch, (p["dx"], p["dy"]), p["gamma"], 0.1 * p["dx"]) for t in (0, 64)]
            assert_same(a, b, "2D %dx%d odr %d walls %d" % (nx, ny, odr, walls))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", MIXED)
@pytest.mark.parametrize("flux", FLUXES)
@pytest.mark.parametrize("nz,ny,nx", sorted(SIZES_3D))
def test_3d_any_march(gpu, monkeypatch, nz, ny, nx, flux, precision):
    g, p = P.ot_vortex_3d(max(nx, ny, nz))
    f0 = np.ascontiguousarray(g[:, :nz + 8, :ny + 8, :nx + 8])
    P.periodic_fill(f0)
    for odr in (1, 2, 3, 4):
        sch = M.scheme(odr, 3, flux, 1, precision=precision)
        a, b = [one_way(monkeypatch, t, f0, sch, (p["dx"], p["dy"], p["dz"]), p["gamma"], 5e-4) for t in (0, 64)]
        assert_same(a, b, "3D %dx%dx%d odr %d" % (nx, ny, nz, odr))


def tube(n, copies):
    """Waves in every field and a contact in each half of n cells, and the same with the middle
    cell repeated over the length of copies - 1 more of them."""
    x = np.arange(n + 8) / n
    ro = 1.0 + 0.3 * np.sin(9 * x + 1) + 0.5 * ((x > 0.2) & (x < 0.8))
    v = [0.4 * np.sin(5 * x), 0.3 * np.cos(7 * x), 0.2 * np.sin(4 * x + 2)]
    by, bz, pr = 0.6 + 0.3 * np.cos(6 * x), 0.2 * np.sin(11 * x), 1.0 + 0.2 * np.cos(8 * x)
    p = {"gamma": 5.0 / 3.0, "bx": 0.75}
    en = pr / (p["gamma"] - 1) + 0.5 * (ro * sum(c * c for c in v) + p["bx"] ** 2 + by ** 2 + bz ** 2)
    f = np.array([ro] + [ro * c for c in v] + [en, by, bz])
    m = n // 2 + 4
    return f, np.concatenate([f[:, :m]] + [f[:, m:m + 1]] * ((copies - 1) * n) + [f[:, m:]], axis=1), p


# whole steps per launch up to 393216 cells in FP64, a launch or two per stage above: the
# same cells in a short grid and in a long one, as far from the cut as the stencils
# reach; periodic: ghosts from the other end, and ghosts filled otherwise
@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64"] + MIXED)
@pytest.mark.parametrize("flux", FLUXES)
@pytest.mark.parametrize("n", [600, 1499])
def test_1d_any_length(gpu, n, flux, precision):
    short, long, p = tube(n, 400000 // n + 1)
    for odr in (1, 2, 3, 4):
        for rk, steps in ((1, 3), (2, 2), (3, 5)):
            for bc in ("open", "periodic", "periodic, other ghosts"):
                out = []
                for f in (short, long):
                    f0 = f.copy()
                    if bc == "periodic":
                        P.periodic_fill(f0)
                    s = M.Solver(f0, M.scheme(odr, rk, flux, 1, precision=precision, bc1d=bc.split(",")[0]), 1.0 / n,
                                 gamma=p["gamma"], bx=p["bx"])
                    s.set_dt(0.05 / n)
                    s.step(steps)
                    out.append(s.download())
                    s.close()
                k = n // 2 - 4 * rk * steps
                what = "odr %d rk %d %s" % (odr, rk, bc)
                assert_same(out[0][:, :k], out[1][:, :k], what + ", low end")
                assert_same(out[0][:, -k:], out[1][:, -k:], what + ", high end")


# members with an open boundary at odr <= 2: windows of whole steps while a group's
# windows (running members of the mean size) fill the 256 CUs at most three times,
# stage launches above.  Alone, beside a member of 3500 windows that runs as long, and
# beside one of 870 that ends after two steps.
@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64"] + MIXED)
@pytest.mark.parametrize("flux", FLUXES)
@pytest.mark.parametrize("odr,rk", [(1, 2), (1, 3), (2, 2), (2, 3)])
def test_1d_members_in_windows_or_stages(gpu, odr, rk, flux, precision):
    sch = M.scheme(odr, rk, flux, 1, precision=precision)
    out = {}
    for beside in ("alone", "long", "short"):
        ens = E.Ensemble(budget_bytes=1 << 29)
        ens.kernel_timing(True)
        ids = []
        for n, steps in ((5, 7), (183, 0), (700, 14)):
            f, _, p = tube(n, 1)
            m = E.member(f, sch, 1.0 / n, tend=4.0 / n, cfl=0.4, vfloor=1.0, gamma=p["gamma"], bx=p["bx"], max_steps=steps)
            ids.append(ens.add(f, m))
        if beside != "alone":
            n = (870 if beside == "short" else 3500) * (182 if rk == 3 else 206)
            f, _, p = tube(n, 1)
            ens.add(f, E.member(f, sch, 1.0 / n, tend=1.0, cfl=0.4, vfloor=1.0, gamma=p["gamma"], bx=p["bx"],
                                max_steps=2 if beside == "short" else 40))
        steps = 0
        while any(ens.status(i)[0] == E.RUNNING for i in ids):
            ens.run(5)
            steps += 5
        st = {k: v[1] for k, v in ens.kernel_stats().items()}
        sweeps, stages = st.get("ens_xsweep", 0), st.get("ens_stage", 0)
        if beside == "alone":
            assert sweeps == 0 and stages > 0, st
        elif beside == "long":
            assert sweeps == steps and stages == steps * (rk - 1), st
        else:
            assert sweeps == 5 and stages > 5 * (rk - 1), st
        out[beside] = [ens.download(i) for i in ids], [ens.status(i) for i in ids]
        ens.close()
    for beside in ("long", "short"):
        assert out[beside][1] == out["alone"][1], beside
        for a, b in zip(out[beside][0], out["alone"][0]):
            assert_same(a, b, "member, companion %s" % beside)
