"""Length of the server's rounds (next_round in mlau_amd/csrc/mlau_server.hip), compiled
for the host from its source text: while the running requests stand it grows to
rounds of at most 2 ms and stays there, follows steps that get longer or shorter, and is
never below the number the server was made with."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "mlau_amd", "csrc", "mlau_server.hip")

DRIVER = r"""
#include <algorithm>
#include <cstdio>
#include <cstdlib>
%s
// least, then pairs of rounds and us per step; a round costs 200 us beside its steps
int main(int argc, char **v)
{
  const int least = atoi(v[1]);
  int n = least;
  for (int a = 2; a + 1 < argc; a += 2)
    for (int k = 0; k < atoi(v[a]); k++) {
      const double s = 200e-6 + n * atof(v[a + 1]) * 1e-6;
      printf("%%d %%.9f\n", n, s);
      n = next_round(least, n, s);
    }
  return next_round(least, 0, 1e-3) != least || next_round(least, 100, 0.0) != least;
}
"""


@pytest.fixture(scope="module")
def rounds(tmp_path_factory):
    src = re.search(r"^int next_round\(.*?^\}", open(SRC).read(), flags=re.S | re.M).group(0)
    d = tmp_path_factory.mktemp("rounds")
    (d / "r.cpp").write_text(DRIVER % src)
    subprocess.run(["g++", "-O1", "-std=c++17", str(d / "r.cpp"), "-o", str(d / "r")], check=True)

    def run(least, *phases):
        out = subprocess.run([str(d / "r"), str(least)] + [str(x) for p in phases for x in p], capture_output=True,
                             text=True, check=True).stdout
        return [(int(a), float(b)) for a, b in (line.split() for line in out.splitlines())]

    return run


@pytest.mark.parametrize("least", [1, 4, 8, 50])
@pytest.mark.parametrize("us", [2, 13, 17, 31, 60, 150, 400])
def test_settles(rounds, least, us):
    r = rounds(least, (30, us))
    assert all(n >= least for n, _ in r)
    assert all(b <= 4 * a for (a, _), (b, _) in zip(r, r[1:]))
    tail = r[8:]
    assert len(set(n for n, _ in tail)) == 1, r
    n, s = tail[0]
    assert n == least or s <= 2e-3, r
    # the next length up (8 or 32 steps more) would be over, or is what the least number gives
    assert (n + (32 if n >= 64 else 8 if n >= 8 else 1)) * (us + 200.0 / n) * 1e-6 > 2e-3, r


def test_follows_the_steps(rounds):
    r = rounds(4, (12, 13), (12, 100), (12, 3000), (12, 13))
    assert r[11][0] == 128 and r[23][0] == 16 and r[35][0] == 4 and r[47][0] == 128, r
    assert min(n for n, _ in r[8:23]) >= 8, r  # shorter steps ask for shorter rounds, not for the shortest
