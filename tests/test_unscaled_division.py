"""Division and square root without operand scaling (mlau_amd/csrc/mlau_dev.h), compiled for the
host from their source text with g++: over the ranges that their comments state they
give the correctly rounded result of / and sqrt, from any first approximation as
close as the hardware's (v_rcp_f64 and v_rsq_f64 are documented to 2^29 ulp); so do zeros,
infinities, NaN and quotients that overflow.  ratio_class and any_ge1 against the
quotient and the reference's nested max."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HDR = os.path.join(ROOT, "mlau_amd", "csrc", "mlau_dev.h")

DRIVER = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#define MLAU_DEV static
static std::mt19937_64 rng(7);
static double error() { return ((int64_t)(rng() >> 11) - (1ll << 52)) * 0x1p-52 * 0x1p-23; }  // 2^29 ulp
static double approx(double y) { return std::isfinite(y) && y != 0.0 ? y * (1.0 + error()) : y; }
static double model_rcp(double d) { return approx(1.0 / d); }
static double model_rsq(double x) { return approx(1.0 / std::sqrt(x)); }
// v_div_fixup_f64: special operands, and the quotient's sign; any other value passes
static double model_fixup(double q, double d, double n)
{
  const double s = std::signbit(n) != std::signbit(d) ? -1.0 : 1.0, inf = std::numeric_limits<double>::infinity();
  if (std::isnan(n) || std::isnan(d)) return NAN;
  if ((n == 0.0 && d == 0.0) || (std::isinf(n) && std::isinf(d))) return NAN;
  if (d == 0.0 || std::isinf(n)) return s * inf;
  if (std::isinf(d) || n == 0.0) return s * 0.0;
  return std::isnan(q) ? q : s * std::fabs(q);
}
static bool model_class(double x, int mask)  // +-0 and +inf only
{
  return mask == 0x260 && (x == 0.0 || (std::isinf(x) && x > 0.0));
}
#define __builtin_amdgcn_rcp model_rcp
#define __builtin_amdgcn_rsq model_rsq
#define __builtin_amdgcn_div_fixup model_fixup
#define __builtin_amdgcn_class model_class
%s
static bool same(double a, double b) { return (std::isnan(a) && std::isnan(b)) || std::memcmp(&a, &b, 8) == 0; }
// 2^lo <= |x| < 2^hi, mantissas near 1 and 2 among them, but none of all ones: there the last
// step's tie goes by the first approximation, in the compiler's scaled sequence too
static double random_in(int lo, int hi)
{
  uint64_t m = rng() >> 12;
  const int kind = rng() %% 8;
  if (kind == 0) m = rng() %% 4;
  if (kind == 1) m = (1ull << 52) - 2 - rng() %% 4;
  return std::ldexp((rng() & 1 ? -1.0 : 1.0) * (1.0 + m * 0x1p-52), lo + (int)(rng() %% (uint64_t)(hi - lo)));
}
static int bad(const char *what, double a, double b, double got, double want)
{
  printf("%%s(%%a, %%a) = %%a, not %%a\n", what, a, b, got, want);
  return 1;
}
static double ref_max(double a, double b) { return (a >= b) ? a : b; }
int main()
{
  const double inf = std::numeric_limits<double>::infinity(), sp[] = {0.0, -0.0, inf, -inf, NAN, 1.0, -3.0, 0.1};
  for (double d : sp) {
    if (!same(rcp_ieee(d), 1.0 / d)) return bad("rcp", d, 0, rcp_ieee(d), 1.0 / d);
    if (d > -1.0 && !same(sqrt_ieee(d), std::sqrt(d))) return bad("sqrt", d, 0, sqrt_ieee(d), std::sqrt(d));
    for (double n : sp)
      if (!same(quot_ieee(n, d), n / d)) return bad("quot", n, d, quot_ieee(n, d), n / d);
  }
  for (long k = 0; k < 3000000; k++) {
    const double d = random_in(-1021, 1022), r = rcp_ieee(d);
    if (!same(r, 1.0 / d)) return bad("rcp", d, 0, r, 1.0 / d);
    const double n = random_in(-967, 1023), q = n / d;
    if (std::isinf(q) ? std::fabs(n * (1.0 / d)) == inf : std::fabs(q) >= 0x1p-1022 && std::fabs(q) < 0x1p1023)
      if (!same(quot_ieee(n, d), q)) return bad("quot", n, d, quot_ieee(n, d), q);
    const double x = std::fabs(random_in(-766, 1023)), s = sqrt_ieee(x);
    if (!same(s, std::sqrt(x))) return bad("sqrt", x, 0, s, std::sqrt(x));
    // near 1, and the special values
    double a = std::fabs(k & 1 ? random_in(-3, 3) : sp[rng() %% 8]), b = k & 2 ? a * (1.0 + 0x1p-52 * (int)(rng() %% 5 - 2)) : sp[rng() %% 8];
    if (std::isnan(a)) b = a;  // b is formed from a pressure that holds a
    const double t = a / b;
    if (ratio_class(a, b) != (t >= 1.0 ? 1 : std::isnan(t) ? 2 : 0)) return bad("ratio_class", a, b, ratio_class(a, b), t);
    const double v[] = {0.5, 1.0, NAN, inf, -1.0}, m0 = v[rng() %% 5], m1 = v[rng() %% 5], m2 = v[rng() %% 5];
    auto cl = [](double m) { return m >= 1.0 ? 1 : std::isnan(m) ? 2 : 0; };
    if (any_ge1(cl(m0), cl(m1), cl(m2)) != (ref_max(m0, ref_max(m1, m2)) >= 1.0)) return bad("any_ge1", m0, m1, m2, 0);
  }
  printf("ok\n");
  return 0;
}
"""


def test_correctly_rounded(tmp_path):
    text = open(HDR).read()
    src = text[text.index("MLAU_DEV double rcp_ieee"):text.index("// include/interp.h:30-37")]
    c, exe = tmp_path / "d.cpp", tmp_path / "d"
    c.write_text(DRIVER % src)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", str(c), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
