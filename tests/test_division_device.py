"""div_rn, div_const and rcp_checked as cf_device.hpp has them, compiled for
the host.

Within the range that their comments state they equal the IEEE quotient bit for
bit.  Out of it div_rn may return NaN or miss the last bit (a tiny operand or
quotient, a reciprocal that is subnormal), and nothing else: the kernels' check
for NaN relies on that.  K is a divisor of
div_const in the sweeps, so its reciprocal's bound is checked too."""
from fractions import Fraction
import re
import subprocess

from conftest import ROOT

MAIN = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
%s
static int same(double a, double b) { return memcmp(&a, &b, sizeof a) == 0 || (a != a && b != b); }
/* the sign of a zero quotient is kept for d > 0 */
static int right(double q, double x, double d) { return x == 0 && d < 0 && q == 0 ? 1 : same(q, x / d); }
static uint64_t s = 88172645463325252ULL;
static uint64_t xr(void) { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s; }
static double bits(uint64_t u) { double d; memcpy(&d, &u, sizeof d); return d; }
int main(void) {
  long in = 0, in_bad = 0, out = 0, out_nan = 0, out_ulp = 0, out_bad = 0, c = 0, c_bad = 0;
  const double special[] = {0.0, 1.0, INFINITY, NAN, 0x1p-1074, 0x1.8p-1040, 0x1p-1022, 0x1p-1024, 0x1.fffffffffffffp1023,
                            0x1p1023, 0x1p-969, 0x1p-500, 0x1.23456p600};
  const int ns = sizeof special / sizeof special[0];
  for (long k = 0; k < 6000000; k++) {
    /* every exponent, subnormals, infinities and NaN among them; every second
       pair has exponents that leave the quotient in range */
    uint64_t ux = xr(), ud = xr();
    if (k & 1) ud = (ud & 0x800fffffffffffffULL) | (((ux >> 52 & 0x7ff) / 2 + 300) << 52);
    double x = bits(ux), d = bits(ud);
    if (k < ns * ns * 4) {
      x = special[k / 4 %% ns] * ((k & 1) ? -1 : 1);
      d = special[k / 4 / ns] * ((k & 2) ? -1 : 1);
    }
    double r = 1.0 / d, q = div_rn(x, d, r), t = x / d;
    int normal = isfinite(x) && isnormal(d) && isnormal(r) && (x == 0 || fabs(x) >= 0x1p-969) &&
                 (t == 0 ? x == 0 : isnormal(t));
    if (normal) {
      in++;
      in_bad += !right(q, x, d);
    } else {
      out++;
      if (right(q, x, d)) continue;
      if (q != q) { out_nan++; continue; }
      if (isfinite(q) && isfinite(t) && (fabs(x) < 0x1p-969 || fabs(t) < 0x1p-969 || !isnormal(r)) &&
          (q == nextafter(t, INFINITY) || q == nextafter(t, -INFINITY))) { out_ulp++; continue; }
      out_bad++;
    }
    if (normal && rcp_checked(d) != 0) { c++; c_bad += !right(div_const(x, d, r), x, d); }
  }
  printf("%%ld %%ld %%ld %%ld %%ld %%ld %%ld %%ld\n", in, in_bad, out, out_nan, out_ulp, out_bad, c, c_bad);
  return 0;
}
"""


def _device(name):
    src = (ROOT / "channel_flow_amd" / "csrc" / "cf_device.hpp").read_text()
    f = re.search(r"^(?:__host__ )?__device__ __forceinline__ (double %s\(.*?\n\})" % name, src, re.S | re.M)
    assert f, name
    return "static " + f.group(1)


def test_device_quotients(tmp_path):
    c = tmp_path / "d.c"
    c.write_text(MAIN % "\n".join(map(_device, ("div_const", "rcp_checked", "div_rn"))))
    exe = tmp_path / "d"
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-o", str(exe), str(c), "-lm"], check=True)
    n = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    inside, in_bad, outside, out_nan, out_ulp, out_bad, checked, c_bad = map(int, n)
    assert inside > 2_000_000 and outside > 500_000 and checked > 500_000
    assert in_bad == 0 and c_bad == 0 and out_bad == 0
    assert out_nan > 0 and out_ulp > 0  # the ends of the range are reached


def test_reciprocal_bound_for_K():
    """|RN(1/K) K - 1| <= 2^-54, exactly: div_const's condition."""
    kg = 1.4
    assert abs(Fraction(1.0 / kg) * Fraction(kg) - 1) <= Fraction(1, 2 ** 54)
