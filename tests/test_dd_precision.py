"""The double-double quotient and square root of the converged-root inversion
(hg_dd.h), compiled for the host, over random operands against 113-bit
arithmetic: at most 4 units of 2^-106 of the result, which three quotient terms
and a remainder kept in double-double hold and shorter forms do not.  The hardware's reciprocal and reciprocal square root
estimates are stood in for by values cut to 27 bits."""
import os
import subprocess

REPO = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))

SOURCE = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#define __device__
#define __host__
#define __forceinline__ inline
static double cut27(double x) {
  uint64_t b;
  memcpy(&b, &x, 8);
  b &= ~((1ull << 26) - 1);
  memcpy(&x, &b, 8);
  return x;
}
#define __builtin_amdgcn_rcp(x) cut27(1.0 / (x))
#define __builtin_amdgcn_rsq(x) cut27(1.0 / std::sqrt(x))
using std::fma;
using std::sqrt;
#include "hg_dd.h"
using namespace hg;

static uint64_t state = 88172645463325252ull;
static double uniform() {  // in [0.5, 1)
  state ^= state << 13;
  state ^= state >> 7;
  state ^= state << 17;
  return 0.5 + (double)(state >> 11) * 0x1p-54;
}
static dd operand() {
  const double hi = uniform() * std::exp2(std::floor(uniform() * 80.0) - 60.0);
  return fast_two_sum(hi, hi * 0x1p-53 * (4.0 * uniform() - 3.0));
}
static double units(__float128 e) { return std::fabs((double)(e * (__float128)0x1p106)); }

int main() {
  double qmax = 0, rmax = 0;
  for (int n = 0; n < 400000; n++) {
    const dd a = operand(), b = operand(), q = dd_div(a, b), r = dd_sqrt(a);
    const __float128 A = (__float128)a.hi + a.lo, B = (__float128)b.hi + b.lo;
    const __float128 Q = (__float128)q.hi + q.lo, R = (__float128)r.hi + r.lo, T = A / B;
    const double eq = units((Q - T) / T), er = units((R * R - A) / A / 2);
    if (!(eq <= qmax)) qmax = eq;
    if (!(er <= rmax)) rmax = er;
  }
  printf("%.3f %.3f\n", qmax, rmax);
}
"""


def test_quotient_and_root_keep_their_bits(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text("")
    (tmp_path / "dd.cpp").write_text(SOURCE)
    exe = str(tmp_path / "dd")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-I", str(tmp_path), "-I",
                    os.path.join(REPO, "harm_finalwham_amd", "csrc"), str(tmp_path / "dd.cpp"), "-o", exe], check=True)
    quotient, root = map(float, subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split())
    print("units of 2^-106: quotient", quotient, "root", root)
    assert quotient <= 4.0
    assert root <= 4.0
