// Double-double arithmetic: a value is the unevaluated sum hi + lo of two
// doubles with |lo| <= ulp(hi) / 2, about 106 bits of significand.
//
// Built from the error-free transformations: Knuth's two-sum (any a, b),
// Dekker's fast two-sum (|a| >= |b|) and the exact product a * b = p + e with
// e = fma(a, b, -p).  The addition is the accurate one (both halves summed
// with error-free transformations), so cancellation between the operands
// keeps full relative precision; multiplication, division and square root
// are the usual one-correction forms (Dekker 1971; Hida, Li and Bailey,
// "Library for double-double and quad-double arithmetic", 2007).
//
// The library compiles with -ffp-contract=off, so every operation below is
// evaluated as written; fma() is an explicit fused multiply-add.
#pragma once
#include <hip/hip_runtime.h>

#include "hg_div.h"

namespace hg {

struct dd {
  double hi, lo;
};

__device__ __forceinline__ dd dd_of(double a) { return dd{a, 0.0}; }
__device__ __forceinline__ double dd_val(dd a) { return a.hi + a.lo; }

__device__ __forceinline__ dd two_sum(double a, double b) {
  double s = a + b;
  double bb = s - a;
  return dd{s, (a - (s - bb)) + (b - bb)};
}

__device__ __forceinline__ dd fast_two_sum(double a, double b) {
  double s = a + b;
  return dd{s, b - (s - a)};
}

__device__ __forceinline__ dd two_prod(double a, double b) {
  double p = a * b;
  return dd{p, fma(a, b, -p)};
}

__device__ __forceinline__ dd dd_neg(dd a) { return dd{-a.hi, -a.lo}; }

__device__ __forceinline__ dd dd_add(dd a, dd b) {
  dd s = two_sum(a.hi, b.hi);
  dd t = two_sum(a.lo, b.lo);
  s.lo += t.hi;
  s = fast_two_sum(s.hi, s.lo);
  s.lo += t.lo;
  return fast_two_sum(s.hi, s.lo);
}

__device__ __forceinline__ dd dd_sub(dd a, dd b) { return dd_add(a, dd_neg(b)); }

__device__ __forceinline__ dd dd_mul(dd a, dd b) {
  dd p = two_prod(a.hi, b.hi);
  p.lo += a.hi * b.lo + a.lo * b.hi;
  return fast_two_sum(p.hi, p.lo);
}

__device__ __forceinline__ dd dd_mul_d(dd a, double b) {
  dd p = two_prod(a.hi, b);
  p.lo += a.lo * b;
  return fast_two_sum(p.hi, p.lo);
}

// 1 / b to about one ulp: the hardware estimate and two Newton steps
__device__ __forceinline__ double rcp_1ulp(double b) { return rcp_refined(b); }

// 1 / sqrt(a) to about one ulp: the hardware estimate and two coupled steps
// for sqrt(a) and 1 / (2 sqrt(a))
__device__ __forceinline__ double rsqrt_1ulp(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  double g = a * y, h = 0.5 * y;
  double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  r = fma(-h, g, 0.5);
  h = fma(h, r, h);
  return h + h;
}

// a / b from r = 1 / b.hi to a few ulp: the quotient of the leading parts
// and one term from its remainder, which the exact product gives to 2^-104 of
// a (a third term would follow the rounding of the second)
__device__ __forceinline__ dd dd_div_r(dd a, dd b, double r) {
  const double q1 = a.hi * r;
  const dd p = two_prod(b.hi, q1);
  const double rem = ((a.hi - p.hi) - p.lo) + fma(-b.lo, q1, a.lo);
  return fast_two_sum(q1, rem * r);
}
__device__ __forceinline__ dd dd_div(dd a, dd b) { return dd_div_r(a, b, rcp_1ulp(b.hi)); }

// sqrt(a) for a > 0: a.hi / sqrt(a.hi) and one correction
__device__ __forceinline__ dd dd_sqrt(dd a) {
  const double y = rsqrt_1ulp(a.hi);
  const double s = a.hi * y;
  const dd p = two_prod(s, s);
  const double e = ((a.hi - p.hi) - p.lo) + a.lo;
  return fast_two_sum(s, e * (0.5 * y));
}

}  // namespace hg
