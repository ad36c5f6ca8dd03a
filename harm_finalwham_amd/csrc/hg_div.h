// Correctly rounded FP64 division with the reciprocal part of the
// hardware's sequence shared by several numerators of one divisor.
#pragma once
#include <hip/hip_runtime.h>

#include <cfloat>

namespace hg {

// Division through the steps of the hardware's correctly rounded FP64
// division with the reciprocal part done once per divisor.  hipcc lowers
// x / d to v_div_scale of d and of x, v_rcp_f64, two Newton steps on the
// reciprocal, the quotient, its residual, v_div_fmas and v_div_fixup.  For
// a divisor of magnitude in [2^-300, 2^300] (div_den_ok) and a numerator
// that is zero or of magnitude in [2^-660, 2^300] (div_num_ok), v_div_scale
// changes neither operand nor sets the flag that makes v_div_fmas rescale,
// and v_div_fixup returns the corrected quotient: rcp_refined and div_core
// are then the whole sequence and give x / d bit for bit, except that a zero
// numerator gives +0 for both signs.  div_group and div_weights look at the
// ranges and divide in full outside them; the callers of the others have
// operands that cannot leave theirs, or look themselves (newton_dx).
// hg_check_division compares each of them with the full way on the device.
__device__ __forceinline__ double rcp_refined(double d) {
  double y = __builtin_amdgcn_rcp(d);
  double e = fma(-d, y, 1.0);
  y = fma(y, e, y);
  e = fma(-d, y, 1.0);
  return fma(y, e, y);
}
__device__ __forceinline__ double div_core(double x, double d, double y) {
  const double q = x * y;
  const double r = fma(-d, q, x);
  return fma(r, y, q);
}
// sqrt(x) for x in [2^-60, 2^60]: the steps hipcc lowers it to, without the
// scaling of tiny arguments and the choice of 0 and infinity around them
__device__ __forceinline__ double sqrt_core(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  double d = fma(-g, g, x);
  g = fma(d, h, g);
  d = fma(-g, g, x);
  return fma(d, h, g);
}

// 1 / d for |d| in [2^-300, 2^300] (div_core with a numerator of 1)
__device__ __forceinline__ double rcp_core(double d) {
  const double y = rcp_refined(d);
  return fma(fma(-d, y, 1.0), y, y);
}

// x[k] / d for K numerators whose ranges the caller knows
template <int K>
__device__ __forceinline__ void div_bounded(double *x, double d) {
  const double y = rcp_refined(d);
#pragma unroll
  for (int k = 0; k < K; k++) x[k] = div_core(x[k], d, y);
}

// WENO5BND's indicators si >= e >= 0 over d = their sum ss + DBL_MIN: in the
// steps' range when e >= 2^-600 and d <= 2^600 (si / d is then at least
// 1e-29: e is 1e-26 of a sum of squares that bounds ss), or when ss = 0 (a line
// of zeros: every quotient is +0); full divisions otherwise
template <int K>
__device__ __forceinline__ void div_weights(double *si, double ss, double e) {
  const double d = ss + DBL_MIN;
  double q[K];
#pragma unroll
  for (int k = 0; k < K; k++) q[k] = si[k];
  div_bounded<K>(q, d);
  if (__builtin_expect((e >= 0x1p-600 && d <= 0x1p600) || ss == 0.0, 1)) {
#pragma unroll
    for (int k = 0; k < K; k++) si[k] = q[k];
  } else {
#pragma unroll
    for (int k = 0; k < K; k++) si[k] /= d;
  }
}

__device__ __forceinline__ bool div_num_ok(double x) {
  const double a = fabs(x);
  return a == 0.0 || (a >= 0x1p-660 && a <= 0x1p300);
}

__device__ __forceinline__ bool div_den_ok(double d) { return d >= 0x1p-300 && d <= 0x1p300; }

// x[k] / d for K numerators of one divisor, whose reciprocal y = rcp_refined(d)
// the caller formed; a divisor that is not positive takes full divisions.  The
// residual is taken as d q - x: where it is zero its negative is -0, which
// leaves a zero quotient's sign alone, so unlike div_core this keeps x / d for
// x = -0 too.
template <int K>
__device__ __forceinline__ void div_group(double *x, double d, double y) {
  double q[K];
  bool ok = div_den_ok(d);
#pragma unroll
  for (int k = 0; k < K; k++) {
    const double q0 = x[k] * y;
    q[k] = fma(-fma(d, q0, -x[k]), y, q0);
    ok = ok && div_num_ok(x[k]);
  }
  if (ok) {
#pragma unroll
    for (int k = 0; k < K; k++) x[k] = q[k];
  } else {
#pragma unroll
    for (int k = 0; k < K; k++) x[k] /= d;
  }
}

}  // namespace hg
