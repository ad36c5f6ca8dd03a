// Device self-check of the arithmetic that leaves out parts of the hardware's
// division and square root (hg_div.h), and of the Newton loop's decisions that
// take a product in place of a quotient (hg_c2p.h), against the full way on
// generated operands: exponents over the whole range (zeros, denormals and the
// values outside the checked ranges included) or, for functions whose callers
// keep a range, over that range; random and structured mantissas, both signs, and
// the ranges' edges.
#include <hip/hip_runtime.h>

#include "harmgpu.h"
#include "hg_c2p.h"
#include "hg_div.h"
#include "hg_host.h"

using namespace hg;

namespace {

__device__ __forceinline__ uint64_t mixh(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// random, just below or just above a power of two, or a pattern
__device__ __forceinline__ uint64_t mantissa(uint64_t h) {
  const uint64_t h2 = mixh(h);
  switch ((h >> 56) & 3) {
    case 0: return h2 & 0xFFFFFFFFFFFFFull;
    case 1: return 0xFFFFFFFFFFFFFull - (h2 & 0xFF);
    case 2: return h2 & 0xFF;
    default: return h2 & 0x5555555555555ull;
  }
}

// a positive operand in [2^lo, 2^hi], every 64th one of the two ends
__device__ __forceinline__ double between(uint64_t h, int lo, int hi) {
  if ((h & 63) == 0) return ldexp(1.0, (h & 64) ? lo : hi);
  const uint64_t e = 1023 + lo + (int64_t)((h >> 40) % (uint64_t)(hi - lo));
  return __longlong_as_double((long long)((e << 52) | mantissa(h)));
}

// an operand from hash h: the biased exponent anywhere, inside the divisor's
// range, around the numerator's range or at the edges of both
__device__ __forceinline__ double operand(uint64_t h) {
  int e;
  switch ((h >> 60) & 3) {
    case 0: e = (int)((h >> 40) % 2047); break;
    case 1: e = 1023 - 300 + (int)((h >> 40) % 601); break;
    case 2: e = 1023 - 680 + (int)((h >> 40) % 1000); break;
    default: {
      const int edges[8] = {1023 - 300, 1023 + 300, 1023 - 660, 1023 + 299,
                            1023 - 301, 1023 - 661, 1023 + 301, 1};
      e = edges[(h >> 40) % 8] + (int)((h >> 36) & 1);
    }
  }
  uint64_t bits = ((uint64_t)e << 52) | mantissa(h);
  if ((h & 0x3FF) == 7) bits = 0;  // zeros of either sign
  if ((h >> 12) & 1) bits |= 0x8000000000000000ull;
  return __longlong_as_double((long long)bits);
}

__device__ __forceinline__ bool same(double a, double b) {
  return __double_as_longlong(a) == __double_as_longlong(b) || (a != a && b != b);
}

// mismatches of the functions whose callers keep the ranges: quotients
__device__ __forceinline__ unsigned check_bounded(uint64_t h) {
  unsigned bad = 0;
  // div_core: the divisor's range, numerators of either sign (a zero one +0)
  const double d = between(mixh(h + 21), -300, 300);
  const uint64_t hx = mixh(h + 22);
  double x = between(hx, -660, 300);
  if ((hx >> 7) & 1) x = -x;
  if (((hx >> 8) & 63) == 0) x = 0.0;
  bad += !same(div_core(x, d, rcp_refined(d)), x / d);
  // WENO5BND: indicators from squares of numbers anywhere (and of zeros) ...
  double u2[3], si[3], r[3];
  const uint64_t hu = mixh(h + 23);
  const int scale = (int)((hu >> 32) % 900) - 450;
  for (int k = 0; k < 3; k++) {
    const uint64_t hk = mixh(hu + k);
    const double u = (hu & 127) == 0 || (hk & 15) == 0 ? 0.0 : ldexp(between(hk, -30, 1), scale);
    u2[k] = u * u;
  }
  const double e = ((u2[0] + u2[2]) + u2[1]) * 1e-26;
  for (int k = 0; k < 3; k++) si[k] = ((hu >> (8 + k)) & 1 ? u2[k] : 0.0) + e;
  const double ss = (si[0] + si[2]) + si[1];
  for (int k = 0; k < 3; k++) r[k] = si[k] / (ss + DBL_MIN);
  div_weights<3>(si, ss, e);
  for (int k = 0; k < 3; k++) bad += !same(si[k], r[k]);
  // ... the weights from those, over their sum and over one of themselves
  double w[3], v[3], t[2];
  for (int k = 0; k < 3; k++) {
    t[0] = r[k] + 1e-26;
    t[0] *= t[0];
    w[k] = rcp_core(t[0]);
    bad += !same(w[k], 1.0 / t[0]);
    v[k] = w[k];
  }
  const double sw = (w[0] + w[2]) + w[1];
  div_bounded<3>(v, sw);
  for (int k = 0; k < 3; k++) bad += !same(v[k], w[k] / sw);
  t[0] = v[0] + 1e-26;
  t[1] = v[2] + 1e-26;
  const double q = t[0] / t[1];
  div_bounded<1>(t, t[1]);
  return bad + !same(t[0], q);
}

// reciprocals and square roots
__device__ __forceinline__ unsigned check_roots(uint64_t h) {
  const uint64_t hd = mixh(h + 31);
  double d = between(hd, -300, 300);
  if ((hd >> 7) & 1) d = -d;
  const double x = between(mixh(h + 32), -60, 60);
  return !same(rcp_core(d), 1.0 / d) + !same(sqrt_core(x), sqrt(x));
}

// the Newton loop's stopping test and its cap on W, at their lines and with
// iterates and steps that are zero, infinite or not a number
__device__ __forceinline__ unsigned check_decisions(uint64_t h) {
  const uint64_t hx = mixh(h + 41), hd = mixh(h + 42);
  const double special[4] = {0.0, HUGE_VAL, -HUGE_VAL, HUGE_VAL - HUGE_VAL};
  double x0 = operand(hx), dx0 = operand(hd);
  if ((hd & 3) == 1) dx0 = NEWT_TOL * x0 * (1.0 + ldexp((double)(int64_t)((hd >> 20) % 65) - 32.0, -45 + (int)(hd >> 60)));
  if ((hx & 31) == 3) x0 = special[(hx >> 5) & 3];
  if ((hd & 31) == 7) dx0 = special[(hd >> 5) & 3];
  unsigned bad = 0;
  const double errx = (x0 == 0.) ? fabs(dx0) : fabs(dx0 / x0);
  for (int last = 0; last < 2; last++) {
    bool far;
    bad += newton_converged(x0, dx0, last != 0, far) != (errx <= NEWT_TOL);
    if (last) bad += far != (errx > MIN_NEWT_TOL);
  }
  C2PInv c;
  c.D = 1.0;
  c.Bsq = 0.0;
  c.w = operand(mixh(h + 43));
  newton_ranges(c);
  const double big = GAMMAFAIL * GAMMAFAIL;
  double W = fabs(x0);
  if ((hx & 3) == 2) W = fabs(c.w) * big * (1.0 + ldexp((double)(int64_t)((hx >> 20) % 65) - 32.0, -45 + (int)(hx >> 60)));
  return bad + (w_too_big(c, W) != (W / c.w > big));
}

// out: [0] mismatches of div_group<3> (one divisor, either sign; a negative one
// takes full divisions) and of check_bounded, [1] of 1 / d through div_group<1>
// and of check_roots, [2] of div_group<4> by 12 and of check_decisions, [3]
// operand sets the first took its shortcut for
__global__ void k_check_div(int64_t n, uint64_t seed, unsigned long long *out) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  unsigned long long bad = 0, badr = 0, badc = 0, fast = 0;
  if (t < n) {
    const uint64_t h = mixh(seed ^ mixh((uint64_t)t));
    const double d = (h & 0xC00) ? fabs(operand(h)) : operand(h);
    double x[3], ref[3];
    bool ok = div_den_ok(d);
    for (int k = 0; k < 3; k++) {
      x[k] = operand(mixh(h + 1 + k));
      ref[k] = x[k] / d;
      ok = ok && div_num_ok(x[k]);
    }
    fast = ok ? 1ull : 0ull;
    div_group<3>(x, d, rcp_refined(d));
    for (int k = 0; k < 3; k++) bad += !same(x[k], ref[k]);
    double r[1] = {1.0};
    div_group<1>(r, d, rcp_refined(d));
    badr += !same(r[0], 1.0 / d);
    double nn[4], q[4];
    for (int k = 0; k < 4; k++) nn[k] = q[k] = operand(mixh(h + 11 + k));
    div_group<4>(q, 12., rcp_refined(12.));
    for (int k = 0; k < 4; k++) badc += !same(q[k], nn[k] / 12.);
    bad += check_bounded(h);
    badr += check_roots(h);
    badc += check_decisions(h);
  }
  if (bad) atomicAdd(&out[0], bad);
  if (badr) atomicAdd(&out[1], badr);
  if (badc) atomicAdd(&out[2], badc);
  if (fast) atomicAdd(&out[3], fast);
}

}  // namespace

extern "C" int hg_check_division(int64_t n, uint64_t seed, int64_t result[4]) {
  if (n < 0 || n > ((int64_t)1 << 32) || !result) {
    set_error("hg_check_division: bad arguments");
    return 1;
  }
  unsigned long long *out = nullptr;
  hipError_t e = hipMalloc((void **)&out, 4 * sizeof(unsigned long long));
  if (e == hipSuccess) e = hipMemset(out, 0, 4 * sizeof(unsigned long long));
  if (e == hipSuccess && n > 0)
    hipLaunchKernelGGL(k_check_div, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, n, seed, out);
  if (e == hipSuccess) e = hipGetLastError();
  unsigned long long h[4] = {0, 0, 0, 0};
  if (e == hipSuccess) e = hipMemcpy(h, out, sizeof h, hipMemcpyDeviceToHost);
  if (out) (void)hipFree(out);
  if (e != hipSuccess) {
    set_error("hg_check_division: %s", hipGetErrorString(e));
    return 1;
  }
  for (int k = 0; k < 4; k++) result[k] = (int64_t)h[k];
  return 0;
}
