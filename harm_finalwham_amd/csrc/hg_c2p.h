// Device Noble et al. (2006) "2D" conserved-to-primitive inversion.
//
// utoprimgen.c:23 Utoprimgen -> utoprim_2d_final.c:34 Utoprim_2d_final ->
// utoprim_2d_final.c:152 Utoprim_new_body -> :573 find_root_2D_gen ->
// :736 general_newton_raphson (no line search) with :1189 func_vsq2 and the
// ideal-gas EOS of utoprim_jon_eos.c / eos.c.  FP64 throughout: same
// operations in the same order as the reference, hence the same iterates,
// iteration counts and failure codes.
#pragma once
#include "hg_dd.h"
#include "hg_phys.h"

namespace hg {

constexpr int MAX_NEWT_ITER = 200;                 // u2p_defs.h:38
constexpr double NEWT_TOL = 1E3 * DBL_EPS;         // u2p_defs.h:39
constexpr double MIN_NEWT_TOL = 1E-6;              // u2p_defs.h:47
constexpr double MAXNEGUTSQ = 1E-10;               // u2p_defs.h:123
constexpr double GAMMAFAIL = 100.0 * 25.0;         // initbase.c:471-476
constexpr double FAIL_VAL = 1.e30;

// Invariants of one inversion (the file statics of utoprim_2d_final.c:13-15)
struct C2PInv {
  double Bsq, QdotB, QdotBsq, Qtsq, Qdotn, D, w;
  double Qcon[4], ncon[4], Bcon[4];
  // set by newton_ranges: what the Newton steps need of D, Bsq and w to leave
  // out the scaling of their divisions
  bool nice;    // D in [2^-150, 2^150], Bsq zero or in [2^-150, 2^150]
  double wlim;  // x0 < wlim makes x0 / w <= gsq_big certain
};

// utoprim_2d_final.c:457 vsq_calc
__device__ __forceinline__ double vsq_of_W(const C2PInv &c, double W) {
  double Wsq = W * W;
  double Xsq = (c.Bsq + W) * (c.Bsq + W);
  return ((Wsq * c.Qtsq + c.QdotBsq * (c.Bsq + 2. * W)) / (Wsq * Xsq));
}

__device__ __forceinline__ void newton_ranges(C2PInv &c) {
  constexpr double gsq_big = GAMMAFAIL * GAMMAFAIL;
  c.nice = c.D >= 0x1p-150 && c.D <= 0x1p150 && (c.Bsq == 0. || (c.Bsq >= 0x1p-150 && c.Bsq <= 0x1p150));
  c.wlim = (c.w >= 0x1p-200 && c.w <= 0x1p200) ? c.w * (gsq_big * (1. - 0x1p-40)) : -1.;
}

// x0 / w > gsq_big of the reference's loop for x0 >= 0: decided by a product
// wherever the quotient is further than its rounding from gsq_big
__device__ __forceinline__ bool w_too_big(const C2PInv &c, double x0) {
  if (x0 < c.wlim) return false;
  return x0 / c.w > GAMMAFAIL * GAMMAFAIL;
}

// One Newton step of utoprim_2d_final.c:1189 func_vsq2 (with the EOS of
// utoprim_jon_eos.c:107,230,346); returns dx[0..1] and f, df.
__device__ __forceinline__ void newton_dx_full(const C2PInv &c, double igr, double W, double vsq,
                                               double &dx0, double &dx1, double &f, double &df) {
  double Wsq = W * W, D = c.D, Bsq = c.Bsq, QdotBsq = c.QdotBsq;
  double Wp = W - D;
  double gamma = 1.0 / sqrt(1.0 - vsq);
  double gammasq = gamma * gamma;
  double wmrho0 = Wp / gammasq - D * vsq / (1.0 + gamma);
  double p_tmp = igr * wmrho0;
  double dPdW = 0.0 * 0.0 + (1.0 - vsq) * igr;
  double Wp2 = W - D;
  double gamma2 = 1.0 / sqrt(1.0 - vsq);
  double dwmrho0dvsq = (D * (gamma2 * 0.5 - 1.0) - Wp2);
  double drho0dvsq = -D * gamma2 * 0.5;
  double dPdvsq = drho0dvsq * 0.0 + dwmrho0dvsq * igr;
  double t2 = -0.5 * Bsq + dPdvsq;
  double t3 = Bsq + W;
  double t4 = t3 * t3;
  double t9 = 1 / Wsq;
  double t11 = c.Qtsq - vsq * t4 + QdotBsq * (Bsq + 2.0 * W) * t9;
  double t16 = QdotBsq * t9;
  double t18 = -c.Qdotn - 0.5 * Bsq * (1.0 + vsq) + 0.5 * t16 - W + p_tmp;
  double t21 = 1 / t3;
  double t23 = 1 / W;
  double t24 = t16 * t23;
  double t25 = -1.0 + dPdW - t24;
  double t35 = t25 * t3 + (Bsq - 2.0 * dPdvsq) * (QdotBsq + vsq * Wsq * W) * t9 * t23;
  double t36 = 1 / t35;
  dx0 = -(t2 * t11 + t4 * t18) * t21 * t36;
  double t40 = (vsq + t24) * t3;
  dx1 = -(-t25 * t11 - 2.0 * t40 * t18) * t21 * t36;
  df = -t11 * t11 - t18 * t18;
  f = -0.5 * df;
}

// newton_dx_full bit for bit.  The iteration is a serial chain of seven
// divisions and a square root, and the instruction count sets its time both
// where lanes fill the SIMDs and where one wavefront walks the last zones;
// the scaling around the hardware's division and square root is about a
// third of it and changes nothing for operands of ordinary size.  The
// bounds: 1 - vsq in [2^-60, 2^60] and W in [2^-150, 2^150] with D and Bsq as
// newton_ranges has them keep W^2, Bsq + W, gamma, gamma^2 and 1 + gamma in
// div_core's ranges; W - D is zero or at least 2^-202; |D vsq| is zero or at
// least 2^-450.  dPdrho0 = 0 drops out: its products are zeros, added to
// terms that are not (-0).  A zone outside takes the full step.  2^24 zones
// in HG_C2P_FP64 take 1.80 ms instead of 2.12 ms.
__device__ __forceinline__ void newton_dx(const C2PInv &c, double igr, double W, double vsq,
                                          double &dx0, double &dx1, double &f, double &df) {
  const double D = c.D, Bsq = c.Bsq, QdotBsq = c.QdotBsq;
  const double omv = 1.0 - vsq;
  const double Wsq = W * W;
  const double Wp = W - D;
  const double gamma = rcp_core(sqrt_core(omv));
  const double gammasq = gamma * gamma;
  const double opg = 1.0 + gamma;
  const double wmrho0 = div_core(Wp, gammasq, rcp_refined(gammasq)) - div_core(D * vsq, opg, rcp_refined(opg));
  const double p_tmp = igr * wmrho0;
  const double dPdW = omv * igr;
  const double dPdvsq = (D * (gamma * 0.5 - 1.0) - Wp) * igr;
  const double t2 = -0.5 * Bsq + dPdvsq;
  const double t3 = Bsq + W;
  const double t4 = t3 * t3;
  const double t9 = rcp_core(Wsq);
  double t11 = c.Qtsq - vsq * t4 + QdotBsq * (Bsq + 2.0 * W) * t9;
  const double t16 = QdotBsq * t9;
  double t18 = -c.Qdotn - 0.5 * Bsq * (1.0 + vsq) + 0.5 * t16 - W + p_tmp;
  const double t21 = rcp_core(t3);
  const double t23 = rcp_core(W);
  const double t24 = t16 * t23;
  const double t25 = -1.0 + dPdW - t24;
  const double t35 = t25 * t3 + (Bsq - 2.0 * dPdvsq) * (QdotBsq + vsq * Wsq * W) * t9 * t23;
  const double t36 = rcp_core(t35);
  const double t40 = (vsq + t24) * t3;
  double e0 = -(t2 * t11 + t4 * t18) * t21 * t36;
  double e1 = -(-t25 * t11 - 2.0 * t40 * t18) * t21 * t36;
  const bool ok = c.nice && omv >= 0x1p-60 && omv <= 0x1p60 && W >= 0x1p-150 && W <= 0x1p150 &&
                  (vsq == 0. || fabs(vsq) >= 0x1p-300) && fabs(t35) >= 0x1p-300 && fabs(t35) <= 0x1p300;
  if (ok) {
    dx0 = e0;
    dx1 = e1;
    df = -t11 * t11 - t18 * t18;
    f = -0.5 * df;
  } else {
    newton_dx_full(c, igr, W, vsq, dx0, dx1, f, df);
  }
}

// Setup of Utoprim_new_body up to the Newton guess (utoprim_2d_final.c:152-300).
// U is alpha * U_geomfree; prim holds the guess.  Returns a failure code (4)
// when the guess is unusable, else 0, and sets W_last and the invariants.
template <class GT>
__device__ __forceinline__ int c2p_setup(const double *U, const GT &G, const double *prim,
                                         double gam, C2PInv &c, double &W_last) {
  double Bcov[4], Qcov[4];
  c.Bcon[0] = 0.;
  c.Bcon[1] = U[B1];
  c.Bcon[2] = U[B2];
  c.Bcon[3] = U[B3];
#pragma unroll
  for (int i = 1; i < 4; i++) {
    Bcov[i] = 0.;
#pragma unroll
    for (int j = 1; j < 4; j++)
      if (!GT::cov0(i, j)) Bcov[i] += G.gcov[i][j] * c.Bcon[j];
  }
#pragma unroll
  for (int i = 0; i < 4; i++) Qcov[i] = U[UU + i];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    c.Qcon[i] = 0.;
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (!GT::con0(i, j)) c.Qcon[i] += G.gcon[i][j] * Qcov[j];
  }
  c.Bsq = 0.;
#pragma unroll
  for (int i = 1; i < 4; i++) c.Bsq += c.Bcon[i] * Bcov[i];
  c.QdotB = 0.;
#pragma unroll
  for (int i = 1; i < 4; i++) c.QdotB += Qcov[i] * c.Bcon[i];  // B^t = 0
  c.QdotBsq = c.QdotB * c.QdotB;
  const double ncov0 = -sqrt(-1. / G.gcon[0][0]);  // the only nonzero n_mu
#pragma unroll
  for (int i = 0; i < 4; i++) c.ncon[i] = GT::con0(i, 0) ? 0. : 0. + G.gcon[i][0] * ncov0;
  c.Qdotn = c.Qcon[0] * ncov0;
  double Qsq = 0.;
#pragma unroll
  for (int i = 0; i < 4; i++) Qsq += Qcov[i] * c.Qcon[i];
  c.Qtsq = Qsq + c.Qdotn * c.Qdotn;
  c.D = U[RHO];

  double utsq = 0.;
#pragma unroll
  for (int i = 1; i < 4; i++)
#pragma unroll
    for (int j = 1; j < 4; j++)
      if (!GT::cov0(i, j)) utsq += G.gcov[i][j] * prim[U1 + i - 1] * prim[U1 + j - 1];
  if ((utsq < 0.) && (fabs(utsq) < MAXNEGUTSQ)) utsq = 0.0;
  const double utsq_too_big = (GAMMAFAIL - 1.0) * (GAMMAFAIL - 1.0);
  if (utsq < 0. || utsq > utsq_too_big) return FAIL_CONVGUESSUTSQ;
  double gammasq = 1. + utsq;
  double gamma = sqrt(gammasq);
  double rho0 = c.D / gamma;
  double u = prim[UU];
  double p = (gam - 1.) * u;
  double w = rho0 + u + p;
  W_last = w * gammasq;
  int i_increase = 0;
  while (((W_last * W_last * W_last * (W_last + 2. * c.Bsq) - c.QdotBsq * (2. * W_last + c.Bsq)) <=
          W_last * W_last * (c.Qtsq - c.Bsq * c.Bsq)) &&
         (i_increase < 10)) {
    W_last *= 10.;
    i_increase++;
  }
  c.w = w;
  newton_ranges(c);
  return 0;
}

// Post-solve of Utoprim_new_body (utoprim_2d_final.c:335-441): from the
// converged W to primitives.  Writes prim[0..4] when the inversion returns 0.
__device__ __forceinline__ int c2p_finish(const C2PInv &c, double W, int retval, double igr,
                                          double *prim_out, bool &assign) {
  const double gsq_big = GAMMAFAIL * GAMMAFAIL;
  const double vsq_big = (gsq_big - 1.0) / (gsq_big);
  const double maxnegvsq = (1.0 - 1.0 / (MAXNEGUTSQ + 1.0));
  assign = false;
  if ((retval != 0) || (W == FAIL_VAL)) return retval * 100 + 1;
  assign = true;  // remaining failures return 0 from Utoprim_new_body: guess kept
  if (!(W >= 0x1p-150 && W < c.wlim)) {  // else 0 < W / w <= gsq_big
    double Wtest = W / c.w;
    if (Wtest <= 0. || Wtest > gsq_big) { assign = false; return FAIL_CONVW; }
  }
  double vsq = vsq_of_W(c, W);
  if ((vsq < 0.) && (fabs(vsq) < maxnegvsq)) vsq = 0.0;
  if ((vsq > vsq_big) || (vsq < 0.0)) { assign = false; return FAIL_CONVUTSQ; }
  double gtmp = sqrt(1. - vsq);
  double gamma = 1. / gtmp;
  double rho0 = c.D * gtmp;
  double w = W * (1. - vsq);
  double p = igr * (w - rho0);
  double u = w - (rho0 + p);
  int flag = 0;
  if ((rho0 <= 0.) || (u < 0.)) {
    if ((rho0 <= 0.) && (u >= 0.)) flag = FAIL_RHONEG;
    if ((rho0 > 0.) && (u < 0.)) flag = FAIL_UNEG;
    if ((rho0 <= 0.) && (u < 0.)) flag = FAIL_RHOUNEG;
  }
  prim_out[RHO] = rho0;
  prim_out[UU] = u;
  double bw[3];
#pragma unroll
  for (int i = 0; i < 3; i++) bw[i] = c.QdotB * c.Bcon[i + 1];
  div_by<3>(bw, W, div_rcp(W));
  const double gx = gamma / (W + c.Bsq);
#pragma unroll
  for (int i = 1; i < 4; i++) {
    double Qtcon = c.Qcon[i] + c.ncon[i] * c.Qdotn;
    prim_out[U1 + i - 1] = gx * (Qtcon + bw[i - 1]);
  }
  return flag;
}

// Utoprimgen's scaling of the evolved conserved variables (utoprimgen.c:23):
// Ug = U / gdet with the rest mass taken out of the energy, Ut = alpha Ug;
// returns alpha
template <class GT>
__device__ __forceinline__ double c2p_scale(const double *U, const GT &G, double *Ug, double *Ut) {
#pragma unroll
  for (int i = 0; i < NPR; i++) Ug[i] = U[i];
  div_by<NPR>(Ug, G.g, div_rcp(G.g));
  Ug[UU] -= Ug[RHO];
  const double alpha = 1.0 / sqrt(-G.gcon[0][0]);
#pragma unroll
  for (int i = 0; i < NPR; i++) Ut[i] = alpha * Ug[i];
  return alpha;
}

// The reference's stopping test errx = |dx0 / x0| <= NEWT_TOL of the iterate x0
// that the step dx0 led to: by a product, but for tiny iterates and quotients
// within 2^-40 of the tolerance.  An infinite step makes both sides infinite and
// errx a NaN, which is no convergence (the reference puts W back and goes on):
// the comparison is strict.  far, whether errx is above MIN_NEWT_TOL, is asked
// of the last step allowed alone.
__device__ __forceinline__ bool newton_converged(double x0, double dx0, bool last, bool &far) {
  const double a0 = fabs(x0), ad = fabs(dx0), lim = NEWT_TOL * a0;
  bool conv = ad < lim * (1. - 0x1p-40);
  far = false;
  if (!(a0 >= 0x1p-900) || !(conv || ad >= lim * (1. + 0x1p-40)) || last) {
    const double errx = (x0 == 0.) ? ad : fabs(dx0 / x0);
    conv = errx <= NEWT_TOL;
    far = errx > MIN_NEWT_TOL;
  }
  return conv;
}

// Full FP64 inversion of one zone (utoprimgen.c:23 with UTOPRIM2DFINAL).
// U: evolved conserved variables (with gdet); pr: guess in, solution out.
// The core also returns the invariants and the final Newton iterate (x0 = W,
// x1 = vsq); newton is false when the set-up failed before the iteration.
template <class GT>
__device__ __forceinline__ int utoprimgen_fp64_core(const double *U, const GT &G, double gam, double *pr,
                                                    int &iters, C2PInv &c, double &x0, double &x1,
                                                    bool &newton) {
  double Ug[NPR], Ut[NPR];
  c2p_scale(U, G, Ug, Ut);
#pragma unroll
  for (int i = B1; i <= B3; i++) pr[i] = Ug[i];
  const double igr = (gam - 1.0) / gam;
  const double gsq_big = GAMMAFAIL * GAMMAFAIL;
  const double vsq_big = (gsq_big - 1.0) / (gsq_big);
  double W_last;
  iters = 0;
  newton = false;
  int code = c2p_setup(Ut, G, pr, gam, c, W_last);
  if (code) return code;
  newton = true;
  // find_root_2D_gen + general_newton_raphson without line search
  x0 = fabs(W_last);
  double v0 = vsq_of_W(c, W_last);
  x1 = (v0 > 1.) ? vsq_big : v0;
  double f = 1., df = 1.;
  bool keep = true, far = false;
  while (keep) {
    iters++;
    double dx0, dx1;
    newton_dx(c, igr, x0, x1, dx0, dx1, f, df);
    double xo0 = x0;
    x0 += dx0;
    x1 += dx1;
    const double a0 = fabs(x0);
    const bool conv = newton_converged(x0, dx0, iters >= MAX_NEWT_ITER, far);
    x0 = w_too_big(c, a0) ? xo0 : a0;
    x1 = (x1 > 1.) ? vsq_big : x1;
    if (conv || (iters >= MAX_NEWT_ITER)) keep = false;
  }
  int retval = 0;
  if (!isfinite(f) || !isfinite(df) || !isfinite(x0) || !isfinite(x1)) retval = 1;
  else if (far) retval = 1;
  double out[NPR];
  bool assign;
  code = c2p_finish(c, x0, retval, igr, out, assign);
  if (assign) {
#pragma unroll
    for (int i = 0; i < B1; i++) pr[i] = out[i];
  }
  return code;
}

template <class GT>
__device__ __forceinline__ int utoprimgen_fp64(const double *U, const GT &G, double gam, double *pr,
                                               int &iters) {
  C2PInv c;
  double x0 = 0., x1 = 0.;
  bool newton;
  return utoprimgen_fp64_core(U, G, gam, pr, iters, c, x0, x1, newton);
}

}  // namespace hg

namespace hg {

// ---------------------------------------------------------------------------
// The converged root and the mixed-precision path.
//
// The reference iteration stops at |dW/W| <= NEWT_TOL with W where the FP64
// residual is still within rounding noise of zero; at Lorentz factors near 50
// and magnetisations near 1e3 that noise moves the primitives by up to ~1e-9
// (vsq is recomputed from W and 1 / (1 - vsq) amplifies it), and two FP64
// iterations from different starts land at different points of the noise.
// The converged root of the same FP64 system (the invariants exactly as the
// reference sets them up) is found by Newton steps whose residuals are
// evaluated in double-double arithmetic (hg_dd.h) with the FP64 Jacobian of
// newton_dx, and the primitives are formed from it in double-double:
//   c2p_polish     FP64 steps to |dW/W| <= 1e-9, then double-double steps
//                  until one moves W by at most 1e-12 of itself (false when
//                  either is not reached).  Newton converges quadratically
//                  there: a step of 1e-12 W leaves an error near 1e-24 W, so
//                  that step's W is the root to the last bit and needs no
//                  further step to confirm it
//   c2p_finish_dd  c2p_finish with vsq, 1 - vsq, rho0, w, p, u and the
//                  velocities in double-double, rounded once
// The mixed-precision path runs the Newton iteration in FP32 from the
// reference's FP64 set-up and start, to |dW/W| <= MIXED_TOL_F32, then polishes
// and finishes as above; a zone whose FP32 phase or polish does not converge
// is inverted again by the reference path (and polished), by the caller.
// ---------------------------------------------------------------------------
constexpr int MIXED_MAX_F32 = 40;         // FP32 Newton steps before falling back
constexpr float MIXED_TOL_F32 = 2e-6f;    // |dW/W| that ends the FP32 phase
constexpr float MIXED_STALL_F32 = 1e-3f;  // below it, a step that shrank less than 4x ends it too
constexpr int POLISH_MAX_F64 = 8;         // FP64 steps of the polish (to |dW/W| <= 1e-9); from the
                                          // FP32 floor at Lorentz factors near 50 (|dW/W| ~ 1e-3) it
                                          // can take six
constexpr int POLISH_MAX_DD = 3;          // double-double steps (until one is <= 1e-12 W)

struct C2PInvF {
  float Bsq, QdotBsq, Qtsq, Qdotn, D;
};

// newton_dx in FP32 (same algebra) with the hardware reciprocal and
// reciprocal square root (about 1 ulp): the FP32 phase only has to bring W
// within MIXED_TOL_F32 of the root, the polish does the rest
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ void newton_dx_f32(const C2PInvF &c, float igr, float W, float vsq, float &dx0,
                                              float &dx1) {
  float Wsq = W * W, D = c.D, Bsq = c.Bsq, QdotBsq = c.QdotBsq;
  float Wp = W - D;
  float gamma = __builtin_amdgcn_rsqf(1.0f - vsq);
  float gammasq = gamma * gamma;
  float wmrho0 = Wp * frcp(gammasq) - D * vsq * frcp(1.0f + gamma);
  float p_tmp = igr * wmrho0;
  float dPdW = (1.0f - vsq) * igr;
  float dwmrho0dvsq = (D * (gamma * 0.5f - 1.0f) - Wp);
  float dPdvsq = dwmrho0dvsq * igr;
  float t2 = -0.5f * Bsq + dPdvsq;
  float t3 = Bsq + W;
  float t4 = t3 * t3;
  float t9 = frcp(Wsq);
  float t11 = c.Qtsq - vsq * t4 + QdotBsq * (Bsq + 2.0f * W) * t9;
  float t16 = QdotBsq * t9;
  float t18 = -c.Qdotn - 0.5f * Bsq * (1.0f + vsq) + 0.5f * t16 - W + p_tmp;
  float t21 = frcp(t3);
  float t23 = frcp(W);
  float t24 = t16 * t23;
  float t25 = -1.0f + dPdW - t24;
  float t35 = t25 * t3 + (Bsq - 2.0f * dPdvsq) * (QdotBsq + vsq * Wsq * W) * t9 * t23;
  float t36 = frcp(t35);
  dx0 = -(t2 * t11 + t4 * t18) * t21 * t36;
  float t40 = (vsq + t24) * t3;
  dx1 = -(-t25 * t11 - 2.0f * t40 * t18) * t21 * t36;
}

// The start of utoprimgen_fp64's Newton loop from the set-up's W_last
__device__ __forceinline__ void newton_start(const C2PInv &c, double W_last, double &x0, double &x1) {
  const double gsq_big = GAMMAFAIL * GAMMAFAIL;
  const double vsq_big = (gsq_big - 1.0) / (gsq_big);
  x0 = fabs(W_last);
  double v0 = vsq_of_W(c, W_last);
  x1 = (v0 > 1.) ? vsq_big : v0;
}

// FP32 Newton from (x0, x1) with the guards of the reference loop; true when
// |dW/W| <= MIXED_TOL_F32 was reached with finite iterates; iters counts steps
__device__ __forceinline__ bool newton_f32(const C2PInv &c, double igr, double &x0, double &x1, int &iters) {
  const double gsq_big = GAMMAFAIL * GAMMAFAIL;
  const double vsq_big = (gsq_big - 1.0) / (gsq_big);
  C2PInvF cf = {(float)c.Bsq, (float)c.QdotBsq, (float)c.Qtsq, (float)c.Qdotn, (float)c.D};
  const float igrf = (float)igr, wf = (float)c.w;
  const float gsq_bigf = (float)gsq_big, vsq_bigf = (float)vsq_big;
  float w0 = (float)x0, w1 = (float)x1;
  bool conv = false;
  int n32 = 0;
  float errp = 1e30f;
  while (n32 < MIXED_MAX_F32) {
    float d0, d1;
    newton_dx_f32(cf, igrf, w0, w1, d0, d1);
    float wo = w0;
    w0 += d0;
    w1 += d1;
    float err = (w0 == 0.f) ? fabsf(d0) : fabsf(d0 * frcp(w0));
    w0 = fabsf(w0);
    w0 = (w0 > gsq_bigf * wf) ? wo : w0;
    w1 = (w1 > 1.f) ? vsq_bigf : w1;
    n32++;
    if (!isfinite(w0) || !isfinite(w1)) break;
    // converged; or near the root (|dW/W| <= MIXED_STALL_F32) with the
    // steps no longer shrinking quadratically: FP32 rounding of the
    // residual (amplified by 1 / (1 - vsq)) sets the floor, the FP64 polish
    // takes it from here
    if (err <= MIXED_TOL_F32 || (err <= MIXED_STALL_F32 && err > 0.25f * errp)) {
      conv = true;
      break;
    }
    errp = err;
  }
  iters += n32;
  x0 = (double)w0;
  x1 = (double)w1;
  return conv;
}

// One Newton step with the residuals t11, t18 of func_vsq2 in double-double
// and the FP64 Jacobian (newton_dx's terms)
__device__ __forceinline__ void newton_dx_dd(const C2PInv &c, double igr, double W, double vsq, double &dx0,
                                             double &dx1) {
  const double Wsq = W * W, D = c.D, Bsq = c.Bsq, QdotBsq = c.QdotBsq;
  const double gamma = 1.0 / sqrt(1.0 - vsq);
  const double dPdW = (1.0 - vsq) * igr;
  const double dPdvsq = (D * (gamma * 0.5 - 1.0) - (W - D)) * igr;
  const double t2 = -0.5 * Bsq + dPdvsq, t3 = Bsq + W, t4 = t3 * t3, t9 = 1 / Wsq;
  const double t16 = QdotBsq * t9, t21 = 1 / t3, t23 = 1 / W, t24 = t16 * t23, t25 = -1.0 + dPdW - t24;
  const double t35 = t25 * t3 + (Bsq - 2.0 * dPdvsq) * (QdotBsq + vsq * Wsq * W) * t9 * t23;
  const double t36 = 1 / t35;
  // residuals: t11 = Qtsq - vsq (Bsq + W)^2 + QdotBsq (Bsq + 2 W) / W^2,
  // t18 = -Qdotn - Bsq (1 + vsq) / 2 + QdotBsq / (2 W^2) - W + p(W, vsq)
  const dd Wd = dd_of(W), vd = dd_of(vsq);
  const dd T3 = two_sum(Bsq, W);
  const dd q = dd_div(dd_of(QdotBsq), two_prod(W, W));
  const dd r11 = dd_add(dd_sub(dd_of(c.Qtsq), dd_mul(vd, dd_mul(T3, T3))), dd_mul(q, two_sum(Bsq, 2.0 * W)));
  const dd omv = two_sum(1.0, -vsq);
  const dd gd = dd_div(dd_of(1.0), dd_sqrt(omv));
  const dd wm = dd_sub(dd_mul(two_sum(W, -D), omv), dd_div(two_prod(vsq, D), dd_add(dd_of(1.0), gd)));
  const dd r18 = dd_add(dd_add(dd_add(dd_of(-c.Qdotn), dd_mul_d(two_sum(1.0, vsq), -0.5 * Bsq)), dd_mul_d(q, 0.5)),
                        dd_add(dd_neg(Wd), dd_mul_d(wm, igr)));
  const double t11 = dd_val(r11), t18 = dd_val(r18);
  dx0 = -(t2 * t11 + t4 * t18) * t21 * t36;
  const double t40 = (vsq + t24) * t3;
  dx1 = -(-t25 * t11 - 2.0 * t40 * t18) * t21 * t36;
}

// The polish: FP64 steps (at most n64; none when n64 = 0) until |dW/W| <=
// 1e-9, then double-double steps until one moves W by <= 1e-12 W.  True when both
// tolerances were reached with finite iterates.
__device__ __forceinline__ bool c2p_polish(const C2PInv &c, double igr, double &x0, double &x1, int n64,
                                           int &iters) {
  const double gsq_big = GAMMAFAIL * GAMMAFAIL;
  const double vsq_big = (gsq_big - 1.0) / (gsq_big);
  bool ok = (n64 == 0);
  for (int k = 0; k < n64 && !ok; k++) {
    double dx0, dx1, f, df;
    newton_dx(c, igr, x0, x1, dx0, dx1, f, df);
    const double xo0 = x0, xn = x0 + dx0;
    x0 = fabs(xn);
    // W put back, or turned round from below zero: not converged, however little
    // it moved (a step of -2 W does not move it)
    const bool big = w_too_big(c, x0), held = big || xn < 0.;
    x0 = big ? xo0 : x0;
    x1 += dx1;
    x1 = (x1 > 1.) ? vsq_big : x1;
    iters++;
    ok = !held && fabs(x0 - xo0) <= 1e-9 * x0;
  }
  if (!ok) return false;
  ok = false;
  for (int k = 0; k < POLISH_MAX_DD && !ok; k++) {
    double dx0, dx1;
    newton_dx_dd(c, igr, x0, x1, dx0, dx1);
    const double xo0 = x0, xn = x0 + dx0;
    x0 = fabs(xn);
    const bool big = w_too_big(c, x0), held = big || xn < 0.;
    x0 = big ? xo0 : x0;
    x1 += dx1;
    x1 = (x1 > 1.) ? vsq_big : x1;
    iters++;
    ok = !held && fabs(x0 - xo0) <= 1e-12 * x0;
  }
  return ok && isfinite(x0) && isfinite(x1);
}

// c2p_finish from a converged W with the primitives formed in double-double
// (the checks and failure codes of c2p_finish, on the rounded values)
__device__ __forceinline__ int c2p_finish_dd(const C2PInv &c, double W, double igr, double *prim_out,
                                             bool &assign) {
  const double gsq_big = GAMMAFAIL * GAMMAFAIL;
  const double vsq_big = (gsq_big - 1.0) / (gsq_big);
  const double maxnegvsq = (1.0 - 1.0 / (MAXNEGUTSQ + 1.0));
  assign = false;
  if (W == FAIL_VAL) return 101;
  double Wtest = W / c.w;
  assign = true;
  if (Wtest <= 0. || Wtest > gsq_big) { assign = false; return FAIL_CONVW; }
  const dd Wsq = two_prod(W, W), X = two_sum(c.Bsq, W);
  dd vd = dd_div(dd_add(dd_mul_d(Wsq, c.Qtsq), dd_mul_d(two_sum(c.Bsq, 2.0 * W), c.QdotBsq)),
                 dd_mul(Wsq, dd_mul(X, X)));
  double vsq = dd_val(vd);
  if ((vsq < 0.) && (fabs(vsq) < maxnegvsq)) {
    vsq = 0.0;
    vd = dd_of(0.0);
  }
  if ((vsq > vsq_big) || (vsq < 0.0)) { assign = false; return FAIL_CONVUTSQ; }
  const dd omv = dd_sub(dd_of(1.0), vd);
  const dd gt = dd_sqrt(omv);
  const dd rho0 = dd_mul_d(gt, c.D);
  const dd w = dd_mul_d(omv, W);
  const dd p = dd_mul_d(dd_sub(w, rho0), igr);
  const dd u = dd_sub(w, dd_add(rho0, p));
  const double r = dd_val(rho0), uu = dd_val(u);
  int flag = 0;
  if ((r <= 0.) || (uu < 0.)) {
    if ((r <= 0.) && (uu >= 0.)) flag = FAIL_RHONEG;
    if ((r > 0.) && (uu < 0.)) flag = FAIL_UNEG;
    if ((r <= 0.) && (uu < 0.)) flag = FAIL_RHOUNEG;
  }
  prim_out[RHO] = r;
  prim_out[UU] = uu;
  const dd f = dd_div(dd_div(dd_of(1.0), gt), X);  // gamma / (W + Bsq)
  const dd iW = dd_div(dd_of(1.0), dd_of(W));
#pragma unroll
  for (int i = 1; i < 4; i++) {
    dd Qt = dd_add(dd_of(c.Qcon[i]), two_prod(c.ncon[i], c.Qdotn));
    dd v = dd_add(Qt, dd_mul(two_prod(c.QdotB, c.Bcon[i]), iW));
    prim_out[U1 + i - 1] = dd_val(dd_mul(f, v));
  }
  return flag;
}

// The reference inversion of one zone with a converged root: utoprimgen_fp64
// (its failure code, its iteration count and, for a failed zone, its
// values), then, for a zone it solves, the polish from its final iterate and
// the primitives in double-double; these replace the reference's values
// when the polish converges.  *polished tells whether they did.
template <class GT>
__device__ __forceinline__ int utoprimgen_refined(const double *U, const GT &G, double gam, double *pr,
                                                  int &iters, bool &polished) {
  C2PInv c;
  double x0 = 0., x1 = 0.;
  bool newton;
  polished = false;
  int code = utoprimgen_fp64_core(U, G, gam, pr, iters, c, x0, x1, newton);
  if (code != 0 || !newton) return code;
  const double igr = (gam - 1.0) / gam;
  int it = 0;
  if (!c2p_polish(c, igr, x0, x1, POLISH_MAX_F64, it)) return code;
  double out[NPR];
  bool assign;
  if (c2p_finish_dd(c, x0, igr, out, assign) == 0 && assign) {
#pragma unroll
    for (int i = 0; i < B1; i++) pr[i] = out[i];
    iters += it;
    polished = true;
  }
  return code;
}

// |dW / W| that the rounding of newton_dx's residuals can make at the root:
// half an ulp of each of their terms through the Jacobian
__device__ __forceinline__ double newton_noise(const C2PInv &c, double igr, double W, double vsq) {
  const double D = c.D, Bsq = c.Bsq;
  const double gamma = rsqrt_1ulp(1.0 - vsq);
  const double dPdvsq = (D * (gamma * 0.5 - 1.0) - (W - D)) * igr;
  const double t2 = -0.5 * Bsq + dPdvsq, t3 = Bsq + W, t4 = t3 * t3, t23 = rcp_1ulp(W), t9 = t23 * t23;
  const double t16 = c.QdotBsq * t9, t24 = t16 * t23, t25 = -1.0 + (1.0 - vsq) * igr - t24;
  const double t35 = t25 * t3 + (Bsq - 2.0 * dPdvsq) * (c.QdotBsq + vsq * W * W * W) * t9 * t23;
  const double s11 = fabs(c.Qtsq) + vsq * t4 + t16 * (Bsq + 2.0 * W);
  const double s18 = fabs(c.Qdotn) + 0.5 * Bsq * (1.0 + vsq) + t16 + W + igr * (W + D);
  return 0.5 * DBL_EPS * (fabs(t2) * s11 + t4 * s18) * fabs(rcp_1ulp(t3) * rcp_1ulp(t35)) * t23;
}

constexpr int LISTED_MAX_F64 = 48;       // FP64 steps before the reference's own iteration takes over
constexpr double LISTED_NOISE = 1e-9;    // largest rounding noise of W the short way accepts
constexpr double LISTED_MARGIN = 16.0;   // W moved by this many times its noise keeps the code 0

// A zone the FP32 phase or its polish left: utoprimgen_refined's root and
// primitives without the part of the reference's iteration that walks in the
// rounding noise of its residual.  Where that noise is above NEWT_TOL
// (Lorentz factors near 50, magnetisations near 1e3) the reference goes on to
// 200 steps, 100 us and more for one zone, and the polish then discards where
// it stopped.  The first steps are the reference's own iterates, to |dW/W| <=
// 1e-9; from there the polish.  Taken only where every stopping point of the
// reference inside the noise would give code 0: the FP64 primitives at W and
// at W moved either way by LISTED_MARGIN times the noise all do.  Every other
// zone is inverted by utoprimgen_refined from the guess, and so is every zone of a
// caller that asks for the counts: they are the reference's, walk included.  The
// list of 1e6 zones of the benchmark distribution (154, gamma 5/3) takes 42 us
// instead of 168 us without them; 1.5e6 listed zones gave the same bits and codes
// either way.
template <bool COUNTED, class GT>
__device__ __forceinline__ int utoprimgen_listed(const double *U, const GT &G, double gam, double *pr, int &iters) {
  C2PInv c;
  double Ug[NPR], Ut[NPR], W_last;
  c2p_scale(U, G, Ug, Ut);
  if (!COUNTED && c2p_setup(Ut, G, pr, gam, c, W_last) == 0) {
    const double igr = (gam - 1.0) / gam;
    double x0, x1;
    newton_start(c, W_last, x0, x1);
    int it = 0;
    if (c2p_polish(c, igr, x0, x1, LISTED_MAX_F64, it)) {
      const double noise = newton_noise(c, igr, x0, x1);
      bool in = noise <= LISTED_NOISE, assign;
      double out[NPR];
      for (int k = -1; k <= 1 && in; k++)
        in = c2p_finish(c, x0 * (1.0 + k * (LISTED_MARGIN * noise)), 0, igr, out, assign) == 0;
      if (in && c2p_finish_dd(c, x0, igr, out, assign) == 0 && assign) {
#pragma unroll
        for (int i = 0; i < B1; i++) pr[i] = out[i];
#pragma unroll
        for (int i = B1; i <= B3; i++) pr[i] = Ug[i];
        return 0;
      }
    }
  }
  bool polished;
  return utoprimgen_refined(U, G, gam, pr, iters, polished);
}

}  // namespace hg
