// kf_pose_math.hpp — FP64 rigid-transform helpers compiled for host and device.
//
// Replaces the host Eigen FP32 4x4 inverse of General::UpdateTransforms and
// ICP::Iterate_ICP (Source/src/General.cpp:27-36, Source/src/ICP.cpp:106-115) with
// the rigid inverse (R^T, -R^T t), and Cpu_buildNewTransformMatrix
// (Source/src/ICP.cu:266-321) with an FP64 Euler-ZYX increment left-multiplied
// onto the pose.  Operation order is fixed, contraction is off and the fused
// multiply-adds are explicit (fma, correctly rounded on both sides), so host and
// device produce identical bits but for the solve's reciprocals (pivot_inverse).
#pragma once

#include <math.h>

#include "kinfu.h"

#if defined(__HIPCC__)
#define KF_HD __host__ __device__ inline
#else
#define KF_HD inline
#endif

namespace kf {

// Row r of -R^T t for the rigid transform T (row-major 4x4).
KF_HD double rigid_inverse_t(const double* T, int r) {
  return -((T[0 * 4 + r] * T[3] + T[1 * 4 + r] * T[7]) + T[2 * 4 + r] * T[11]);
}

// Ti = inverse of the rigid transform T (row-major 4x4).
KF_HD void rigid_inverse(const double* T, double* Ti) {
  for (int r = 0; r < 3; ++r) {
    for (int c = 0; c < 3; ++c) Ti[r * 4 + c] = T[c * 4 + r];
    Ti[r * 4 + 3] = rigid_inverse_t(T, r);
  }
  Ti[12] = 0.0;
  Ti[13] = 0.0;
  Ti[14] = 0.0;
  Ti[15] = 1.0;
}

// Entry (i, j) of A * B (row-major 4x4).
KF_HD double mat4_mul_entry(const double* A, const double* B, int i, int j) {
  return ((A[i * 4 + 0] * B[0 * 4 + j] + A[i * 4 + 1] * B[1 * 4 + j]) + A[i * 4 + 2] * B[2 * 4 + j]) +
         A[i * 4 + 3] * B[3 * 4 + j];
}

// C = A * B (row-major 4x4); C must not alias A or B.
KF_HD void mat4_mul(const double* A, const double* B, double* C) {
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 4; ++j) C[i * 4 + j] = mat4_mul_entry(A, B, i, j);
}

// One Newton step of the polar decomposition on the rotation block,
// R <- R (3I - R^T R) / 2: removes the (quadratically small) drift from
// orthonormality that repeated pose products accumulate.  The constant-velocity
// prediction T1 (T0^-1 T1) would otherwise amplify it by ~2.4x per frame.
KF_HD void orthonormalize(double* T) {
  double S[9];  // R^T R
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j)
      S[i * 3 + j] = (T[0 * 4 + i] * T[0 * 4 + j] + T[1 * 4 + i] * T[1 * 4 + j]) + T[2 * 4 + i] * T[2 * 4 + j];
  double R[9];
  for (int r = 0; r < 3; ++r)
    for (int c = 0; c < 3; ++c) {
      const double rs = (T[r * 4 + 0] * S[0 * 3 + c] + T[r * 4 + 1] * S[1 * 3 + c]) + T[r * 4 + 2] * S[2 * 3 + c];
      R[r * 3 + c] = 1.5 * T[r * 4 + c] - 0.5 * rs;
    }
  for (int r = 0; r < 3; ++r)
    for (int c = 0; c < 3; ++c) T[r * 4 + c] = R[r * 3 + c];
}

// Fills the FP32 fields of p from p->T_wc.
KF_HD void pose_finish_fields(kf_pose* p) {
  double Ti[16];
  rigid_inverse(p->T_wc, Ti);
  for (int r = 0; r < 3; ++r) {
    for (int c = 0; c < 3; ++c) {
      p->wc.r[r * 3 + c] = (float)p->T_wc[r * 4 + c];
      p->cw.r[r * 3 + c] = (float)Ti[r * 4 + c];
    }
    p->wc.t[r] = (float)p->T_wc[r * 4 + 3];
    p->cw.t[r] = (float)Ti[r * 4 + 3];
  }
}

// Constant-velocity guess: T_{k-1} (T_{k-2}^-1 T_{k-1}), orthonormalised, with the
// FP32 fields.
KF_HD kf_pose constant_velocity_pose(const kf_pose& p2, const kf_pose& p1) {
  double Ti[16], Dl[16];
  kf_pose g;
  rigid_inverse(p2.T_wc, Ti);
  mat4_mul(Ti, p1.T_wc, Dl);
  mat4_mul(p1.T_wc, Dl, g.T_wc);
  orthonormalize(g.T_wc);
  pose_finish_fields(&g);
  return g;
}

// Euler-ZYX increment R = Rz(g) Ry(b) Rx(a) with translation t (same element
// formulas as the reference's incremental transform).
KF_HD double euler_zyx_entry(int e, double ca, double sa, double cb, double sb, double cg, double sg, double tx,
                             double ty, double tz) {
  switch (e) {
    case 0: return cg * cb;
    case 1: return -sg * ca + (cg * sb) * sa;
    case 2: return sg * sa + (cg * sb) * ca;
    case 3: return tx;
    case 4: return sg * cb;
    case 5: return cg * ca + (sg * sb) * sa;
    case 6: return -cg * sa + (sg * sb) * ca;
    case 7: return ty;
    case 8: return -sb;
    case 9: return cb * sa;
    case 10: return cb * ca;
    case 11: return tz;
    case 15: return 1.0;
    default: return 0.0;
  }
}

KF_HD void small_sincos(double x, double* c, double* s);

KF_HD void euler_zyx(double a, double b, double g, double tx, double ty, double tz, double* D) {
  double ca, sa, cb, sb, cg, sg;
  small_sincos(a, &ca, &sa);
  small_sincos(b, &cb, &sb);
  small_sincos(g, &cg, &sg);
  for (int e = 0; e < 16; ++e) D[e] = euler_zyx_entry(e, ca, sa, cb, sb, cg, sg, tx, ty, tz);
}

KF_HD double pivot_inverse(double d) {
#if defined(__HIP_DEVICE_COMPILE__)
  double r = __builtin_amdgcn_rcp(d);
  r = fma(r, fma(-d, r, 1.0), r);
  return fma(r, fma(-d, r, 1.0), r);
#else
  return 1.0 / d;
#endif
}

// Solves the 6x6 SPD system A x = g (A given by its 21 upper-triangle entries,
// row-major i <= j) by the square-root-free Cholesky factorisation A = L D L^T
// (L unit lower triangular).  Returns false if a pivot D_j is not above
// rel_eps * max diagonal (or NaN) — the pivot a Cholesky factorisation would take
// the square root of.  Each column divides once (1 / D_j) and multiplies, so the
// critical path holds six divisions and no square root.  W holds L D (the
// unscaled column entries), so no product is formed twice.  The updates are fused
// multiply-adds (one rounding each).  On the device 1 / D_j is the hardware reciprocal
// refined by two Newton steps (within an ulp of the quotient; D_j is a normal number
// where it counts) and there is no early return: a bad pivot is remembered.
KF_HD bool ldlt_solve6(const double* upper21, const double* g, double rel_eps, double* x) {
  double A[6][6];
  int k = 0;
  double dmax = 0.0;
  for (int i = 0; i < 6; ++i)
    for (int j = i; j < 6; ++j) {
      A[i][j] = upper21[k];
      A[j][i] = upper21[k];
      ++k;
    }
  for (int i = 0; i < 6; ++i) dmax = A[i][i] > dmax ? A[i][i] : dmax;
  const double thr = rel_eps * dmax;
  bool ok = true;
  double L[6][6], W[6][6], inv[6];
  for (int j = 0; j < 6; ++j) {
    double d = A[j][j];
    for (int m = 0; m < j; ++m) d = fma(-W[j][m], L[j][m], d);
    ok = ok && d > thr;
    inv[j] = pivot_inverse(d);
    for (int i = j + 1; i < 6; ++i) {
      double w = A[i][j];
      for (int m = 0; m < j; ++m) w = fma(-W[i][m], L[j][m], w);
      W[i][j] = w;
      L[i][j] = w * inv[j];
    }
  }
  double z[6];
  for (int i = 0; i < 6; ++i) {
    double s = g[i];
    for (int m = 0; m < i; ++m) s = fma(-L[i][m], z[m], s);
    z[i] = s;
  }
  for (int i = 5; i >= 0; --i) {
    double s = z[i] * inv[i];
    for (int m = 5; m > i; --m) s = fma(-L[m][i], x[m], s);  // the newest x last: one step of the chain each
    x[i] = s;
  }
  return ok;
}

// cos and sin of a small angle: Taylor series through x^14 / x^13 (Horner in x^2)
// for |x| <= 0.25, where the truncation error is below 1e-20; libm otherwise.  On the
// device the series is formed without a branch, and libm's code is entered only when a
// lane of the wave needs it (800 cycles against 200 with the test around the series).
KF_HD void small_sincos(double x, double* c, double* s) {
  const double z = x * x;
  double ps = 1.0 / 6227020800.0, pc = -1.0 / 87178291200.0;  // Horner steps as fused multiply-adds
  ps = fma(z, ps, -1.0 / 39916800.0);
  pc = fma(z, pc, 1.0 / 479001600.0);
  ps = fma(z, ps, 1.0 / 362880.0);
  pc = fma(z, pc, -1.0 / 3628800.0);
  ps = fma(z, ps, -1.0 / 5040.0);
  pc = fma(z, pc, 1.0 / 40320.0);
  ps = fma(z, ps, 1.0 / 120.0);
  pc = fma(z, pc, -1.0 / 720.0);
  ps = fma(z, ps, -1.0 / 6.0);
  pc = fma(z, pc, 1.0 / 24.0);
  ps = fma(z, ps, 1.0);
  pc = fma(z, pc, -0.5);
  *s = x * ps;
  *c = fma(z, pc, 1.0);
  const bool large = !(fabs(x) <= 0.25);
#if defined(__HIP_DEVICE_COMPILE__)
  if (__builtin_expect(__any(large), 0))
#endif
    if (large) {
      *c = cos(x);
      *s = sin(x);
    }
}

}  // namespace kf
