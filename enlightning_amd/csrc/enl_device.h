// enl_device.h -- device-side building blocks of the per-patch update path
// for gfx950 (CDNA4).  What decides something (the sensor, tag_cells) and the
// pressure keep the operations of the reference Fortran (fortran/rhs_*.m4,
// update_state.m4, tag_cells.m4) and give its bits; flux differences, the
// source and the temperature are algebraically equal forms that agree with
// it to rounding.  Compiled with -ffp-contract=off: every fused multiply-add
// is written out, so all kernels that share an expression round alike.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#pragma clang fp contract(off)

namespace enl {

// Fortran default-REAL literals are folded in single precision and widened.
constexpr double kC13_12 = (double)(13.0f / 12.0f);
constexpr double kW01 = (double)0.1f;
constexpr double kW06 = (double)0.6f;
constexpr double kW03 = (double)0.3f;
constexpr double kEpsWeno = (double)10.0e-6f;
constexpr double kC1_6 = (double)(1.0f / 6.0f);
constexpr double kC1_3 = (double)(1.0f / 3.0f);
constexpr double kC2_3 = (double)(2.0f / 3.0f);
constexpr double kC4_3 = (double)(4.0f / 3.0f);
constexpr double kA1 = (double)0.79926643f;
constexpr double kA2 = (double)-0.18941314f;
constexpr double kA3 = (double)0.02651995f;
constexpr double kC078 = (double)0.78f;
constexpr double kC09 = (double)0.9f;
constexpr double kThresh = (double)0.9999f;

// rhs variants, one per fortran/rhs_*.m4 file.
enum Variant : int {
  kHybridHighLlf = 0,
  kHybridHigh = 1,
  kHybridLowLlf = 2,
  kHybridLow = 3,
  kWenoHighLlf = 4,
  kWenoHigh = 5,
  kWenoLowLlf = 6,
  kWenoLow = 7,
  kDrp = 8,
  kNumVariants = 9
};

// Compile-time description of a variant (what differs between the nine
// Fortran files; the flux and source blocks are common to all of them).
template <int V>
struct Scheme {
  static constexpr bool hybrid = V <= kHybridLow;
  static constexpr bool drp = V <= kHybridLow || V == kDrp;
  static constexpr bool weno = V != kDrp;
  static constexpr int order = (V == kHybridLowLlf || V == kHybridLow || V == kWenoLowLlf || V == kWenoLow) ? 3 : 5;
  static constexpr bool llf = (V == kHybridHighLlf || V == kHybridLowLlf || V == kWenoHighLlf || V == kWenoLowLlf);
  // flux stencil half width: rhs_weno_low*.m4 build F(0:4) (q=-2..2)
  static constexpr int reach = (V == kWenoLowLlf || V == kWenoLow) ? 2 : 3;
  // LLF window half width: q=-3..3 (*_high_llf) or -2..2 (*_low_llf)
  static constexpr int llf_reach = order == 5 ? 3 : 2;
};

// The order of a variant's WENO scheme (rhs_*_low*.m4: 3).
__host__ inline int variant_order(int v) {
  return v == kHybridLowLlf || v == kHybridLow || v == kWenoLowLlf || v == kWenoLow ? 3 : 5;
}

__host__ __device__ inline double sq(double x) { return x * x; }

// FP64 division through a shared reciprocal.  hipcc expands n / d into
// v_div_scale of both operands (range scaling), v_rcp_f64 and two Newton
// steps on the reciprocal, the quotient n*r, its residual, the corrected
// quotient (v_div_fmas) and v_div_fixup (special operands).  When neither
// operand needs scaling, both v_div_scale return their input, v_div_fmas is
// a plain fma and v_div_fixup returns the quotient: rcp_nr and div_nr below
// are then that same sequence, so div_nr(n, d, rcp_nr(d)) == n / d bit for
// bit, and one reciprocal serves every quotient by d.  No scaling happens
// when |d| is in [2^-50, 2^50] (den_ok) and n is zero or |n| is in
// [2^-960, 2^700] (num_ok): the exponents differ by less than 768, the
// exponent of n is above the sequence's tiny-numerator bound (2^-969) and
// 1/d, n/d are normal.  A zero numerator gives +0 (n / d gives -0 for
// n = -0, d > 0; the two compare equal).
__device__ inline double rcp_nr(double d) {
  double r = __builtin_amdgcn_rcp(d);
  double e = fma(-d, r, 1.0);
  r = fma(r, e, r);
  e = fma(-d, r, 1.0);
  return fma(r, e, r);
}
__device__ inline double div_nr(double n, double d, double r) {
  const double q = n * r;
  const double e = fma(-d, q, n);
  return fma(e, r, q);
}
__host__ __device__ inline bool den_ok(double d) {
  const double m = fabs(d);
  return m >= 0x1p-50 && m <= 0x1p50;
}
__host__ __device__ inline bool num_ok(double n) {
  const double m = fabs(n);
  return (m >= 0x1p-960 && m <= 0x1p700) || n == 0;
}
// 1/d within an ulp: rcp_nr where den_ok, else the IEEE division.
__device__ inline double rcp_any(double d) { return den_ok(d) ? rcp_nr(d) : 1.0 / d; }
// A reciprocal to full precision in one cubic step: with e = 1 - d r the
// error of r(1 + e + e^2) is e^3, far below an ulp (v_rcp_f64 is good to
// about 2^-24).  Zero, infinite and NaN d give no finite result.
__device__ inline double rcp_cubic(double d) {
  const double r = __builtin_amdgcn_rcp(d);
  const double e = fma(-d, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

// WENO flux differences from the differences of the split fluxes.
//
// One direction of the reference's WENO branch forms the split fluxes
// f+- = (F +- alpha w) / 2 at 2R + 1 points, four reconstructions and
// pf1 + mf1 - pf2 - mf2 (rhs_hybrid_high_llf.m4:286-354).  The smoothness
// indicators, and the candidates less the middle one f_1, are functions of
// the differences of neighbouring f alone: with e_m = 2 (f_{m+1} - f_m), the
// second differences c_m = e_m - e_{m-1} and t_m = c_{m+1} - c_m,
//   16 beta = 4 (13/12) c^2 + (second term)^2,
//   pf = f_1 - (1/12) q1 (t_0 q2 + 4 r2 t_2 q0) / (q1 (q2 + 2 r2 q0) + 2 q0 q2)
// with q_k = (16 eps + 16 beta_k)^2 (the common factor 256 cancels), r2 =
// w01 / w06 and w03 / w06 = 1/2 exactly (0.6f = 2 * 0.3f).  The four second
// differences and their squares serve both reconstructions of a sign, and
// their two fractions share one division.  The minus side is the plus side
// on the differences in reverse order.  Beside needing less than half the
// operations of four separate reconstructions, the large common part of F
// and alpha w (the pressure, a stratified ambient) cancels in the first
// subtraction, before anything is rounded at its size.  Where the products
// leave the finite range (16 beta beyond ~1e38, or non-finite data) the
// result is not finite and the caller evaluates the reference's expressions
// instead (weno_dir_ref).  A pass of one all-WENO RK3 step at 1024^2:
// 398 us with four separate reconstructions of one division each, 291 us in
// this form, 307 us with the candidates taken relative to their middle point
// instead of f_1 (three more operations per sign, no smaller error on any
// tested field).
//
// weno_pair5 returns (pf1 - pf2) / (kC1_6 / 2).
constexpr double kR2 = kW01 / kW06;
static_assert(kW03 / kW06 == 0.5, "the float literals 0.3 and 0.6 differ by an exact factor of two");

// The reference's reconstruction wenop5 (rhs_hybrid_high_llf.m4:400-433) by its
// own expressions; wenom5 (365-398) is its mirror image, (e, d, c, b, a).
__device__ inline double wenop5_ref(double a, double b, double c, double d, double e) {
  const double b0 = kC13_12 * sq(c - 2 * d + e) + 0.25 * sq(3 * c - 4 * d + e);
  const double b1 = kC13_12 * sq(b - 2 * c + d) + 0.25 * sq(b - d);
  const double b2 = kC13_12 * sq(a - 2 * b + c) + 0.25 * sq(a - 4 * b + 3 * c);
  const double z0 = kW03 / sq(kEpsWeno + b0), z1 = kW06 / sq(kEpsWeno + b1), z2 = kW01 / sq(kEpsWeno + b2);
  const double sigma = z0 + z1 + z2;
  return (z0 / sigma) * (kC1_6 * (2 * c + 5 * d - e)) + (z1 / sigma) * (kC1_6 * (-b + 5 * c + 2 * d)) +
         (z2 / sigma) * (kC1_6 * (2 * a - 7 * b + 11 * c));
}

__device__ inline double weno_pair5(double e0, double e1, double e2, double e3, double e4) {
  constexpr double kC = 4 * kC13_12, kE = 16 * kEpsWeno;
  const double c1 = e1 - e0, c2 = e2 - e1, c3 = e3 - e2, c4 = e4 - e3;
  const double t1 = c2 - c1, t2 = c3 - c2, t3 = c4 - c3;
  const double s1 = fma(kC * c1, c1, kE), s2 = fma(kC * c2, c2, kE), s3 = fma(kC * c3, c3, kE),
               s4 = fma(kC * c4, c4, kE);
  auto quad = [](double l, double s) { return sq(fma(l, l, s)); };
  double n1, d1, n2, d2;
  {
    const double q0 = quad(fma(-3.0, e2, e3), s3), q1 = quad(e1 + e2, s2), q2 = quad(fma(3.0, e1, -e0), s1);
    n1 = q1 * fma(4 * kR2 * q0, t1, t2 * q2);
    d1 = fma(q1, fma(2 * kR2, q0, q2), 2 * (q0 * q2));
  }
  {
    const double q0 = quad(fma(-3.0, e3, e4), s4), q1 = quad(e2 + e3, s3), q2 = quad(fma(3.0, e2, -e1), s2);
    n2 = q1 * fma(4 * kR2 * q0, t2, t3 * q2);
    d2 = fma(q1, fma(2 * kR2, q0, q2), 2 * (q0 * q2));
  }
  return fma(fma(n2, d1, -(n1 * d2)), rcp_cubic(d1 * d2), fma(-2.0, e3, fma(-5.0, e2, e1)));
}

// The same for the third-order scheme (rhs_hybrid_low_llf.m4:349-399): with
// q = (4 eps + e^2)^2, w(2/3) = 2 w(1/3) exactly and e_m as above, the convex
// combination of the two neighbouring differences
//   pf = f_c + (1/4) (2 q(e_1) e_2 + q(e_2) e_1) / (2 q(e_1) + q(e_2))
// (f_c the value at the middle point); weno_pair3 returns 4 (pf1 - pf2).
// Relative to a candidate, as the fifth-order form is, it needs as many
// operations and its error on random data is 1.4 times the reference's.
static_assert(kC2_3 == 2 * kC1_3, "float(2/3) = 2 float(1/3)");

// wenop3 (rhs_hybrid_low_llf.m4:375-399); wenom3 (349-373) is its mirror image.
__device__ inline double wenop3_ref(double a, double b, double c) {
  const double z0 = kC2_3 / sq(kEpsWeno + sq(c - b)), z1 = kC1_3 / sq(kEpsWeno + sq(b - a));
  const double sigma = z0 + z1;
  return (z0 / sigma) * (0.5 * (b + c)) + (z1 / sigma) * (0.5 * (-a + 3 * b));
}
__device__ inline double weno_pair3(double e1, double e2, double e3) {
  constexpr double kE = 4 * kEpsWeno;
  const double q1 = sq(fma(e1, e1, kE)), q2 = sq(fma(e2, e2, kE)), q3 = sq(fma(e3, e3, kE));
  const double p1 = 2 * q1, p2 = 2 * q2;
  const double n1 = fma(p1, e2, q2 * e1), d1 = p1 + q2;
  const double n2 = fma(p2, e3, q3 * e2), d2 = p2 + q3;
  return fma(fma(n1, d2, -(n2 * d1)), rcp_cubic(d1 * d2), -2 * e2);
}

// One direction of the WENO branch for one component: F and W at the points
// m = -R..R of the stencil (index m + 3), alpha the LLF speed; returns
// (pf1 + mf1 - pf2 - mf2) / kWenoUnit<ORDER>.
template <int ORDER>
constexpr double kWenoUnit = ORDER == 5 ? 0.5 * kC1_6 : 0.25;

template <int ORDER>
__device__ inline double weno_dir(const double* F, const double* W, double alpha) {
  constexpr int R = ORDER == 5 ? 3 : 2;
  double dF[6], dW[6];
#pragma unroll
  for (int m = 3 - R; m < 3 + R; m++) {
    dF[m] = F[m + 1] - F[m];
    dW[m] = W[m + 1] - W[m];
  }
  auto ep = [&](int m) { return fma(alpha, dW[m], dF[m]); };
  auto em = [&](int m) { return fma(-alpha, dW[m], dF[m]); };
  if constexpr (ORDER == 5) {
    const double p = weno_pair5(ep(0), ep(1), ep(2), ep(3), ep(4));
    __builtin_amdgcn_sched_barrier(0);
    return p + weno_pair5(em(5), em(4), em(3), em(2), em(1));
  } else
    return weno_pair3(ep(1), ep(2), ep(3)) + weno_pair3(em(4), em(3), em(2));
}

// The same by the reference's expressions, for where weno_dir's is not finite:
// its weights vanish for a candidate across a jump whose smoothness leaves the
// range, and the other candidates are summed as they are (the differences of
// weno_dir would hold the jump and lose them in it).  point(m, F, W) gives F
// and W at point m.  pf1, mf1, pf2 and mf2 come from one rolled loop that reads
// its points again: rare, and no registers of the path before it are held for
// it (dense kernel 81 VGPRs, 114 with the four written out; the list kernel 154
// and no spills, 168 and 36 B with the stencil selected into registers:
// channel at 2048^2 2.70 -> 2.63 ms).
template <int ORDER, class Point>
__device__ inline double weno_dir_ref(Point point, double alpha) {
  constexpr int R = ORDER == 5 ? 3 : 2;
  double sum = 0;
#pragma unroll 1
  for (int r = 0; r < 4; r++) {
    const bool minus = r & 1, second = r >> 1;
    const int first = (minus ? R - 1 : -R) + second, step = minus ? -1 : 1;
    const double s = minus ? -alpha : alpha;
    double f[2 * R - 1];
#pragma unroll
    for (int q = 0; q < 2 * R - 1; q++) {
      double F, W;
      point(first + q * step, F, W);
      f[q] = 0.5 * (F + s * W);
    }
    double v;
    if constexpr (ORDER == 5)
      v = wenop5_ref(f[0], f[1], f[2], f[3], f[4]);
    else
      v = wenop3_ref(f[0], f[1], f[2]);
    sum = r == 0 ? v : second ? sum - v : sum + v;
  }
  return sum / kWenoUnit<ORDER>;
}

// Smoothness ratio of the hybrid sensor and of tag_cells
// (rhs_hybrid_high_llf.m4:246, tag_cells.m4:71).
__device__ inline double smooth_ratio(double tmp1, double tmp2, double ep) {
  return (2 * fabs(tmp1 * tmp2) + ep) / (sq(tmp1) + sq(tmp2) + ep);
}

// ep = 0.9*tol*(xi**2)/(1-0.9*(tol**2)), xi = 1 (rhs_hybrid_high_llf.m4:114-115)
__host__ __device__ inline double sensor_eps(double tol) {
  double xi = 1;
  return kC09 * tol * sq(xi) / (1 - kC09 * sq(tol));
}

// What update_state needs of the gas, with the constants' quotients formed
// once on the host (make_eos).
struct Eos {
  double c, c_lr, rho0, c_p, p0, T0, c_v, R;
  double k1;              // (gamma1 - 1) / (2 * rho0)
  double inv_cp, inv_cv;  // IEEE reciprocals
  bool ok;                // rho0, c_p, c_v pass div_nr's range conditions
};
__host__ inline Eos make_eos(double c, double c_lr, double rho0, double gamma1, double c_p, double p0, double T0,
                             double c_v, double R) {
  Eos e = {c, c_lr, rho0, c_p, p0, T0, c_v, R, (gamma1 - 1) / (2 * rho0), 1.0 / c_p, 1.0 / c_v, false};
  e.ok = rho0 > 0 && den_ok(rho0) && den_ok(c_p) && den_ok(c_v);
  return e;
}

// Pressure and temperature of one cell, update_state.m4:88-105 (xc1 is the
// cell-centre height xylo(1)+dxy(1)*(j-ifirst1+0.5)).
__device__ inline void eos_p_T_ref(const Eos& E, double xc1, double w0, double w3, double& p, double& T) {
  p = sq(E.c + E.c_lr * xc1) *
          ((w0 - E.rho0) + E.k1 * sq(w0 - E.rho0) + (w0 / E.c_p) * (w3 / w0)) +
      E.p0;
  T = E.T0 * exp((w3 / w0 - E.R * log(E.rho0 / w0)) / E.c_v);
}

// log of y in [2^-101, 2^101], within 2.1 ulps (a model of these operations on
// the CPU against extended precision, 2e6 values each of eight ranges: at most
// 2.03 near y = 0.7, RMS 0.6 around 1 and less beyond): y = 2^e m with m in [1/sqrt 2,
// sqrt 2), log m = 2 atanh(s) = 2 s + s^3 P(s^2) with s = (m - 1) / (m + 1), P
// the interpolant of the atanh series at Chebyshev nodes of its range (error
// below 5e-18 of the result).  A third of the library function's
// instructions.
__device__ inline double log_mid(double y) {
  double m = __builtin_amdgcn_frexp_mant(y);
  int e = __builtin_amdgcn_frexp_exp(y);
  if (m < 0x1.6a09e667f3bcdp-1) {
    m = m + m;
    e--;
  }
  const double d = m + 1, n = m - 1, r = rcp_cubic(d);
  const double q = n * r, s = fma(fma(-d, q, n), r, q);
  const double z = s * s;
  double P = 0x1.2b583bc0f4a07p-3;
  P = fma(P, z, 0x1.39fe61b2d9627p-3);
  P = fma(P, z, 0x1.7462b4a01ca9cp-3);
  P = fma(P, z, 0x1.c71c62e5ac92cp-3);
  P = fma(P, z, 0x1.2492492df11e1p-2);
  P = fma(P, z, 0x1.99999999952e4p-2);
  P = fma(P, z, 0x1.5555555555558p-1);
  return fma((double)e, 0x1.62e42fefa39efp-1, fma(s * z, P, s + s));
}

// eos_p_T_ref with its quotients through reciprocals where the operands
// allow it: the same p bit for bit (div_nr is IEEE division there); T = T0
// exp(x) with x's quotient by c_v a product and its logarithm log_mid, so a
// relative error of some ulps times 1 + |x|, as eos_p_T_ref's is (RMS over
// waves, shocks and stratified states 0.98-1.00 of it).
// want_T false leaves T alone.
__device__ inline void eos_p_T(const Eos& E, double xc1, double w0, double w3, double& p, double& T,
                               bool want_T = true) {
  if (E.ok && w0 > 0 && den_ok(w0) && num_ok(w3)) {
    const double rw = rcp_nr(w0);
    const double s = div_nr(w3, w0, rw);
    const double d = w0 - E.rho0;
    p = sq(E.c + E.c_lr * xc1) * (d + E.k1 * sq(d) + div_nr(w0, E.c_p, E.inv_cp) * s) + E.p0;
    if (want_T) T = E.T0 * exp(fma(-E.R, log_mid(div_nr(E.rho0, w0, rw)), s) * E.inv_cv);
    return;
  }
  eos_p_T_ref(E, xc1, w0, w3, p, T);
}

}  // namespace enl
