// swm_numerics.hpp -- per-point FP64 arithmetic of the mPDeC5 / WENO5 PATANKAR
// step, shared by every kernel of the library.
//
// Each function evaluates the reference expression in the reference's order
// (Fortran: left to right, parentheses honoured) and the whole library is
// built with -ffp-contract=off, so no multiply-add is fused; '/' and sqrt are
// the IEEE correctly rounded FP64 operations.  Together that makes the device
// results bitwise equal to a contraction-free build of the reference.
// MAX/MIN follow the reference compiler's lowering, which fixes NaN
// behaviour: MAX(a,b) = (a > b) ? a : b, MIN(a,b) = (a < b) ? a : b.
#pragma once

#include <hip/hip_runtime.h>

namespace swm {

constexpr double kWenoEps = 1.0E-24;     // src/finitevolume_vars.f90:97
constexpr double kMinDepth = 1.0E-6;     // src/finitevolume_vars.f90:104
constexpr double kMinTimestep = 1.0E-30; // src/finitevolume_vars.f90:106
constexpr double kWLobatto = 1. / 12.;   // src/finitevolume_vars.f90:96
constexpr double kHuge = 1.7976931348623157e308;  // HUGE(1.0), real(8)

__device__ __forceinline__ double max_r(double a, double b) { return (a > b) ? a : b; }
__device__ __forceinline__ double min_r(double a, double b) { return (a < b) ? a : b; }

// ------------------------------------------------------------------------
// Division with a reciprocal shared between quotients of one denominator.
//
// gfx950 evaluates the IEEE quotient a/b as
//   sb = div_scale(b), sa = div_scale(a), r = rcp(sb),
//   r = fma(r, fma(-sb, r, 1), r)  (twice),  q = sa*r,
//   div_fixup(div_fmas(fma(-sb, q, sa), r, q), b, a).
// When a and b are normal, a/b is normal and their exponents are far from
// the ranges where the hardware rescales (|a|, |b| in [2^-500, 2^500] with
// |a/b| >= 2^-900 is far inside them), div_scale returns its operand,
// div_fmas is a plain fma and div_fixup returns its value, so recip_refined
// once per denominator followed by div_by per numerator yields the same bits
// as '/', with 5 + 3 instructions instead of 11 per quotient.  Callers check
// the range first and use '/' otherwise.
// ------------------------------------------------------------------------
#ifndef SWM_SHARED_RECIP
#define SWM_SHARED_RECIP 1
#endif
constexpr double kRecipLo = 0x1p-400;
constexpr double kRecipHi = 0x1p+400;

// 1 when kRecipLo <= b <= kRecipHi (0 for NaN); combined with '&' so that the
// three checks of a reconstruction need no branches.
__device__ __forceinline__ int recip_range(double b) {
  return (int)(b >= kRecipLo) & (int)(b <= kRecipHi);
}

__device__ __forceinline__ double recip_refined(double b) {
  double r = __builtin_amdgcn_rcp(b);
  double e = fma(-b, r, 1.0);
  r = fma(r, e, r);
  e = fma(-b, r, 1.0);
  r = fma(r, e, r);
  return r;
}

// Reciprocals of two, three or four denominators from one hardware reciprocal
// of their product: R = 1/(b1 b2 ..) takes the first refinement, R times the
// other denominators approximates each 1/b_k to 2^-48 (as one refined rcp
// does: its seed is good to 2^-24.4), and the last refinement is the one of
// recip_refined.  v_rcp_f64 takes the issue time of 3.4 multiplications
// (7.2 against 2.1 ns per wave and SIMD), so three reciprocals cost 17 slots
// instead of 22 and four 22 instead of 29.  Callers keep the product inside
// the exponent range (kWenoLo, kWenoHi).
__device__ __forceinline__ double newton(double b, double r) { return fma(r, fma(-b, r, 1.0), r); }

__device__ __forceinline__ void recip2(double b1, double b2, double& r1, double& r2) {
  const double P = b1 * b2;
  const double R = newton(P, __builtin_amdgcn_rcp(P));
  r1 = newton(b1, R * b2);
  r2 = newton(b2, R * b1);
}

__device__ __forceinline__ void recip3(double b1, double b2, double b3, double& r1, double& r2,
                                       double& r3) {
  const double p = b1 * b2, P = p * b3;
  const double R = newton(P, __builtin_amdgcn_rcp(P));
  const double t = R * b3;
  r1 = newton(b1, t * b2);
  r2 = newton(b2, t * b1);
  r3 = newton(b3, R * p);
}

__device__ __forceinline__ void recip4(const double b[4], double r[4]) {
  const double p = b[0] * b[1], q = b[2] * b[3], P = p * q;
  const double R = newton(P, __builtin_amdgcn_rcp(P));
  const double tp = R * q, tq = R * p;
  r[0] = newton(b[0], tp * b[1]);
  r[1] = newton(b[1], tp * b[0]);
  r[2] = newton(b[2], tq * b[3]);
  r[3] = newton(b[3], tq * b[2]);
}

__device__ __forceinline__ double div_by(double a, double b, double rb) {
  double q = a * rb;
  double e = fma(-b, q, a);
  return fma(e, rb, q);
}

// a/b for a positive b in [2^-400, 2^400] with rb = recip_refined(b): the
// same bits as '/'.  A zero numerator needs no division (the quotient is a
// itself); numerators beyond the range of div_by (tiny, huge, NaN, Inf) take
// the IEEE quotient.
__device__ __forceinline__ double div_pos(double a, double b, double rb) {
#if SWM_SHARED_RECIP
  const double m = fabs(a);
  if ((int)(m >= kRecipLo) & (int)(m <= kRecipHi)) return div_by(a, b, rb);
  if (a == 0.) return a;
#endif
  return a / b;
}

// The smaller of two values, the other one where one is NaN, in one
// instruction (fmin() first quiets each operand with one of its own).
__device__ __forceinline__ double min_n(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// ConsToPrim, src/equation.f90:912-945:  ht = h + MIN_DEPTH/h; u = hu/ht.
__device__ __forceinline__ void cons_to_prim(double h, double hu, double hv, double& u,
                                             double& v) {
  double ht = h + kMinDepth / h;
  u = hu / ht;
  v = hv / ht;
}

// Smoothness indicators shared by both WENO5 sweeps,
// src/reconstruction.f90:699-704 and :1024-1029, and (eps + beta)^2, with the
// reference's operations one by one.
__device__ __forceinline__ void weno5_den(double qm2, double qm1, double q0, double qp1,
                                          double qp2, double& d1, double& d2, double& d3) {
  double b1 = (1.0 / 3.0) * (4.0 * qm2 * qm2 - 19.0 * qm2 * qm1 + 25.0 * qm1 * qm1 +
                             11.0 * qm2 * q0 - 31.0 * qm1 * q0 + 10.0 * q0 * q0);
  double b2 = (1.0 / 3.0) * (4.0 * qm1 * qm1 - 13.0 * qm1 * q0 + 13.0 * q0 * q0 +
                             5.0 * qm1 * qp1 - 13.0 * q0 * qp1 + 4.0 * qp1 * qp1);
  double b3 = (1.0 / 3.0) * (10.0 * q0 * q0 - 31.0 * q0 * qp1 + 25.0 * qp1 * qp1 +
                             11.0 * q0 * qp2 - 19.0 * qp1 * qp2 + 4.0 * qp2 * qp2);
  d1 = (kWenoEps + b1) * (kWenoEps + b1);
  d2 = (kWenoEps + b2) * (kWenoEps + b2);
  d3 = (kWenoEps + b3) * (kWenoEps + b3);
}

// The same d1..d3 bit for bit wherever weno5_regular accepts them, with the
// factors 4 folded into exact FMAs: 4*q*q = 4*(q*q) and fma(4, q*q, y) rounds
// 4*q*q + y once, as the separate addition does.  Scaling by 4 commutes with
// rounding unless q*q is subnormal; an error there is at most 2^-1074 and can
// pass through a rounded sum only where the sum is below 2^-960 (a later sum
// of this chain: below 2^-690), so it never reaches eps + beta with
// eps = 10^-24 = 2^-79.7.
__device__ __forceinline__ void weno5_den_exact(double qm2, double qm1, double q0, double qp1,
                                                double qp2, double& d1, double& d2, double& d3) {
  const double s1 = qm1 * qm1, sp1 = qp1 * qp1;
  const double x0 = 13.0 * q0, c0 = 10.0 * q0 * q0;
  const double b1 = (1.0 / 3.0) * (fma(4.0, qm2 * qm2, -(19.0 * qm2 * qm1)) + 25.0 * qm1 * qm1 +
                                   11.0 * qm2 * q0 - 31.0 * qm1 * q0 + c0);
  const double b2 = (1.0 / 3.0) * fma(4.0, sp1, fma(4.0, s1, -(13.0 * qm1 * q0)) + x0 * q0 +
                                                    5.0 * qm1 * qp1 - x0 * qp1);
  const double b3 = (1.0 / 3.0) * fma(4.0, qp2 * qp2, c0 - 31.0 * q0 * qp1 + 25.0 * qp1 * qp1 +
                                                          11.0 * q0 * qp2 - 19.0 * qp1 * qp2);
  d1 = (kWenoEps + b1) * (kWenoEps + b1);
  d2 = (kWenoEps + b2) * (kWenoEps + b2);
  d3 = (kWenoEps + b3) * (kWenoEps + b3);
}

// The range in which a reconstruction takes the shared reciprocals: the three
// (eps + beta)^2 in [2^-240, 2^240).  Then the products of recip3 and recip4
// lie in 2^+-976, the alphas in [2^-244, 2^240], their sums in
// [2^-244, 2^242] and the weights above 2^-486; and every q is finite, since an
// Inf or NaN q would make one of the three Inf or NaN, and below 2^512, where
// the squares overflow (mostly far below: a q of 2^100 needs neighbours equal to
// it, the betas being differences), so that the candidates are finite too.
// They are squares, so their high words compare as unsigned integers (a NaN
// of either sign is above the range): two three-operand min/max and two
// compares instead of six FP64 compares.
constexpr unsigned kWenoLo = (1023u - 240u) << 20;
constexpr unsigned kWenoHi = (1023u + 240u) << 20;
__device__ __forceinline__ bool weno5_regular(double d1, double d2, double d3) {
  const unsigned h1 = __double2hiint(d1), h2 = __double2hiint(d2), h3 = __double2hiint(d3);
  return (int)(min(min(h1, h2), h3) >= kWenoLo) & (int)(max(max(h1, h2), h3) < kWenoHi);
}

// WENO5_FirstSweep, src/reconstruction.f90:673-755: cell average line values
// at the left (wm) and right (wp) faces.
__device__ __forceinline__ void weno5_first(double qm2, double qm1, double q0, double qp1,
                                            double qp2, double& wm, double& wp) {
  double d1, d2, d3;
#if SWM_SHARED_RECIP
  weno5_den_exact(qm2, qm1, q0, qp1, qp2, d1, d2, d3);
  if (weno5_regular(d1, d2, d3)) {
    double r1, r2, r3;
    recip3(d1, d2, d3, r1, r2, r3);
    const double am1 = div_by(3.0 / 10.0, d1, r1), ap1 = div_by(1.0 / 10.0, d1, r1);
    const double a2 = div_by(3.0 / 5.0, d2, r2);
    const double am3 = div_by(1.0 / 10.0, d3, r3), ap3 = div_by(3.0 / 10.0, d3, r3);
    const double sm = am1 + a2 + am3, sp = ap1 + a2 + ap3;
    double rm, rp;
    recip2(sm, sp, rm, rp);
    // doubling is exact, so 2*q + y is one FMA
    {
      const double o1 = div_by(am1, sm, rm), o2 = div_by(a2, sm, rm), o3 = div_by(am3, sm, rm);
      const double w1 = (1.0 / 6.0) * fma(2.0, q0, -qm2 + 5.0 * qm1);
      const double w2 = (1.0 / 6.0) * (fma(2.0, qm1, 5.0 * q0) - qp1);
      const double w3 = (1.0 / 6.0) * fma(2.0, qp2, 11.0 * q0 - 7.0 * qp1);
      wm = o1 * w1 + o2 * w2 + o3 * w3;
    }
    {
      const double o1 = div_by(ap1, sp, rp), o2 = div_by(a2, sp, rp), o3 = div_by(ap3, sp, rp);
      const double w1 = (1.0 / 6.0) * (fma(2.0, qm2, -(7.0 * qm1)) + 11.0 * q0);
      const double w2 = (1.0 / 6.0) * fma(2.0, qp1, -qm1 + 5.0 * q0);
      const double w3 = (1.0 / 6.0) * (fma(2.0, q0, 5.0 * qp1) - qp2);
      wp = o1 * w1 + o2 * w2 + o3 * w3;
    }
    return;
  }
#endif
  weno5_den(qm2, qm1, q0, qp1, qp2, d1, d2, d3);
  {
    double a1 = (3.0 / 10.0) / d1;
    double a2 = (3.0 / 5.0) / d2;
    double a3 = (1.0 / 10.0) / d3;
    double s = a1 + a2 + a3;
    double o1 = a1 / s, o2 = a2 / s, o3 = a3 / s;
    double w1 = (1.0 / 6.0) * (-qm2 + 5.0 * qm1 + 2.0 * q0);
    double w2 = (1.0 / 6.0) * (2.0 * qm1 + 5.0 * q0 - qp1);
    double w3 = (1.0 / 6.0) * (11.0 * q0 - 7.0 * qp1 + 2.0 * qp2);
    wm = o1 * w1 + o2 * w2 + o3 * w3;
  }
  {
    double a1 = (1.0 / 10.0) / d1;
    double a2 = (3.0 / 5.0) / d2;
    double a3 = (3.0 / 10.0) / d3;
    double s = a1 + a2 + a3;
    double o1 = a1 / s, o2 = a2 / s, o3 = a3 / s;
    double w1 = (1.0 / 6.0) * (2.0 * qm2 - 7.0 * qm1 + 11.0 * q0);
    double w2 = (1.0 / 6.0) * (-qm1 + 5.0 * q0 + 2.0 * qp1);
    double w3 = (1.0 / 6.0) * (2.0 * q0 + 5.0 * qp1 - qp2);
    wp = o1 * w1 + o2 * w2 + o3 * w3;
  }
}

// Coefficients of one Gauss point of WENO5_SecondSweep,
// src/reconstruction.f90:1036-1133.  The literals are the reference's decimal
// strings; signed literals are folded into the coefficients (a - c*q ==
// a + (-c)*q exactly).  c13, c14, c20, c24, c30, c31 are the reference's
// 0.0*Q terms.
struct Weno2Coef {
  double g1, g2, g3;
  double c10, c11, c12, c13, c14, c20, c21, c22, c23, c24, c30, c31, c32, c33, c34;
};

template <int G>
__device__ constexpr Weno2Coef weno2_coef() {
  if constexpr (G == 0)
    return {0.2658420974778319, 0.6112504900322486, 0.1229074124899195,
            -0.1642562761719537, 0.7590807081409336, 0.4051755680310201, 0.0000000000000000, 0.0000000000000000,
            +0.0000000000000000, 0.2663118796250726, 0.8979443965468811, -0.1642562761719537, 0.0000000000000000,
            +0.0000000000000000, 0.0000000000000000, 1.6968800354220990, -0.9631919150471715, 0.2663118796250726};
  else if constexpr (G == 1)
    return {0.1281641584355059, 0.5219691498503563, 0.3498666917141379,
            -0.1122135388132497, 0.3944175994189276, 0.7177959393943222, 0.0000000000000000, 0.0000000000000000,
            +0.0000000000000000, 0.0577769829791784, 1.0544365558340714, -0.1122135388132497, 0.0000000000000000,
            +0.0000000000000000, 0.0000000000000000, 1.2277675047716066, -0.2855444877507849, 0.0577769829791784};
  else if constexpr (G == 2)
    return {0.3498666917141379, 0.5219691498503563, 0.1281641584355059,
            +0.0577769829791784, -0.2855444877507849, 1.2277675047716066, 0.0000000000000000, 0.0000000000000000,
            +0.0000000000000000, -0.1122135388132497, 1.0544365558340714, 0.0577769829791784, 0.0000000000000000,
            +0.0000000000000000, 0.0000000000000000, 0.7177959393943222, 0.3944175994189276, -0.1122135388132497};
  else
    return {0.1229074124899195, 0.6112504900322486, 0.2658420974778319,
            +0.2663118796250726, -0.9631919150471715, 1.6968800354220990, 0.0000000000000000, 0.0000000000000000,
            +0.0000000000000000, -0.1642562761719537, 0.8979443965468811, 0.2663118796250726, 0.0000000000000000,
            +0.0000000000000000, 0.0000000000000000, 0.4051755680310201, 0.7590807081409336, -0.1642562761719537};
}

// The three candidate values, every term kept: the 0.0*Q terms propagate
// NaN/Inf and fix the sign of zero exactly as the reference does (the
// compiler shares the four distinct 0.0*q products between the Gauss points).
template <int G>
__device__ __forceinline__ void weno2_cand(double qm2, double qm1, double q0, double qp1,
                                           double qp2, double& w1, double& w2, double& w3) {
  constexpr Weno2Coef C = weno2_coef<G>();
  w1 = C.c10 * qm2 + C.c11 * qm1 + C.c12 * q0 + C.c13 * qp1 + C.c14 * qp2;
  w2 = C.c20 * qm2 + C.c21 * qm1 + C.c22 * q0 + C.c23 * qp1 + C.c24 * qp2;
  w3 = C.c30 * qm2 + C.c31 * qm1 + C.c32 * q0 + C.c33 * qp1 + C.c34 * qp2;
}

// The same candidates without the 0.0*Q terms, for finite q: they can change
// only the sign of a zero sum, and every sum has a positive coefficient
// (at least 0.4) on q0, so no sum is -0 unless q0 is -0 or a negative
// subnormal that the product rounds to -0 (weno5_second sends those to the
// full form).
template <int G>
__device__ __forceinline__ void weno2_cand_nz(double qm2, double qm1, double q0, double qp1,
                                              double qp2, double& w1, double& w2, double& w3) {
  constexpr Weno2Coef C = weno2_coef<G>();
  static_assert(C.c13 == 0. && C.c14 == 0. && C.c20 == 0. && C.c24 == 0. && C.c30 == 0. &&
                    C.c31 == 0. && C.c12 > 0.4 && C.c22 > 0.4 && C.c32 > 0.4,
                "the terms left out are zeros");
  w1 = C.c10 * qm2 + C.c11 * qm1 + C.c12 * q0;
  w2 = C.c21 * qm1 + C.c22 * q0 + C.c23 * qp1;
  w3 = C.c32 * q0 + C.c33 * qp1 + C.c34 * qp2;
}

// alpha_k = gamma_k / (eps + beta_k)^2 (src/reconstruction.f90:1030-1032)
// through the shared reciprocals, and their sum.
template <int G>
__device__ __forceinline__ double weno2_alpha(double d1, double d2, double d3, double r1,
                                              double r2, double r3, double a[3]) {
  constexpr Weno2Coef C = weno2_coef<G>();
  a[0] = div_by(C.g1, d1, r1);
  a[1] = div_by(C.g2, d2, r2);
  a[2] = div_by(C.g3, d3, r3);
  return a[0] + a[1] + a[2];
}

// omega_k = alpha_k / sum(alpha) (src/reconstruction.f90:1033-1035) and the
// weighted candidates.
template <int G>
__device__ __forceinline__ double weno2_blend(double qm2, double qm1, double q0, double qp1,
                                              double qp2, const double a[3], double s, double rs) {
  const double o1 = div_by(a[0], s, rs), o2 = div_by(a[1], s, rs), o3 = div_by(a[2], s, rs);
  double w1, w2, w3;
  weno2_cand_nz<G>(qm2, qm1, q0, qp1, qp2, w1, w2, w3);
  return (o1 * w1 + o2 * w2 + o3 * w3);
}

// One Gauss point with '/' and every term.
template <int G>
__device__ __forceinline__ double weno5_second_gp(double qm2, double qm1, double q0, double qp1,
                                                  double qp2, double d1, double d2, double d3) {
  constexpr Weno2Coef C = weno2_coef<G>();
  double a1 = C.g1 / d1;
  double a2 = C.g2 / d2;
  double a3 = C.g3 / d3;
  double s = a1 + a2 + a3;
  double o1 = a1 / s, o2 = a2 / s, o3 = a3 / s;
  double w1, w2, w3;
  weno2_cand<G>(qm2, qm1, q0, qp1, qp2, w1, w2, w3);
  return (o1 * w1 + o2 * w2 + o3 * w3);
}

// WENO5_SecondSweep, src/reconstruction.f90:999-1136: point values at the
// four Gauss nodes of the cell.
__device__ __forceinline__ void weno5_second(double qm2, double qm1, double q0, double qp1,
                                             double qp2, double w[4]) {
  double d1, d2, d3;
#if SWM_SHARED_RECIP
  weno5_den_exact(qm2, qm1, q0, qp1, qp2, d1, d2, d3);
  // the gammas lie in [0.12, 0.62]: the ranges of weno5_regular hold
  if ((int)weno5_regular(d1, d2, d3) &
      (int)((unsigned)__double2hiint(q0) != 0x80000000u)) {
    double r1, r2, r3, a[4][3], s[4], rs[4];
    recip3(d1, d2, d3, r1, r2, r3);
    s[0] = weno2_alpha<0>(d1, d2, d3, r1, r2, r3, a[0]);
    s[1] = weno2_alpha<1>(d1, d2, d3, r1, r2, r3, a[1]);
    s[2] = weno2_alpha<2>(d1, d2, d3, r1, r2, r3, a[2]);
    s[3] = weno2_alpha<3>(d1, d2, d3, r1, r2, r3, a[3]);
    recip4(s, rs);
    w[0] = weno2_blend<0>(qm2, qm1, q0, qp1, qp2, a[0], s[0], rs[0]);
    w[1] = weno2_blend<1>(qm2, qm1, q0, qp1, qp2, a[1], s[1], rs[1]);
    w[2] = weno2_blend<2>(qm2, qm1, q0, qp1, qp2, a[2], s[2], rs[2]);
    w[3] = weno2_blend<3>(qm2, qm1, q0, qp1, qp2, a[3], s[3], rs[3]);
    return;
  }
#endif
  weno5_den(qm2, qm1, q0, qp1, qp2, d1, d2, d3);
  w[0] = weno5_second_gp<0>(qm2, qm1, q0, qp1, qp2, d1, d2, d3);
  w[1] = weno5_second_gp<1>(qm2, qm1, q0, qp1, qp2, d1, d2, d3);
  w[2] = weno5_second_gp<2>(qm2, qm1, q0, qp1, qp2, d1, d2, d3);
  w[3] = weno5_second_gp<3>(qm2, qm1, q0, qp1, qp2, d1, d2, d3);
}

// PositivityLimiterX/Y body, src/finitevolume.f90:671-691: theta-scaling of
// the h values at the Gauss points of one cell towards the cell mean vh.
// Returns the smallest of the unlimited values and csi (a NaN among them may
// hide behind the others; then csi is NaN too).
//
// A theta is 1 without a division where |num| >= |den| with num finite (the
// rounded |num/den| is then at least 1).  Every den_g = vh - mmin_g has mmin_g
// between the smallest of all nine values and csi, and rounding is monotonic,
// so comparing num with those two ends settles the four thetas at once -- the
// usual case, the Gauss values lying close to the mean: 30 instructions
// instead of 80.  A NaN or Inf among the values makes csi one, which fails
// the comparison.
__device__ __forceinline__ double positivity_limit(double vh, const double wbnd[4], double wm[4],
                                                   double wp[4]) {
  double alpha = wbnd[0] * wm[0], beta = wbnd[0] * wp[0];
  double mn = min_n(wm[0], wp[0]);
#pragma unroll
  for (int g = 1; g < 4; ++g) {
    alpha = alpha + wbnd[g] * wm[g];
    beta = beta + wbnd[g] * wp[g];
    mn = min_n(mn, min_n(wm[g], wp[g]));
  }
  constexpr double c = 1. - 2. * kWLobatto;
  const double csi = div_pos(vh - kWLobatto * alpha - kWLobatto * beta, c, 1. / c);
  mn = min_n(mn, csi);
  const double num = vh - kMinDepth;
  if ((int)(fabs(num) >= fabs(vh - csi)) & (int)(fabs(num) >= fabs(vh - mn))) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      wp[g] = vh + (wp[g] - vh);
      wm[g] = vh + (wm[g] - vh);
    }
    return mn;
  }
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    double mmin = min_r(min_r(csi, wm[g]), wp[g]);
    const double den = vh - mmin;
    double theta;
    if (vh == mmin)
      theta = 1.;
    else if ((int)(fabs(num) >= fabs(den)) & (int)(fabs(num) <= kHuge))
      theta = 1.;
    else
      theta = min_r(1., fabs(num / den));
    wp[g] = vh + theta * (wp[g] - vh);
    wm[g] = vh + theta * (wm[g] - vh);
  }
  return mn;
}

// 1 when every limited depth of a cell is certain to lie in the range of
// sqrt_regular: with the unlimited ones at least 2^-40 vh (mn is their
// minimum), the limited ones, between them and vh but for two roundings of
// vh, are at least 2^-41 vh.
__device__ __forceinline__ bool depths_regular(double vh, double mn) {
  return (int)(mn >= vh * 0x1p-40) & (int)(vh >= 0x1p-600);
}

// sqrt(x) for finite x in [2^-767, 2^1023): y ~ 1/sqrt(x) to 2^-24, one
// Goldschmidt step for s ~ sqrt(x) and h ~ 1/(2 sqrt(x)), then two residual
// corrections s + (x - s*s)*h with the residual exact in one FMA; the last
// rounds a value accurate to 2^-99, the bits of sqrt().  sqrt() adds the
// scaling of subnormal operands and the cases of 0 and Inf: 8 instructions
// of 18.
__device__ __forceinline__ double sqrt_regular(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double s = x * y, h = 0.5 * y;
  const double e = fma(-h, s, 0.5);
  s = fma(s, e, s);
  h = fma(h, e, h);
  s = fma(fma(-s, s, x), h, s);
  return fma(fma(-s, s, x), h, s);
}

// EvaluateFlux1D, src/equation.f90:1014-1016
__device__ __forceinline__ void flux_1d(double h, double vx, double vy, double g, double& f1,
                                        double& f2, double& f3) {
  f1 = h * vx;
  f2 = h * (vx * vx) + (0.5 * g) * (h * h);
  f3 = (h * vx) * vy;
}

// RiemannSolver + RiemannSolverByRusanov at one Gauss point,
// src/equation.f90:1048-1069 and :1096-1103.  (n1,n2),(t1,t2) are the face's
// NormVect/TangVect (src/mesh.f90:74-110); they are compile-time constants
// here, and the products with 0 and 1 are kept as in the reference.
template <int N1, int N2, int T1, int T2>
__device__ __forceinline__ void rusanov(double hl, double ul, double vl, double hr, double ur,
                                        double vr, double g, double& F1, double& F2, double& F3) {
  const double n1 = N1, n2 = N2, t1 = T1, t2 = T2;
  double pl1 = hl, pl2 = n1 * ul + n2 * vl, pl3 = t1 * ul + t2 * vl;
  double pr1 = hr, pr2 = n1 * ur + n2 * vr, pr3 = t1 * ur + t2 * vr;
  double cl2 = pl1 * pl2, cl3 = pl1 * pl3;  // PrimToCons
  double cr2 = pr1 * pr2, cr3 = pr1 * pr3;
  double fl1, fl2, fl3, fr1, fr2, fr3;
  flux_1d(pl1, pl2, pl3, g, fl1, fl2, fl3);
  flux_1d(pr1, pr2, pr3, g, fr1, fr2, fr3);
  double fastl = pl2 + sqrt(g * pl1);
  double fastr = pr2 + sqrt(g * pr1);
  double lmax = max_r(fabs(fastl), fabs(fastr));
  double f1 = 0.5 * ((fl1 + fr1) - lmax * (pr1 - pl1));
  double f2 = 0.5 * ((fl2 + fr2) - lmax * (cr2 - cl2));
  double f3 = 0.5 * ((fl3 + fr3) - lmax * (cr3 - cl3));
  F1 = f1;
  F2 = n1 * f2 + t1 * f3;
  F3 = n2 * f2 + t2 * f3;
}

// The same flux by normal velocity n* and tangential velocity t*, for finite
// states with depths in the range of sqrt_regular: mass, normal and tangential
// momentum.  The rotation's products with 0 only fix signs of zeros here, and
// those die in the Gauss sum, which starts at +0; so they are left out, and
// hl*nl serves as conserved momentum and as mass flux.
__device__ __forceinline__ void rusanov_regular(double hl, double nl, double tl, double hr,
                                                double nr, double tr, double g, double& F1,
                                                double& Fn, double& Ft) {
  const double ml = hl * nl, mr = hr * nr;
  const double lmax =
      max_r(fabs(nl + sqrt_regular(g * hl)), fabs(nr + sqrt_regular(g * hr)));
  const double hg = 0.5 * g;
  F1 = 0.5 * ((ml + mr) - lmax * (hr - hl));
  Fn = 0.5 * (((hl * (nl * nl) + hg * (hl * hl)) + (hr * (nr * nr) + hg * (hr * hr))) -
              lmax * (mr - ml));
  Ft = 0.5 * ((ml * tl + mr * tr) - lmax * (hr * tr - hl * tl));
}

__device__ __forceinline__ bool is_finite(double a) {
  return __builtin_amdgcn_class(a, 0x1F8);  // zero, subnormal or normal
}

// JamesonIndicator, src/shocksindicator.f90:93-129, on the depths of three
// neighbouring cells.
__device__ __forceinline__ bool jameson_shock(double hm, double h0, double hp) {
  double ind = fabs(hm + hp - 2.0 * h0);
  ind = ind / (fabs(hm) + fabs(hp) + fabs(2.0 * h0));
  return ind > 0.5E-03;
}

// MINMOD, src/reconstruction.f90:387-402; SIGN(1.0, x) is copysign(1.0, x).
__device__ __forceinline__ double minmod(double x, double y) {
  return 0.5 * (copysign(1.0, x) + copysign(1.0, y)) * min_r(fabs(x), fabs(y));
}

// ReconstructionFixX/Y (src/reconstruction.f90:219-242, :298-321) for one
// variable of a flagged cell, from the cell's value q0 and its neighbours
// along the sweep direction: recfix 1 puts q0 at every Gauss point, 2 the
// MUSCL values (src/reconstruction.f90:348-381) with d = MESH_DX(dir).
__device__ __forceinline__ void reconstruction_fix(int recfix, double qm1, double q0, double qp1,
                                                   double d, double wm[4], double wp[4]) {
  double m = q0, p = q0;
  if (recfix == 2) {
    double sp = (qp1 - q0) / d;
    double sm = (q0 - qm1) / d;
    double slope = minmod(sm, sp);
    m = q0 - 0.5 * slope * d;
    p = q0 + 0.5 * slope * d;
  }
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    wm[g] = m;
    wp[g] = p;
  }
}

// PATANKAR_DIV, src/timediscretization.f90:913-924
__device__ __forceinline__ double patankar_div(double prod, double h) {
  if (h < kMinDepth) return 0.;
  return 2. * h * prod / (h * h + max_r(h * h, kMinDepth));
}

}  // namespace swm
