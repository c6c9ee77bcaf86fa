// Correctly rounded acos and sincos for the RMHD quartic's resolvent cubic
// (Src/RMHD/rmhd.hpp:441-444: theta = acos(arg)/3, cos(theta), sin(theta)).
//
// The reference's CPU build takes these from the host libm (glibc), whose
// acos, sin and cos return the correctly rounded double for all but a tiny
// fraction of arguments.  The device math library is faithful (about 1 ulp),
// so its last bit differs often, and the RMHD state drifts from the
// reference's at the 1e-12 level.  These routines compute the value to about
// 2^-100 relative accuracy in double-double arithmetic and round it once, so
// they return the correctly rounded double unless the exact value lies within
// ~2^-100 of a rounding midpoint.  The same source runs on the host (tests
// compare it with glibc on 1e8 arguments) and on the device.
//
// Method (the classical table + polynomial evaluation, e.g. Muller,
// "Elementary Functions: Algorithms and Implementation", ch. 6 and 11, with
// error-free transformations from Dekker 1971 and Ogita, Rump & Oishi 2005):
//  - sincos(x), 0 <= x <= 2.19: x = t_k + r with t_k = k/64 and |r| <= 1/128
//    (r exact by Sterbenz); sin(t_k), cos(t_k) as double-doubles from the
//    table; sin r and cos r by their Taylor series to r^11 and r^10, the two
//    leading correction terms in double-double; the addition formulas in
//    double-double.
//  - acos(x): one Newton step in double-double from the library's acos of
//    |x|, whose error (a few ulp) becomes ~2^-104 after the step.
//    |x| <= 1/2: theta = theta0 + (cos theta0 - x)/sin theta0.  |x| > 1/2:
//    acos x = 2 phi (x > 0) or pi - 2 phi (x < 0) with sin^2 phi = h =
//    (1 - |x|)/2 (exact), phi = phi0 - (sin^2 phi0 - h)/sin(2 phi0),
//    phi0 = acos(|x|)/2, which keeps full relative accuracy as x -> +-1.
// Both functions try a quick phase first: about 2^-73 in plain doubles with an
// error bound, and a test whether that decides the rounding.  It nearly always
// does, so the double-double evaluation is a branch that wavefronts skip.  RMHD
// HLL at 128^3, us per x, y, z sweep, which solve two quartics per face: 154, 194,
// 210 with double-double forms and the library's acos as the seed, 132, 169, 186
// with the quick phase and a seed of 2^-38 (the z sweep 229 where the compiler
// hoists the constants out of the march: mhd3d_fp64_nohoist.hip).
// Explicit fma() calls are the error-free products; they are exact on both
// sides regardless of -ffp-contract.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#include "crmath_table.hpp"

namespace gpl { namespace cr {

#define GPL_CR_HD __host__ __device__ __forceinline__

struct dd { double hi, lo; };

// Knuth's TwoSum: hi + lo == a + b exactly
GPL_CR_HD dd two_sum(double a, double b)
{
  const double s = a + b;
  const double bb = s - a;
  const double e = (a - (s - bb)) + (b - bb);
  return {s, e};
}
// Dekker's FastTwoSum, |a| >= |b|
GPL_CR_HD dd fast_two_sum(double a, double b)
{
  const double s = a + b;
  return {s, b - (s - a)};
}
// hi + lo == a*b exactly
GPL_CR_HD dd two_prod(double a, double b)
{
  const double p = a*b;
  return {p, fma(a, b, -p)};
}
GPL_CR_HD dd dd_add(dd a, dd b)
{
  dd s = two_sum(a.hi, b.hi);
  s.lo += a.lo + b.lo;
  return fast_two_sum(s.hi, s.lo);
}
GPL_CR_HD dd dd_mul(dd a, dd b)
{
  dd p = two_prod(a.hi, b.hi);
  p.lo += a.hi*b.lo + a.lo*b.hi;
  return fast_two_sum(p.hi, p.lo);
}
GPL_CR_HD dd dd_mul_d(dd a, double b)
{
  dd p = two_prod(a.hi, b);
  p.lo += a.lo*b;
  return fast_two_sum(p.hi, p.lo);
}

GPL_CR_HD const double *table_row(int k)
{
#if defined(__HIP_DEVICE_COMPILE__)
  return kSinCosDev[k];
#else
  return kSinCosHost[k];
#endif
}

// sin and cos of x, 0 <= x <= 2.19 (table index k <= 140), as double-doubles (~2^-100 relative for
// sin and cos away from their zeros; absolute ~2^-105 near cos's zero)
GPL_CR_HD void dd_sincos(double x, dd &s, dd &c)
{
  const int k = (int)(x*64.0 + 0.5);
  const double r = x - k*0.015625;               // exact
  const double zh = r*r, zl = fma(r, r, -zh);     // z = r^2 = zh + zl
  // sin r = r (1 + z (s1 + z (s2 + z (s3 + z (s4 + z s5)))))
  const double st = -1.0/5040.0 + zh*(1.0/362880.0 + zh*(-1.0/39916800.0));
  dd t = fast_two_sum(kS2Hi, zh*st);
  t.lo += kS2Lo;                                   // s2 + z st
  dd w = dd_mul(dd{zh, zl}, t);
  w = dd_add(dd{kS1Hi, kS1Lo}, w);                 // s1 + z (...)
  w = dd_mul(dd{zh, zl}, w);                       // z (...)
  const dd rw = dd_mul_d(w, r);                    // |r w| < 2^-16 |r|
  dd sr = fast_two_sum(r, rw.hi);
  sr.lo += rw.lo;                                  // sin r = r + r w
  // cos r = 1 + z (-1/2 + z (c2 + z (c3 + z (c4 + z c5)))), cw = cos r - 1
  const double ct = -1.0/720.0 + zh*(1.0/40320.0 + zh*(-1.0/3628800.0));
  dd u = fast_two_sum(kC2Hi, zh*ct);
  u.lo += kC2Lo;                                   // c2 + z ct
  u = dd_mul(dd{zh, zl}, u);
  u = dd_add(dd{-0.5, 0.0}, u);
  const dd cw = dd_mul(dd{zh, zl}, u);
  // addition formulas: sin x = S + S cw + C sin r, cos x = C + C cw - S sin r
  const double *row = table_row(k);
  const dd S{row[0], row[1]}, C{row[2], row[3]};
  s = dd_add(dd_add(S, dd_mul(S, cw)), dd_mul(C, sr));
  const dd msr{-sr.hi, -sr.lo};
  c = dd_add(dd_add(C, dd_mul(C, cw)), dd_mul(S, msr));
}

// The quick phase (Ziv's strategy; Muller, "Elementary Functions", ch. 10): sin
// and cos of x as unevaluated sums sh + sl and ch + cl with |sl| < 2^-23, in plain
// double arithmetic with exact products and sums where a rounding would count.
// With |r| <= 2^-7, the corrections being S cw + C r w for sin x (w = sin r/r - 1,
// cw = cos r - 1), the largest rounded terms are r w <= 2^-23.6 (relative error of
// w 2^-51.2: 2^-74.8) and the last addition (2^-76.6): absolute error below 2^-73.5
// for both; for k = 0 (S = 0, C = 1) sin x = r + r w has relative error below
// 2^-67.8.
struct sincos_sum { double sh, sl, ch, cl; int k; };
GPL_CR_HD sincos_sum quick_sincos(double x)
{
  sincos_sum q;
  q.k = (int)(x*64.0 + 0.5);
  const double r = x - q.k*0.015625;              // exact
  const double zh = r*r, zl = fma(r, r, -zh);
  const double w = zh*fma(zh, fma(zh, fma(zh, 1.0/362880.0, -1.0/5040.0), 1.0/120.0), -1.0/6.0);
  const double rw = r*w;
  const double hz = -0.5*zh;                       // cos r - 1 = hz + t
  const double t = fma(zh*zh, fma(zh, fma(zh, 1.0/40320.0, -1.0/720.0), 1.0/24.0), -0.5*zl);
  const double *row = table_row(q.k);
  const double S = row[0], Sl = row[1], C = row[2], Cl = row[3];
  {
    const dd p = two_prod(C, r), h = two_prod(S, hz);
    const dd a = fast_two_sum(S, p.hi);            // S >= |C r|, or S = 0 (k = 0)
    const dd b = fast_two_sum(a.hi, h.hi);
    double lo = fma(Sl, hz, fma(Cl, r, Sl));
    lo = fma(S, t, lo + (p.lo + h.lo)) + (a.lo + b.lo);
    q.sh = b.hi;
    q.sl = fma(C, rw, lo);
  }
  {
    const dd p = two_prod(S, -r), h = two_prod(C, hz);
    const dd a = two_sum(C, p.hi);                 // C passes through 0
    const dd b = two_sum(a.hi, h.hi);
    double lo = fma(Cl, hz, fma(Sl, -r, Cl));
    lo = fma(C, t, lo + (p.lo + h.lo)) + (a.lo + b.lo);
    q.ch = b.hi;
    q.cl = fma(-S, rw, lo);
  }
  return q;
}
constexpr double kE72 = 0x1p-72, kE71 = 0x1p-71, kE66 = 0x1p-66, kE65 = 0x1p-65;

// sin(x) and cos(x) correctly rounded for 0 <= x <= 2.19 (the resolvent
// cubic's theta lies in [0, pi/3]); other arguments (NaN) give NaN.
// The quick phase decides unless hi + (lo - e) and hi + (lo + e) round apart, e
// its error bound (about once in 2^14 arguments); then the double-double form.
GPL_CR_HD void sincos_cr(double x, double *sn, double *cs)
{
  if (!(x >= 0.0 && x <= 2.19)) { *sn = *cs = __builtin_nan(""); return; }
  const sincos_sum q = quick_sincos(x);
  const double es = q.k ? kE72 : q.sh*kE66;
  const double s1 = q.sh + (q.sl + es), c1 = q.ch + (q.cl + kE72);
  *sn = s1;
  *cs = c1;
  if (s1 == q.sh + (q.sl - es) && c1 == q.ch + (q.cl - kE72)) return;
  dd s, c;
  dd_sincos(x, s, c);
  *sn = s.hi + s.lo;
  *cs = c.hi + c.lo;
}

// The Newton step of acos_cr for -1 < x < 1 from its seed (acos_seed).  A
// seed a few ulp off still gives the correctly rounded result (the step
// squares its relative error).  Both forms of the step are evaluated from one
// double-double sincos of the seed and the right one is selected, so lanes of
// a wavefront that take different forms do not run the expensive part twice.
//  |x| <= 1/2: theta = theta0 + (cos theta0 - x)/sin theta0, theta0 in [pi/3, 2pi/3];
//  |x| >  1/2: acos x = 2 phi (x > 0) or pi - 2 phi (x < 0) with sin^2 phi = h =
//              (1 - |x|)/2 (exact), phi = phi0 - (sin^2 phi0 - h)/sin(2 phi0),
//              phi0 in (0, pi/6], which keeps full relative accuracy as x -> +-1.
GPL_CR_HD double acos_refine(double x, double seed)
{
  dd s, c;
  dd_sincos(seed, s, c);
  const double d1 = (c.hi - x) + c.lo;             // cos t0 - x
  const double r_mid = seed + d1/s.hi;
  const double h = (1.0 - fabs(x))*0.5;            // sin^2 phi, exact
  const dd s2 = dd_mul(s, s);
  const double d2 = (s2.hi - h) + s2.lo;           // sin^2 phi0 - h
  const double delta = -d2/(2.0*s.hi*c.hi);
  const double r_pos = 2.0*(seed + delta);         // exact doubling of RN(phi)
  dd t = two_sum(kPiHi, -2.0*seed);                // pi - 2 phi
  t.lo += kPiLo - 2.0*delta;
  const double r_neg = t.hi + t.lo;
  return fabs(x) <= 0.5 ? r_mid : (x > 0.0 ? r_pos : r_neg);
}

// The seed of the Newton step from one library acos of |x| (a few ulp):
// theta0 = acos x for |x| <= 1/2, phi0 = acos(|x|)/2 otherwise.
GPL_CR_HD double acos_seed(double x)
{
  const double t = acos(fabs(x));
  if (fabs(x) <= 0.5) return x >= 0.0 ? t : kPiHi - t;
  return 0.5*t;
}

// 1/x and sqrt(x) to about 2^-44 for the places below that need no more: on the
// device the hardware's estimate (2^-23) and one Newton step instead of the IEEE
// sequences.  x is positive and far from the ends of the range.  RMHD HLL sweeps of
// 64^3, us: x 23.9 -> 22.7, y 26.7 -> 25.9.
GPL_CR_HD double near_rcp(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
  const double r = __builtin_amdgcn_rcp(x);
  return fma(fma(-x, r, 1.0), r, r);
#else
  return 1.0/x;
#endif
}
GPL_CR_HD double near_sqrt(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
  const double r = __builtin_amdgcn_rsq(x), z = x*r;
  return fma(fma(-z, z, x), 0.5*r, z);
#else
  return sqrt(x);
#endif
}

// A seed for the quick phase, one polynomial for either form: asin(z) = z + z y P(y),
// y = z^2 <= 1/4, with z = |x| or sqrt((1 - |x|)/2), P the Chebyshev interpolant of
// degree 7 of (asin(z)/z - 1)/y (relative error of the seed 2^-38).
GPL_CR_HD double quick_acos_seed(double x)
{
  const double ax = fabs(x), h = (1.0 - ax)*0.5;
  const bool mid = ax <= 0.5;
  const double y = mid ? x*x : h;
  const double z = mid ? x : near_sqrt(h);
  double P = 0.02930523970533579;
  P = fma(P, y, 0.0054431851027481075);
  P = fma(P, y, 0.019306260869368045);
  P = fma(P, y, 0.022132443623426794);
  P = fma(P, y, 0.030397634130580702);
  P = fma(P, y, 0.044642358484883196);
  P = fma(P, y, 0.07500000598829049);
  P = fma(P, y, 0.16666666665495086);
  const double a = fma(z*y, P, z);
  return mid ? kPiHi*0.5 - a : a;
}

// The same step from the quick phase, with one division for either form; false
// if the bound of its error leaves two roundings.  The step's own second-order
// term is below 2^-77 (relative to phi for |x| > 1/2).  |x| <= 1/2: the error of cos
// over sin theta >= 0.86, below 2^-73.  |x| > 1/2: that of sin^2 over sin 2 phi,
// below 2^-73, for k = 0 phi 2^-67.8.
GPL_CR_HD bool quick_acos(double x, double seed, double *res)
{
  const sincos_sum q = quick_sincos(seed);
  const dd s = fast_two_sum(q.sh, q.sl);
  const double ax = fabs(x), h = (1.0 - ax)*0.5;
  const bool mid = ax <= 0.5;
  dd s2 = two_prod(s.hi, s.hi);
  s2.lo += 2.0*s.hi*s.lo;
  const double num = mid ? (q.ch - x) + q.cl : (h - s2.hi) - s2.lo;
  const double den = mid ? s.hi : 2.0*s.hi*(q.ch + q.cl);
  const double delta = num*near_rcp(den);       // below 2^-38 seed, so to 2^-80 of it
  const double e = q.k ? kE71 : seed*kE65;
  const bool neg = !mid && x < 0.0;
  dd t = two_sum(kPiHi, -2.0*seed);
  t.lo += kPiLo - 2.0*delta;
  const double hi = neg ? t.hi : seed, lo = neg ? t.lo : delta, err = neg ? 2.0*e : e;
  const double r1 = hi + (lo + err), r2 = hi + (lo - err);
  *res = !mid && !neg ? 2.0*r1 : r1;
  return r1 == r2;
}

// acos(x) correctly rounded for -1 <= x <= 1, else NaN.
GPL_CR_HD double acos_cr(double x)
{
  if (!(x >= -1.0 && x <= 1.0)) return __builtin_nan("");
  if (x == 1.0) return 0.0;
  if (x == -1.0) return kPiHi;
  double r;
  if (quick_acos(x, quick_acos_seed(x), &r)) return r;
  return acos_refine(x, acos_seed(x));
}

#undef GPL_CR_HD

}}  // namespace gpl::cr
