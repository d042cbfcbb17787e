// iz_math.h -- FP64 exp, log and reciprocal of the kinetics and transport
// kernels.
//
// These kernels evaluate tens of exponentials per cell and call with
// arguments of moderate size, so what they pay in a general library function
// is the handling of its corner cases.  The forms here are the textbook
// ones: Cody and Waite's two-part reduction by ln 2 with a polynomial in the
// remainder (exp), and log m = 2 artanh((m - 1) / (m + 1)) (log); the
// polynomials interpolate at Chebyshev points, with relative errors below
// 2e-18 (exp, degree 11 on |r| <= ln 2 / 2) and 2e-17 (log).  Against exact
// values they are within 0.8 ulp (exp) and 1.1 ulp (log) over the ranges below
// (tests/test_math_cpu.py; the host library: 0.5 ulp).
//   d_exp   any finite x up to 1e9 in magnitude: overflow to inf and
//           underflow through the denormals to 0 as exp; NaN to NaN
//   d_log   x > 0 finite; NaN otherwise
//   d_rcp   1 / x by Newton's iteration for finite nonzero x whose
//           reciprocal is finite and normal, within 1 ulp; 0, inf and NaN
//           give NaN
#pragma once

#include <math.h>

#ifndef IZ_HD
#define IZ_HD __device__
#endif

IZ_HD inline double d_rcp(double x) {
#ifdef __HIP_DEVICE_COMPILE__
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
#else
  return 1.0 / x;
#endif
}

// e with |x| = m 2^e, 1/2 <= m < 1, for finite nonzero x
IZ_HD inline int d_exponent(double x) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_frexp_exp(x);
#else
  int e;
  (void)frexp(x, &e);
  return e;
#endif
}

IZ_HD inline double d_exp(double x) {
  const double t = rint(x * 1.4426950408889634);
  const double a = fma(t, -0.6931471803691238, x);
  const double r = fma(t, -1.9082149292705877e-10, a);
  double p = 2.5100424157005067e-08;
  p = fma(p, r, 2.7620138719733994e-07);
  p = fma(p, r, 2.7557268378684192e-06);
  p = fma(p, r, 2.480152119021773e-05);
  p = fma(p, r, 0.00019841269863105968);
  p = fma(p, r, 0.0013888888917281794);
  p = fma(p, r, 0.008333333333330051);
  p = fma(p, r, 0.04166666666662399);
  p = fma(p, r, 0.16666666666666669);
  p = fma(p, r, 0.5000000000000001);
  // 1 + r + r^2 p with the roundings of r and of 1 + r put back
  const double s = 1.0 + r, dr = fma(t, -1.9082149292705877e-10, a - r);
  p = s + fma(r * r, p, ((1.0 - s) + r) + dr);
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_ldexp(p, (int)t);
#else
  return (x != x) ? x : ldexp(p, t > 4e3 ? 4000 : (t < -4e3 ? -4000 : (int)t));
#endif
}

IZ_HD inline double d_log(double x) {
  int e;
  double m = frexp(x, &e);
  const bool low = m < 0.70710678118654752;
  m = low ? m + m : m;
  e = low ? e - 1 : e;
  const double n = m - 1.0, d = m + 1.0, r = d_rcp(d);
  double s = n * r;
  s = fma(fma(-d, s, n), r, s);
  const double z = s * s, k = (double)e;
  double p = 0.13088034850927555;
  p = fma(p, z, 0.13268638369266825);
  p = fma(p, z, 0.15386244737621665);
  p = fma(p, z, 0.18181795547521137);
  p = fma(p, z, 0.22222222392581045);
  p = fma(p, z, 0.28571428570799784);
  p = fma(p, z, 0.40000000000000885);
  p = fma(p, z, 0.6666666666666666);
  // 2 s = n - s n with n exact: the rounding of s enters through s n only
  const double l = fma(s, fma(z, -p, n), k * -1.9082149292705877e-10);
  return x > 0.0 ? fma(k, 0.6931471803691238, n - l) : NAN;
}
