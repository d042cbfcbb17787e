// iz_weno.h -- the WENO5 face reconstruction of izem_flux_mode 1 with one
// reciprocal (device code, host-compilable for the tests).
#pragma once

#include "iz_math.h"

// module_weno.f90:114-190
#define IZ_Z1 (13.0 / 12.0)
#define IZ_Z2 (1.0 / 4.0)
#define IZ_EPS_WENO 1.0e-10

// gl + gr of a face from the split fluxes scaled by two, gp2 = g + lam w and
// gm2 = g - lam w: what wenorec (js) or wenorec_nw gives for gp2 / 2 and
// gm2 / 2, added.  The smoothness indicators scale with the square, so eps
// does too.  The weights are brought to a common denominator, which leaves
// one reciprocal of the eight divisions; its terms, products of eight
// indicators and a flux, are finite for fluxes up to 1e17 times the unit
// scale.  Where a result is not finite the caller asks again with WIDE.

// one side: q[0..4] in its upwind order
struct IzWeno5 {
  double t0, t1, t2;  // eps + smoothness indicators of candidates q2 q3 q4, q1 q2 q3, q0 q1 q2
  double v0, v1, v2;  // the candidates, times 6
};
IZ_HD inline IzWeno5 d_weno5_side(double q0, double q1, double q2, double q3, double q4) {
#pragma clang fp contract(on)
  const double e4 = 4.0 * IZ_EPS_WENO;
  const double a0 = (q2 + q4) - 2.0 * q3, b0 = 3.0 * q2 - 4.0 * q3 + q4;
  const double a1 = (q1 + q3) - 2.0 * q2, b1 = q1 - q3;
  const double a2 = (q0 + q2) - 2.0 * q1, b2 = q0 - 4.0 * q1 + 3.0 * q2;
  IzWeno5 s;
  s.t0 = IZ_Z1 * (a0 * a0) + (IZ_Z2 * (b0 * b0) + e4);
  s.t1 = IZ_Z1 * (a1 * a1) + (IZ_Z2 * (b1 * b1) + e4);
  s.t2 = IZ_Z1 * (a2 * a2) + (IZ_Z2 * (b2 * b2) + e4);
  s.v0 = 2.0 * q2 + (5.0 * q3 - q4);
  s.v1 = 5.0 * q2 + (2.0 * q3 - q1);
  s.v2 = 11.0 * q2 + (2.0 * q0 - 7.0 * q1);
  return s;
}
// its numerator and denominator of the weighted candidates
IZ_HD inline void d_weno5_sums(IzWeno5 s, double &num, double &den) {
#pragma clang fp contract(on)
  s.t0 = s.t0 * s.t0;
  s.t1 = s.t1 * s.t1;
  s.t2 = s.t2 * s.t2;
  const double w0 = 3.0 * (s.t1 * s.t2), w1 = 6.0 * (s.t0 * s.t2), w2 = s.t0 * s.t1;
  den = w0 + w1 + w2;
  num = w0 * s.v0 + w1 * s.v1 + w2 * s.v2;
}
// a side of a face with large fluxes: the indicators scaled by the power of
// two that brings their sum into [1/2, 1), which cancels in the quotient.
// Finite up to 1e70 (the reference's form: 1e76).
IZ_HD inline double d_weno5_side_wide(double q0, double q1, double q2, double q3, double q4) {
  IzWeno5 s = d_weno5_side(q0, q1, q2, q3, q4);
  const int e = -d_exponent(s.t0 + s.t1 + s.t2);
  s.t0 = ldexp(s.t0, e);
  s.t1 = ldexp(s.t1, e);
  s.t2 = ldexp(s.t2, e);
  double num, den;
  d_weno5_sums(s, num, den);
  return num / den;
}
// WIDE: the same face for fluxes beyond the range above
template <bool WIDE>
IZ_HD inline double d_weno5_face_fused(bool js, const double *gp, const double *gm) {
#pragma clang fp contract(on)
  if (js) {
    if constexpr (WIDE)
      return (d_weno5_side_wide(gp[0], gp[1], gp[2], gp[3], gp[4]) +
              d_weno5_side_wide(gm[5], gm[4], gm[3], gm[2], gm[1])) * (1.0 / 12.0);
    double n1, d1, n2, d2;
    d_weno5_sums(d_weno5_side(gp[0], gp[1], gp[2], gp[3], gp[4]), n1, d1);
    d_weno5_sums(d_weno5_side(gm[5], gm[4], gm[3], gm[2], gm[1]), n2, d2);
    return (n1 * d2 + n2 * d1) * (d_rcp(d1 * d2) * (1.0 / 12.0));
  }
  const double a = 2.0 * (gp[4] + gm[1]) - 13.0 * (gp[3] + gm[2]) + 47.0 * (gp[2] + gm[3]) +
                   27.0 * (gp[1] + gm[4]) - 3.0 * (gp[0] + gm[5]);
  return a * (1.0 / 120.0);
}
