// flow.hip -- FP64 HIP kernels of the IZEM reacting-flow right-hand side and
// SSP-RK3 time step for CDNA4 (gfx950).
//
// Compiled with -ffp-contract=off.  The Euler faces of izem_flux_mode 0, the
// WENO7 build's other kernels, the stencils and the stage update evaluate the
// reference's expressions in the reference's order, so their results are the
// reference algorithm's own roundings.  With ng = 3 the Newton inversion and
// the transport properties (in either flux mode) and the Euler faces of mode
// 1 are re-associated and contracted where a pragma says so: they agree with
// the reference to rounding.  Reference: saras13015/Phd devel-izem/src
// (file:line cited per kernel).
#include "flow_device.h"
#include "iz_math.h"
#include "izem_ctx.h"

#include <stdlib.h>
#include <string.h>
#include <type_traits>
#include <utility>

__constant__ IzThd c_thd;
__constant__ IzThx c_thx;

// ===================================================================
// Euler fluxes (euler_LLF_x/_y/_z: module_weno.f90:537-1044, 1055-1584,
// 1595-2118): one thread per cell face in 256-thread blocks.  The cells of
// a block's stencils are staged once in LDS, with the per-cell quantities
// every stencil point needs (u_n, P, c), so a cell is read from HBM once per
// block instead of once per face and stencil point:
//   x:    each wave takes 64 consecutive faces of the (face, j, k) order
//         (they may wrap into the next row); its tile is the run of cells
//         their stencils cover;
//   y, z: a block takes IZ_EU_TX cells along x by IZ_EU_TF faces along the
//         direction and stages IZ_EU_TF + 5 cell rows; logical tiles are
//         numbered so that tiles adjacent along the direction run on the
//         same XCD, whose L2 then serves the shared halo rows.
// The face value F^ of the 14 equations goes to a face array; the flux
// difference is a separate pass (k_euler_apply).
// ===================================================================
#define IZ_EU_BLOCK 256
#define IZ_EU_TX 32
#define IZ_EU_TF (IZ_EU_BLOCK / IZ_EU_TX)
#define IZ_EU_ROWS (IZ_EU_TF + IZ_S - 1)
#define IZ_EU_NQ (IZ_NV + 3)  // staged per cell: the conserved variables, u_n, P, c
#define IZ_QU IZ_NV           // staged slots of u_n, P, c
#define IZ_QP (IZ_NV + 1)
#define IZ_QC (IZ_NV + 2)
#ifndef IZ_EULER_WAVES
#define IZ_EULER_WAVES 2
#endif
#ifndef IZ_EULER_FAST_WAVES
#define IZ_EULER_FAST_WAVES 2
#endif

// per-cell part of the stencil presolve (module_weno.f90:634-650), with the
// expressions of the per-stencil loop evaluated once per cell
__device__ inline void eu_stage_cell(const double *__restrict__ v, const double *__restrict__ T,
                                     const double *__restrict__ W_i,
                                     const double *__restrict__ cp, long nc, long c, int cn,
                                     double *dst, int fs, int &neg) {
  const double r0 = v[c];
  const double rho_i = 1.0 / r0;
  dst[0] = r0;
#pragma unroll
  for (int l = 1; l < IZ_NV; l++) dst[l * fs] = v[l * nc + c];
  const double un = v[cn * nc + c] * rho_i;
  const double P = r0 * T[c] * W_i[c];
  if (P <= 0.0) neg = 1;
  double gam = c_thd.gam2 * W_i[c] / cp[c];
  gam = 1.0 / (1.0 - gam);
  const double cs = sqrt(gam * P * rho_i);
  dst[IZ_QU * fs] = un;
  dst[IZ_QP * fs] = P;
  dst[IZ_QC * fs] = cs;
}

// rows of the left eigenvector matrix projected together (eu_face_ref):
// the sums of four fit the registers of two waves per SIMD with six stencil
// points (244 VGPRs), those of two with eight
#define IZ_EU_GROUP (IZ_NG == 3 ? 4 : 2)
template <int M>
using EuRow = std::integral_constant<int, M>;
template <int M0, class F, int... I>
__device__ inline void eu_row_group(F &f, std::integer_sequence<int, I...>) {
  f(EuRow<M0 + I>{}...);
}
// f on the rows M0 .. IZ_NV - 1, a group at a time
template <int M0, class F>
__device__ inline void eu_species_rows(F &f) {
  if constexpr (M0 < IZ_NV) {
    constexpr int G = IZ_NV - M0 < IZ_EU_GROUP ? IZ_NV - M0 : IZ_EU_GROUP;
    eu_row_group<M0>(f, std::make_integer_sequence<int, G>{});
    eu_species_rows<M0 + G>(f);
  }
}

// F^ of one face from its IZ_S staged stencil cells: Q(q, st) is staged
// quantity q of stencil point st (st = ng - 1 is i_l, st = ng is i_r); cL, cR are
// the HBM indices of i_l, i_r (for h_k); F^ goes to F[m * nfaces + fidx].
// The reference's dense projections (w = el . U, g = el . F over all 14
// columns, in its summation order: bit parity with the oracle).  SITE gives every calling
// kernel an instantiation of its own: with a single caller each is inlined
// as before, where a shared one is left out of line.
template <int DIR, int QS, int SS, int SITE>
__device__ inline void eu_face_ref(const double *tile, int off, bool js,
                               const double *__restrict__ ha, long nc, long cL, long cR,
                               double *__restrict__ F, long nfaces, long fidx) {
  // staged quantity q of stencil point st
  auto Q = [&](int q, int st) { return tile[off + q * QS + st * SS]; };
  constexpr int cn = 1 + DIR;             // normal momentum column
  constexpr int t1 = (DIR == 0) ? 2 : 1;  // tangential columns (el rows 4, 5)
  constexpr int t2 = (DIR == 2) ? 2 : 3;
  double lmax0 = -1.0, lmax1 = -1.0, lmax2 = -1.0;
#pragma unroll
  for (int st = 0; st < IZ_S; st++) {
    const double u = Q(IZ_QU, st), cs = Q(IZ_QC, st);
    lmax0 = fmax(fabs(u - cs), lmax0);
    lmax1 = fmax(fabs(u), lmax1);
    lmax2 = fmax(fabs(u + cs), lmax2);
  }
  // Roe average of i_l and i_r (module_weno.f90:654-667, 726-735)
  double uc[3], Yc[IZ_NRV], ht_c, et_c, r, r1;
  {
    constexpr int SL = IZ_NG - 1, SR = IZ_NG;  // stencil points of i_l, i_r
    const double riL = 1.0 / Q(0, SL), riR = 1.0 / Q(0, SR);
    double uL[3], uR[3];
#pragma unroll
    for (int q = 0; q < 3; q++) { uL[q] = Q(1 + q, SL) * riL; uR[q] = Q(1 + q, SR) * riR; }
    double htL = 0.0, htR = 0.0;
    r = sqrt(Q(0, SR) * riL);
    r1 = 1.0 / (r + 1.0);
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++) {
      const double yL = Q(IZ_NIV + l, SL) * riL, yR = Q(IZ_NIV + l, SR) * riR;
      htL = htL + ha[l * nc + cL] * yL;
      htR = htR + ha[l * nc + cR] * yR;
      Yc[l] = (r * (yR) + yL) * r1;
    }
    htL = htL + 0.5 * (uL[0] * uL[0] + uL[1] * uL[1] + uL[2] * uL[2]);
    htR = htR + 0.5 * (uR[0] * uR[0] + uR[1] * uR[1] + uR[2] * uR[2]);
    const double etL = Q(4, SL) * riL, etR = Q(4, SR) * riR;
#pragma unroll
    for (int q = 0; q < 3; q++) uc[q] = (r * uR[q] + uL[q]) * r1;
    ht_c = (r * htR + htL) * r1;
    et_c = (r * etR + etL) * r1;
  }
  // EOS-compatible average state (module_weno.f90:750-761)
  const double W_i_c = d_wmix_scalar(Yc);
  const double T_c = (ht_c - et_c) / W_i_c;
  const double cp_c = d_cp_scalar(T_c, Yc);
  double gam_c = c_thd.gam2 * W_i_c / cp_c;
  gam_c = 1.0 / (1.0 - gam_c);
  const double cs_c = sqrt(gam_c * T_c * W_i_c);
  double psi[IZ_NRV];
  {
    double ha_c[IZ_NRV];
    d_ha_scalar(T_c, ha_c);
    const double wrk = (gam_c / (gam_c - 1.0)) * T_c;
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++) {
      psi[l] = -(r * ha_c[l] + ha_c[l]) * r1;
      psi[l] = psi[l] + wrk * c_thd.Wc_i[l];
    }
  }
  const double cs_c_i = 1.0 / cs_c, cs_c_2 = cs_c * cs_c;
  const double ux_c = uc[0], vy_c = uc[1], wz_c = uc[2];
  const double q = 0.5 * (ux_c * ux_c + vy_c * vy_c + wz_c * wz_c);
  const double b2 = (gam_c - 1.0) / cs_c_2;
  const double b1 = b2 * q;
  const double xi = b1 - b2 * ht_c;
  const double un_c = uc[cn - 1];
  const double hb2 = 0.5 * b2;

  // entry (m, c) of the left eigenvector matrix (module_weno.f90:775-874),
  // rows 3 and 4 excepted (two nonzeros, below)
  auto el = [&](auto mc, int c) -> double {
    constexpr int m = decltype(mc)::value;
    if constexpr (m == 0 || m == 2) {
      if (c == 0) return m == 0 ? 0.5 * (b1 + un_c * cs_c_i) : 0.5 * (b1 - un_c * cs_c_i);
      if (c == cn)
        return m == 0 ? -0.5 * (b2 * uc[c - 1] + cs_c_i) : -0.5 * (b2 * uc[c - 1] - cs_c_i);
      if (c <= 3) return -0.5 * (b2 * uc[c - 1]);
      if (c == 4) return 0.5 * b2;
      return hb2 * psi[c - IZ_NIV];
    } else if constexpr (m == 1) {
      if (c == 0) return 1.0 - b1;
      if (c <= 3) return b2 * uc[c - 1];
      if (c == 4) return -b2;
      const double a = hb2 * psi[c - IZ_NIV];
      return -a - a;
    } else if constexpr (m == 5) {
      const double opx = (1 + xi);
      if (c == 0) return opx * q;
      if (c <= 3) return -opx * uc[c - 1];
      if (c == 4) return opx;
      return xi * psi[c - IZ_NIV];
    } else {
      const double y = Yc[m - 6];
      if (c == 0) return -b1 * y;
      if (c <= 3) return b2 * uc[c - 1] * y;
      if (c == 4) return -b2 * y;
      const double x = -((b2 * y) * psi[c - IZ_NIV]);
      return c - IZ_NIV == m - 6 ? x + 1.0 : x;
    }
  };
  double ghat[IZ_NV];
  // Characteristic fields M of one group: w = el . U and g = el . F of every
  // stencil point, summed column by column (each sum in the reference's
  // order).  A staged value and its flux are read and formed once for the
  // group, so the LDS, which held this kernel up with one row at a time, is
  // read a group's size less often: 1.68 -> 1.35 (x), 1.82 -> 1.40 (y, z) ms
  // per launch at 160^3; groups of two 1.47 and 1.54.  The opaque offset keeps
  // the compiler from carrying a group's reads to the next one in registers.
  auto project = [&](auto... M) {
    constexpr int G = sizeof...(M);
    int offm = off;
    asm volatile("" : "+v"(offm));
    auto Qm = [&](int q, int st) { return tile[offm + q * QS + st * SS]; };
    double w[G][IZ_S], g[G][IZ_S], u[IZ_S], p[IZ_S];
#pragma unroll
    for (int st = 0; st < IZ_S; st++) {
      u[st] = Qm(IZ_QU, st);
      p[st] = Qm(IZ_QP, st);
    }
#pragma unroll
    for (int c = 0; c < IZ_NV; c++) {
      const double e[G] = {el(M, c)...};
#pragma unroll
      for (int st = 0; st < IZ_S; st++) {
        const double v = Qm(c, st);
        double f;
        if (c == 0) f = Qm(cn, st);
        else if (c == cn) f = v * u[st] + p[st];
        else if (c == 4) f = u[st] * (v + p[st]);
        else f = v * u[st];
#pragma unroll
        for (int k = 0; k < G; k++) {
          w[k][st] = c == 0 ? e[k] * v : w[k][st] + e[k] * v;
          g[k][st] = c == 0 ? e[k] * f : g[k][st] + e[k] * f;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // the sums are complete here: left to itself the compiler moves a row's
    // additions past the reconstruction of the rows before and spills the terms
#pragma unroll
    for (int k = 0; k < G; k++)
#pragma unroll
      for (int st = 0; st < IZ_S; st++) asm volatile("" : "+v"(w[k][st]), "+v"(g[k][st]));
    constexpr int rows[G] = {decltype(M)::value...};
#pragma unroll
    for (int k = 0; k < G; k++) {
      const double lam = rows[k] == 0 ? lmax0 : rows[k] == 2 ? lmax2 : lmax1;
      double gp[IZ_S], gm[IZ_S];
#pragma unroll
      for (int st = 0; st < IZ_S; st++) {
        gp[st] = 0.5 * (g[k][st] + lam * w[k][st]);
        gm[st] = g[k][st] - gp[st];
      }
      double gl, gr;
      d_weno_face(js, gp, gm, gl, gr);
      ghat[rows[k]] = gl + gr;
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if constexpr (IZ_EU_GROUP == 4) {
    project(EuRow<0>{}, EuRow<1>{}, EuRow<2>{}, EuRow<5>{});
  } else {
    project(EuRow<0>{}, EuRow<2>{});
    project(EuRow<1>{}, EuRow<5>{});
  }
  eu_species_rows<6>(project);
  // rows 3 and 4: a tangential momentum and the mass
#pragma unroll
  for (int m = 3; m <= 4; m++) {
    int offm = off;
    asm volatile("" : "+v"(offm));
    auto Qm = [&](int q, int st) { return tile[offm + q * QS + st * SS]; };
    const int tc = (m == 3) ? t1 : t2;
    const double et0 = -uc[tc - 1];
    double gp[IZ_S], gm[IZ_S];
#pragma unroll
    for (int st = 0; st < IZ_S; st++) {
      const double u = Qm(IZ_QU, st);
      const double v0 = Qm(0, st), vt = Qm(tc, st);
      const double f0 = Qm(cn, st), ft = vt * u;
      const double wc = et0 * v0 + vt, gc = et0 * f0 + ft;
      gp[st] = 0.5 * (gc + lmax1 * wc);
      gm[st] = gc - gp[st];
    }
    double gl, gr;
    d_weno_face(js, gp, gm, gl, gr);
    ghat[m] = gl + gr;
  }

  // F^ = er . ghat with the nonzero pattern of er (module_weno.f90:881-989)
  double fh;
  fh = ghat[0] + ghat[1];
  fh = fh + ghat[2];
  F[fidx] = fh;
#pragma unroll
  for (int c = 1; c <= 3; c++) {
    const double u = uc[c - 1];
    const double e0 = (c == cn) ? u - cs_c : u;
    const double e2 = (c == cn) ? u + cs_c : u;
    fh = e0 * ghat[0] + u * ghat[1];
    fh = fh + e2 * ghat[2];
    if (c == t1) fh = fh + ghat[3];
    if (c == t2) fh = fh + ghat[4];
    F[(long)c * nfaces + fidx] = fh;
  }
  fh = (ht_c - un_c * cs_c) * ghat[0] + q * ghat[1];
  fh = fh + (ht_c + un_c * cs_c) * ghat[2];
  fh = fh + uc[t1 - 1] * ghat[3];
  fh = fh + uc[t2 - 1] * ghat[4];
  fh = fh + ghat[5];
  F[4 * nfaces + fidx] = fh;
#pragma unroll
  for (int l = 0; l < IZ_NRV - 1; l++) {
    fh = Yc[l] * ghat[0] + Yc[l] * ghat[2];
    fh = fh + ghat[6 + l];
    F[(long)(IZ_NIV + l) * nfaces + fidx] = fh;
  }
  {
    const double wrk = -1.0 / psi[IZ_NRV - 1];
    fh = Yc[IZ_NRV - 1] * ghat[0] + Yc[IZ_NRV - 1] * ghat[2];
    fh = fh + wrk * ghat[5];
#pragma unroll
    for (int l = 0; l < IZ_NRV - 1; l++) fh = fh + (wrk * psi[l]) * ghat[6 + l];
    F[(long)(IZ_NV - 1) * nfaces + fidx] = fh;
  }
}

// The same face through the structure of el (izem_flux_mode 1): with
//   S = -b1 U_0 + b2 (u . m) - b2 E - b2 sum_l psi_l U_l   (and the same of F)
// every row but the tangential ones is S-plus-few-terms: row 1 is U_0 + S,
// rows 0 and 2 are -S/2 -+ (u_n U_0 - U_n) / (2 c), row 5 is
// -(1 + xi) / b2 S - sum_l psi_l U_l, and species row 6 + s is U_{5+s} + Y_s S.
// The characteristic projections then cost about a tenth of the dense ones.
// FMA contraction, the folded thermodynamic polynomials and one reciprocal
// per reconstructed field; fields are taken one after the other and enter F^
// as they come, so that few of them are live at a time: 204 VGPRs, two waves
// per SIMD (three or four spill: 3.6 and 4.3 ms).  The kernel is bound by FP64
// issue: 4.5 -> 2.0 (x), 2.2 (y, z) ms per launch at 256^3.  Results
// differ from the dense order by rounding only.
template <int DIR, int QS, int SS, int SITE, bool WIDE = false>
__device__ __forceinline__ void eu_face_fast(const double *tile, int off, bool js,
                                    const double *__restrict__ ha, long nc, long cL, long cR,
                                    double *__restrict__ F, long nfaces, long fidx) {
#pragma clang fp contract(on)
  // The stencil is read from LDS again by every field: an opaque copy of the
  // offset, taken anew by fresh(), keeps the compiler from holding the values
  // of an earlier reading in registers (which spills), and the scheduling
  // barrier from moving a field's reads ahead of the fields before it.
  int offm = off;
  auto fresh = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+v"(offm));
  };
  auto Q = [&](int q, int st) { return tile[offm + q * QS + st * SS]; };
  constexpr int cn = 1 + DIR;             // normal momentum column
  constexpr int t1 = (DIR == 0) ? 2 : 1;  // tangential columns (el rows 4, 5)
  constexpr int t2 = (DIR == 2) ? 2 : 3;
  // Roe average of i_l and i_r (module_weno.f90:654-667, 726-735)
  double uc[3], Yc[IZ_NRV], ht_c, et_c;
  {
    constexpr int SL = IZ_NG - 1, SR = IZ_NG;  // stencil points of i_l, i_r
    const double riL = 1.0 / Q(0, SL), riR = 1.0 / Q(0, SR);
    const double r = sqrt(Q(0, SR) * riL);
    const double r1 = 1.0 / (r + 1.0), r2 = r * r1;
    double htL = 0.0, htR = 0.0, kL = 0.0, kR = 0.0;
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++) {
      const double yL = Q(IZ_NIV + l, SL) * riL, yR = Q(IZ_NIV + l, SR) * riR;
      htL += ha[l * nc + cL] * yL;
      htR += ha[l * nc + cR] * yR;
      Yc[l] = r2 * yR + r1 * yL;
    }
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const double uL = Q(1 + q, SL) * riL, uR = Q(1 + q, SR) * riR;
      kL += uL * uL;
      kR += uR * uR;
      uc[q] = r2 * uR + r1 * uL;
    }
    ht_c = r2 * (htR + 0.5 * kR) + r1 * (htL + 0.5 * kL);
    et_c = r2 * (Q(4, SR) * riR) + r1 * (Q(4, SL) * riL);
  }
  // EOS-compatible average state (module_weno.f90:750-761)
  double W_i_c = 0.0;
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) W_i_c += Yc[l] * c_thd.Wc_i[l];
  const double T_c = (ht_c - et_c) / W_i_c;
  double cp_c, psi[IZ_NRV];
#if IZ_NG == 3
  if (d_thermo_in_range(T_c)) {
    d_thermo(T_c, Yc, cp_c, psi);
  } else
#endif
  {
    cp_c = d_cp_scalar(T_c, Yc);
    d_ha_scalar(T_c, psi);
  }
  const double gam_c = 1.0 / (1.0 - c_thd.gam2 * W_i_c / cp_c);
  const double cs_c_2 = gam_c * T_c * W_i_c;
  const double cs_c = sqrt(cs_c_2);
  {
    const double wrk = (gam_c / (gam_c - 1.0)) * T_c;
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++) psi[l] = wrk * c_thd.Wc_i[l] - psi[l];
  }
  const double hc = 0.5 / cs_c;
  const double q = 0.5 * (uc[0] * uc[0] + uc[1] * uc[1] + uc[2] * uc[2]);
  const double b2 = (gam_c - 1.0) / cs_c_2;
  const double b1 = b2 * q;
  const double un_c = uc[cn - 1];
  fresh();
  double lmax0 = 0.0, lmax1 = 0.0, lmax2 = 0.0;
  double u[IZ_S], sw[IZ_S], sg[IZ_S];
  double gp[IZ_S], gm[IZ_S], g0, g1, g2, g5;
  {
    // per stencil point, S and sum_l psi_l U_l of U and of F, and u_n U_0 -
    // U_n with its F counterpart
    double pw[IZ_S], dw[IZ_S], dg[IZ_S];
#pragma unroll
    for (int st = 0; st < IZ_S; st++) {
      u[st] = Q(IZ_QU, st);
      const double cs = Q(IZ_QC, st), p = Q(IZ_QP, st);
      lmax0 = fmax(fabs(u[st] - cs), lmax0);
      lmax1 = fmax(fabs(u[st]), lmax1);
      lmax2 = fmax(fabs(u[st] + cs), lmax2);
      const double u0 = Q(0, st), un = Q(cn, st), u4 = Q(4, st);
      double m = uc[0] * Q(1, st) + uc[1] * Q(2, st) + uc[2] * Q(3, st) - u4;
      double ps = 0.0;
#pragma unroll
      for (int l = 0; l < IZ_NRV; l++) ps += psi[l] * Q(IZ_NIV + l, st);
      pw[st] = ps;
      // F = u U + p (e_n + u e_4), and U_n = u U_0
      const double s0 = b2 * (m - ps);
      sw[st] = s0 - b1 * u0;
      sg[st] = u[st] * s0 + (b2 * (p * (un_c - u[st])) - b1 * un);
      dw[st] = un_c * u0 - un;
      dg[st] = un_c * un - (un * u[st] + p);
    }
    // rows 0 and 2
#pragma unroll
    for (int st = 0; st < IZ_S; st++) {
      const double w = hc * dw[st] - 0.5 * sw[st], g = hc * dg[st] - 0.5 * sg[st];
      gp[st] = g + lmax0 * w;
      gm[st] = g - lmax0 * w;
    }
    g0 = d_weno_face_fused<WIDE>(js, gp, gm);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int st = 0; st < IZ_S; st++) {
      const double w = -hc * dw[st] - 0.5 * sw[st], g = -hc * dg[st] - 0.5 * sg[st];
      gp[st] = g + lmax2 * w;
      gm[st] = g - lmax2 * w;
    }
    g2 = d_weno_face_fused<WIDE>(js, gp, gm);
    __builtin_amdgcn_sched_barrier(0);
    // row 5: -(1 + xi) / b2 with xi = b1 - b2 ht
    const double k = (1.0 + (b1 - b2 * ht_c)) / b2;
#pragma unroll
    for (int st = 0; st < IZ_S; st++) {
      const double w = -k * sw[st] - pw[st], g = -k * sg[st] - pw[st] * u[st];
      gp[st] = g + lmax1 * w;
      gm[st] = g - lmax1 * w;
    }
    g5 = d_weno_face_fused<WIDE>(js, gp, gm);
  }
  // row 1
  fresh();
#pragma unroll
  for (int st = 0; st < IZ_S; st++) {
    const double w = Q(0, st) + sw[st], g = Q(cn, st) + sg[st];
    gp[st] = g + lmax1 * w;
    gm[st] = g - lmax1 * w;
  }
  g1 = d_weno_face_fused<WIDE>(js, gp, gm);
  const double g02 = g0 + g2, gs = g02 + g1, gd = cs_c * (g2 - g0);
  F[fidx] = gs;
  F[(long)cn * nfaces + fidx] = un_c * gs + gd;
  double f4 = ht_c * g02 + un_c * gd + q * g1 + g5;
  // the tangential rows: U_t - u_t U_0, carried by u
#pragma unroll
  for (int tt = 0; tt < 2; tt++) {
    const int tc = tt == 0 ? t1 : t2;
    const double ut = uc[tc - 1];
    fresh();
#pragma unroll
    for (int st = 0; st < IZ_S; st++) {
      const double w = Q(tc, st) - ut * Q(0, st), g = u[st] * w;
      gp[st] = g + lmax1 * w;
      gm[st] = g - lmax1 * w;
    }
    const double gt = d_weno_face_fused<WIDE>(js, gp, gm);
    F[(long)tc * nfaces + fidx] = ut * gs + gt;
    f4 += ut * gt;
  }
  F[4 * nfaces + fidx] = f4;
  // species rows; the last species from row 5 and the others
  const double wrk = -1.0 / psi[IZ_NRV - 1];
  double last = g5;
#pragma unroll
  for (int l = 0; l < IZ_NRV - 1; l++) {
    const double y = Yc[l];
    fresh();
#pragma unroll
    for (int st = 0; st < IZ_S; st++) {
      const double vs = Q(IZ_NIV + l, st);
      const double w = vs + y * sw[st], g = vs * u[st] + y * sg[st];
      gp[st] = g + lmax1 * w;
      gm[st] = g - lmax1 * w;
    }
    const double gl = d_weno_face_fused<WIDE>(js, gp, gm);
    F[(long)(IZ_NIV + l) * nfaces + fidx] = y * g02 + gl;
    last += psi[l] * gl;
  }
  F[(long)(IZ_NV - 1) * nfaces + fidx] = Yc[IZ_NRV - 1] * g02 + wrk * last;
  // f4 and last hold every reconstructed field: the face is formed again where
  // the short reconstruction left its range (iz_weno.h).  Of an inert step at
  // 193 x 129 x 97 this test of a face takes nothing measurable, one of every
  // field 0.6 %, the wide form throughout 2 %.
  if constexpr (IZ_NG == 3 && !WIDE) {
    if (__builtin_expect(!(fabs(f4 + last) < INFINITY), 0))
      eu_face_fast<DIR, QS, SS, SITE, true>(tile, off, js, ha, nc, cL, cR, F, nfaces, fidx);
  }
}

template <int DIR, int QS, int SS, bool FAST, int SITE>
__device__ inline void eu_face(const double *tile, int off, bool js,
                               const double *__restrict__ ha, long nc, long cL, long cR,
                               double *__restrict__ F, long nfaces, long fidx) {
  if constexpr (FAST)
    eu_face_fast<DIR, QS, SS, SITE>(tile, off, js, ha, nc, cL, cR, F, nfaces, fidx);
  else
    eu_face_ref<DIR, QS, SS, SITE>(tile, off, js, ha, nc, cL, cR, F, nfaces, fidx);
}

// LDS bytes of one block of k_euler_faces<DIR>; tile0 = cells staged per
// wave for x (64 + IZ_S - 1, and IZ_S - 1 more per row boundary that 64
// consecutive faces can cross)
static inline int eu_tile0(const IzDims &d) {
  return (64 + IZ_S - 1) + (IZ_S - 1) * (63 / (d.nx + 1) + 1);
}
static inline size_t eu_lds_bytes(int dir, int tile0) {
  if (dir == 0) return (size_t)4 * tile0 * (IZ_EU_NQ * sizeof(double) + 1);
  return (size_t)IZ_EU_ROWS * IZ_EU_TX * (IZ_EU_NQ * sizeof(double) + 1);
}
// logical tiles of k_euler_faces<1/2> (x tiles * face tiles * other index)
static inline long eu_ntiles(const IzDims &d, int dir) {
  const int nd = dir == 1 ? d.ny : d.nz;
  const long ntf = (nd + 1 + IZ_EU_TF - 1) / IZ_EU_TF;
  const long ntx = (d.nx + IZ_EU_TX - 1) / IZ_EU_TX;
  return ntf * ntx * (dir == 1 ? d.nz : d.ny);
}

// The flags a face sees in a decomposed run: those of its stencil cells
// (left cell il, points il - ng + 1 .. il + ng) that the viewing rank rv
// owns -- the sensor is neither set on ghosts nor exchanged between ranks
// (module_tools.f90:2733-2814 per rank, then module_weno.f90:955-989).
// tsn[st * stride] is stencil point st's flag.
__device__ inline int eu_flags_view(const uint8_t *tsn, int stride, int il, int n, int np,
                                    int rv) {
  const int lo = iz_rank_lo(rv, n, np), hi = iz_rank_lo(rv + 1, n, np) - 1;
  int shk = 0;
#pragma unroll
  for (int st = 0; st < IZ_S; st++) {
    const int p = il - IZ_NG + 1 + st;
    if (p >= lo && p <= hi) shk |= tsn[st * stride];
  }
  return shk;
}

// RANKS: the run reproduces a decomposed one (d.np[DIR] > 1): a face takes
// the flag view of the rank of its right cell
template <int DIR, bool FAST, bool RANKS>
__global__ void __attribute__((amdgpu_flat_work_group_size(IZ_EU_BLOCK, IZ_EU_BLOCK),
                               amdgpu_waves_per_eu(FAST ? IZ_EULER_FAST_WAVES : IZ_EULER_WAVES)))
k_euler_faces(IzDims d, const double *__restrict__ v, const double *__restrict__ T,
              const double *__restrict__ W_i, const double *__restrict__ cp,
              const double *__restrict__ ha, const uint8_t *__restrict__ sensor, int weno_avg,
              double *__restrict__ F, long nfaces, int *__restrict__ status, int tile0,
              long ntiles) {
  extern __shared__ double lds[];
  int neg = 0;
  if constexpr (DIR == 0) {
    // face, row and slot numbers fit 32 bits (faces < 2^31 is checked at
    // context creation); only HBM cell indices are 64-bit
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned f0 = (blockIdx.x * 4u + wave) * 64u;  // first face of this wave
    const unsigned nf = d.nx + 1, NXc = d.nx + 2 * IZ_NG;  // faces, cells per row
    const unsigned nrows = (unsigned)d.ny * d.nz, nfc = (unsigned)nfaces;
    // cell-major tile (slot * IZ_EU_NQ + q): every stencil access is a
    // compile-time offset from the lane's first stencil cell
    double *tl = lds + wave * tile0 * IZ_EU_NQ;
    uint8_t *tsn = (uint8_t *)(lds + 4 * tile0 * IZ_EU_NQ) + wave * tile0;
    // cells in row-flattened order r * NXc + (x + ng); face f's stencil
    // starts at S(f) = r * NXc + x + 1 for its left cell x
    unsigned S0 = 0;
    if (f0 < nfc) S0 = (f0 / nf) * NXc + (f0 % nf);
    for (int t = lane; t < tile0; t += 64) {
      const unsigned cf = S0 + t;
      const unsigned r = cf / NXc;
      if (f0 < nfc && r < nrows) {
        const int xc = (int)(cf - r * NXc) - IZ_NG;
        const long c = iz_cidx(d, xc, (int)(r % d.ny), (int)(r / d.ny));
        eu_stage_cell(v, T, W_i, cp, d.nc, c, 1, tl + t * IZ_EU_NQ, 1, neg);
        tsn[t] = sensor[c];
      }
    }
    __syncthreads();
    const unsigned f = f0 + lane;
    if (f < nfc) {
      const unsigned r = f / nf;
      const int x = (int)(f - r * nf) - 1;
      const int o = (int)(r * NXc + x + 1 - S0);
      const long cL = iz_cidx(d, x, (int)(r % d.ny), (int)(r / d.ny));
      int shk = 0;
      if constexpr (RANKS) {
        shk = eu_flags_view(tsn + o, 1, x, d.nx, d.np[0], iz_rank_of(x + 1, d.nx, d.np[0]));
      } else {
#pragma unroll
        for (int st = 0; st < IZ_S; st++) shk |= tsn[o + st];
      }
      eu_face<0, 1, IZ_EU_NQ, FAST, RANKS>(lds, (wave * tile0 + o) * IZ_EU_NQ, shk && weno_avg, ha, d.nc,
                              cL, cL + 1, F, nfaces, (long)f);
    }
  } else {
    // hardware blocks b, b + 8, ... run on one XCD: give them consecutive
    // logical tiles, face tiles fastest
    const long per = (ntiles + 7) / 8;
    const long L = (long)(blockIdx.x % 8) * per + blockIdx.x / 8;
    const bool blk_ok = L < ntiles;
    const int nd = DIR == 1 ? d.ny : d.nz;
    const int ntf = (nd + 1 + IZ_EU_TF - 1) / IZ_EU_TF;
    const int ntx = (d.nx + IZ_EU_TX - 1) / IZ_EU_TX;
    const int tf = (int)(L % ntf);
    const int tx = (int)((L / ntf) % ntx);
    const int oth = (int)(L / ((long)ntf * ntx));  // k for y faces, j for z faces
    const int row0 = tf * IZ_EU_TF - IZ_NG;          // first staged cell along DIR
    constexpr int FS = IZ_EU_ROWS * IZ_EU_TX;        // field stride in LDS
    uint8_t *tsn = (uint8_t *)(lds + (long)IZ_EU_NQ * FS);
    for (int t = threadIdx.x; t < FS; t += IZ_EU_BLOCK) {
      const int rr = t / IZ_EU_TX, cx = tx * IZ_EU_TX + t % IZ_EU_TX;
      const int cdir = row0 + rr;
      if (blk_ok && cx < d.nx && cdir <= nd + IZ_NG - 1) {
        const long c = DIR == 1 ? iz_cidx(d, cx, cdir, oth) : iz_cidx(d, cx, oth, cdir);
        eu_stage_cell(v, T, W_i, cp, d.nc, c, 1 + DIR, lds + t, FS, neg);
        tsn[t] = sensor[c];
      }
    }
    __syncthreads();
    const int xl = threadIdx.x % IZ_EU_TX, fl = threadIdx.x / IZ_EU_TX;
    const int x = tx * IZ_EU_TX + xl;
    const int f = tf * IZ_EU_TF + fl - 1;  // left cell of the face along DIR
    if (blk_ok && x < d.nx && f <= nd - 1) {
      // stencil point st of this face is staged row fl + st
      int shk = 0;
      if constexpr (RANKS) {
        shk = eu_flags_view(tsn + fl * IZ_EU_TX + xl, IZ_EU_TX, f, nd, d.np[DIR],
                            iz_rank_of(f + 1, nd, d.np[DIR]));
      } else {
#pragma unroll
        for (int st = 0; st < IZ_S; st++) shk |= tsn[(fl + st) * IZ_EU_TX + xl];
      }
      long cL, cR, fidx;
      if (DIR == 1) {
        cL = iz_cidx(d, x, f, oth);
        cR = cL + d.NX;
        fidx = x + (long)d.nx * ((f + 1) + (long)(d.ny + 1) * oth);
      } else {
        cL = iz_cidx(d, x, oth, f);
        cR = cL + d.NX * d.NY;
        fidx = x + (long)d.nx * (oth + (long)d.ny * (f + 1));
      }
      eu_face<DIR, FS, IZ_EU_TX, FAST, RANKS>(lds, fl * IZ_EU_TX + xl, shk && weno_avg, ha, d.nc, cL, cR, F,
                                 nfaces, fidx);
    }
  }
  if (neg) atomicOr(status, IZ_ST_NEG_PRESSURE);
}

// The face between two ranks along DIR formed a second time, with the left
// rank's flag view: each rank of a decomposed run forms its boundary faces
// itself, and the left rank's last cell takes its right face from its own
// view (module_weno.f90:955-1020 per rank).  One thread per seam face
// t = (r) + (np - 1) line, r the left rank; F^ goes to Fs[m * nseam + t].
// Each thread stages its IZ_S stencil cells in its own LDS run, quantity
// q of stencil point st at q * IZ_S + st.
#define IZ_SEAM_BLOCK 32
template <int DIR, bool FAST>
__global__ void __launch_bounds__(IZ_SEAM_BLOCK)
k_euler_seams(IzDims d, const double *__restrict__ v, const double *__restrict__ T,
              const double *__restrict__ W_i, const double *__restrict__ cp,
              const double *__restrict__ ha, const uint8_t *__restrict__ sensor, int weno_avg,
              double *__restrict__ Fs, long nseam, int *__restrict__ status) {
  extern __shared__ double lds[];
  const long t = (long)blockIdx.x * IZ_SEAM_BLOCK + threadIdx.x;
  int neg = 0;
  if (t < nseam) {
    const int np = d.np[DIR];
    const int n = DIR == 0 ? d.nx : (DIR == 1 ? d.ny : d.nz);
    const int r = (int)(t % (np - 1));
    const long line = t / (np - 1);
    // x lines are (j, k), y lines (i, k), z lines (i, j)
    const int a = DIR == 0 ? (int)(line % d.ny) : (int)(line % d.nx);
    const int b = DIR == 0 ? (int)(line / d.ny) : (int)(line / d.nx);
    auto cell = [&](int p) {
      return DIR == 0 ? iz_cidx(d, p, a, b) : (DIR == 1 ? iz_cidx(d, a, p, b) : iz_cidx(d, a, b, p));
    };
    const int il = iz_rank_lo(r + 1, n, np) - 1;  // the left rank's last cell
    const int off = threadIdx.x * IZ_S * IZ_EU_NQ;
    uint8_t fl[IZ_S];
#pragma unroll
    for (int st = 0; st < IZ_S; st++) {
      const long c = cell(il - IZ_NG + 1 + st);
      eu_stage_cell(v, T, W_i, cp, d.nc, c, 1 + DIR, lds + off + st, IZ_S, neg);
      fl[st] = sensor[c];
    }
    const int shk = eu_flags_view(fl, 1, il, n, np, r);
    eu_face<DIR, IZ_S, 1, FAST, 2>(lds, off, shk && weno_avg, ha, d.nc, cell(il), cell(il + 1),
                                    Fs, nseam, t);
  }
  if (neg) atomicOr(status, IZ_ST_NEG_PRESSURE);
}

// seam face arrays of the three directions (d.np > 1)
struct IzSeams {
  const double *F[3];
  long n[3];
};

// fl = (F^_r - F^_l) * d_i  (x assigns, y/z accumulate): module_weno.f90:998-1020;
// a rank's last cell takes its right face from the seam array
template <int DIR>
__global__ void k_euler_apply(IzDims d, const double *__restrict__ F, long nfaces,
                              const double *__restrict__ d_i, int accumulate,
                              double *__restrict__ fl, const double *__restrict__ Fs, long nseam) {
  long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long ncin = (long)d.nx * d.ny * d.nz;
  if (tid >= ncin) return;
  int i = (int)(tid % d.nx);
  long r = tid / d.nx;
  int j = (int)(r % d.ny), k = (int)(r / d.ny);
  long fr, fl_;
  double di;
  if (DIR == 0) { fl_ = i + (long)(d.nx + 1) * (j + (long)d.ny * k); fr = fl_ + 1; di = d_i[i + d.ng]; }
  else if (DIR == 1) { fl_ = i + (long)d.nx * (j + (long)(d.ny + 1) * k); fr = fl_ + d.nx; di = d_i[j + d.ng]; }
  else { fl_ = i + (long)d.nx * (j + (long)d.ny * k); fr = fl_ + (long)d.nx * d.ny; di = d_i[k + d.ng]; }
  long c = iz_cidx(d, i, j, k);
  long sr = -1;
  if (d.np[DIR] > 1) {
    if (DIR == 0) sr = iz_seam(i, d.nx, d.np[0], j + (long)d.ny * k);
    else if (DIR == 1) sr = iz_seam(j, d.ny, d.np[1], i + (long)d.nx * k);
    else sr = iz_seam(k, d.nz, d.np[2], i + (long)d.nx * j);
  }
#pragma unroll
  for (int m = 0; m < IZ_NV; m++) {
    const double Fr = sr >= 0 ? Fs[m * nseam + sr] : F[m * nfaces + fr];
    double df = (Fr - F[m * nfaces + fl_]) * di;
    if (accumulate) fl[m * d.nc + c] = fl[m * d.nc + c] + df * 1.0;
    else fl[m * d.nc + c] = df * 1.0;
  }
}

// ===================================================================
// Primitive variables: force_sumY, Newton with the reference's global exit.
// ===================================================================
struct IzBox { int i0, i1, j0, j1, k0, k1; };

__device__ inline bool box_cell(const IzBox &b, long tid, int &i, int &j, int &k) {
  int ni = b.i1 - b.i0 + 1, nj = b.j1 - b.j0 + 1, nk = b.k1 - b.k0 + 1;
  if (tid >= (long)ni * nj * nk) return false;
  i = b.i0 + (int)(tid % ni);
  long r = tid / ni;
  j = b.j0 + (int)(r % nj);
  k = b.k0 + (int)(r / nj);
  return true;
}

// The domains of one pass (interior and ghost slabs, domain_select) in one
// launch: thread indices [first[q], first[q+1]) are the cells of box[q].
// A slab alone is too small a grid to fill the device.
struct IzDomSet {
  IzBox box[7];
  int dom[7];
  long first[8];
  int n;
};
__device__ inline bool domset_cell(const IzDomSet &s, long tid, int &dom, int &i, int &j,
                                   int &k) {
  if (tid >= s.first[s.n]) return false;
  IzBox b = s.box[0];
  int dm = s.dom[0];
  long f0 = s.first[0];
  // compile-time indices only, so the set stays in scalar registers
#pragma unroll
  for (int p = 1; p < 7; p++)
    if (p < s.n && tid >= s.first[p]) { b = s.box[p]; dm = s.dom[p]; f0 = s.first[p]; }
  dom = dm;
  return box_cell(b, tid - f0, i, j, k);
}

// The domains of one Newton pass (the interior, a Dirichlet row, or all ghost
// slabs together) in one launch, with blocks of their own per domain, so
// that a block's reduction goes to one domain's mask: blocks [first[q],
// first[q + 1]) walk the cells of box[q].  A slab alone is a few tens of
// blocks; the six of a 3-D box one by one took 18 launches a pass.
struct IzNewtonSet {
  IzBox box[6];
  int dom[6], slot[6];
  unsigned first[7];
  int n;
};
__device__ inline int nset_domain(const IzNewtonSet &s, IzBox &b, unsigned &blk, unsigned &nblk) {
  b = s.box[0];
  int q = 0;
  unsigned f0 = 0, f1 = s.first[1];
  // compile-time indices only, so the set stays in scalar registers
#pragma unroll
  for (int p = 1; p < 6; p++)
    if (p < s.n && blockIdx.x >= s.first[p]) {
      b = s.box[p];
      q = p;
      f0 = s.first[p];
      f1 = s.first[p + 1];
    }
  blk = blockIdx.x - f0;
  nblk = f1 - f0;
  return q;
}
__device__ inline int nset_slot(const IzNewtonSet &s, int q) {
  int v = s.slot[0];
#pragma unroll
  for (int p = 1; p < 6; p++) v = (p == q) ? s.slot[p] : v;
  return v;
}
__device__ inline int nset_dom(const IzNewtonSet &s, int q) {
  int v = s.dom[0];
#pragma unroll
  for (int p = 1; p < 6; p++) v = (p == q) ? s.dom[p] : v;
  return v;
}

// force_sumY (npv = 0): module_thermodynamics.f90:1709-1760
__device__ inline void d_force_sumY(double *vc) {
  double rho = vc[0], rho_i = 1.0 / rho, sum = 0.0, Y;
#pragma unroll
  for (int l = 0; l < IZ_NRV - 1; l++) {
    Y = vc[IZ_NIV + l] * rho_i;
    Y = fmin(fmax(Y, 0.0), 1.0);
    vc[IZ_NIV + l] = rho * Y;
    sum = sum + Y;
  }
  Y = 1.0 - sum;
  Y = fmin(fmax(Y, 0.0), 1.0);
  vc[IZ_NIV + IZ_NRV - 1] = rho * Y;
}

// Newton probe: iterate one cell and record in bit (it-1) whether its
// increment blocks the global exit test sqrt(max DF^2) < eps at iteration it
// (module_thermodynamics.f90:111-150), and in bit (it-1) of neg whether its
// T is negative after iteration it (the repair branch, :120-139).  Cells
// stop once their increment has fallen far below eps: Newton's quadratic
// contraction keeps all later increments below it.
template <bool FRESH>
__device__ inline unsigned long long d_newton_probe(const double *vc, double T, double eps,
                                                    unsigned long long &neg) {
  unsigned long long mask = 0ull;
  for (int it = 1; it <= 64; it++) {
    double cpv, h[IZ_NRV];
    double DF = d_newton_cell<FRESH>(vc, T, cpv, h);
    T = T + DF;
    if (T < 0.0) neg |= 1ull << (it - 1);
    double e = sqrt(DF * DF);
    if (!(e < eps)) mask |= 1ull << (it - 1);
    else if (e < eps * 1.0e-3) break;
  }
  return mask;
}

// Block-wide reductions that end in one atomic per block.  Kernels that
// reduce walk the cells with a grid-stride loop over a grid capped at a
// few blocks per CU, so a launch issues a few thousand atomics on the
// target words instead of one per wave (same-address atomics serialise in
// L2).  blockDim.x is a multiple of 64 and at most 1024; every thread of
// the block calls these.
__device__ inline void block_or_u64(unsigned long long m, unsigned long long *dst) {
  __shared__ unsigned long long s_or[16];
  for (int off = 32; off > 0; off >>= 1) m |= __shfl_xor(m, off, 64);
  if ((threadIdx.x & 63) == 0) s_or[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long a = 0ull;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) a |= s_or[w];
    if (a) atomicOr(dst, a);
  }
}
// the Newton probe's two masks: blocking iterations into dst[0], negative
// temperatures into dst[IZ_NEG_MASKS]
#define IZ_NEG_MASKS 8
__device__ inline void block_or_probe(unsigned long long m, unsigned long long neg,
                                      unsigned long long *dst) {
  __shared__ unsigned long long s_or2[2][16];
  for (int off = 32; off > 0; off >>= 1) {
    m |= __shfl_xor(m, off, 64);
    neg |= __shfl_xor(neg, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    s_or2[0][threadIdx.x >> 6] = m;
    s_or2[1][threadIdx.x >> 6] = neg;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long a = 0ull, b = 0ull;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) {
      a |= s_or2[0][w];
      b |= s_or2[1][w];
    }
    if (a) atomicOr(dst, a);
    if (b) atomicOr(dst + IZ_NEG_MASKS, b);
  }
}

__device__ inline void atomic_max_pos(double *addr, double val) {
  // non-negative doubles order like their bit patterns
  atomicMax((unsigned long long *)addr, (unsigned long long)__double_as_longlong(val));
}
__device__ inline void atomic_min_pos(double *addr, double val) {
  atomicMin((unsigned long long *)addr, (unsigned long long)__double_as_longlong(val));
}

// x[0..N) reduced over the block by max (MAXR) or min, then one atomic per
// value into dst[0..N); values are non-negative (or +inf)
template <int N, bool MAXR>
__device__ inline void block_extreme_pos(double *x, double *dst) {
  __shared__ double s_ex[N][16];
#pragma unroll
  for (int q = 0; q < N; q++) {
    double a = x[q];
    for (int off = 32; off > 0; off >>= 1) {
      const double b = __shfl_xor(a, off, 64);
      a = MAXR ? fmax(a, b) : fmin(a, b);
    }
    if ((threadIdx.x & 63) == 0) s_ex[q][threadIdx.x >> 6] = a;
  }
  __syncthreads();
  if (threadIdx.x < N) {
    const int q = threadIdx.x;
    double a = s_ex[q][0];
    for (int w = 1; w < (int)(blockDim.x >> 6); w++) a = MAXR ? fmax(a, s_ex[q][w]) : fmin(a, s_ex[q][w]);
    if (MAXR) atomic_max_pos(&dst[q], a);
    else atomic_min_pos(&dst[q], a);
  }
}

// force_sumY and the Newton probe on the domains of a set.  fill: the cells
// are ghost cells of a periodic or extrapolated face and first take their
// source cell's conserved variables (k_ghost_fill's copy), so that the ghost
// layers are read and written once.
__global__ void __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(2, 2)))
k_force_probe(IzDims d, IzNewtonSet s, int fill, int forcesum, double *__restrict__ v,
              const double *__restrict__ T, double eps, unsigned long long *__restrict__ masks) {
  IzBox b;
  unsigned blk, nblk;
  const int q = nset_domain(s, b, blk, nblk), dom = nset_dom(s, q);
  int i, j, k;
  unsigned long long m = 0ull, neg = 0ull;
  for (long tid = (long)blk * 256 + threadIdx.x; box_cell(b, tid, i, j, k);
       tid += (long)nblk * 256) {
    const long c = iz_cidx(d, i, j, k);
    long cs = c;
    if (fill) {
      int si = i, sj = j, sk = k;
      if (dom == -1) si = (d.phys & 1) ? 0 : i + d.nx;
      else if (dom == 1) si = (d.phys & 2) ? d.nx - 1 : i - d.nx;
      else if (dom == -2) sj = (d.phys & 4) ? 0 : j + d.ny;
      else if (dom == 2) sj = (d.phys & 8) ? d.ny - 1 : j - d.ny;
      else if (dom == -3) sk = (d.phys & 16) ? 0 : k + d.nz;
      else sk = (d.phys & 32) ? d.nz - 1 : k - d.nz;
      cs = iz_cidx(d, si, sj, sk);
    }
    double vc[IZ_NV];
#pragma unroll
    for (int l = 0; l < IZ_NV; l++) vc[l] = v[l * d.nc + cs];
    if (forcesum) d_force_sumY(vc);
    if (fill) {
#pragma unroll
      for (int l = 0; l < IZ_NIV; l++) v[l * d.nc + c] = vc[l];
    }
    if (fill || forcesum) {
#pragma unroll
      for (int l = IZ_NIV; l < IZ_NV; l++) v[l * d.nc + c] = vc[l];
    }
    if (eps > 0.0) m |= d_newton_probe<true>(vc, T[c], eps, neg);
  }
  block_or_probe(m, neg, masks + nset_slot(s, q));
}

// number of global iterations from the OR of all probes: the first
// iteration with no blocking cell; itmax when every probed iteration blocked
__device__ inline int d_newton_count(unsigned long long mask, int itmax) {
  if (~mask == 0ull) return itmax;
  return __builtin_ctzll(~mask) + 1;
}

// whether a cell's T turns negative before the global exit: the first
// negative iteration (neg mask) is not after the exit iteration N
__device__ inline bool d_newton_repairs(unsigned long long mask, unsigned long long neg,
                                        int itmax) {
  return neg && __builtin_ctzll(neg) + 1 <= d_newton_count(mask, itmax);
}

// Apply exactly N iterations, write T, W_i, cp (last evaluation, i.e. at the
// pre-update T), ha (module_thermodynamics.f90:79-186, Wmix_i :700-728).
// When a cell turns negative before the exit, nothing is written here and
// k_newton_repair runs the domain's iterations instead.
__global__ void __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(2, 2)))
k_newton_apply(IzDims d, IzNewtonSet s, const double *__restrict__ v,
                               double *__restrict__ T, double *__restrict__ W_i,
                               double *__restrict__ cp, double *__restrict__ ha,
                               const unsigned long long *__restrict__ masks, int itmax,
                               int repair, int *__restrict__ status, int *__restrict__ iters) {
  IzBox b;
  unsigned blk, nblk;
  const int slot = nset_slot(s, nset_domain(s, b, blk, nblk));
  const unsigned long long *mask = masks + slot;
  const long tid = (long)blk * 256 + threadIdx.x;
  int i, j, k;
  if (!box_cell(b, tid, i, j, k)) return;
  if (repair && d_newton_repairs(*mask, mask[IZ_NEG_MASKS], itmax)) return;
  const int N = d_newton_count(*mask, itmax);
  if (tid == 0) iters[slot] = N;
  long c = iz_cidx(d, i, j, k);
  double vc[IZ_NV];
#pragma unroll
  for (int l = 0; l < IZ_NV; l++) vc[l] = v[l * d.nc + c];
  double w = 0.0;
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) w = w + (vc[IZ_NIV + l] / vc[0]) * c_thd.Wc_i[l];
  W_i[c] = w;
  double Tc = T[c], cpv = 0.0, h[IZ_NRV];
  for (int it = 0; it < N; it++) {
    double DF = d_newton_cell<true>(vc, Tc, cpv, h);
    Tc = Tc + DF;
  }
  T[c] = Tc;
  cp[c] = cpv;
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) ha[l * d.nc + c] = h[l];
  int st = 0;
  // with the repair: negative only after iteration 64, beyond what the
  // probe records; without (prim_inv_var_err_mach): the reference's warning
  if (Tc < 0.0) st |= repair ? IZ_ST_NEG_T_ABORT : IZ_ST_NEG_TEMPERATURE;
  if (Tc != Tc) st |= IZ_ST_NAN;
  if (N >= itmax) st |= IZ_ST_NEWTON_ITMAX;
  if (st) atomicOr(status, st);
}

// The negative-temperature repair of prim_inv_var (module_thermodynamics.f90:
// 79-186), run when the probe saw a cell of the domain turn negative before
// the global exit: one block redoes the domain's iterations from the
// caller's T in the reference's order.  Each iteration evaluates every
// cell's increment (cp, ha at the pre-update T), adds it, and collects the
// cells whose T is negative; those are then taken in storage order:
// recorded, their conserved variables replaced by the mean of their x
// neighbours (a negative neighbour met earlier in the sweep enters with its
// replaced values), the iteration count restarted.  After the exit test
// every recorded cell gets T = mean of its x neighbours' T.  W_i comes from
// the conserved variables before any replacement (:102).  A rare, slow path
// (one block; seconds on a 256^3 domain): status IZ_ST_NEG_TEMPERATURE
// marks it; IZ_ST_NEG_T_ABORT marks a repair the reference aborts on (more
// than IZ_NEGT_MAX cells, :131), one that would read outside the array (a
// cell at its x edge) or more than IZ_NEGT_SWEEP negative cells in one
// iteration.  One block per domain of the set (a domain's repair reads no
// cell that another's writes: slabs meet at edges, and x neighbours of a y
// or z slab's cells are its own).  As the last kernel of a Newton pass it
// also clears the domain's masks for the next one.
#define IZ_NEGT_MAX 40000
#define IZ_NEGT_SWEEP 1024
__global__ void __launch_bounds__(1024)
k_newton_repair(IzDims d, IzNewtonSet set, int repair, double *__restrict__ v,
                double *__restrict__ T, double *__restrict__ W_i, double *__restrict__ cp,
                double *__restrict__ ha, unsigned long long *__restrict__ masks, int itmax,
                double eps, int *__restrict__ recs, int *__restrict__ status,
                int *__restrict__ iters) {
  const int slot = nset_slot(set, blockIdx.x);
  IzBox b = set.box[0];
#pragma unroll
  for (int p = 1; p < 6; p++)
    if (p == (int)blockIdx.x) b = set.box[p];
  const unsigned long long m0 = masks[slot], n0 = masks[slot + IZ_NEG_MASKS];
  __syncthreads();
  if (threadIdx.x == 0) {
    masks[slot] = 0ull;
    masks[slot + IZ_NEG_MASKS] = 0ull;
  }
  if (!repair || !d_newton_repairs(m0, n0, itmax)) return;
  int *rec = recs + (long)slot * IZ_NEGT_MAX;
  __shared__ int s_neg[IZ_NEGT_SWEEP];
  __shared__ int s_nneg, s_it, s_ipt, s_correct, s_stop, s_bad;
  __shared__ double s_max[16], s_err;
  __shared__ int s_nan[16];
  const int ni = b.i1 - b.i0 + 1, nj = b.j1 - b.j0 + 1;
  const long n = (long)ni * nj * (b.k1 - b.k0 + 1);
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, w = tid >> 6;
  for (long t = tid; t < n; t += nt) {
    int i, j, k;
    box_cell(b, t, i, j, k);
    const long c = iz_cidx(d, i, j, k);
    double wsum = 0.0;
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++)
      wsum = wsum + (v[(IZ_NIV + l) * d.nc + c] / v[c]) * c_thd.Wc_i[l];
    W_i[c] = wsum;
  }
  if (tid == 0) {
    s_it = 0;
    s_ipt = 0;
    s_correct = 0;
    s_bad = 0;
    s_err = 0.0;
  }
  __syncthreads();
  for (;;) {
    if (tid == 0) {
      s_it = s_it + 1;
      s_stop = s_it > itmax;
      s_nneg = 0;
    }
    __syncthreads();
    if (s_stop) break;
    double mx = -INFINITY;
    int nan = 0;
    for (long t = tid; t < n; t += nt) {
      int i, j, k;
      box_cell(b, t, i, j, k);
      const long c = iz_cidx(d, i, j, k);
      double vc[IZ_NV];
#pragma unroll
      for (int l = 0; l < IZ_NV; l++) vc[l] = v[l * d.nc + c];
      double cpv, h[IZ_NRV];
      const double DF = d_newton_cell<true>(vc, T[c], cpv, h);
      cp[c] = cpv;
#pragma unroll
      for (int l = 0; l < IZ_NRV; l++) ha[l * d.nc + c] = h[l];
      const double Tn = T[c] + DF;
      T[c] = Tn;
      const double d2 = DF * DF;
      if (Tn < 0.0) {
        const int q = atomicAdd(&s_nneg, 1);
        if (q < IZ_NEGT_SWEEP) s_neg[q] = (int)t;
      }
      if (d2 != d2) nan = 1;
      mx = fmax(mx, d2);
    }
    for (int off = 32; off > 0; off >>= 1) {
      mx = fmax(mx, __shfl_xor(mx, off, 64));
      nan |= __shfl_xor(nan, off, 64);
    }
    if (lane == 0) {
      s_max[w] = mx;
      s_nan[w] = nan;
    }
    __syncthreads();
    if (tid == 0) {
      double m = s_max[0];
      int nn = s_nan[0];
      for (int q = 1; q < (nt >> 6); q++) {
        m = fmax(m, s_max[q]);
        nn |= s_nan[q];
      }
      const double error = nn ? NAN : sqrt(m);
      s_err = error;
      const int nneg = s_nneg;
      if (nneg > IZ_NEGT_SWEEP) s_bad = 1;
      // this sweep's negative cells in storage order
      for (int a = 1; a < nneg && !s_bad; a++) {
        const int x = s_neg[a];
        int q = a - 1;
        while (q >= 0 && s_neg[q] > x) {
          s_neg[q + 1] = s_neg[q];
          q--;
        }
        s_neg[q + 1] = x;
      }
      for (int q = 0; q < nneg && !s_bad; q++) {
        int i, j, k;
        box_cell(b, s_neg[q], i, j, k);
        const long c = iz_cidx(d, i, j, k);
        const int ia = i + d.ng;
        s_ipt = s_ipt + 1;
        if (s_ipt > IZ_NEGT_MAX || ia < 1 || ia > (int)d.NX - 2) {
          s_bad = 1;
          break;
        }
        rec[s_ipt - 1] = (int)c;
        s_it = 0;
        s_correct = 1;
        for (int l = 0; l < IZ_NV; l++)
          v[l * d.nc + c] = 0.5 * (v[l * d.nc + c - 1] + v[l * d.nc + c + 1]);
      }
      s_stop = s_bad || error < eps;
      if (!s_stop && s_correct)
        for (int l = 0; l < s_ipt; l++) {
          const long c = rec[l];
          T[c] = 0.5 * (T[c - 1] + T[c + 1]);
        }
    }
    __syncthreads();
    if (s_stop) break;
  }
  if (tid == 0) {
    int st = IZ_ST_NEG_TEMPERATURE;
    if (s_bad) st |= IZ_ST_NEG_T_ABORT;
    if (s_err != s_err) st |= IZ_ST_NAN;
    if (s_it > itmax) st |= IZ_ST_NEWTON_ITMAX;
    atomicOr(status, st);
    iters[slot] = s_it;
  }
}


// upd_prim_var_woT: module_thermodynamics.f90:522-689
__global__ void k_upd_prim_woT(IzDims d, IzBox b, const double *__restrict__ v,
                               const double *__restrict__ T, double *__restrict__ W_i,
                               double *__restrict__ cp, double *__restrict__ ha) {
  long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int i, j, k;
  if (!box_cell(b, tid, i, j, k)) return;
  long c = iz_cidx(d, i, j, k);
  double vc[IZ_NV];
#pragma unroll
  for (int l = 0; l < IZ_NV; l++) vc[l] = v[l * d.nc + c];
  double w = 0.0;
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) w = w + (vc[IZ_NIV + l] / vc[0]) * c_thd.Wc_i[l];
  W_i[c] = w;
  double cpv, h[IZ_NRV];
  (void)d_newton_cell<false>(vc, T[c], cpv, h);
  cp[c] = cpv;
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) ha[l * d.nc + c] = h[l];
}

// Face-ghost fill of nf fields on one rank: comm_cons's periodic self-exchange
// (module_parallel.f90:1715-1777) or, on a physical face, upd_boundaries'
// bc_extrapolation (module_BCs.f90:327-412: the ng ghost layers take the
// edge value).  Threads cover the 2*ng slabs of direction dir.
// wall (the conserved variables, nf = IZ_NV, with face S a post-shock slip
// wall): bc_postshock_slipwall (module_BCs.f90:1065-1172) on that face: the
// first nfix cells take the post-shock state on the ghost rows and on the
// first interior row, the others mirror rows 1..ng (rho v odd).
// mode bit 1: the periodic faces (comm_cons); bit 2: the physical faces'
// conditions (upd_boundaries), a characteristic outflow face excepted.
__global__ void k_ghost_fill(IzDims d, double *__restrict__ a, int nf, int dir,
                             const double *__restrict__ wall, int mode) {
  long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int n0, n1, n;  // transverse sizes and the direction length
  if (dir == 0) { n0 = d.ny; n1 = d.nz; n = d.nx; }
  else if (dir == 1) { n0 = d.nx; n1 = d.nz; n = d.ny; }
  else { n0 = d.nx; n1 = d.ny; n = d.nz; }
  long per = (long)n0 * n1 * 2 * d.ng;
  if (tid >= per * nf) return;
  int f = (int)(tid / per);
  long r = tid % per;
  int s = (int)(r % (2 * d.ng));
  r /= (2 * d.ng);
  int p0 = (int)(r % n0), p1 = (int)(r / n0);
  const int face = 2 * dir + (s < d.ng ? 0 : 1);
  const int phys = (d.phys >> face) & 1;
  if (!(mode & (phys ? 2 : 1))) return;
  if (face == 1 && d.nscbc) return;
  if (wall && dir == 1 && s < d.ng) {
    if (p0 < d.nfix) {
      a[f * d.nc + iz_cidx(d, p0, -1 - s, p1)] = wall[f];
      if (s == 0) a[f * d.nc + iz_cidx(d, p0, 0, p1)] = wall[f];
    } else {
      const double val = a[f * d.nc + iz_cidx(d, p0, 1 + s, p1)];
      a[f * d.nc + iz_cidx(d, p0, -1 - s, p1)] = (f == 2) ? -val : val;
    }
    return;
  }
  int dst, src;
  if (s < d.ng) {
    dst = -1 - s;
    src = ((d.phys >> (2 * dir)) & 1) ? 0 : n - 1 - s;
  } else {
    int q = s - d.ng;
    dst = n + q;
    src = ((d.phys >> (2 * dir + 1)) & 1) ? n - 1 : q;
  }
  long cd, cs;
  if (dir == 0) { cd = iz_cidx(d, dst, p0, p1); cs = iz_cidx(d, src, p0, p1); }
  else if (dir == 1) { cd = iz_cidx(d, p0, dst, p1); cs = iz_cidx(d, p0, src, p1); }
  else { cd = iz_cidx(d, p0, p1, dst); cs = iz_cidx(d, p0, p1, src); }
  a[f * d.nc + cd] = a[f * d.nc + cs];
}

// bc_nscbc_out (module_BCs.f90:2331-2516), face E: per row, the one-sided
// fourth-order x derivatives of rho, u, v, w, p and Y over the last five
// cells, the characteristic amplitudes L1..L5 of a subsonic outflow with
// L1 relaxed toward pinf (sigma (1 - M^2) c / Lx, sigma = 0.28), and the
// last cell's state advanced by -dt d(.) written to it and to the ghosts.
// One thread per (j, k) row; the row's reads all precede its writes.
__global__ void k_nscbc_out(IzDims d, double *__restrict__ v, const double *__restrict__ T,
                            const double *__restrict__ W_i, const double *__restrict__ cp,
                            const double *__restrict__ dtp, double scale, double Lx,
                            double pinf, double dxi) {
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= (long)d.ny * d.nz) return;
  const int j = (int)(tid % d.ny), k = (int)(tid / d.ny);
  const int ex = d.nx - 1;
  const long nc = d.nc;
  // alph4or(-4..0)
  const double a4[5] = {-3.0 / 12.0, 16.0 / 12.0, -36.0 / 12.0, 48.0 / 12.0, -25.0 / 12.0};
  const double sigma1 = 0.28;
  const double dtime = *dtp * scale;
  const long ce = iz_cidx(d, ex, j, k);
  double rho = v[ce], rho_i = 1.0 / rho;
  double ux = v[nc + ce] * rho_i, vy = v[2 * nc + ce] * rho_i, wz = v[3 * nc + ce] * rho_i;
  double Pres = v[ce] * T[ce] * W_i[ce];
  double gam = c_thd.gam2 * W_i[ce] / cp[ce];
  gam = 1.0 / (1.0 - gam);
  double cs = sqrt(gam * Pres * rho_i);
  const double Mach = sqrt(ux * ux + vy * vy + wz * wz) / cs;
  const double Machm = fmax(0.0, Mach);
  double drho = 0.0, dux = 0.0, dvy = 0.0, dwz = 0.0, dPres = 0.0, dYa[IZ_NRV], Ya[IZ_NRV];
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) dYa[l] = 0.0;
#pragma unroll
  for (int m = 0; m < 5; m++) {
    const long c = ce - 4 + m;
    rho = v[c];
    rho_i = 1.0 / rho;
    ux = v[nc + c] * rho_i;
    vy = v[2 * nc + c] * rho_i;
    wz = v[3 * nc + c] * rho_i;
    Pres = v[c] * T[c] * W_i[c];
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++) Ya[l] = v[(IZ_NIV + l) * nc + c] * rho_i;
    drho = drho + a4[m] * rho;
    dux = dux + a4[m] * ux;
    dvy = dvy + a4[m] * vy;
    dwz = dwz + a4[m] * wz;
    dPres = dPres + a4[m] * Pres;
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++) dYa[l] = dYa[l] + a4[m] * Ya[l];
  }
  drho = -drho * dxi;
  dux = -dux * dxi;
  dvy = -dvy * dxi;
  dwz = -dwz * dxi;
  dPres = -dPres * dxi;
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) dYa[l] = -dYa[l] * dxi;
  double L1 = 0.0, L2 = 0.0, L3 = 0.0, L4 = 0.0, L5 = 0.0, L5Y[IZ_NRV];
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) L5Y[l] = 0.0;
  gam = c_thd.gam2 * W_i[ce] / cp[ce];
  gam = 1.0 / (1.0 - gam);
  cs = sqrt(gam * Pres * rho_i);
  if (ux - cs < 0.0) L1 = sigma1 * (1.0 - Machm * Machm) * cs / Lx * (Pres - pinf);
  else L1 = (ux - cs) * (dPres - rho * cs * dux);
  if (ux + cs > 0.0) L5 = (ux + cs) * (dPres + rho * cs * dux);
  else L5 = (ux + cs) * (2.0 * dPres - L1 / (ux - cs));
  if (ux > 0.0) {
    L2 = ux * (cs * cs * drho - dPres);
    L3 = ux * dvy;
    L4 = ux * dwz;
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++) L5Y[l] = ux * dYa[l];
  } else {
    L2 = ux * cs * cs * drho - 0.5 * ux * (L5 / (ux + cs) + L1 / (ux - cs));
  }
  const double d2 = 0.5 * (L5 + L1);
  const double d1 = (L2 + d2) / (cs * cs);
  const double d3 = 0.5 * (L5 - L1) / (cs * rho);
  const double d4 = L3, d5 = L4;
  double has[IZ_NRV];
  d_ha_scalar(T[ce], has);
  double hm = 0.0;
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) hm = hm + has[l] * Ya[l];
  const double q2 = ux * ux + vy * vy + wz * wz;
  double out[IZ_NV];
  out[0] = rho - d1 * dtime;
  out[1] = (rho * ux) - (ux * d1 + rho * d3) * dtime;
  out[2] = (rho * vy) - (vy * d1 + rho * d4) * dtime;
  out[3] = (rho * wz) - (wz * d1 + rho * d5) * dtime;
  out[4] = (rho * hm - Pres + 0.5 * rho * q2) -
           (0.5 * q2 * d1 + rho * (ux * d3 + vy * d4 + wz * d5) + d2 / (gam - 1.0)) * dtime;
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++)
    out[IZ_NIV + l] = (rho * Ya[l]) - (Ya[l] * d1 + rho * L5Y[l]) * dtime;
  for (int i = ex; i <= ex + d.ng; i++) {
    const long c = iz_cidx(d, i, j, k);
#pragma unroll
    for (int l = 0; l < IZ_NV; l++) v[l * nc + c] = out[l];
  }
}

// force_sumY on one Dirichlet row, right after its face's condition (the
// reference's order: module_BCs.f90:131 before the next face)
__global__ void k_force_row(IzDims d, IzBox b, double *__restrict__ v) {
  long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int i, j, k;
  if (!box_cell(b, tid, i, j, k)) return;
  const long c = iz_cidx(d, i, j, k);
  double vc[IZ_NV];
#pragma unroll
  for (int m = 0; m < IZ_NV; m++) vc[m] = v[m * d.nc + c];
  d_force_sumY(vc);
#pragma unroll
  for (int m = IZ_NIV; m < IZ_NV; m++) v[m * d.nc + c] = vc[m];
}

// shock_sensor_modified_adams_shariff (sticky): module_tools.f90:2733-2814
__global__ void k_sensor(IzDims d, double max_rel_weight, const double *__restrict__ v,
                         const double *__restrict__ T, const double *__restrict__ W_i,
                         uint8_t *__restrict__ sensor) {
  long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long ncin = (long)d.nx * d.ny * d.nz;
  if (tid >= ncin) return;
  int i = (int)(tid % d.nx);
  long r = tid / d.nx;
  int j = (int)(r % d.ny), k = (int)(r / d.ny);
  long c = iz_cidx(d, i, j, k);
  double ri = 1.0 / v[c];
  double P = v[c] * T[c] * W_i[c];
  bool flag = false;
  for (int dd = 0; dd < d.ndim; dd++) {
    int p = (dd == 0) ? i : (dd == 1 ? j : k);
    int n = (dd == 0) ? d.nx : (dd == 1 ? d.ny : d.nz);
    // the sweep of each rank stops one short of its last cell
    if (p >= iz_rank_lo(iz_rank_of(p, n, d.np[dd]) + 1, n, d.np[dd]) - 1) continue;
    long c2 = c + ((dd == 0) ? 1 : (dd == 1 ? d.NX : d.NX * d.NY));
    double ri2 = 1.0 / v[c2];
    double P2 = v[c2] * T[c2] * W_i[c2];
    double drho = fabs(v[c2] - v[c]) * fmin(ri, ri2);
    double dpres = fabs(P2 - P) / fmin(P, P2);
    if (drho > max_rel_weight && dpres > max_rel_weight) flag = true;
  }
  if (flag) sensor[c] = 1;
}

// shock_sensor_ducros (sticky) with compute_duixj's velocity gradients:
// module_tools.f90:2665-2719, 2521-2651.  The gradients are d?_fixed1's
// sixth-order central differences (alpha6, in z as well: the reference's z
// operator reads k +- 4 of an ng = 3 halo); velocities m / rho in the
// reference's form m * (1 / rho).
__global__ void k_sensor_ducros(IzDims d, double treduc, const double *__restrict__ dx_i,
                                const double *__restrict__ dy_i, const double *__restrict__ dz_i,
                                const double *__restrict__ v, uint8_t *__restrict__ sensor) {
  long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long ncin = (long)d.nx * d.ny * d.nz;
  if (tid >= ncin) return;
  int i = (int)(tid % d.nx);
  long r = tid / d.nx;
  int j = (int)(r % d.ny), k = (int)(r / d.ny);
  const long c = iz_cidx(d, i, j, k);
  const long st[3] = {1, d.NX, (long)d.NX * d.NY};
  const double dinv[3] = {dx_i[i + d.ng], dy_i[j + d.ng], dz_i[k + d.ng]};
  // g[a][b] = d u_a / d x_b
  double g[3][3];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) {
      if (a >= d.ndim || b >= d.ndim) { g[a][b] = 0.0; continue; }
      const long s = st[b];
      auto u = [&](int l) {
        const long cc = c + l * s;
        const double rho_i = 1.0 / v[cc];
        return v[(long)(1 + a) * d.nc + cc] * rho_i;
      };
      if (d.phys) {
        const int pos = b == 0 ? i : (b == 1 ? j : k), n = b == 0 ? d.nx : (b == 1 ? d.ny : d.nz);
        g[a][b] = d_deriv_line(u, dinv[b], pos, n, (d.phys >> (2 * b)) & 1,
                               (d.phys >> (2 * b + 1)) & 1);
        continue;
      }
      g[a][b] = d_deriv_central(u, dinv[b]);
    }
  double div, vort, wrk;
  if (d.ndim == 2) {
    div = g[0][0] + g[1][1];
    div = div * div;
    wrk = g[1][0] - g[0][1];
    vort = wrk * wrk;
  } else {
    div = g[0][0] + g[1][1] + g[2][2];
    div = div * div;
    wrk = g[2][1] - g[1][2];
    vort = wrk * wrk;
    wrk = g[0][2] - g[2][0];
    wrk = wrk * wrk;
    vort = vort + wrk;
    wrk = g[1][0] - g[0][1];
    wrk = wrk * wrk;
    vort = vort + wrk;
  }
  const double ducloc = div / (div + vort + 1.0e-30);
  if (ducloc > treduc) sensor[c] = 1;
}

// Block order of the kernels that take 7-point stencils along y and z of
// tens of fields (k_visc_fused, k_rhs_update).  In storage order the seven
// planes of a z stencil are tens of MB apart and every XCD's L2 (4 MB) sees
// all of them, so each plane comes from beyond the L2 seven times.  Here the
// interior is cut into bands of rows that are walked along z, and each
// XCD (hardware blocks b, b + 8, ... share one) takes a contiguous part of
// that walk: the planes that its blocks in flight need are a few rows wide
// and mostly stay in its L2 (256^3: 24 GB fetched per k_rhs_update launch
// against 38 in storage order).  Launches at 256^3 with bands of 8 / 16 / 32
// rows, and one band: k_visc_fused 4.71 / 4.75 / 4.77 / 5.32 ms,
// k_rhs_update 6.44 / 6.43 / 6.38 / 7.22 (6.57 in storage order); at 193 x
// 129 x 97 0.81 / 0.79 / 0.79 / 0.82 and 1.05 / 0.99 / 0.98 / 1.08.
struct IzBand {
  int n;     // bands of about IZ_BAND_ROWS rows, one row more or less
  int bpk;   // blocks per band and plane
  long nb;   // blocks in all (bands x planes x bpk)
};
#ifndef IZ_BAND_ROWS
#define IZ_BAND_ROWS 32
#endif
static IzBand band_of(const IzDims &d, int bs) {
  IzBand b;
  b.n = (d.ny + IZ_BAND_ROWS / 2) / IZ_BAND_ROWS;
  if (b.n < 1) b.n = 1;
  b.bpk = (int)iz_blocks((long)((d.ny + b.n - 1) / b.n) * d.nx, bs);
  b.nb = (long)b.n * d.nz * b.bpk;
  return b;
}
static unsigned band_grid(const IzBand &b) { return (unsigned)(((b.nb + 7) / 8) * 8); }
// the cell of thread t of block blk (bs threads); false: none
__device__ inline bool band_cell(const IzDims &d, const IzBand &b, unsigned blk, int bs, int t,
                                 int &i, int &j, int &k) {
  const long per = (b.nb + 7) / 8, L = (long)(blk % 8) * per + blk / 8;
  if (L >= b.nb) return false;
  const long bp = (long)b.bpk * d.nz;
  const int band = (int)(L / bp), r = (int)(L - band * bp);
  k = r / b.bpk;
  const int idx = (r - k * b.bpk) * bs + t;
  const int j0 = (int)((long)band * d.ny / b.n), rows = (int)((long)(band + 1) * d.ny / b.n) - j0;
  if (idx >= rows * d.nx) return false;
  const int q = idx / d.nx;
  j = j0 + q;
  i = idx - q * d.nx;
  return true;
}

// ===================================================================
// Viscous and species-diffusion fluxes: viscflux_xy / viscflux_xyz
// (module_viscflux.f90:721-1135, 1660-2189), periodic faces.
// ===================================================================

// velocities and mole fractions on a domain (molefrac :1669-1698)
__global__ void k_visc_prim(IzDims d, IzDomSet ds, const double *__restrict__ v,
                            const double *__restrict__ W_i, double *__restrict__ prim) {
  long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int i, j, k, dom;
  if (!domset_cell(ds, tid, dom, i, j, k)) return;
  long c = iz_cidx(d, i, j, k);
  double r0 = v[c];
  for (int l = 0; l < IZ_NRV; l++)
    prim[(3 + l) * d.nc + c] = v[(IZ_NIV + l) * d.nc + c] / (r0 * W_i[c] * c_thd.Wc[l]);
  double rho_i = 1.0 / r0;
  for (int q = 0; q < d.ndim; q++) prim[q * d.nc + c] = v[(1 + q) * d.nc + c] * rho_i;
}

// mixture-averaged transport of one cell (prim_vis_vars :989-1230)
#if IZ_NG == 4
// WENO7 keeps the reference's expressions: its weights lift differences in
// the last bit of the transport to 2e-10 of the state over 66 iterations of a
// shock tube, and its time is in the faces.
// FRESH: the tables at an index offset by z, see d_newton_cell
template <bool FRESH = false>
__device__ inline void d_transport(double rho, double T, double W_i, const double *Xa, double *dm,
                                   double &mu, double &ct, bool want_mu, int sym,
                                   int z = 0) {
  const double eps = 1.0e-12;
  double Kl = 0.5 * 1.0e-5 / c_thd.laminf;
  double Ku = 1.0e-1 / c_thd.muinf;
  double lt1 = log(T * c_thd.Tinf);
  double lt2 = lt1 * lt1;
  double lt3 = lt2 * lt1;
  double P = rho * T * W_i;
  double Kd = 1.0e-4 * c_thd.p0 / (c_thd.pinf * c_thd.Dinf);
  for (int m = 0; m < IZ_NRV; m++) {
    double wrk1 = 0.0, s = 0.0;
    for (int l = 0; l < IZ_NRV; l++) {
      if (m == l) continue;
      const double *cf = c_thd.CofD[m][l];
      double dkj = 0.0;
      dkj = dkj + cf[0] * 1.0;
      dkj = dkj + cf[1] * lt1;
      dkj = dkj + cf[2] * lt2;
      dkj = dkj + cf[3] * lt3;
      double xe = Xa[l] + eps;
      wrk1 = wrk1 + xe * c_thd.Wc[l] * W_i;
      s = s + xe * (1.0 / exp(dkj));
    }
    dm[m] = wrk1 * Kd / (s * P);
  }
  double w1 = 0.0, cc = 0.0;
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) {
    const double *cf = c_thd.CofLam[l];
    double s = 0.0;
    s = s + cf[0] * 1.0;
    s = s + cf[1] * lt1;
    s = s + cf[2] * lt2;
    s = s + cf[3] * lt3;
    double c1 = exp(s), c2 = Xa[l];
    cc = cc + c2 / c1;
    w1 = w1 + c2 * c1;
  }
  ct = Kl * (1.0 / cc + w1);
  mu = 0.0;
  if (!want_mu) return;
  double eta[IZ_NRV];
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) {
    const double *cf = c_thd.CofEta[l];
    double s = 0.0;
    s = s + cf[0] * 1.0;
    s = s + cf[1] * lt1;
    s = s + cf[2] * lt2;
    s = s + cf[3] * lt3;
    eta[l] = exp(s);
  }
  double mus = 0.0;
#pragma unroll
  for (int m = 0; m < IZ_NRV; m++) {
    double c4 = 0.0;
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++) {
      double c3 = 1.0 + c_thd.wilke_c1[m][l] * sqrt(eta[m] / eta[l]);
      double c2 = c3 * c3 * c_thd.wilke_c2[m][l];
      c4 = c4 + c2 * Xa[l];
    }
    mus = mus + Ku * (eta[m] * Xa[m] / c4);
  }
  mu = mus;
}
#else
// The exponentials are most of the work: D_kl is symmetric where the fits are
// (sym, checked when the context is made), so 36 serve the 72 pairs, 1 / D_kl
// is the exponential of the negated fit, and the ratios sqrt(eta_m / eta_l) of
// Wilke's rule are products of exp(+-s / 2).  54 exponentials and 36
// reciprocals per cell where the reference's expressions take 90, 162
// divisions and 81 square roots (k_visc_fused at 160^3 1.53 -> 1.31 ms, of
// which the rest is memory).
// FRESH: the tables at an index offset by z, see d_newton_cell
template <bool FRESH = false>
__device__ inline void d_transport(double rho, double T, double W_i, const double *Xa, double *dm,
                                   double &mu, double &ct, bool want_mu, int sym,
                                   int z = 0) {
#pragma clang fp contract(on)
  const double eps = 1.0e-12;
  const double lt1 = d_log(T * c_thd.Tinf);
  const double lt2 = lt1 * lt1;
  const double lt3 = lt2 * lt1;
  auto fit = [&](const double *cf) { return cf[0] + cf[1] * lt1 + cf[2] * lt2 + cf[3] * lt3; };
  {
    const double P = rho * T * W_i;
    const double Kd = 1.0e-4 * c_thd.p0 / (c_thd.pinf * c_thd.Dinf);
    double s[IZ_NRV], xe[IZ_NRV];
#pragma unroll
    for (int m = 0; m < IZ_NRV; m++) {
      s[m] = 0.0;
      xe[m] = Xa[m] + eps;
    }
#pragma unroll
    for (int m = 0; m < IZ_NRV; m++)
#pragma unroll
      for (int l = m + 1; l < IZ_NRV; l++) {
        const double e = d_exp(-fit(c_thd.CofD[FRESH ? m + z : m][l]));
        double f = e;
        if (!sym) f = d_exp(-fit(c_thd.CofD[FRESH ? l + z : l][m]));
        s[m] += xe[l] * e;
        s[l] += xe[m] * f;
      }
    // sum over the other species of xe W, from both ends (a difference
    // from the total would cancel where one species is nearly all)
    double up[IZ_NRV], dn = 0.0;
    up[0] = 0.0;
#pragma unroll
    for (int m = 1; m < IZ_NRV; m++) up[m] = up[m - 1] + xe[m - 1] * c_thd.Wc[m - 1];
    const double kp = Kd * W_i / P;
#pragma unroll
    for (int m = IZ_NRV - 1; m >= 0; m--) {
      dm[m] = (up[m] + dn) * kp * d_rcp(s[m]);
      dn += xe[m] * c_thd.Wc[m];
    }
  }
  double w1 = 0.0, cc = 0.0;
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) {
    const double c1 = d_exp(fit(c_thd.CofLam[FRESH ? l + z : l]));
    cc += Xa[l] * d_rcp(c1);
    w1 += Xa[l] * c1;
  }
  ct = (0.5 * 1.0e-5 / c_thd.laminf) * (1.0 / cc + w1);
  mu = 0.0;
  if (!want_mu) return;
  double h[IZ_NRV], g[IZ_NRV];  // sqrt(eta) and its reciprocal
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) {
    h[l] = d_exp(0.5 * fit(c_thd.CofEta[FRESH ? l + z : l]));
    g[l] = d_rcp(h[l]);
  }
  double mus = 0.0;
#pragma unroll
  for (int m = 0; m < IZ_NRV; m++) {
    double c4 = 0.0;
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++) {
      const double c3 = 1.0 + c_thd.wilke_c1[FRESH ? m + z : m][l] * (h[m] * g[l]);
      c4 += c3 * c3 * c_thd.wilke_c2[FRESH ? m + z : m][l] * Xa[l];
    }
    mus += h[m] * h[m] * Xa[m] / c4;
  }
  mu = (1.0e-1 / c_thd.muinf) * mus;
}
#endif

// Gradients and viscous fluxes in one pass (d?_fixed1 + the flux part of
// viscflux_xy/_xyz, module_viscflux.f90:721-1135, 1660-2189).  The
// reference stores the first derivatives of u, v, w, T and X_k for the
// interior, copies them to the ghost slabs (comm) and evaluates the fluxes on
// the interior and on each ghost slab.  Here each cell takes its derivatives
// straight from the primitives: an interior cell at itself, a ghost-slab cell
// at its periodic image in the interior, which is the value the copy would
// have brought.  Everything else (transport, v, T, W_i, h_k) is read at the
// cell itself, as in the reference.  Only the diffusion fluxes rho Y_k V_k
// (into the species slots of fd) and the stresses and heat flux (sf) are
// stored; the derivative slots of fd are not written.
template <bool PHYS>
__global__ void __attribute__((amdgpu_flat_work_group_size(128, 128), amdgpu_waves_per_eu(2)))
k_visc_fused(IzDims d, IzBand bd, IzDomSet ds, int sym, double sqgmr, double rvd0, double rlam0,
             const double *__restrict__ v, const double *__restrict__ T,
             const double *__restrict__ W_i, const double *__restrict__ ha,
             const double *__restrict__ prim, const double *__restrict__ dx_i,
             const double *__restrict__ dy_i, const double *__restrict__ dz_i,
             double *__restrict__ fd, double *__restrict__ sf) {
  // the interior in band order, then the ghost slabs
  int i, j, k, dom = 0;
  const unsigned nbi = (unsigned)(((bd.nb + 7) / 8) * 8);
  if (blockIdx.x < nbi) {
    if (!band_cell(d, bd, blockIdx.x, 128, threadIdx.x, i, j, k)) return;
  } else {
    const long tid = (long)(blockIdx.x - nbi) * 128 + threadIdx.x;
    if (!domset_cell(ds, tid, dom, i, j, k)) return;
  }
  const long nc = d.nc;
  const long c = iz_cidx(d, i, j, k);
  // derivative location: the periodic image of a ghost-slab cell
  int ii = i, jj = j, kk = k;
  if (dom == -1) ii += d.nx; else if (dom == 1) ii -= d.nx;
  else if (dom == -2) jj += d.ny; else if (dom == 2) jj -= d.ny;
  else if (dom == -3) kk += d.nz; else if (dom == 3) kk -= d.nz;
  const long cd = iz_cidx(d, ii, jj, kk);
  const long sx = 1, sy = d.NX, sz = d.NX * d.NY;
  const double dxi = dx_i[ii + d.ng], dyi = dy_i[jj + d.ng], dzi = dz_i[kk + d.ng];
  const double twothirds = 2.0 / 3.0;
  double X[IZ_NRV], dm[IZ_NRV], mu, ct;
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) X[l] = prim[(3 + l) * nc + c];
  const double r0 = v[c], Wi = W_i[c];
  d_transport(r0, T[c], Wi, X, dm, mu, ct, true, sym);
  double rho_i = 1.0 / r0;
  double uxs = v[nc + c] * rho_i, vys = v[2 * nc + c] * rho_i, wzs = v[3 * nc + c] * rho_i;
  double rmu = -sqgmr * mu;
  double rvd = rvd0 * r0;
  double rlam = -rlam0 * ct;
  if (d.ndim == 3) {
    const int nfluid = 12;
    const double f1 = d_deriv_dir<PHYS>(d, prim, cd, 0, ii, dxi), f2 = d_deriv_dir<PHYS>(d, prim, cd, 1, jj, dyi),
                 f3 = d_deriv_dir<PHYS>(d, prim, cd, 2, kk, dzi);
    const double f4 = d_deriv_dir<PHYS>(d, prim + nc, cd, 0, ii, dxi), f5 = d_deriv_dir<PHYS>(d, prim + nc, cd, 1, jj, dyi),
                 f6 = d_deriv_dir<PHYS>(d, prim + nc, cd, 2, kk, dzi);
    const double f7 = d_deriv_dir<PHYS>(d, prim + 2 * nc, cd, 0, ii, dxi),
                 f8 = d_deriv_dir<PHYS>(d, prim + 2 * nc, cd, 1, jj, dyi),
                 f9 = d_deriv_dir<PHYS>(d, prim + 2 * nc, cd, 2, kk, dzi);
    double sxx = twothirds * rmu * (f1 + f1 - (f5 + f9));
    double sxy = rmu * (f4 + f2);
    double sxz = rmu * (f7 + f3);
    double syy = twothirds * rmu * (f5 + f5 - (f1 + f9));
    double syz = rmu * (f8 + f6);
    double szz = twothirds * rmu * (f9 + f9 - (f1 + f5));
    double gx[IZ_NRV], gy[IZ_NRV], gz[IZ_NRV];
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++) {
      const double *a = prim + (3 + l) * nc;
      gx[l] = d_deriv_dir<PHYS>(d, a, cd, 0, ii, dxi);
      gy[l] = d_deriv_dir<PHYS>(d, a, cd, 1, jj, dyi);
      gz[l] = d_deriv_dir<PHYS>(d, a, cd, 2, kk, dzi);
    }
    double vdcx = 0.0, vdcy = 0.0, vdcz = 0.0;
#pragma unroll
    for (int l = 1; l <= IZ_NRV; l++) {
      double wrk = dm[l - 1] * c_thd.Wc[l - 1] * Wi;
      vdcx = vdcx + wrk * gx[l - 1];
      vdcy = vdcy + wrk * gy[l - 1];
      vdcz = vdcz + wrk * gz[l - 1];
    }
    double vdhx = 0.0, vdhy = 0.0, vdhz = 0.0;
#pragma unroll
    for (int l = 1; l <= IZ_NRV; l++) {
      double Ya = v[(IZ_NIV + l - 1) * nc + c] * rho_i;
      double vdtx = vdcx * Ya, vdty = vdcy * Ya, vdtz = vdcz * Ya;
      double wrk = -dm[l - 1] * c_thd.Wc[l - 1] * Wi;
      vdtx = vdtx + wrk * gx[l - 1];
      vdty = vdty + wrk * gy[l - 1];
      vdtz = vdtz + wrk * gz[l - 1];
      double jx = rvd * vdtx, jy = rvd * vdty, jz = rvd * vdtz;
      fd[(long)(nfluid + 3 * l - 3) * nc + c] = jx;
      fd[(long)(nfluid + 3 * l - 2) * nc + c] = jy;
      fd[(long)(nfluid + 3 * l - 1) * nc + c] = jz;
      double h = ha[(long)(l - 1) * nc + c];
      vdhx = vdhx + h * jx;
      vdhy = vdhy + h * jy;
      vdhz = vdhz + h * jz;
    }
    const double tx = d_deriv_dir<PHYS>(d, T, cd, 0, ii, dxi), ty = d_deriv_dir<PHYS>(d, T, cd, 1, jj, dyi),
                 tz = d_deriv_dir<PHYS>(d, T, cd, 2, kk, dzi);
    sf[0 * nc + c] = sxx; sf[1 * nc + c] = sxy; sf[2 * nc + c] = sxz;
    sf[3 * nc + c] = syy; sf[4 * nc + c] = syz; sf[5 * nc + c] = szz;
    sf[6 * nc + c] = uxs * sxx + vys * sxy + wzs * sxz + rlam * tx + vdhx;
    sf[7 * nc + c] = uxs * sxy + vys * syy + wzs * syz + rlam * ty + vdhy;
    sf[8 * nc + c] = uxs * sxz + vys * syz + wzs * szz + rlam * tz + vdhz;
  } else {
    const int nfluid = 6;
    const double f1 = d_deriv_dir<PHYS>(d, prim, cd, 0, ii, dxi), f2 = d_deriv_dir<PHYS>(d, prim, cd, 1, jj, dyi);
    const double f3 = d_deriv_dir<PHYS>(d, prim + nc, cd, 0, ii, dxi), f4 = d_deriv_dir<PHYS>(d, prim + nc, cd, 1, jj, dyi);
    double sxx = twothirds * rmu * (f1 + f1 - f4);
    double sxy = rmu * (f3 + f2);
    double syy = twothirds * rmu * (f4 + f4 - f1);
    double gx[IZ_NRV], gy[IZ_NRV];
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++) {
      const double *a = prim + (3 + l) * nc;
      gx[l] = d_deriv_dir<PHYS>(d, a, cd, 0, ii, dxi);
      gy[l] = d_deriv_dir<PHYS>(d, a, cd, 1, jj, dyi);
    }
    double vdcx = 0.0, vdcy = 0.0;
#pragma unroll
    for (int l = 1; l <= IZ_NRV; l++) {
      double wrk = dm[l - 1] * c_thd.Wc[l - 1] * Wi;
      vdcx = vdcx + wrk * gx[l - 1];
      vdcy = vdcy + wrk * gy[l - 1];
    }
    double vdhx = 0.0, vdhy = 0.0;
#pragma unroll
    for (int l = 1; l <= IZ_NRV; l++) {
      double Ya = v[(IZ_NIV + l - 1) * nc + c] * rho_i;
      double vdtx = vdcx * Ya, vdty = vdcy * Ya;
      double wrk = -dm[l - 1] * c_thd.Wc[l - 1] * Wi;
      vdtx = vdtx + wrk * gx[l - 1];
      vdty = vdty + wrk * gy[l - 1];
      double jx = rvd * vdtx, jy = rvd * vdty;
      fd[(long)(nfluid + 2 * l - 2) * nc + c] = jx;
      fd[(long)(nfluid + 2 * l - 1) * nc + c] = jy;
      double h = ha[(long)(l - 1) * nc + c];
      vdhx = vdhx + h * jx;
      vdhy = vdhy + h * jy;
    }
    const double tx = d_deriv_dir<PHYS>(d, T, cd, 0, ii, dxi), ty = d_deriv_dir<PHYS>(d, T, cd, 1, jj, dyi);
    sf[0 * nc + c] = sxx; sf[1 * nc + c] = sxy; sf[2 * nc + c] = syy;
    sf[3 * nc + c] = uxs * sxx + vys * sxy + rlam * tx + vdhx;
    sf[4 * nc + c] = uxs * sxy + vys * syy + rlam * ty + vdhy;
  }
}

// viscous divergence of one cell into out[0..13] (0 for the continuity and,
// in 2-D, the z-momentum equations), :2087-2183
template <bool PHYS>
__device__ inline void d_visc_div(const IzDims &d, long c, int i, int j, int k,
                                  const double *__restrict__ sf, const double *__restrict__ fd,
                                  const double *__restrict__ dx_i, const double *__restrict__ dy_i,
                                  const double *__restrict__ dz_i, double *out, bool *has) {
  const long nc = d.nc, sx = 1, sy = d.NX, sz = d.NX * d.NY;
  const double dxi = dx_i[i + d.ng], dyi = dy_i[j + d.ng], dzi = dz_i[k + d.ng];
  for (int m = 0; m < IZ_NV; m++) { out[m] = 0.0; has[m] = false; }
  if (d.ndim == 3) {
    const int nf = 12;
    double wx, wy, wz;
    wx = d_deriv_dir<PHYS>(d, sf + 0 * nc, c, 0, i, dxi); wy = d_deriv_dir<PHYS>(d, sf + 1 * nc, c, 1, j, dyi);
    wz = d_deriv_dir<PHYS>(d, sf + 2 * nc, c, 2, k, dzi); out[1] = wx + wy + wz;
    wx = d_deriv_dir<PHYS>(d, sf + 1 * nc, c, 0, i, dxi); wy = d_deriv_dir<PHYS>(d, sf + 3 * nc, c, 1, j, dyi);
    wz = d_deriv_dir<PHYS>(d, sf + 4 * nc, c, 2, k, dzi); out[2] = wx + wy + wz;
    wx = d_deriv_dir<PHYS>(d, sf + 2 * nc, c, 0, i, dxi); wy = d_deriv_dir<PHYS>(d, sf + 4 * nc, c, 1, j, dyi);
    wz = d_deriv_dir<PHYS>(d, sf + 5 * nc, c, 2, k, dzi); out[3] = wx + wy + wz;
    wx = d_deriv_dir<PHYS>(d, sf + 6 * nc, c, 0, i, dxi); wy = d_deriv_dir<PHYS>(d, sf + 7 * nc, c, 1, j, dyi);
    wz = d_deriv_dir<PHYS>(d, sf + 8 * nc, c, 2, k, dzi); out[4] = wx + wy + wz;
    has[1] = has[2] = has[3] = has[4] = true;
    for (int l = 1; l <= IZ_NRV; l++) {
      wx = d_deriv_dir<PHYS>(d, fd + (long)(nf + 3 * l - 3) * nc, c, 0, i, dxi);
      wy = d_deriv_dir<PHYS>(d, fd + (long)(nf + 3 * l - 2) * nc, c, 1, j, dyi);
      wz = d_deriv_dir<PHYS>(d, fd + (long)(nf + 3 * l - 1) * nc, c, 2, k, dzi);
      out[IZ_NIV + l - 1] = wx + wy + wz;
      has[IZ_NIV + l - 1] = true;
    }
  } else {
    const int nf = 6;
    double wx, wy;
    wx = d_deriv_dir<PHYS>(d, sf + 0 * nc, c, 0, i, dxi); wy = d_deriv_dir<PHYS>(d, sf + 1 * nc, c, 1, j, dyi);
    out[1] = wx + wy;
    wx = d_deriv_dir<PHYS>(d, sf + 1 * nc, c, 0, i, dxi); wy = d_deriv_dir<PHYS>(d, sf + 2 * nc, c, 1, j, dyi);
    out[2] = wx + wy;
    wx = d_deriv_dir<PHYS>(d, sf + 3 * nc, c, 0, i, dxi); wy = d_deriv_dir<PHYS>(d, sf + 4 * nc, c, 1, j, dyi);
    out[4] = wx + wy;
    has[1] = has[2] = has[4] = true;
    for (int l = 1; l <= IZ_NRV; l++) {
      wx = d_deriv_dir<PHYS>(d, fd + (long)(nf + 2 * l - 2) * nc, c, 0, i, dxi);
      wy = d_deriv_dir<PHYS>(d, fd + (long)(nf + 2 * l - 1) * nc, c, 1, j, dyi);
      out[IZ_NIV + l - 1] = wx + wy;
      has[IZ_NIV + l - 1] = true;
    }
  }
}

template <bool PHYS>
__global__ void k_visc_apply(IzDims d, const double *__restrict__ sf,
                             const double *__restrict__ fd, const double *__restrict__ dx_i,
                             const double *__restrict__ dy_i, const double *__restrict__ dz_i,
                             double *__restrict__ fl) {
  long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long ncin = (long)d.nx * d.ny * d.nz;
  if (tid >= ncin) return;
  int i = (int)(tid % d.nx);
  long r = tid / d.nx;
  int j = (int)(r % d.ny), k = (int)(r / d.ny);
  long c = iz_cidx(d, i, j, k);
  double out[IZ_NV];
  bool has[IZ_NV];
  d_visc_div<PHYS>(d, c, i, j, k, sf, fd, dx_i, dy_i, dz_i, out, has);
  for (int m = 0; m < IZ_NV; m++)
    if (has[m]) fl[m * d.nc + c] = fl[m * d.nc + c] + out[m];
}

// ===================================================================
// Fused right-hand side + SSP-RK3 stage update + force_sumY + Newton probe
// (rk3, module_solver.f90:769-847).  mode 0: write f only; mode 1: update;
// mode 2: update from the step's first state, which is kept in v0.
// ===================================================================
#ifndef IZ_RHS_WAVES
#define IZ_RHS_WAVES 2
#endif
// SEAMS: the run reproduces a decomposed one (d.np > 1); a rank's last cell
// takes its right face from the seam arrays
template <bool PHYS, bool SEAMS>
__global__ void __attribute__((amdgpu_flat_work_group_size(256, 256),
                               amdgpu_waves_per_eu(IZ_RHS_WAVES, IZ_RHS_WAVES)))
k_rhs_update(IzDims d, IzBand bd, int mode, const double *__restrict__ Fx, const double *__restrict__ Fy,
             const double *__restrict__ Fz, IzSeams sm, int vis, const double *__restrict__ sf,
             const double *__restrict__ fd, const double *__restrict__ dx_i,
             const double *__restrict__ dy_i, const double *__restrict__ dz_i,
             const double *__restrict__ dtp, double bk, double ck,
             double *__restrict__ v0, double *__restrict__ v, double *__restrict__ fout,
             int forcesum, const double *__restrict__ T, double eps,
             unsigned long long *__restrict__ mask) {
  // one cell per thread (a grid-stride loop here was 2.7x slower: the
  // y/z face and viscous stencil neighbours lose their L2 reuse)
  unsigned long long msk = 0ull, neg = 0ull;
  int i, j, k;
  if (band_cell(d, bd, blockIdx.x, 256, threadIdx.x, i, j, k)) {
    long c = iz_cidx(d, i, j, k);
    const long nfx = (long)(d.nx + 1) * d.ny * d.nz, nfy = (long)d.nx * (d.ny + 1) * d.nz,
               nfz = (long)d.nx * d.ny * (d.nz + 1);
    const long fxl = i + (long)(d.nx + 1) * (j + (long)d.ny * k);
    const long fyl = i + (long)d.nx * (j + (long)(d.ny + 1) * k);
    const long fzl = i + (long)d.nx * (j + (long)d.ny * k);
    const double dxi = dx_i[i + d.ng], dyi = dy_i[j + d.ng], dzi = dz_i[k + d.ng];
    double f[IZ_NV];
    if constexpr (SEAMS) {
      const long sx = iz_seam(i, d.nx, d.np[0], j + (long)d.ny * k);
      const long sy = iz_seam(j, d.ny, d.np[1], i + (long)d.nx * k);
      const long sz = iz_seam(k, d.nz, d.np[2], i + (long)d.nx * j);
#pragma unroll
      for (int m = 0; m < IZ_NV; m++) {
        double Fr = sx >= 0 ? sm.F[0][m * sm.n[0] + sx] : Fx[m * nfx + fxl + 1];
        double df = (Fr - Fx[m * nfx + fxl]) * dxi;
        f[m] = df * 1.0;
        if (d.ndim >= 2) {
          Fr = sy >= 0 ? sm.F[1][m * sm.n[1] + sy] : Fy[m * nfy + fyl + d.nx];
          df = (Fr - Fy[m * nfy + fyl]) * dyi;
          f[m] = f[m] + df * 1.0;
        }
        if (d.ndim == 3) {
          Fr = sz >= 0 ? sm.F[2][m * sm.n[2] + sz] : Fz[m * nfz + fzl + (long)d.nx * d.ny];
          df = (Fr - Fz[m * nfz + fzl]) * dzi;
          f[m] = f[m] + df * 1.0;
        }
      }
    } else {
#pragma unroll
      for (int m = 0; m < IZ_NV; m++) {
        double df = (Fx[m * nfx + fxl + 1] - Fx[m * nfx + fxl]) * dxi;
        f[m] = df * 1.0;
        if (d.ndim >= 2) {
          df = (Fy[m * nfy + fyl + d.nx] - Fy[m * nfy + fyl]) * dyi;
          f[m] = f[m] + df * 1.0;
        }
        if (d.ndim == 3) {
          df = (Fz[m * nfz + fzl + (long)d.nx * d.ny] - Fz[m * nfz + fzl]) * dzi;
          f[m] = f[m] + df * 1.0;
        }
      }
    }
    if (vis) {
      double out[IZ_NV];
      bool has[IZ_NV];
      d_visc_div<PHYS>(d, c, i, j, k, sf, fd, dx_i, dy_i, dz_i, out, has);
#pragma unroll
      for (int m = 0; m < IZ_NV; m++)
        if (has[m]) f[m] = f[m] + out[m];
    }
    if (mode == 0) {
#pragma unroll
      for (int m = 0; m < IZ_NV; m++) fout[m * d.nc + c] = f[m];
    } else {
      const double dt = *dtp;
      double vc[IZ_NV];
#pragma unroll
      for (int m = 0; m < IZ_NV; m++) {
        const double vs = v[m * d.nc + c];
        double vb = vs;
        if (mode == 2) v0[m * d.nc + c] = vs;
        else vb = v0[m * d.nc + c];
        vc[m] = vb * bk + ck * (vs - dt * f[m]);
      }
      if (forcesum) d_force_sumY(vc);
#pragma unroll
      for (int m = 0; m < IZ_NV; m++) v[m * d.nc + c] = vc[m];
      msk = d_newton_probe<false>(vc, T[c], eps, neg);
    }
  }
  if (mode != 0) block_or_probe(msk, neg, mask);
}

// ===================================================================
// Time step: timestep (module_solver.f90:202-408)
// ===================================================================
// the convective limit's rate of one cell
__device__ inline double d_dt_conv(const IzDims &d, const double *__restrict__ v, double T, double Wi,
                                   double cp, long c, double dxi, double dyi, double dzi) {
  const double rho_i = 1.0 / v[c];
  const double ux = v[d.nc + c] * rho_i, vy = v[2 * d.nc + c] * rho_i,
               wz = v[3 * d.nc + c] * rho_i;
  double gamma = c_thd.gam2 * Wi / cp;
  gamma = 1.0 / (1.0 - gamma);
  const double P = v[c] * T * Wi;
  const double cs = sqrt(gamma * P * rho_i);
  return fmax(fmax((fabs(ux) + cs) * dxi, (fabs(vy) + cs) * dyi), (fabs(wz) + cs) * dzi);
}
__global__ void k_dt_conv(IzDims d, const double *__restrict__ v, const double *__restrict__ T,
                          const double *__restrict__ W_i, const double *__restrict__ cp,
                          const double *__restrict__ dx_i, const double *__restrict__ dy_i,
                          const double *__restrict__ dz_i, double *__restrict__ red) {
  const long ncin = (long)d.nx * d.ny * d.nz;
  double dtc = 0.0;
  for (long tid = (long)blockIdx.x * blockDim.x + threadIdx.x; tid < ncin;
       tid += (long)gridDim.x * blockDim.x) {
    int i = (int)(tid % d.nx);
    long r = tid / d.nx;
    int j = (int)(r % d.ny), k = (int)(r / d.ny);
    long c = iz_cidx(d, i, j, k);
    dtc = fmax(dtc, d_dt_conv(d, v, T[c], W_i[c], cp[c], c, dx_i[i + d.ng], dy_i[j + d.ng],
                              dz_i[k + d.ng]));
  }
  block_extreme_pos<1, true>(&dtc, red);
}

__device__ inline double d_filter_delta2(const IzDims &d, const double *dx_i, const double *dy_i,
                                         const double *dz_i, int i, int j, int k) {
  double delta;
  if (d.ndim == 3)
    delta = 1.0 / pow(dx_i[i + d.ng] * dy_i[j + d.ng] * dz_i[k + d.ng], 1.0 / 3.0);
  else if (d.ndim == 2)
    delta = 1.0 / sqrt(dx_i[i + d.ng] * dy_i[j + d.ng]);
  else
    delta = 1.0 / dx_i[i + d.ng];
  return delta * delta;
}

// the convective limit and one pass over the transport properties: per species the maximum of the
// mixture diffusivity and the minimum of Delta^2 / D_l, and the minimum of
// Delta^2 rho / (lambda / cp).  The species whose diffusivity maximum is
// the largest is only known after the whole grid is reduced; keeping the
// minimum for every species lets k_dt_final pick that species' value, which
// is the minimum the reference takes over that one species.
__global__ void __attribute__((amdgpu_flat_work_group_size(128, 128), amdgpu_waves_per_eu(2, 2)))
k_dt_visc(IzDims d, int sym, const double *__restrict__ v, const double *__restrict__ T,
                          const double *__restrict__ W_i, const double *__restrict__ cp,
                          const double *__restrict__ dx_i, const double *__restrict__ dy_i,
                          const double *__restrict__ dz_i, double *__restrict__ red) {
  const long ncin = (long)d.nx * d.ny * d.nz;
  double dmax[IZ_NRV], mins[IZ_NRV + 1], dtc = 0.0;
#pragma unroll
  for (int l = 0; l < IZ_NRV; l++) dmax[l] = 0.0;
#pragma unroll
  for (int l = 0; l <= IZ_NRV; l++) mins[l] = __longlong_as_double(0x7ff0000000000000LL);
  for (long tid = (long)blockIdx.x * blockDim.x + threadIdx.x; tid < ncin;
       tid += (long)gridDim.x * blockDim.x) {
    int i = (int)(tid % d.nx);
    long r = tid / d.nx;
    int j = (int)(r % d.ny), k = (int)(r / d.ny);
    long c = iz_cidx(d, i, j, k);
    double X[IZ_NRV], dm[IZ_NRV], mu, ct;
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++)
      X[l] = v[(IZ_NIV + l) * d.nc + c] / (v[c] * W_i[c] * c_thd.Wc[l]);
    int z = 0;
    asm volatile("" : "+s"(z));
    d_transport<true>(v[c], T[c], W_i[c], X, dm, mu, ct, false, sym, z);
    const double d2 = d_filter_delta2(d, dx_i, dy_i, dz_i, i, j, k);
#pragma unroll
    for (int l = 0; l < IZ_NRV; l++) {
      dmax[l] = fmax(dmax[l], dm[l]);
      mins[l] = fmin(mins[l], d2 / (dm[l] + 0.0));
    }
    mins[IZ_NRV] = fmin(mins[IZ_NRV], d2 * v[c] / (ct / cp[c] + 0.0));
    dtc = fmax(dtc, d_dt_conv(d, v, T[c], W_i[c], cp[c], c, dx_i[i + d.ng], dy_i[j + d.ng],
                              dz_i[k + d.ng]));
  }
  block_extreme_pos<1, true>(&dtc, red);
  block_extreme_pos<IZ_NRV, true>(dmax, red + 1);
  block_extreme_pos<IZ_NRV + 1, false>(mins, red + 12);
}

// red layout: [0] dtc, [1..9] dm max, [12..20] min d2/D_l per species,
// [21] min d2 rho cp/lambda
// ts: [0..3] dt_4, [4] dtmin (in: previous), [5] DTmax (K)
__device__ inline void d_dt_init(double *red, int t) {
  if (t == 0) red[0] = 1.0;
  if (t >= 1 && t <= 9) red[t] = 0.0;
  if (t >= 12 && t <= 21) red[t] = __longlong_as_double(0x7ff0000000000000LL);
}
__global__ void k_dt_init(double *red) { d_dt_init(red, threadIdx.x); }

// the limits from the reductions, which are reset for the next call (64
// threads)
__global__ void k_dt_final(double *__restrict__ red, double CFL, double CFLmin, double Fo,
                           double CPR, int visdt, int reaction, double rvd0_i, double rlamcp0_i,
                           double *__restrict__ ts) {
  if (threadIdx.x == 0) {
    double dt4[4] = {1.0, 1.0, 1.0, 1.0};
    dt4[0] = CFL / red[0];
    if (visdt) {
      // species of the global diffusivity maximum: the first in species order
      double gmax = red[1];
      int ldmax = 0;
      for (int l = 1; l < IZ_NRV; l++)
        if (gmax < red[1 + l]) { gmax = red[1 + l]; ldmax = l; }
      dt4[1] = rvd0_i * Fo * red[12 + ldmax];
      dt4[2] = rlamcp0_i * Fo * red[12 + IZ_NRV];
    }
    if (reaction) {
      dt4[3] = ts[4] * CPR / ts[5];
      dt4[3] = fmin(dt4[3], 1.0);
      dt4[3] = fmax(dt4[3], dt4[0] * CFLmin / CFL);
    }
    double mn = dt4[0];
    for (int q = 1; q < 4; q++) mn = fmin(mn, dt4[q]);
    for (int q = 0; q < 4; q++) ts[q] = dt4[q];
    ts[4] = mn;
  }
  __syncthreads();
  d_dt_init(red, threadIdx.x);
}


// the functions of iz_math.h for their unit tests
__global__ void k_math_batch(int f, int n, const double *__restrict__ x, double *__restrict__ y) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  y[t] = f == 0 ? d_exp(x[t]) : f == 1 ? d_log(x[t]) : d_rcp(x[t]);
}

// batched wenorec for unit tests of the reconstruction itself
__global__ void k_wenorec_batch(int n, int js, const double *__restrict__ vp,
                                const double *__restrict__ vm, double *__restrict__ out) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  double a[6], b[6];
  for (int s = 0; s < 6; s++) { a[s] = vp[6 * t + s]; b[s] = vm[6 * t + s]; }
  double gl, gr;
  if (js) d_wenorec(a, b, gl, gr);
  else d_wenorec_nw(a, b, gl, gr);
  out[2 * t] = gl;
  out[2 * t + 1] = gr;
}

// explicit instantiations used by the API
template __global__ void k_euler_apply<0>(IzDims, const double *, long, const double *, int, double *,
                                              const double *, long);
template __global__ void k_euler_apply<1>(IzDims, const double *, long, const double *, int, double *,
                                              const double *, long);
template __global__ void k_euler_apply<2>(IzDims, const double *, long, const double *, int, double *,
                                              const double *, long);

// ===================================================================
// C ABI (include/izem_hip.h)
// ===================================================================
static IzBox domain_box(const IzDims &d, int dom) {
  IzBox b{0, d.nx - 1, 0, d.ny - 1, 0, d.nz - 1};
  switch (dom) {
    case -1: b.i0 = -d.ng; b.i1 = -1; break;
    case 1: b.i0 = d.nx; b.i1 = d.nx + d.ng - 1; break;
    case -2: b.j0 = -d.ng; b.j1 = -1; break;
    case 2: b.j0 = d.ny; b.j1 = d.ny + d.ng - 1; break;
    case -3: b.k0 = -d.ng; b.k1 = -1; break;
    case 3: b.k0 = d.nz; b.k1 = d.nz + d.ng - 1; break;
    // the Dirichlet rows: a face's first interior layer
    // (module_parallel.f90:1946-1957, 1983-1994)
    case -10: b.i1 = 0; break;
    case 10: b.i0 = d.nx - 1; break;
    case -20: b.j1 = 0; break;
    case 20: b.j0 = d.ny - 1; break;
    case -30: b.k1 = 0; break;
    case 30: b.k0 = d.nz - 1; break;
    default: break;
  }
  return b;
}
// probe-mask and iteration-count slot of a domain (slot 7 serves the
// Dirichlet rows, one per call)
static int mask_slot(int dom) { return (dom <= -10 || dom >= 10) ? 7 : dom + 3; }
static long box_count(const IzBox &b) {
  return (long)(b.i1 - b.i0 + 1) * (b.j1 - b.j0 + 1) * (b.k1 - b.k0 + 1);
}
static long n_interior(const IzDims &d) { return (long)d.nx * d.ny * d.nz; }
// the interior (where asked for) and the 2 * ndim ghost slabs, in domain_select's order; the
// slabs of a direction with physical faces are left out (the viscous fluxes
// there are never read: the derivative closures next to a physical face use
// interior points only)
static IzDomSet domain_set(const IzDims &d, bool interior) {
  IzDomSet s{};
  s.n = 0;
  s.first[0] = 0;
  for (int dom = -d.ndim; dom <= d.ndim; dom++) {
    const int dir = (dom < 0 ? -dom : dom) - 1;
    if (dom == 0 ? !interior : ((d.phys >> (2 * dir)) & 3)) continue;
    s.box[s.n] = domain_box(d, dom);
    s.dom[s.n] = dom;
    s.first[s.n + 1] = s.first[s.n] + box_count(s.box[s.n]);
    s.n++;
  }
  return s;
}

// the set of nd domains; capped: at most 16 blocks per CU and domain (kernels
// that reduce walk their cells), else one thread per cell
static IzNewtonSet newton_set(const izem_ctx *c, const int *doms, int nd, int capped) {
  IzNewtonSet s{};
  s.n = nd;
  s.first[0] = 0;
  for (int q = 0; q < 6; q++) {
    if (q < nd) {
      s.box[q] = domain_box(c->d, doms[q]);
      s.dom[q] = doms[q];
      s.slot[q] = mask_slot(doms[q]);
      const long n = box_count(s.box[q]);
      s.first[q + 1] = s.first[q] + (capped ? iz_blocks_capped(c, n, 256, 16) : iz_blocks(n, 256));
    } else {
      s.first[q + 1] = s.first[q];
    }
  }
  return s;
}

extern "C" int izem_create(izem_ctx **out, const izem_grid *g, const double *thd, long nthd,
                           const izem_opts *opts) {
  if (!out || !g || !thd || !opts) return IZEM_E_ARG;
  if (nthd != (long)(sizeof(IzThd) / sizeof(double))) return IZEM_E_ARG;
  if (g->ng != IZ_NG || g->ndim < 2 || g->ndim > 3 || g->nx < 2 * IZ_NG + 1 ||
      g->ny < 2 * IZ_NG + 1)
    return IZEM_E_ARG;
  if (g->ndim == 3 && g->nz < 2 * IZ_NG + 1) return IZEM_E_ARG;
  if (g->ndim == 2 && g->nz != 1) return IZEM_E_ARG;
  // face indices of a direction are 32-bit in the Euler kernels
  if ((long)(g->nx + 1) * (g->ny + 1) * (g->nz + 1) >= (1L << 31)) return IZEM_E_ARG;
  izem_ctx *c = (izem_ctx *)calloc(1, sizeof(izem_ctx));
  if (!c) return IZEM_E_NOMEM;
  {
    int dev = 0;
    c->ncu = 256;
    if (hipGetDevice(&dev) == hipSuccess)
      (void)hipDeviceGetAttribute(&c->ncu, hipDeviceAttributeMultiprocessorCount, dev);
  }
  IzDims &d = c->d;
  d.nx = g->nx; d.ny = g->ny; d.nz = g->nz; d.ng = g->ng; d.ndim = g->ndim;
  d.NX = d.nx + 2 * d.ng; d.NY = d.ny + 2 * d.ng; d.NZ = d.nz + 2 * d.ng;
  d.nc = d.NX * d.NY * d.NZ;
  d.np[0] = d.np[1] = d.np[2] = 1;
  c->o = *opts;
  if (hipStreamCreate(&c->own_stream) != hipSuccess) { free(c); return IZEM_E_HIP; }
  c->stream = c->own_stream;
  if (hipMemcpyToSymbol(HIP_SYMBOL(c_thd), thd, sizeof(IzThd)) != hipSuccess) {
    izem_destroy(c);
    return IZEM_E_HIP;
  }
  {
    const IzThd *t = (const IzThd *)thd;
    c->dsym = 1;
    for (int m = 0; m < IZ_NRV; m++)
      for (int l = 0; l < m; l++)
        if (memcmp(t->CofD[m][l], t->CofD[l][m], sizeof t->CofD[m][l])) c->dsym = 0;
  }
  {
    // see IzThx
    const IzThd *t = (const IzThd *)thd;
    IzThx x;
    x.tlo = t->Tpolymin[0];
    x.thi = t->Tpolymax[0];
    x.tlim = t->Tpolylim[0];
    for (int l = 0; l < IZ_NRV; l++) {
      if (t->Tpolymin[l] > x.tlo) x.tlo = t->Tpolymin[l];
      if (t->Tpolymax[l] < x.thi) x.thi = t->Tpolymax[l];
      if (t->Tpolylim[l] != x.tlim) x.thi = -1.0;  // no common range: never taken
      for (int r = 0; r < 2; r++) {
        const double *a = t->HeatCap[l][r];
        const double f = t->Wc_i[l] / t->Tinf, g = t->gam2 * t->Wc_i[l];
        for (int q = 0; q < 5; q++) {
          x.h[r][l][q] = f * a[q] / (q + 1);
          x.c[r][l][q] = g * a[q];
        }
        x.h[r][l][5] = f * a[5];
      }
    }
    if (hipMemcpyToSymbol(HIP_SYMBOL(c_thx), &x, sizeof x) != hipSuccess) {
      izem_destroy(c);
      return IZEM_E_HIP;
    }
  }
  c->nfaces[0] = (long)(d.nx + 1) * d.ny * d.nz;
  c->nfaces[1] = (long)d.nx * (d.ny + 1) * d.nz;
  c->nfaces[2] = (long)d.nx * d.ny * (d.nz + 1);
  c->nderiv = d.ndim * (d.ndim + 1) + d.ndim * IZ_NRV;
  c->nsf = (d.ndim == 3) ? 9 : 5;
  bool ok = true;
  for (int q = 0; q < d.ndim; q++)
    ok = ok && hipMalloc(&c->F[q], sizeof(double) * IZ_NV * c->nfaces[q]) == hipSuccess;
  ok = ok && hipMalloc(&c->prim, sizeof(double) * (3 + IZ_NRV) * d.nc) == hipSuccess;
  ok = ok && hipMalloc(&c->fd, sizeof(double) * c->nderiv * d.nc) == hipSuccess;
  ok = ok && hipMalloc(&c->sf, sizeof(double) * c->nsf * d.nc) == hipSuccess;
  ok = ok && hipMalloc(&c->v0, sizeof(double) * IZ_NV * d.nc) == hipSuccess;
  ok = ok && hipMalloc(&c->masks, sizeof(unsigned long long) * 2 * IZ_NEG_MASKS) == hipSuccess;
  ok = ok && hipMalloc(&c->negT_rec, sizeof(int) * IZ_NEG_MASKS * IZ_NEGT_MAX) == hipSuccess;
  ok = ok && hipMalloc(&c->status, sizeof(int) * 2) == hipSuccess;
  ok = ok && hipMalloc(&c->iters, sizeof(int) * 8) == hipSuccess;
  ok = ok && hipMalloc(&c->red, sizeof(double) * 24) == hipSuccess;
  ok = ok && hipMalloc(&c->ts, sizeof(double) * 6) == hipSuccess;
  if (!ok) { izem_destroy(c); return IZEM_E_NOMEM; }
  // fields are read at ghost edges/corners never; keep scratch defined
  ok = hipMemsetAsync(c->prim, 0, sizeof(double) * (3 + IZ_NRV) * d.nc, c->stream) == hipSuccess;
  ok = ok && hipMemsetAsync(c->fd, 0, sizeof(double) * c->nderiv * d.nc, c->stream) == hipSuccess;
  ok = ok && hipMemsetAsync(c->sf, 0, sizeof(double) * c->nsf * d.nc, c->stream) == hipSuccess;
  ok = ok && hipMemsetAsync(c->status, 0, sizeof(int) * 2, c->stream) == hipSuccess;
  // zero between Newton passes: k_newton_repair clears what a pass has set
  ok = ok && hipMemsetAsync(c->masks, 0, sizeof(unsigned long long) * 2 * IZ_NEG_MASKS,
                            c->stream) == hipSuccess;
  if (ok) hipLaunchKernelGGL(k_dt_init, dim3(1), dim3(64), 0, c->stream, c->red);
  double ts0[6] = {1.0, 1.0, 1.0, 1.0, 1.0, 0.0};
  ok = ok && hipMemcpyAsync(c->ts, ts0, sizeof(ts0), hipMemcpyHostToDevice, c->stream) ==
                 hipSuccess;
  if (!ok || hipStreamSynchronize(c->stream) != hipSuccess) { izem_destroy(c); return IZEM_E_HIP; }
  *out = c;
  return IZEM_OK;
}

extern "C" int izem_profile(izem_ctx *c, int capacity) {
  if (!c || capacity < 0) return IZEM_E_ARG;
  IzProf &p = c->prof;
  IZ_CHECK(hipStreamSynchronize(c->stream));
  if (p.ev) {
    for (int k = 0; k < 2 * p.cap; k++) (void)hipEventDestroy(p.ev[k]);
    free(p.ev);
    free(p.cls);
    p.ev = nullptr;
    p.cls = nullptr;
  }
  p.on = 0; p.n = 0; p.cap = 0;
  if (capacity == 0) return IZEM_OK;
  p.ev = (hipEvent_t *)calloc(2 * capacity, sizeof(hipEvent_t));
  p.cls = (int *)calloc(capacity, sizeof(int));
  if (!p.ev || !p.cls) return IZEM_E_NOMEM;
  for (int k = 0; k < 2 * capacity; k++) IZ_CHECK(hipEventCreate(&p.ev[k]));
  p.cap = capacity;
  p.on = 1;
  return IZEM_OK;
}

extern "C" int izem_profile_read(izem_ctx *c, double *ms, int *count) {
  if (!c || !ms || !count) return IZEM_E_ARG;
  IzProf &p = c->prof;
  IZ_CHECK(hipStreamSynchronize(c->stream));
  for (int q = 0; q < IZP_NCLASS; q++) { ms[q] = 0.0; count[q] = 0; }
  for (int k = 0; k < p.n; k++) {
    float t = 0.f;
    IZ_CHECK(hipEventElapsedTime(&t, p.ev[2 * k], p.ev[2 * k + 1]));
    ms[p.cls[k]] += t;
    count[p.cls[k]] += 1;
  }
  p.n = 0;
  return IZEM_OK;
}

extern "C" int izem_destroy(izem_ctx *c) {
  if (!c) return IZEM_OK;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  izem_profile(c, 0);
  iz_graph_destroy(c);
  iz_chem_destroy(c);
  for (int q = 0; q < 3; q++) if (c->F[q]) (void)hipFree(c->F[q]);
  for (int q = 0; q < 3; q++) if (c->Fs[q]) (void)hipFree(c->Fs[q]);
  if (c->wall_state) (void)hipFree(c->wall_state);
  if (c->prim) (void)hipFree(c->prim);
  if (c->fd) (void)hipFree(c->fd);
  if (c->sf) (void)hipFree(c->sf);
  if (c->v0) (void)hipFree(c->v0);
  if (c->masks) (void)hipFree(c->masks);
  if (c->negT_rec) (void)hipFree(c->negT_rec);
  if (c->status) (void)hipFree(c->status);
  if (c->iters) (void)hipFree(c->iters);
  if (c->red) (void)hipFree(c->red);
  if (c->ts) (void)hipFree(c->ts);
  if (c->own_stream) (void)hipStreamDestroy(c->own_stream);
  free(c);
  return IZEM_OK;
}

extern "C" int izem_flux_mode(izem_ctx *c, int mode) {
  if (!c || mode < 0 || mode > 1) return IZEM_E_ARG;
  c->flux_mode = mode;
  return IZEM_OK;
}

// GRID%BCXMIN .. BCZMAX (module_input.f90, bc(1:6)): 0 periodic, 1
// extrapolation (bc_extrapolation + the one-sided derivative closures of a
// face without a neighbour, module_BCs.f90:327-412, module_deriv.f90:268-469)
extern "C" int izem_set_bc(izem_ctx *c, const int bc[6]) {
  if (!c || !bc) return IZEM_E_ARG;
  int phys = 0, wall = 0, nscbc = 0;
  for (int f = 0; f < 6; f++) {
    if (bc[f] != IZEM_BC_PERIODIC && bc[f] != IZEM_BC_EXTRAPOLATION &&
        bc[f] != IZEM_BC_POSTSHOCK_SLIPWALL && bc[f] != IZEM_BC_NSCBC_OUT)
      return IZEM_E_ARG;
    // the post-shock slip wall is declared for face S only (module_BCs.f90:1163-1168),
    // the characteristic outflow for face E only (:2511-2514)
    if (bc[f] == IZEM_BC_POSTSHOCK_SLIPWALL) {
      if (f != 2) return IZEM_E_ARG;
      wall = 1;
    }
    if (bc[f] == IZEM_BC_NSCBC_OUT) {
      if (f != 1) return IZEM_E_ARG;
      nscbc = 1;
    }
    if (bc[f] != IZEM_BC_PERIODIC) {
      if (f / 2 >= c->d.ndim) return IZEM_E_ARG;
      phys |= 1 << f;
    }
  }
  // a direction is periodic on both faces or on neither
  for (int dir = 0; dir < 3; dir++)
    if (((phys >> (2 * dir)) & 3) == 1 || ((phys >> (2 * dir)) & 3) == 2) return IZEM_E_ARG;
  if (phys != c->d.phys || wall != c->d.wall || nscbc != c->d.nscbc) {
    c->d.phys = phys;
    c->d.wall = wall;
    c->d.nscbc = nscbc;
    iz_graph_destroy(c);  // a captured step holds the old dimensions
  }
  return IZEM_OK;
}

extern "C" int izem_set_nscbc(izem_ctx *c, double Lx, double pinf, double dxi_last) {
  if (!c || !(Lx > 0.0) || !(pinf > 0.0) || !(dxi_last > 0.0)) return IZEM_E_ARG;
  c->nscbc_Lx = Lx;
  c->nscbc_pinf = pinf;
  c->nscbc_dxi = dxi_last;
  c->nscbc_set = 1;
  iz_graph_destroy(c);
  return IZEM_OK;
}

extern "C" int izem_set_wall_state(izem_ctx *c, const double *state, int nfix) {
  if (!c || !state || nfix < 0 || nfix > c->d.nx) return IZEM_E_ARG;
  if (!c->wall_state &&
      hipMalloc(&c->wall_state, sizeof(double) * IZ_NV) != hipSuccess) {
    c->wall_state = nullptr;
    return IZEM_E_NOMEM;
  }
  IZ_CHECK(hipMemcpyAsync(c->wall_state, state, sizeof(double) * IZ_NV, hipMemcpyHostToDevice,
                          c->stream));
  IZ_CHECK(hipStreamSynchronize(c->stream));
  if (nfix != c->d.nfix) iz_graph_destroy(c);
  c->d.nfix = nfix;
  c->wall_set = 1;
  return IZEM_OK;
}

extern "C" int izem_set_decomposition(izem_ctx *c, const int nproc[3]) {
  if (!c || !nproc) return IZEM_E_ARG;
  const int n[3] = {c->d.nx, c->d.ny, c->d.nz};
  for (int q = 0; q < 3; q++) {
    if (nproc[q] < 1 || nproc[q] > n[q]) return IZEM_E_ARG;
    if (q >= c->d.ndim && nproc[q] != 1) return IZEM_E_ARG;
  }
  if (nproc[0] == c->d.np[0] && nproc[1] == c->d.np[1] && nproc[2] == c->d.np[2])
    return IZEM_OK;
  IZ_CHECK(hipStreamSynchronize(c->stream));
  iz_graph_destroy(c);  // a captured step holds the old launches
  const long lines[3] = {(long)c->d.ny * c->d.nz, (long)c->d.nx * c->d.nz,
                         (long)c->d.nx * c->d.ny};
  for (int q = 0; q < 3; q++) {
    if (c->Fs[q]) (void)hipFree(c->Fs[q]);
    c->Fs[q] = nullptr;
    c->nseam[q] = 0;
    c->d.np[q] = 1;
  }
  for (int q = 0; q < 3; q++) {
    if (nproc[q] == 1) continue;
    const long ns = (long)(nproc[q] - 1) * lines[q];
    if (hipMalloc(&c->Fs[q], sizeof(double) * IZ_NV * ns) != hipSuccess) {
      for (int p = 0; p < 3; p++) {
        if (c->Fs[p]) (void)hipFree(c->Fs[p]);
        c->Fs[p] = nullptr;
        c->nseam[p] = 0;
        c->d.np[p] = 1;
      }
      return IZEM_E_NOMEM;
    }
    c->nseam[q] = ns;
  }
  for (int q = 0; q < 3; q++) c->d.np[q] = nproc[q];
  return IZEM_OK;
}

extern "C" int izem_synchronize(izem_ctx *c) {
  if (!c) return IZEM_E_ARG;
  IZ_CHECK(hipStreamSynchronize(c->stream));
  return IZEM_OK;
}

extern "C" int izem_status(izem_ctx *c, int *bits) {
  if (!c || !bits) return IZEM_E_ARG;
  int h = 0;
  IZ_CHECK(hipMemcpyAsync(&h, c->status, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  IZ_CHECK(hipMemsetAsync(c->status, 0, sizeof(int), c->stream));
  IZ_CHECK(hipStreamSynchronize(c->stream));
  *bits = h;
  return IZEM_OK;
}

extern "C" double *izem_time_state(izem_ctx *c) { return c ? c->ts : nullptr; }

extern "C" int izem_set_stream(izem_ctx *c, void *stream) {
  if (!c) return IZEM_E_ARG;
  IZ_CHECK(hipStreamSynchronize(c->stream));
  c->stream = stream ? (hipStream_t)stream : c->own_stream;
  return IZEM_OK;
}

extern "C" int izem_get_time_state(izem_ctx *c, double *h) {
  if (!c || !h) return IZEM_E_ARG;
  IZ_CHECK(hipMemcpyAsync(h, c->ts, 6 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  IZ_CHECK(hipStreamSynchronize(c->stream));
  return IZEM_OK;
}

extern "C" int izem_set_time_state(izem_ctx *c, const double *h) {
  if (!c || !h) return IZEM_E_ARG;
  IZ_CHECK(hipMemcpyAsync(c->ts, h, 6 * sizeof(double), hipMemcpyHostToDevice, c->stream));
  IZ_CHECK(hipStreamSynchronize(c->stream));
  return IZEM_OK;
}

extern "C" int izem_wenorec(izem_ctx *c, int n, int js, const double *vp, const double *vm,
                            double *out) {
  if (!c || n < 0 || !vp || !vm || !out) return IZEM_E_ARG;
  if (n == 0) return IZEM_OK;
  hipLaunchKernelGGL(k_wenorec_batch, dim3(iz_blocks(n, 256)), dim3(256), 0, c->stream, n, js,
                     vp, vm, out);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_math(izem_ctx *c, int f, int n, const double *x, double *y) {
  if (!c || f < 0 || f > 2 || n < 0 || !x || !y) return IZEM_E_ARG;
  if (n == 0) return IZEM_OK;
  hipLaunchKernelGGL(k_math_batch, dim3(iz_blocks(n, 256)), dim3(256), 0, c->stream, f, n, x, y);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

// k_rhs_update for the context's faces and decomposition
typedef void (*IzRhsKernel)(IzDims, IzBand, int, const double *, const double *, const double *, IzSeams,
                            int, const double *, const double *, const double *, const double *,
                            const double *, const double *, double, double, double *,
                            double *, double *, int, const double *, double,
                            unsigned long long *);
static IzRhsKernel rhs_update_kernel(const IzDims &d) {
  const bool seams = d.np[0] > 1 || d.np[1] > 1 || d.np[2] > 1;
  if (seams) return d.phys ? k_rhs_update<true, true> : k_rhs_update<false, true>;
  return d.phys ? k_rhs_update<true, false> : k_rhs_update<false, false>;
}
static IzSeams seams_of(const izem_ctx *c) {
  IzSeams s;
  for (int q = 0; q < 3; q++) { s.F[q] = c->Fs[q]; s.n[q] = c->nseam[q]; }
  return s;
}

static int euler_dir(izem_ctx *c, int dir, const double *d_i, const double *T,
                     const double *W_i, const double *cp, const double *ha,
                     const uint8_t *sensor, const double *v, double *fl, bool apply) {
  if (!c || !d_i || !T || !W_i || !cp || !ha || !sensor || !v) return IZEM_E_ARG;
  if (dir >= c->d.ndim) return IZEM_E_ARG;
  long nf = c->nfaces[dir];
  int wa = c->o.weno_avg;
  const int tile0 = eu_tile0(c->d);
  const size_t lds = eu_lds_bytes(dir, tile0);
  const long ntiles = dir == 0 ? 0 : eu_ntiles(c->d, dir);
  // x: four 64-face waves per block; y, z: logical tiles rounded up to a
  // multiple of the 8 XCDs (blocks past the last tile only pass the barrier)
  const unsigned nb = dir == 0 ? iz_blocks(nf, IZ_EU_BLOCK) : (unsigned)(((ntiles + 7) / 8) * 8);
  int pk = iz_prof_begin(c, IZP_EULER);
#define IZ_EU(D, FAST, RANKS)                                                          \
  hipLaunchKernelGGL((k_euler_faces<D, FAST, RANKS>), dim3(nb), dim3(IZ_EU_BLOCK), lds,   \
                     c->stream, c->d, v, T, W_i, cp, ha, sensor, wa, c->F[D], nf, c->status, \
                     tile0, ntiles)
#define IZ_EU_DIR(FAST, RANKS)            \
  if (dir == 0) IZ_EU(0, FAST, RANKS);    \
  else if (dir == 1) IZ_EU(1, FAST, RANKS); \
  else IZ_EU(2, FAST, RANKS)
  const bool ranks = c->d.np[dir] > 1;
  if (c->flux_mode) {
    if (ranks) { IZ_EU_DIR(true, true); }
    else { IZ_EU_DIR(true, false); }
  } else {
    if (ranks) { IZ_EU_DIR(false, true); }
    else { IZ_EU_DIR(false, false); }
  }
#undef IZ_EU_DIR
#undef IZ_EU
  if (c->d.np[dir] > 1) {
    // the faces between ranks again, with the left rank's view
    const long ns = c->nseam[dir];
    const unsigned nbs = iz_blocks(ns, IZ_SEAM_BLOCK);
    const size_t lds_s = (size_t)IZ_SEAM_BLOCK * IZ_S * IZ_EU_NQ * sizeof(double);
#define IZ_SEAM(D, FAST)                                                                    \
  hipLaunchKernelGGL((k_euler_seams<D, FAST>), dim3(nbs), dim3(IZ_SEAM_BLOCK), lds_s, c->stream, \
                     c->d, v, T, W_i, cp, ha, sensor, wa, c->Fs[D], ns, c->status)
    if (c->flux_mode) {
      if (dir == 0) IZ_SEAM(0, true);
      else if (dir == 1) IZ_SEAM(1, true);
      else IZ_SEAM(2, true);
    } else {
      if (dir == 0) IZ_SEAM(0, false);
      else if (dir == 1) IZ_SEAM(1, false);
      else IZ_SEAM(2, false);
    }
#undef IZ_SEAM
  }
  iz_prof_end(c, pk);
  IZ_CHECK(hipGetLastError());
  if (apply) {
    if (!fl) return IZEM_E_ARG;
    unsigned nbc = iz_blocks(n_interior(c->d), 256);
    int acc = dir > 0;
    if (dir == 0)
      hipLaunchKernelGGL(k_euler_apply<0>, dim3(nbc), dim3(256), 0, c->stream, c->d, c->F[0], nf,
                         d_i, acc, fl, c->Fs[0], c->nseam[0]);
    else if (dir == 1)
      hipLaunchKernelGGL(k_euler_apply<1>, dim3(nbc), dim3(256), 0, c->stream, c->d, c->F[1], nf,
                         d_i, acc, fl, c->Fs[1], c->nseam[1]);
    else
      hipLaunchKernelGGL(k_euler_apply<2>, dim3(nbc), dim3(256), 0, c->stream, c->d, c->F[2], nf,
                         d_i, acc, fl, c->Fs[2], c->nseam[2]);
    IZ_CHECK(hipGetLastError());
  }
  return IZEM_OK;
}

extern "C" int izem_euler_llf_x(izem_ctx *c, const double *dx_i, const double *T,
                                const double *W_i, const double *cp, const double *ha,
                                const uint8_t *sensor, const double *v, double *fl) {
  return euler_dir(c, 0, dx_i, T, W_i, cp, ha, sensor, v, fl, true);
}
extern "C" int izem_euler_llf_y(izem_ctx *c, const double *dy_i, const double *T,
                                const double *W_i, const double *cp, const double *ha,
                                const uint8_t *sensor, const double *v, double *fl) {
  return euler_dir(c, 1, dy_i, T, W_i, cp, ha, sensor, v, fl, true);
}
extern "C" int izem_euler_llf_z(izem_ctx *c, const double *dz_i, const double *T,
                                const double *W_i, const double *cp, const double *ha,
                                const uint8_t *sensor, const double *v, double *fl) {
  return euler_dir(c, 2, dz_i, T, W_i, cp, ha, sensor, v, fl, true);
}

// comm_cons (the periodic exchange of every direction), then, with bcs,
// upd_boundaries' face conditions in the order W, E, S, N, B, F: a face
// that writes its first interior row (a Dirichlet face) has that row's
// force_sumY right after its condition, before the next face reads it
// (module_BCs.f90:71-137); the row's primitives follow in iz_ghost_newton.
int iz_comm_cons(izem_ctx *c, double *a, int nf, int bcs, const double *T, const double *W_i,
                 const double *cp, const double *dtp, double scale) {
  const IzDims &d = c->d;
  if (bcs && (d.wall || d.nscbc) && nf != IZ_NV) return IZEM_E_STATE;
  if (bcs && d.wall && !c->wall_set) return IZEM_E_STATE;
  if (bcs && d.nscbc && (!c->nscbc_set || !T || !W_i || !cp || !dtp)) return IZEM_E_STATE;
  const double *wall = (bcs && d.wall) ? c->wall_state : nullptr;
  int pk = iz_prof_begin(c, IZP_OTHER);
  auto fill = [&](int dir, int mode) {
    long n0 = (dir == 0) ? d.ny : d.nx, n1 = (dir == 2) ? d.ny : d.nz;
    long tot = n0 * n1 * 2 * d.ng * nf;
    hipLaunchKernelGGL(k_ghost_fill, dim3(iz_blocks(tot, 256)), dim3(256), 0, c->stream, d, a,
                       nf, dir, wall, mode);
  };
  for (int dir = 0; dir < d.ndim; dir++) fill(dir, 1);
  if (bcs) {
    for (int dir = 0; dir < d.ndim; dir++) {
      if (!((d.phys >> (2 * dir)) & 3)) continue;
      fill(dir, 2);
      if (dir == 0 && d.nscbc) {
        hipLaunchKernelGGL(k_nscbc_out, dim3(iz_blocks((long)d.ny * d.nz, 64)), dim3(64), 0,
                           c->stream, d, a, T, W_i, cp, dtp, scale, c->nscbc_Lx, c->nscbc_pinf,
                           c->nscbc_dxi);
        if (c->o.forcesum) {
          IzBox b = domain_box(d, 10);
          hipLaunchKernelGGL(k_force_row, dim3(iz_blocks(box_count(b), 256)), dim3(256), 0,
                             c->stream, d, b, a);
        }
      }
      if (dir == 1 && d.wall && c->o.forcesum) {
        IzBox b = domain_box(d, -20);
        hipLaunchKernelGGL(k_force_row, dim3(iz_blocks(box_count(b), 256)), dim3(256), 0,
                           c->stream, d, b, a);
      }
    }
  }
  iz_prof_end(c, pk);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_comm_cons(izem_ctx *c, double *v) {
  if (!c || !v) return IZEM_E_ARG;
  return iz_comm_cons(c, v, IZ_NV, 1);
}

extern "C" int izem_comm_cons_exchange(izem_ctx *c, double *v) {
  if (!c || !v) return IZEM_E_ARG;
  return iz_comm_cons(c, v, IZ_NV, 0);
}

extern "C" int izem_upd_boundaries(izem_ctx *c, const double *dt, const double *T,
                                   const double *W_i, const double *cp, double *v) {
  if (!c || !dt || !T || !W_i || !cp || !v) return IZEM_E_ARG;
  return iz_comm_cons(c, v, IZ_NV, 1, T, W_i, cp, dt, 1.0);
}

// viscous fluxes into the context scratch (prim, fd, sf)
static int visc_fluxes(izem_ctx *c, const double *dx_i, const double *dy_i, const double *dz_i,
                       const double *T, const double *W_i, const double *ha, const double *v) {
  const IzDims &d = c->d;
  int pk = iz_prof_begin(c, IZP_VISC);
  // every domain's primitives are written before any domain's fluxes read
  // them (a slab cell's derivatives come from its interior image)
  const IzDomSet ds = domain_set(d, true);
  const long ncell = ds.first[ds.n];
  hipLaunchKernelGGL(k_visc_prim, dim3(iz_blocks(ncell, 256)), dim3(256), 0, c->stream, d, ds, v,
                     W_i, c->prim);
  const double rvd0 = c->o.sqgmr / c->o.Sc, rlam0 = c->o.sqgmr * c->o.ggmopr;
  const IzBand bd = band_of(d, 128);
  const IzDomSet slabs = domain_set(d, false);
  const dim3 grid(band_grid(bd) + iz_blocks(slabs.first[slabs.n], 128));
  if (d.phys)
    hipLaunchKernelGGL(k_visc_fused<true>, grid, dim3(128), 0, c->stream, d, bd, slabs, c->dsym,
                       c->o.sqgmr, rvd0, rlam0, v, T, W_i, ha, c->prim, dx_i, dy_i, dz_i, c->fd,
                       c->sf);
  else
    hipLaunchKernelGGL(k_visc_fused<false>, grid, dim3(128), 0, c->stream, d, bd, slabs, c->dsym,
                       c->o.sqgmr, rvd0, rlam0, v, T, W_i, ha, c->prim, dx_i, dy_i, dz_i, c->fd,
                       c->sf);
  iz_prof_end(c, pk);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_viscflux(izem_ctx *c, const double *dx_i, const double *dy_i,
                             const double *dz_i, const double *T, const double *W_i,
                             const double *ha, const double *v, double *fl) {
  if (!c || !dx_i || !dy_i || !dz_i || !T || !W_i || !ha || !v || !fl) return IZEM_E_ARG;
  int r = visc_fluxes(c, dx_i, dy_i, dz_i, T, W_i, ha, v);
  if (r) return r;
  if (c->d.phys)
    hipLaunchKernelGGL(k_visc_apply<true>, dim3(iz_blocks(n_interior(c->d), 256)), dim3(256), 0,
                       c->stream, c->d, c->sf, c->fd, dx_i, dy_i, dz_i, fl);
  else
    hipLaunchKernelGGL(k_visc_apply<false>, dim3(iz_blocks(n_interior(c->d), 256)), dim3(256), 0,
                       c->stream, c->d, c->sf, c->fd, dx_i, dy_i, dz_i, fl);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

static int dom_ok(const IzDims &d, int dom) {
  if (dom % 10 == 0 && dom != 0) dom /= 10;
  return dom >= -d.ndim && dom <= d.ndim;
}

extern "C" int izem_force_sumY(izem_ctx *c, int dom, double *v) {
  if (!c || !v || !dom_ok(c->d, dom)) return IZEM_E_ARG;
  // no probe: nothing reaches the masks
  const IzNewtonSet s = newton_set(c, &dom, 1, 1);
  hipLaunchKernelGGL(k_force_probe, dim3(s.first[1]), dim3(256), 0, c->stream, c->d, s, 0, 1, v,
                     (const double *)nullptr, -1.0, c->masks);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

// the iterations of a probed set: apply, then the rare repair, which also
// clears the masks
static void newton_finish(izem_ctx *c, const int *doms, int nd, double *v, double *W_i, double *T,
                          double *cp, double *ha, int mach) {
  const double eps = mach ? 1.0e-10 : 1.0e-5;
  const int itmax = mach ? 100 : 200;
  const IzNewtonSet s = newton_set(c, doms, nd, 0);
  hipLaunchKernelGGL(k_newton_apply, dim3(s.first[nd]), dim3(256), 0, c->stream, c->d, s, v, T,
                     W_i, cp, ha, c->masks, itmax, !mach, c->status, c->iters);
  hipLaunchKernelGGL(k_newton_repair, dim3(nd), dim3(1024), 0, c->stream, c->d, s, !mach, v, T,
                     W_i, cp, ha, c->masks, itmax, eps, c->negT_rec, c->status, c->iters);
}

// force_sumY (optional) + probe + apply on a list of at most six domains;
// prim_inv_var (eps 1e-5, 200 iterations, negative-temperature repair) or,
// with mach, prim_inv_var_err_mach (module_thermodynamics.f90:201-260: eps
// 1e-10, 100 iterations, a negative temperature only warned about).  fill:
// the domains are ghost slabs that take their source cells' conserved
// variables first
static int newton_domains(izem_ctx *c, const int *doms, int nd, int forcesum, double *v,
                          double *W_i, double *T, double *cp, double *ha, int mach = 0,
                          int fill = 0) {
  const IzNewtonSet s = newton_set(c, doms, nd, 1);
  int pk = iz_prof_begin(c, IZP_NEWTON);
  hipLaunchKernelGGL(k_force_probe, dim3(s.first[nd]), dim3(256), 0, c->stream, c->d, s, fill,
                     forcesum, v, T, mach ? 1.0e-10 : 1.0e-5, c->masks);
  newton_finish(c, doms, nd, v, W_i, T, cp, ha, mach);
  iz_prof_end(c, pk);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_prim_inv_var(izem_ctx *c, int dom, double *v, double *W_i, double *T,
                                 double *cp, double *ha, int *iters) {
  if (!c || !v || !W_i || !T || !cp || !ha || !dom_ok(c->d, dom)) return IZEM_E_ARG;
  int r = newton_domains(c, &dom, 1, 0, v, W_i, T, cp, ha);
  if (r) return r;
  if (iters) {
    IZ_CHECK(hipMemcpyAsync(iters, c->iters + mask_slot(dom), sizeof(int), hipMemcpyDeviceToHost,
                            c->stream));
    IZ_CHECK(hipStreamSynchronize(c->stream));
  }
  return IZEM_OK;
}

extern "C" int izem_prim_inv_var_mach(izem_ctx *c, int dom, double *v, double *W_i, double *T,
                                      double *cp, double *ha, int *iters) {
  if (!c || !v || !W_i || !T || !cp || !ha || !dom_ok(c->d, dom)) return IZEM_E_ARG;
  int r = newton_domains(c, &dom, 1, 0, v, W_i, T, cp, ha, 1);
  if (r) return r;
  if (iters) {
    IZ_CHECK(hipMemcpyAsync(iters, c->iters + mask_slot(dom), sizeof(int), hipMemcpyDeviceToHost,
                            c->stream));
    IZ_CHECK(hipStreamSynchronize(c->stream));
  }
  return IZEM_OK;
}

extern "C" int izem_upd_prim_var_woT(izem_ctx *c, int dom, const double *v, const double *T,
                                     double *W_i, double *cp, double *ha) {
  if (!c || !v || !T || !W_i || !cp || !ha || !dom_ok(c->d, dom)) return IZEM_E_ARG;
  return iz_upd_prim_woT(c, dom, v, T, W_i, cp, ha);
}

int iz_upd_prim_woT(izem_ctx *c, int dom, const double *v, const double *T, double *W_i,
                    double *cp, double *ha) {
  IzBox b = domain_box(c->d, dom);
  int pk = iz_prof_begin(c, IZP_NEWTON);
  hipLaunchKernelGGL(k_upd_prim_woT, dim3(iz_blocks(box_count(b), 256)), dim3(256), 0, c->stream,
                     c->d, b, v, T, W_i, cp, ha);
  iz_prof_end(c, pk);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

// upd_prim_var_dirichlet of a post-shock slip wall (its condition wrote the
// first interior row: force_sumY and prim_inv_var there, module_BCs.f90:
// 93-96, 131, 297-314), then upd_prim_var_ghost on the ghost slabs
static const int ghost_faces[6] = {-1, 1, -2, 2, -3, 3};
int iz_ghost_newton(izem_ctx *c, double *T, double *W_i, double *cp, double *ha, double *v) {
  // the Dirichlet rows in face order (their force_sumY came with the fill)
  if (c->d.nscbc) {
    static const int row = 10;
    int r = newton_domains(c, &row, 1, 0, v, W_i, T, cp, ha);
    if (r) return r;
  }
  if (c->d.wall) {
    static const int row = -20;
    int r = newton_domains(c, &row, 1, 0, v, W_i, T, cp, ha);
    if (r) return r;
  }
  return newton_domains(c, ghost_faces, 2 * c->d.ndim, c->o.forcesum, v, W_i, T, cp, ha);
}

// comm_cons + upd_boundaries + the ghost cells' primitives, as a stage or a
// reaction ends.  Without a Dirichlet face the conditions of all faces read
// interior cells only, so the probe's pass over the ghost cells makes the
// copies itself: three launches (2-D 128^2: 32 us a pass where the copies
// and a probe, apply and repair per slab, 15 launches, took 92).
int iz_fill_ghost_newton(izem_ctx *c, double *T, double *W_i, double *cp, double *ha, double *v,
                         const double *dtp, double scale) {
  if (c->d.wall || c->d.nscbc) {
    int r = iz_comm_cons(c, v, IZ_NV, 1, T, W_i, cp, dtp, scale);
    if (r) return r;
    return iz_ghost_newton(c, T, W_i, cp, ha, v);
  }
  return newton_domains(c, ghost_faces, 2 * c->d.ndim, c->o.forcesum, v, W_i, T, cp, ha, 0, 1);
}

extern "C" int izem_upd_prim_var_ghost(izem_ctx *c, double *T, double *W_i, double *cp,
                                       double *ha, double *v) {
  if (!c || !T || !W_i || !cp || !ha || !v) return IZEM_E_ARG;
  return iz_ghost_newton(c, T, W_i, cp, ha, v);
}

extern "C" int izem_shock_sensor(izem_ctx *c, const double *v, const double *T,
                                 const double *W_i, uint8_t *sensor) {
  if (!c || !v || !T || !W_i || !sensor) return IZEM_E_ARG;
  int pk = iz_prof_begin(c, IZP_OTHER);
  hipLaunchKernelGGL(k_sensor, dim3(iz_blocks(n_interior(c->d), 256)), dim3(256), 0, c->stream,
                     c->d, c->o.max_rel_weight, v, T, W_i, sensor);
  iz_prof_end(c, pk);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_shock_sensor_ducros(izem_ctx *c, const double *dx_i, const double *dy_i,
                                        const double *dz_i, const double *v, uint8_t *sensor) {
  if (!c || !dx_i || !dy_i || !dz_i || !v || !sensor || c->d.ndim < 2) return IZEM_E_ARG;
  int pk = iz_prof_begin(c, IZP_OTHER);
  hipLaunchKernelGGL(k_sensor_ducros, dim3(iz_blocks(n_interior(c->d), 256)), dim3(256), 0,
                     c->stream, c->d, c->o.ducros_treduc, dx_i, dy_i, dz_i, v, sensor);
  iz_prof_end(c, pk);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

// sensor + fluxes of one stage into the context scratch
static int stage_fluxes(izem_ctx *c, const double *dx_i, const double *dy_i,
                        const double *dz_i, const double *T, const double *W_i,
                        const double *cp, const double *ha, uint8_t *sensor, const double *v) {
  // module_solver.f90:758-762
  int r = c->o.sensor_type == 1 ? izem_shock_sensor_ducros(c, dx_i, dy_i, dz_i, v, sensor)
                                : izem_shock_sensor(c, v, T, W_i, sensor);
  if (r) return r;
  const double *di[3] = {dx_i, dy_i, dz_i};
  for (int q = 0; q < c->d.ndim; q++) {
    r = euler_dir(c, q, di[q], T, W_i, cp, ha, sensor, v, nullptr, false);
    if (r) return r;
  }
  if (c->o.vis) return visc_fluxes(c, dx_i, dy_i, dz_i, T, W_i, ha, v);
  return IZEM_OK;
}

extern "C" int izem_rhs(izem_ctx *c, const double *dx_i, const double *dy_i, const double *dz_i,
                        const double *T, const double *W_i, const double *cp, const double *ha,
                        uint8_t *sensor, const double *v, double *f) {
  if (!c || !dx_i || !dy_i || !dz_i || !T || !W_i || !cp || !ha || !sensor || !v || !f)
    return IZEM_E_ARG;
  int r = stage_fluxes(c, dx_i, dy_i, dz_i, T, W_i, cp, ha, sensor, v);
  if (r) return r;
  const IzDims &d = c->d;
  const IzBand bd = band_of(d, 256);
  hipLaunchKernelGGL(rhs_update_kernel(d), dim3(band_grid(bd)), dim3(256), 0,
                     c->stream, d, bd, 0, c->F[0], c->F[1], c->F[2], seams_of(c), c->o.vis, c->sf,
                     c->fd, dx_i, dy_i, dz_i,
                     (const double *)nullptr, 0.0, 0.0, (double *)nullptr,
                     (double *)nullptr, f, 0, T, 0.0, (unsigned long long *)nullptr);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_rk3(izem_ctx *c, const double *dt, const double *dx_i, const double *dy_i,
                        const double *dz_i, double *T, double *W_i, double *cp, double *ha,
                        uint8_t *sensor, double *v) {
  if (!c || !dt || !dx_i || !dy_i || !dz_i || !T || !W_i || !cp || !ha || !sensor || !v)
    return IZEM_E_ARG;
  static const double bk3[3] = {0.00, 0.75, 1.00 / 3.00};
  static const double ck3[3] = {1.00, 0.25, 2.00 / 3.00};
  const IzDims &d = c->d;
  for (int ik = 0; ik < 3; ik++) {
    int r = stage_fluxes(c, dx_i, dy_i, dz_i, T, W_i, cp, ha, sensor, v);
    if (r) return r;
    int pk = iz_prof_begin(c, IZP_RHS);
    // the first stage keeps the state it starts from in v0
    const IzBand bd = band_of(d, 256);
    hipLaunchKernelGGL(rhs_update_kernel(d), dim3(band_grid(bd)), dim3(256), 0,
                       c->stream, d, bd, ik == 0 ? 2 : 1, c->F[0], c->F[1], c->F[2], seams_of(c),
                       c->o.vis, c->sf, c->fd, dx_i, dy_i, dz_i, dt,
                       bk3[ik], ck3[ik], c->v0, v, (double *)nullptr, c->o.forcesum, T, 1.0e-5,
                       c->masks + 3);
    iz_prof_end(c, pk);
    static const int interior = 0;
    pk = iz_prof_begin(c, IZP_NEWTON);
    newton_finish(c, &interior, 1, v, W_i, T, cp, ha, 0);
    iz_prof_end(c, pk);
    IZ_CHECK(hipGetLastError());
    r = iz_fill_ghost_newton(c, T, W_i, cp, ha, v, dt, 1.0);
    if (r) return r;
  }
  return IZEM_OK;
}

extern "C" int izem_timestep(izem_ctx *c, const double *dx_i, const double *dy_i,
                             const double *dz_i, const double *cp, const double *W_i,
                             const double *T, const double *v) {
  if (!c || !dx_i || !dy_i || !dz_i || !cp || !W_i || !T || !v) return IZEM_E_ARG;
  const IzDims &d = c->d;
  int pk = iz_prof_begin(c, IZP_OTHER);
  const int visdt = c->o.vis && c->o.vis_dt;
  if (visdt)
    hipLaunchKernelGGL(k_dt_visc, dim3(iz_blocks_capped(c, n_interior(d), 128, 32)), dim3(128),
                       0, c->stream, d, c->dsym, v, T, W_i, cp, dx_i, dy_i, dz_i, c->red);
  else
    hipLaunchKernelGGL(k_dt_conv, dim3(iz_blocks_capped(c, n_interior(d), 256, 16)), dim3(256), 0,
                       c->stream, d, v, T, W_i, cp, dx_i, dy_i, dz_i, c->red);
  double rvd0_i = c->o.Sc / c->o.sqgmr, rlamcp0_i = c->o.Pr / c->o.sqgmr;
  hipLaunchKernelGGL(k_dt_final, dim3(1), dim3(64), 0, c->stream, c->red, c->o.CFL, c->o.CFLmin,
                     c->o.Fo, c->o.CPR, visdt, c->o.reaction, rvd0_i, rlamcp0_i, c->ts);
  iz_prof_end(c, pk);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}
