// Device-side building blocks of the GRMHD substep for gfx950.
//
// Per-point physics of the reference (ReconX, AsterX fluxes/eigenvalues,
// EOSX ideal gas, AsterUtils contractions) as __device__ functions.  The
// expressions keep the reference's evaluation order term for term and the
// library is compiled with -ffp-contract=off, so results agree bit for bit
// with a strict-IEEE CPU evaluation of the same formulas wherever only
// +,-,*,/,sqrt are involved (all correctly rounded on CDNA4).  Deliberate
// exceptions, which agree to rounding level: finite differences multiply by
// a host-computed 1/dx, and the source terms divide by alpha and W once.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "asterx.h"

#define ASX_DEV __device__ __forceinline__
#include "asx_quotient.hpp"

namespace asx {

// The library builds with -ffp-contract=off so that con2prim and the
// reconstruction (whose limiter branches compare computed values) evaluate
// their expressions exactly as written.  The smooth arithmetic after the
// reconstruction -- Riemann fluxes, characteristic speeds, source terms,
// flux divergence, gauge terms, RK combination -- opts in to fused
// multiply-add with ASX_CONTRACT at the top of a function body: it changes
// results by rounding only (no branch depends on it), well inside the
// 1e-12 parity bar, and removes about a third of the FP64 instructions.
#define ASX_CONTRACT _Pragma("clang fp contract(fast)")

// ---------------------------------------------------------------------------
// Patch view passed to kernels by value
// ---------------------------------------------------------------------------
struct KPatch {
  double *g[ASX_NUM_GF];
  int sj[8], sk[8]; // dense strides per centering code (bit d: vertex on d)
  int n[3], ng;
  double dx[3], x0[3];
  double idx[3]; // 1/dx
};

// Centering code of each slot (include/asterx.h enum order).
ASX_DEV constexpr int cent(int s) {
  return (s <= ASX_KZZ)             ? 7
         : (s <= ASX_MASK_CC)       ? 0
         : (s == ASX_MASK_VC)       ? 7
         : (s == ASX_DBX_STAG)      ? 1
         : (s == ASX_DBY_STAG)      ? 2
         : (s == ASX_DBZ_STAG)      ? 4
         : (s == ASX_AVEC_X)        ? 6
         : (s == ASX_AVEC_Y)        ? 5
         : (s == ASX_AVEC_Z)        ? 3
         : (s == ASX_PSI)           ? 7
         : (s <= ASX_FXBZ)          ? 1
         : (s <= ASX_FYBZ)          ? 2
         : (s <= ASX_FZBZ)          ? 4
         : (s <= ASX_VTILDE_Z_XFACE) ? 1
         : (s <= ASX_VTILDE_Z_YFACE) ? 2
         : (s <= ASX_VTILDE_Y_ZFACE) ? 4
         : (s <= ASX_AMIN_XFACE)    ? 1
         : (s <= ASX_AMIN_YFACE)    ? 2
         : (s <= ASX_AMIN_ZFACE)    ? 4
         : (s <= ASX_G)             ? 7
         : (s <= ASX_DYE_RHS)       ? 0
         : (s == ASX_AVEC_X_RHS)    ? 6
         : (s == ASX_AVEC_Y_RHS)    ? 5
         : (s == ASX_AVEC_Z_RHS)    ? 3
         : (s == ASX_REGRID_ERROR)  ? 0
                                    : 7;
}

ASX_DEV int off(const KPatch &p, int c, int i, int j, int k) {
  return i + p.sj[c] * j + p.sk[c] * k;
}
template <int S> ASX_DEV double &at(const KPatch &p, int i, int j, int k) {
  return p.g[S][off(p, cent(S), i, j, k)];
}
ASX_DEV double &at(const KPatch &p, int s, int i, int j, int k) {
  return p.g[s][off(p, cent(s), i, j, k)];
}
// Linear offset of one step along axis d for centering c.
ASX_DEV int step(const KPatch &p, int c, int d) {
  return d == 0 ? 1 : (d == 1 ? p.sj[c] : p.sk[c]);
}

// ---------------------------------------------------------------------------
// Scalar helpers (std::min/max semantics: first operand kept on ties/NaN)
// ---------------------------------------------------------------------------
ASX_DEV double smin(double a, double b) { return (b < a) ? b : a; }
ASX_DEV double smax(double a, double b) { return (a < b) ? b : a; }
ASX_DEV double pow2(double x) { return x * x; }
ASX_DEV int sgn(double v) { return (0.0 < v) - (v < 0.0); }

// Workgroups are handed to the 8 XCDs of the chip round-robin (w % 8), and
// each XCD has its own L2.  Map workgroup w to a tile index such that every
// XCD receives one contiguous run of tiles, so neighbouring tiles (sharing
// halo cells and metric vertices) hit the same L2.  A bijection of [0, nb).
ASX_DEV int xcd_tile(int w, int nb) {
  constexpr int NX = 8;
  const int x = w % NX, l = w / NX, per = (nb + NX - 1) / NX, rem = nb % NX;
  return (rem == 0 || x < rem) ? x * per + l : rem * per + (x - rem) * (per - 1) + l;
}

struct Sym3 {
  double xx, xy, xz, yy, yz, zz;
  ASX_DEV double operator()(int i, int j) const {
    const int a = i < j ? i : j, b = i < j ? j : i;
    return a == 0 ? (b == 0 ? xx : (b == 1 ? xy : xz))
                  : (a == 1 ? (b == 1 ? yy : yz) : zz);
  }
};
// 3x3 symmetric determinant and inverse (cofactors over det)
ASX_DEV double det3(const Sym3 &g) {
  return 2 * g.xy * g.xz * g.yz + g.xx * g.yy * g.zz - g.yy * pow2(g.xz) -
         g.xx * pow2(g.yz) - g.zz * pow2(g.xy);
}
// SPLIT: a branch for each kind of divisor, which ends the live ranges before
// it (con2prim of independent zones 152 -> 124 VGPRs).  Else the quotients in
// line with what surrounds them, put right afterwards where they do not hold:
// for the guided solve, whose registers suffice (2^24 zones 1.36 -> 1.33 ms); con2prim of
// a patch loses its second wave per SIMD (192^3 substep 4.41 -> 5.03 ms).
template <bool SPLIT = true> ASX_DEV Sym3 inv3(const Sym3 &g, double det) {
  auto over = [&](const auto &d) {
    return Sym3{(g.yy * g.zz - pow2(g.yz)) / d, (g.xz * g.yz - g.xy * g.zz) / d,
                (g.xy * g.yz - g.xz * g.yy) / d, (g.xx * g.zz - pow2(g.xz)) / d,
                (g.xy * g.xz - g.xx * g.yz) / d, (g.xx * g.yy - pow2(g.xy)) / d};
  };
  const Divisor d(det);
  if constexpr (SPLIT) {
    return d.holds() ? over(d) : over(det);
  } else {
    Sym3 u = over(d);
    if (!d.holds()) u = over(det);
    return u;
  }
}
ASX_DEV void lower(const Sym3 &g, const double v[3], double o[3]) {
  o[0] = 0.0 + g.xx * v[0] + g.xy * v[1] + g.xz * v[2];
  o[1] = 0.0 + g.xy * v[0] + g.yy * v[1] + g.yz * v[2];
  o[2] = 0.0 + g.xz * v[0] + g.yz * v[1] + g.zz * v[2];
}
ASX_DEV double dot3(const double a[3], const double b[3]) {
  return 0.0 + a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

// ---------------------------------------------------------------------------
// Reconstruction (ReconX)
// ---------------------------------------------------------------------------
struct RParams {
  int ppm_shock_detection, ppm_zone_flattening;
  double kgamma; // poly_k * poly_gamma (PPM contact test uses the ID polytrope)
  double ppm_eta1, ppm_eta2, ppm_eps, ppm_eps_shock, ppm_small, ppm_omega1,
      ppm_omega2, weno_eps, mp5_alpha;
};

// minmod, ReconX/src/minmod.hxx:14-26 (signbit test: -0 differs from +0)
ASX_DEV double minmod(double x, double y) {
  if (__builtin_signbit(x) != __builtin_signbit(y)) return 0.0;
  if (fabs(x) < fabs(y)) return x;
  return y;
}
ASX_DEV double monocentral(double x, double y) {
  if (sgn(x) != sgn(y)) return 0.0;
  return sgn(x) * smin(2 * fabs(x), smin(2 * fabs(y), fabs(x + y) / 2));
}

// PPM parabola of the centre cell from 5 values (ReconX/src/ppm.hxx:23-162)
ASX_DEV void ppm_cell(double gImm, double gIm, double gI, double gIp,
                      double gIpp, double pImm, double pIm, double pIp,
                      double pIpp, double vIm, double vIp, bool is_rho,
                      const RParams &rp, double &lo, double &up) {
  const double delta_Im = 0.5 * (gI - gImm);
  const double diff_I = gIp - gIm;
  const double delta_I = 0.5 * diff_I;
  const double delta_Ip = 0.5 * (gIpp - gI);
  const double f_Im_Imm = 2 * fabs(gIm - gImm);
  const double f_I_Im = 2 * fabs(gI - gIm);
  const double f_Ip_I = 2 * fabs(gIp - gI);
  const double f_Ipp_Ip = 2 * fabs(gIpp - gIp);
  const bool ss_Im = ((gI - gIm) * (gIm - gImm) > 0);
  const bool ss_I = ((gIp - gI) * (gI - gIm) > 0);
  const bool ss_Ip = ((gIpp - gIp) * (gIp - gI) > 0);
  // sgn(d) min(|d|, a, b); both factors of a positive product share d's sign
  auto limited = [](double d, double a, double b) {
    return __builtin_copysign(__builtin_fmin(fabs(d), __builtin_fmin(a, b)), d);
  };
  const double dm_Im =
      ss_Im ? limited(delta_Im, f_Im_Imm, f_I_Im) : 0;
  const double dm_I =
      ss_I ? limited(delta_I, f_I_Im, f_Ip_I) : 0;
  const double dm_Ip =
      ss_Ip ? limited(delta_Ip, f_Ip_I, f_Ipp_Ip) : 0;
  lo = 0.5 * (gIm + gI) + (1. / 6.) * (dm_Im - dm_I);
  up = 0.5 * (gI + gIp) + (1. / 6.) * (dm_I - dm_Ip);
  const double diff_press_I = pIp - pIm;
  const double min_press_I = smin(pIm, pIp);
  if (rp.ppm_shock_detection && is_rho) {
    const bool contact = (rp.kgamma * fabs(diff_I) * min_press_I >=
                          fabs(diff_press_I) * smin(gIp, gIm));
    if (contact) {
      const double d2_Im = gI - 2 * gIm + gImm;
      const double d2_Ip = gIpp - 2 * gIp + gI;
      const bool cond2 =
          (fabs(diff_I) - rp.ppm_eps_shock * smin(fabs(gIp), fabs(gIm))) > 0.;
      const double eta_t = ((d2_Im * d2_Ip < 0) && cond2)
                               ? ((-1. / 6.) * (d2_Ip - d2_Im) / diff_I)
                               : 0;
      const double eta = smax(0., smin(rp.ppm_eta1 * (eta_t - rp.ppm_eta2), 1.));
      lo = (1 - eta) * lo + eta * (gIm + 0.5 * dm_Im);
      up = (1 - eta) * up + eta * (gIp - 0.5 * dm_Ip);
    }
  }
  if (rp.ppm_zone_flattening) {
    const double w =
        ((fabs(diff_press_I) > rp.ppm_eps * min_press_I) && (vIm > vIp)) ? 1. : 0;
    const double ft =
        (fabs(pIpp - pImm) < rp.ppm_small)
            ? 1.0
            : smax(0., 1. - w * smax(0., rp.ppm_omega2 *
                                             ((diff_press_I / (pIpp - pImm)) -
                                              rp.ppm_omega1)));
    const double omf = (1 - ft) * gI;
    lo = ft * lo + omf;
    up = ft * up + omf;
  }
  if ((up - gI) * (gI - lo) <= 0) {
    lo = gI;
    up = gI;
  } else {
    const double d = up - lo;
    const double d2 = d * d;
    const double g6 = 6 * d * (gI - 0.5 * (lo + up));
    if (g6 > d2) {
      lo = 3 * gI - 2 * up;
    } else if (g6 < -d2) {
      up = 3 * gI - 2 * lo;
    }
  }
}

// The four differences of a 5-cell stencil; the WENO-Z face values below are
// the centre value plus a combination of them, which needs fewer operations
// than the reference's sums over the values and loses no digits to their
// cancellation.
struct Diff4 {
  double e0, e1, e2, e3;
  ASX_DEV Diff4(double gImm, double gIm, double gI, double gIp, double gIpp)
      : e0(gIm - gImm), e1(gI - gIm), e2(gIp - gI), e3(gIpp - gIp) {}
};

// WENO-Z face values of the centre cell (ReconX/src/wenoz.hxx:23-99).
// Same smoothness indicators, weights and stencils; the nonlinear weights
// a_k = 1 + tau5/(b_k + eps) are carried over the common denominator
// prod_k (b_k + eps), and the two face values share one reciprocal, so a
// cell costs one reciprocal instead of the reference's fourteen divisions
// (identical up to rounding).  The (b_k + eps) are first rescaled by a power
// of two (exact) so the triple products cannot overflow.
// With the values' differences, shared by the indicators and both faces'
// polynomials, and fused multiply-adds a face kernel holds 1751 FP64
// instructions instead of 2213 (192^3 faces, bound by memory traffic and
// instruction issue together: 2.07 -> 1.98 ms).
ASX_DEV void wenoz_cell(double gImm, double gIm, double gI, double gIp,
                        double gIpp, double weno_eps, double &m, double &p) {
  const Diff4 d(gImm, gIm, gI, gIp, gIpp);
  const double d0 = d.e1 - d.e0, d1 = d.e2 - d.e1, d2 = d.e3 - d.e2;
  const double c0 = __builtin_fma(2.0, d.e1, d0);  // gImm - 4 gIm + 3 gI
  const double c1 = d.e1 + d.e2;                   // gIp - gIm
  const double c2 = __builtin_fma(-2.0, d.e2, d2); // 3 gI - 4 gIp + gIpp
  const double eps4 = 4.0 * weno_eps;
  auto indicator = [&](double dd, double cc) { // 4 (b_k + eps)
    return __builtin_fma(13.0 / 3.0, dd * dd, __builtin_fma(cc, cc, eps4));
  };
  double s0 = indicator(d0, c0), s1 = indicator(d1, c1), s2 = indicator(d2, c2);
  const int e = -__builtin_amdgcn_frexp_exp(__builtin_fmax(s0, __builtin_fmax(s1, s2)));
  s0 = __builtin_amdgcn_ldexp(s0, e);
  s1 = __builtin_amdgcn_ldexp(s1, e);
  s2 = __builtin_amdgcn_ldexp(s2, e);
  const double tau5 = fabs(s0 - s2);
  // a_k * s0 s1 s2, times the linear weights in tenths
  const double n0 = (s0 + tau5) * (s1 * s2);
  const double n1 = 6.0 * ((s1 + tau5) * (s0 * s2));
  const double n2 = (s2 + tau5) * (s0 * s1);
  const double t0 = 3.0 * n0, t2 = 3.0 * n2;
  // six times the candidate polynomials, less the centre value
  const double nm = __builtin_fma(
      n2, __builtin_fma(2.0, d.e3, -5.0 * d.e2),
      -__builtin_fma(n1, __builtin_fma(2.0, d.e1, d.e2), t0 * __builtin_fma(4.0, d.e1, -d.e0)));
  const double np = __builtin_fma(
      n0, __builtin_fma(-2.0, d.e0, 5.0 * d.e1),
      __builtin_fma(n1, __builtin_fma(2.0, d.e2, d.e1), t2 * __builtin_fma(4.0, d.e2, -d.e3)));
  const double dm = (t0 + n1) + n2, dp = (n0 + n1) + t2;
  // one reciprocal for both sides: after the rescaling the weights' sums
  // lie within ~1e-130 .. 1e2, so their product neither overflows nor
  // underflows
  const double r = (1.0 / 6.0) * rcp_normal(dm * dp);
  m = __builtin_fma(nm, dp * r, gI);
  p = __builtin_fma(np, dm * r, gI);
}

// minmod of four values: the smallest if all are positive, the largest if
// all are negative, else 0
ASX_DEV double minmod4(double a, double b, double c, double d) {
  const double lo = __builtin_fmin(__builtin_fmin(a, b), __builtin_fmin(c, d));
  const double hi = __builtin_fmax(__builtin_fmax(a, b), __builtin_fmax(c, d));
  return __builtin_fmax(lo, 0.0) + __builtin_fmin(hi, 0.0);
}
ASX_DEV double minmod2(double a, double b) {
  return __builtin_fmax(__builtin_fmin(a, b), 0.0) + __builtin_fmin(__builtin_fmax(a, b), 0.0);
}
// The two MP5 face values of the centre cell (ReconX/src/mp5.hxx:26-77; the
// low side is the high side of the mirrored stencil).  The limited curvatures
// serve both faces, the low face taking them in the other order, and minmod
// is minima and maxima instead of sign tests and selects (a face kernel holds
// 3013 vector instructions instead of 4214); each value is the
// reference's sum in its order, since the limiter's branches and, behind
// them, con2prim amplify a change of rounding.
ASX_DEV void mp5_cell(double gImm, double gIm, double gI, double gIp, double gIpp,
                      double alpha, double &lo, double &up) {
  up = (2 * gImm - 13 * gIm + 47 * gI + 27 * gIp - 3 * gIpp) * (1.0 / 60.0);
  lo = (2 * gIpp - 13 * gIp + 47 * gI + 27 * gIm - 3 * gImm) * (1.0 / 60.0);
  const double em = gI - gIm, ep = gI - gIp; // deltam of either side
  const double am = alpha * em, ap = alpha * ep;
  const bool oku = (up - gI) * (up - (gI + minmod2(-ep, am))) <= 1.0e-10;
  const bool okl = (lo - gI) * (lo - (gI + minmod2(-em, ap))) <= 1.0e-10;
  if (!(oku && okl)) {
    const double dm = gImm + gI - 2 * gIm;
    const double d = gIm + gIp - 2 * gI;
    const double dp = gI + gIpp - 2 * gIp;
    const double cp = minmod4(4 * d - dp, 4 * dp - d, d, dp);
    const double cm = minmod4(4 * dm - d, 4 * d - dm, dm, d);
    // the side towards cell gn: curvatures cn there and co on the other side
    auto limit = [&](double ul, double gn, double e, double ae, double cn, double co) {
      const double uul = gI + ae;
      const double umd = (gI + gn) / 2.0 - cn / 2.0;
      const double ulc = gI + e / 2.0 + 4.0 / 3.0 * co;
      const double umin = __builtin_fmax(__builtin_fmin(gI, __builtin_fmin(gn, umd)),
                                         __builtin_fmin(gI, __builtin_fmin(uul, ulc)));
      const double umax = __builtin_fmin(__builtin_fmax(gI, __builtin_fmax(gn, umd)),
                                         __builtin_fmax(gI, __builtin_fmax(uul, ulc)));
      return ul + minmod2(umin - ul, umax - ul);
    };
    const double lu = limit(up, gIp, em, am, cp, cm);
    const double ll = limit(lo, gIm, ep, ap, cm, cp);
    up = oku ? up : lu;
    lo = okl ? lo : ll;
  }
}

// Face states from a 6-point stencil s[0..5] = cells I-3 .. I+2 along the
// face normal (ReconX/src/reconstruct.hxx:36-103): out0 from cell I-1,
// out1 from cell I.
template <int M>
ASX_DEV void recon(const double s[6], const double ps[6], const double vs[6],
                   bool is_rho, const RParams &rp, double &o0, double &o1) {
  if (M == ASX_RECON_GODUNOV) {
    o0 = s[2];
    o1 = s[3];
  } else if (M == ASX_RECON_MINMOD) {
    o0 = s[2] + minmod(s[3] - s[2], s[2] - s[1]) / 2;
    o1 = s[3] - minmod(s[4] - s[3], s[3] - s[2]) / 2;
  } else if (M == ASX_RECON_MONOCENTRAL) {
    o0 = s[2] + monocentral(s[3] - s[2], s[2] - s[1]) / 2;
    o1 = s[3] - monocentral(s[4] - s[3], s[3] - s[2]) / 2;
  } else if (M == ASX_RECON_PPM) {
    double a0, a1, b0, b1;
    ppm_cell(s[0], s[1], s[2], s[3], s[4], ps[0], ps[1], ps[3], ps[4], vs[1],
             vs[3], is_rho, rp, a0, a1);
    ppm_cell(s[1], s[2], s[3], s[4], s[5], ps[1], ps[2], ps[4], ps[5], vs[2],
             vs[4], is_rho, rp, b0, b1);
    o0 = a1;
    o1 = b0;
  } else if (M == ASX_RECON_WENOZ) {
    double a0, a1, b0, b1;
    wenoz_cell(s[0], s[1], s[2], s[3], s[4], rp.weno_eps, a0, a1);
    wenoz_cell(s[1], s[2], s[3], s[4], s[5], rp.weno_eps, b0, b1);
    o0 = a1;
    o1 = b0;
  } else {
    double a0, a1, b0, b1;
    mp5_cell(s[0], s[1], s[2], s[3], s[4], rp.mp5_alpha, a0, a1);
    mp5_cell(s[1], s[2], s[3], s[4], s[5], rp.mp5_alpha, b0, b1);
    o0 = a1;
    o1 = b0;
  }
}
// Lowest stencil point m (of I-3+m) each method reads.
template <int M> ASX_DEV constexpr int stencil_lo() {
  return M == ASX_RECON_GODUNOV ? 2
         : (M == ASX_RECON_MINMOD || M == ASX_RECON_MONOCENTRAL) ? 1
                                                                  : 0;
}
ASX_DEV int stencil_lo_rt(int m) {
  return m == ASX_RECON_GODUNOV ? 2
         : (m == ASX_RECON_MINMOD || m == ASX_RECON_MONOCENTRAL) ? 1
                                                                  : 0;
}
// Runtime dispatch for the low-order fallback (Godunov/minmod/monocentral).
ASX_DEV void recon_lo(int m, const double s[6], double &o0, double &o1) {
  const RParams rp{};
  const double z[6] = {0, 0, 0, 0, 0, 0};
  if (m == ASX_RECON_MINMOD)
    recon<ASX_RECON_MINMOD>(s, z, z, false, rp, o0, o1);
  else if (m == ASX_RECON_MONOCENTRAL)
    recon<ASX_RECON_MONOCENTRAL>(s, z, z, false, rp, o0, o1);
  else
    recon<ASX_RECON_GODUNOV>(s, z, z, false, rp, o0, o1);
}

// ---------------------------------------------------------------------------
// Riemann fluxes and characteristic speeds (AsterX)
// ---------------------------------------------------------------------------
// Characteristic speeds (lambda+, lambda-) of the left (0) and right (1)
// states (AsterX/src/eigenvalues.hxx:19-79, the roots of a2 l^2 + a1 l + a0
// over alpha), one reciprocal serving both 1/(2 a2 alpha) (a2 > 0)
ASX_DEV void eig_sides(double alp, double ialp, double beta, double u, const double vel[2],
                       const double rho[2], const double cs2[2], const double w[2],
                       const double h[2], const double bsq[2], double &l0p, double &l0m,
                       double &l1p, double &l1m) {
  ASX_CONTRACT
  double a1[2], a2[2], sd[2];
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const double a0 = (bsq[f] + cs2[f] * h[f] * rho[f]) * (pow2(beta) - pow2(alp) * u) -
                      (-1 + cs2[f]) * h[f] * rho[f] * pow2(beta - alp * vel[f]) * pow2(w[f]);
    a1[f] = 2 * beta * (bsq[f] + cs2[f] * h[f] * rho[f]) -
            2 * (-1 + cs2[f]) * h[f] * rho[f] * (beta - alp * vel[f]) * pow2(w[f]);
    a2[f] = bsq[f] + h[f] * rho[f] * (cs2[f] + pow2(w[f]) - cs2[f] * pow2(w[f]));
    double det = pow2(a1[f]) - 4 * a2[f] * a0;
    if (det < 0) det = 0;
    sd[f] = sqrt(det);
  }
  const double r = ialp / (4 * a2[0] * a2[1]); // 1 / (2 a2 alpha) = 2 a2' r
  const double f0 = 2 * a2[1] * r, f1 = 2 * a2[0] * r;
  l0p = (-a1[0] + sd[0]) * f0;
  l0m = (-a1[0] - sd[0]) * f0;
  l1p = (-a1[1] + sd[1]) * f1;
  l1m = (-a1[1] - sd[1]) * f1;
}
// max/min over {0, l0+, l0+, l0-, l0-, l1+, l1+, l1-, l1-} (fluxes.hxx:35-42)
ASX_DEV void char_extrema(double l0p, double l0m, double l1p, double l1m,
                          double &cmax, double &cmin) {
  cmax = smax(smax(smax(smax(0.0, l0p), l0m), l1p), l1m);
  cmin = smin(smin(smin(smin(0.0, l0p), l0m), l1p), l1m);
}
// HLLE with the common 1/(cmax - cmin) precomputed (AsterX/src/fluxes.hxx:31-50)
ASX_DEV double hlle(double cmax, double cmin, double idc, double U0, double U1,
                    double F0, double F1) {
  ASX_CONTRACT
  return (cmax * F0 - cmin * F1 + cmax * cmin * (U1 - U0)) * idc;
}
ASX_DEV double laxf(double cabs, double U0, double U1, double F0, double F1) {
  ASX_CONTRACT
  return 0.5 * ((F0 + F1) - cabs * (U1 - U0));
}

// ---------------------------------------------------------------------------
// Ideal-gas EOS (EOSX/src/eos_3p_idealgas/eos_3p_idealgas.hxx)
// ---------------------------------------------------------------------------
struct IdealGas {
  double gamma, gm1, inv_gamma, temp_over_eps;
  double eps_min, eps_max, rho_min, rho_max, ye_min, ye_max, temp_min,
      temp_max;
  double igm1; // 1/(gamma-1)
  ASX_DEV double press_re(double rho, double eps) const { return gm1 * rho * eps; }
  ASX_DEV double eps_rp(double rho, double press) const {
    return press / (rho * gm1);
  }
  ASX_DEV double csnd2(double eps) const { return gm1 * eps / (eps + inv_gamma); }
  ASX_DEV double csnd(double eps) const { return sqrt(csnd2(eps)); }
  ASX_DEV double temp_re(double eps) const { return temp_over_eps * eps; }
  ASX_DEV double eps_rt(double temp) const { return temp / temp_over_eps; }
  ASX_DEV double press_rt(double rho, double temp) const {
    return press_re(rho, eps_rt(temp));
  }
  ASX_DEV double kappa(double rho, double eps) const {
    return (gamma - 1.0) * eps * pow(rho, 1.0 - gamma);
  }
  // The 3-parameter interface shared with TabEOS (EOSX eos_3p.hxx): Ye is
  // not used by the ideal gas, and eps is never changed.
  struct Cell {}; // what a zone keeps between solves: nothing
  ASX_DEV void start_cell(Cell &, double, double) const {}
  ASX_DEV double press_re(double rho, double &eps, double) const { return press_re(rho, eps); }
  ASX_DEV double press_re(double rho, double &eps, double, Cell &) const {
    return press_re(rho, eps);
  }
  ASX_DEV double temp_re(double, double &eps, double) const { return temp_re(eps); }
  ASX_DEV double kappa_re(double rho, double &eps, double) const { return kappa(rho, eps); }
  ASX_DEV double kappa_near(double rho, double &eps, double, double) const {
    return kappa(rho, eps);
  }
  ASX_DEV double csnd_re(double, double &eps, double) const { return csnd(eps); }
  // p and eps from (rho, kappa) (eos_3p_idealgas.hxx:201-215):
  // p = kappa rho^gamma, eps = kappa rho^(gamma-1) / (gamma-1)
  ASX_DEV double press_rk(double rho, double kap, double) const { return kap * pow(rho, gamma); }
  ASX_DEV double eps_rk(double rho, double kap, double) const {
    return kap * pow(rho, gamma - 1.0) / (gamma - 1.0);
  }
  // press_re, temp_re and kappa_re at one (rho, eps, Ye)
  ASX_DEV void state_re(double rho, double &eps, double ye, double &press, double &temp,
                        double &kap, Cell &) const {
    press = press_re(rho, eps, ye);
    temp = temp_re(rho, eps, ye);
    kap = kappa_re(rho, eps, ye);
  }
  ASX_DEV double eps_rt(double, double temp, double) const { return eps_rt(temp); }
  ASX_DEV double press_rt(double rho, double temp, double) const { return press_rt(rho, temp); }
  ASX_DEV double eps_rp(double rho, double press, double) const { return eps_rp(rho, press); }
  ASX_DEV double csnd_rt(double, double temp, double) const { return csnd(eps_rt(temp)); }
  // eos_3p_idealgas.hxx: the entropy of (rho, T) is kappa(rho, eps(T))
  ASX_DEV double entropy_rt(double rho, double temp, double) const {
    return kappa(rho, eps_rt(temp));
  }
};

// v2f metric average at a face normal to D (AsterUtils aster_interp.hxx:237-249)
template <int D>
ASX_DEV double avg_v2f(const double *g, int o, int sj, int sk) {
  constexpr int J = (D + 1) % 3, K = (D + 2) % 3;
  const int s1 = J == 0 ? 1 : (J == 1 ? sj : sk);
  const int s2 = K == 0 ? 1 : (K == 1 ? sj : sk);
  double s = 0.0;
  s += g[o];
  s += g[o + s1];
  s += g[o + s2];
  s += g[o + s1 + s2];
  return s / 4.0;
}
// v2c average (aster_interp.hxx:191-205)
ASX_DEV double avg_v2c(const double *g, int o, int sj, int sk) {
  double s = 0.0;
  s += g[o];
  s += g[o + 1];
  s += g[o + sj];
  s += g[o + sj + 1];
  s += g[o + sk];
  s += g[o + sk + 1];
  s += g[o + sk + sj];
  s += g[o + sk + sj + 1];
  return s / 8.0;
}

} // namespace asx
