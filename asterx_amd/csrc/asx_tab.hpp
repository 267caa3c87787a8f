// Tabulated 3-parameter EOS for gfx950 (EOSX eos_3p_tabulated3d): a table
// of log p, log(eps + shift), c_s^2 and entropy over axes log rho, log T,
// Ye (code units; axes uniform), the variable index fastest, and the EOSX interface
// on it (EOSX/src/eos_3p_tabulated3d/eos_3p_tabulated3d.hxx:186-357):
// trilinear interpolation in the order of eos_linear_interp_ND.hxx (rho,
// then T, then Ye) and the same clamping of the inputs, including the
// change of eps the reference makes through its reference argument.  The
// temperature from (rho, eps, Ye) is the root the reference's Brent
// iteration (EOSX/src/utils/eos_brent.hxx, tolerance 1e-14 in log T)
// approaches, solved exactly on the piecewise-linear interpolant.
#pragma once

#include "asx_device.hpp"

namespace asx {

struct TabEOS {
  enum { PRESS = 0, EPS = 1, CS2 = 2, ENT = 3, NV = 4 };
  const double *tab;    // [v + NV * (ir + n0 * (it + n1 * iy))]
  const double *ax[3];  // axis values: log rho, log T, Ye
  int n[3];
  double idx[3];        // 1 / (ax[d][1] - ax[d][0])
  double shift;         // energy shift
  double rho_min, rho_max, temp_min, temp_max, ye_min, ye_max; // rgrho, rgtemp, rgye
  double eps_min, eps_max;                                     // rgeps
  int grows; // eps grows with T along every (rho, Ye) line (asx_eos_table)

  // nearest lower node, uniform axis (eos_linear_interp_ND.hxx:57-73)
  ASX_DEV int find(int d, double x) const {
    const double xl = x - ax[d][0];
    if (!(xl > 0.0)) return 0;
    const double f = xl * idx[d];
    const int last = n[d] - 2;
    return f >= (double)last ? last : (int)f;
  }
  ASX_DEV static double lin(double A, double B, double xA, double xB, double x) {
    const double l = (x - xA) / (xB - xA);
    return (B - A) * l + A;
  }
  // one variable at (log rho, log T, Ye)
  ASX_DEV double interp(int v, double lr, double lt, double ye) const {
    const int i0 = find(0, lr), i1 = find(1, lt), i2 = find(2, ye);
    const int s1 = NV * n[0], s2 = NV * n[0] * n[1];
    const double *p = tab + v + NV * i0 + s1 * i1 + s2 * i2;
    const double r0 = ax[0][i0], r1 = ax[0][i0 + 1];
    const double t0 = ax[1][i1], t1 = ax[1][i1 + 1];
    const double y0 = ax[2][i2], y1 = ax[2][i2 + 1];
    const double a00 = lin(p[0], p[NV], r0, r1, lr);
    const double a10 = lin(p[s1], p[s1 + NV], r0, r1, lr);
    const double a01 = lin(p[s2], p[s2 + NV], r0, r1, lr);
    const double a11 = lin(p[s2 + s1], p[s2 + s1 + NV], r0, r1, lr);
    const double b0 = lin(a00, a10, t0, t1, lt);
    const double b1 = lin(a01, a11, t0, t1, lt);
    return lin(b0, b1, y0, y1, ye);
  }
  // p, eps and c_s^2 at one point (indices found once)
  ASX_DEV void interp3(double lr, double lt, double ye, double out[3]) const {
    const int i0 = find(0, lr), i1 = find(1, lt), i2 = find(2, ye);
    const int s1 = NV * n[0], s2 = NV * n[0] * n[1];
    const double *p = tab + NV * i0 + s1 * i1 + s2 * i2;
    const double r0 = ax[0][i0], r1 = ax[0][i0 + 1];
    const double t0 = ax[1][i1], t1 = ax[1][i1 + 1];
    const double y0 = ax[2][i2], y1 = ax[2][i2 + 1];
#pragma unroll
    for (int v = 0; v < 3; ++v) {
      const double a00 = lin(p[v], p[v + NV], r0, r1, lr);
      const double a10 = lin(p[v + s1], p[v + s1 + NV], r0, r1, lr);
      const double a01 = lin(p[v + s2], p[v + s2 + NV], r0, r1, lr);
      const double a11 = lin(p[v + s2 + s1], p[v + s2 + s1 + NV], r0, r1, lr);
      const double b0 = lin(a00, a10, t0, t1, lt);
      const double b1 = lin(a01, a11, t0, t1, lt);
      out[v] = lin(b0, b1, y0, y1, ye);
    }
  }
  // eps_rt, press_rt and csnd_rt^2 at one (rho, T, Ye) from one lookup; the
  // pressure is looked up again at the unbounded (rho, T) when either lies
  // outside the table (press_rt takes the logs of the inputs)
  ASX_DEV void state_rt(double rho, double temp, double ye, double &eps, double &press,
                        double &cs2) const {
    const double rc = crho(rho), tc = ctemp(temp);
    double v[3];
    interp3(log(rc), log(tc), ye, v);
    eps = exp(v[EPS]) - shift;
    press = (rc == rho && tc == temp) ? exp(v[PRESS]) : press_rt(rho, temp, ye);
    const double cs = sqrt(v[CS2]);
    cs2 = cs * cs;
  }
  // std::fmin / std::fmax as the reference (a NaN argument is dropped)
  ASX_DEV double crho(double rho) const { return fmin(fmax(rho, rho_min), rho_max); }
  ASX_DEV double ctemp(double t) const { return fmin(fmax(t, temp_min), temp_max); }
  ASX_DEV double xmin1() const { return ax[1][0]; }
  ASX_DEV double xmax1() const { return ax[1][n[1] - 1]; }

  // logtemp_from_valid_rho_eps_ye (eos_3p_tabulated3d.hxx:186-218)
  ASX_DEV double logtemp_re(double rho, double &eps, double ye) const {
    const double r = crho(rho);
    eps = fmax(eps + shift, eps_min + shift) - shift;
    const double lrho = log(r);
    const double leps = log(eps + shift);
    const double vmin = interp(EPS, lrho, xmin1(), ye);
    const double vmax = interp(EPS, lrho, xmax1(), ye);
    if (leps <= vmin) {
      eps = exp(vmin) - shift;
      return xmin1();
    }
    if (leps >= vmax) {
      eps = exp(vmax) - shift;
      return xmax1();
    }
    return logtemp_nodes(lrho, leps, ye, vmin, vmax);
  }
  // The table cell of a zone's previous solve, kept in registers between the
  // solves of one zone: node indices (i0 < 0: none yet), the cell's position
  // and inverse width on each axis, and per corner [Ye][T][rho]
  // log(eps + shift) and log p.  full: the next cell may not be looked for
  // from this one, see solve_re.
  struct Cell {
    int i0 = -1, i1 = -1, i2 = 0;
    bool full = false;
    double r0, ri, t0, dt, ly; // log rho: low node, 1 / width; log T: low node, width; Ye weight
    double e[2][2][2], p[2][2][2];
  };
  // Start of a zone's solves: its Ye, and a temperature near which to look.
  // Between the Ye nodes a table that grows with T still grows; beyond them
  // (by more than the rounding of the weight) the difference of two growing
  // lines need not.
  ASX_DEV void start_cell(Cell &c, double ye, double temp) const {
    c.i2 = find(2, ye);
    c.ly = (ye - ax[2][c.i2]) / (ax[2][c.i2 + 1] - ax[2][c.i2]);
    c.full = !(grows && c.ly >= -1e-15 && c.ly <= 1.0 + 1e-15);
    c.i1 = find(1, log(ctemp(temp)));
    c.i0 = -1;
  }
  ASX_DEV void load_cell(Cell &c, int i0, int i1) const {
    const int s1 = NV * n[0], s2 = NV * n[0] * n[1];
    const double *q = tab + NV * i0 + s1 * i1 + s2 * c.i2;
    if (c.i0 != i0) {
      c.r0 = ax[0][i0];
      c.ri = 1.0 / (ax[0][i0 + 1] - c.r0);
    }
    c.t0 = ax[1][i1];
    c.dt = ax[1][i1 + 1] - c.t0;
    c.i0 = i0;
    c.i1 = i1;
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const double *v = q + y * s2 + t * s1 + r * NV; // log p and log eps are adjacent
          c.p[y][t][r] = v[PRESS];
          c.e[y][t][r] = v[EPS];
        }
  }
  // p and log T from (rho, eps, Ye): logtemp_re's root, to rounding.
  // Where eps grows with T along the (rho, Ye) line one cell brackets the
  // root, so the search may start anywhere, and starts from the zone's
  // previous cell.  A zone's consecutive solves (the Brent
  // iterates, then the final state) move rho and eps by less and less, so
  // the cell they end in repeats: its corner values stay in registers and a
  // solve inside it reads no memory.  When the root has left it, the next
  // cell is predicted from the cell's slope d eps / d T (exact for a thermal
  // energy linear in T, so it usually lands on the cell or beside it) and
  // checked at its own nodes; a miss is searched outwards from there by
  // doubling steps, then bisected.  Where eps need not grow (Cell::full)
  // several cells may hold a root: the axis is bisected from its ends, as
  // logtemp_re does it, and no result depends on where a search began.
  // Bound by the latency of dependent table reads: some lane of a wavefront
  // leaves its cell in almost every iteration, and a search from scratch
  // costs the whole wavefront eight dependent probes.  Con2prim of 1 000 003
  // zones on the 234 x 180 x 50 table: 2.75 ms with the search from scratch
  // outside the previous T cell, 0.79 ms with this (table reads per
  // wavefront 1490 -> 436, waves waiting 74 % -> 34 % of their time), 0.75
  // since a predicted cell that holds is not loaded a second time; keeping
  // the corners alone, without the prediction, left it at 2.70.
  ASX_DEV void solve_re(double rho, double &eps, Cell &c, double &lrho, double &lt,
                        double &press) const {
    const double r = crho(rho);
    eps = fmax(eps + shift, eps_min + shift) - shift;
    lrho = log(r);
    const double es = eps + shift, leps = log(es);
    const int i0 = find(0, lrho), last = n[1] - 1;
    if (c.i0 != i0) load_cell(c, i0, c.i1);
    const double lr = (lrho - c.r0) * c.ri;
    auto mix = [&](const double (&v)[2][2][2], int t) {
      const double a0 = (v[0][t][1] - v[0][t][0]) * lr + v[0][t][0];
      const double a1 = (v[1][t][1] - v[1][t][0]) * lr + v[1][t][0];
      return (a1 - a0) * c.ly + a0;
    };
    double elo = mix(c.e, 0), ehi = mix(c.e, 1);
    // outside [elo, ehi): every lane of the wavefront that has left its cell
    auto below = [&] { return !(elo <= leps); };
    auto above = [&] { return !(leps < ehi); };
    if (c.full || (below() && c.i1 > 0) || (above() && c.i1 < last - 1)) {
      const int s1 = NV * n[0];
      const double *row = tab + EPS + NV * i0 + s1 * n[1] * c.i2;
      auto node = [&](int m) {
        const double *q = row + s1 * m;
        const int s2 = s1 * n[1];
        const double a0 = (q[NV] - q[0]) * lr + q[0];
        const double a1 = (q[s2 + NV] - q[s2]) * lr + q[s2];
        return (a1 - a0) * c.ly + a0;
      };
      int lo, hi; // the root's cell is looked for between these nodes
      if (c.full) {
        const bool low = leps <= node(0), high = leps >= node(last);
        lo = high && !low ? last - 1 : 0;
        hi = low ? 1 : last;
      } else {
        // eps linear in T through the cell's nodes, in single precision
        const float k = 1.44269504f;
        const float dlo = __builtin_amdgcn_exp2f(k * (float)(elo - leps));
        const float dhi = __builtin_amdgcn_exp2f(k * (float)(ehi - leps));
        const float th = __builtin_amdgcn_exp2f(k * (float)c.dt);
        // T / T_lo at the target
        const float x = 1.0f + (1.0f - dlo) * (th - 1.0f) / (dhi - dlo);
        const float step = __builtin_amdgcn_logf(fmaxf(x, 1e-30f)) / (k * (float)c.dt);
        int j = c.i1 + (int)fminf(fmaxf(floorf(step), -(float)last), (float)last);
        j = below() ? min(j, c.i1 - 1) : max(j, c.i1 + 1); // past the cell it left
        j = min(max(j, 0), last - 1);
        load_cell(c, i0, j);
        elo = mix(c.e, 0);
        ehi = mix(c.e, 1);
        lo = j;
        hi = j + 1;
        int d = 1;
        if (below()) {
          while (lo > 0 && below()) {
            hi = lo;
            lo = max(lo - d, 0);
            d *= 2;
            elo = node(lo);
          }
        } else {
          while (hi < last && above()) {
            lo = hi;
            hi = min(hi + d, last);
            d *= 2;
            ehi = node(hi);
          }
        }
      }
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (node(mid) <= leps) lo = mid;
        else hi = mid;
      }
      if (lo != c.i1) load_cell(c, i0, lo);
      elo = mix(c.e, 0);
      ehi = mix(c.e, 1);
    }
    double f; // log T weight in the cell
    if (c.i1 == 0 && leps <= elo) { // at or below the table's lowest T
      eps = exp(elo) - shift;
      f = 0.0;
    } else if (c.i1 == last - 1 && leps >= ehi) {
      eps = exp(ehi) - shift;
      f = 1.0;
    } else {
      f = (leps - elo) / (ehi - elo);
    }
    lt = c.t0 + f * c.dt;
    const double b0 = mix(c.p, 0), b1 = mix(c.p, 1);
    press = exp((b1 - b0) * f + b0);
  }
  // E_j at the node row q of the T axis: log(eps + shift) interpolated in
  // log rho, then in Ye (the reference's order)
  ASX_DEV static double enode(const double *q, int s2, double r0, double r1, double y0,
                              double y1, double lrho, double ye) {
    const double a0 = lin(q[0], q[NV], r0, r1, lrho);
    const double a1 = lin(q[s2], q[s2 + NV], r0, r1, lrho);
    return lin(a0, a1, y0, y1, ye);
  }
  // The root in log T of interp(EPS, lrho, lt, ye) = leps for
  // vmin < leps < vmax (the interpolant's values at the ends of the T
  // axis).  At fixed (lrho, ye) the interpolant is linear in lt inside each
  // cell [t_j, t_j+1], between the node values E_j (the bilinear rho, Ye
  // interpolation at T node j, in the reference's order), so the root is
  // found exactly: a bisection over the node index keeps
  // E_lo <= leps < E_hi -- a sign change, hence a root, in between -- down
  // to adjacent nodes, then that cell's linear equation is solved.  Brent's
  // iteration on the same function stops within 2 eps |lt| + 1e-14 of this
  // root, after about twice as many dependent steps of twice the reads.
  ASX_DEV double logtemp_nodes(double lrho, double leps, double ye, double vmin,
                               double vmax) const {
    const int i0 = find(0, lrho), i2 = find(2, ye);
    const int s1 = NV * n[0], s2 = NV * n[0] * n[1];
    const double *p = tab + EPS + NV * i0 + s2 * i2;
    const double r0 = ax[0][i0], r1 = ax[0][i0 + 1];
    const double y0 = ax[2][i2], y1 = ax[2][i2 + 1];
    int lo = 0, hi = n[1] - 1;
    double elo = vmin, ehi = vmax;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      const double em = enode(p + s1 * mid, s2, r0, r1, y0, y1, lrho, ye);
      if (em <= leps) {
        lo = mid;
        elo = em;
      } else {
        hi = mid;
        ehi = em;
      }
    }
    const double t0 = ax[1][lo], t1 = ax[1][hi];
    return t0 + (leps - elo) * (t1 - t0) / (ehi - elo);
  }
  // press_from_valid_rho_temp_ye: the bounded rho, T are not used there
  ASX_DEV double press_rt(double rho, double temp, double ye) const {
    return exp(interp(PRESS, log(rho), log(temp), ye));
  }
  ASX_DEV double press_re(double rho, double &eps, double ye) const {
    const double lr = log(crho(rho));
    const double lt = logtemp_re(rho, eps, ye);
    return exp(interp(PRESS, lr, lt, ye));
  }
  ASX_DEV double press_re(double rho, double &eps, double, Cell &c) const {
    double lr, lt, press;
    solve_re(rho, eps, c, lr, lt, press);
    return press;
  }
  ASX_DEV double eps_rt(double rho, double temp, double ye) const {
    return exp(interp(EPS, log(crho(rho)), log(ctemp(temp)), ye)) - shift;
  }
  ASX_DEV double csnd_rt(double rho, double temp, double ye) const {
    return sqrt(interp(CS2, log(crho(rho)), log(ctemp(temp)), ye));
  }
  ASX_DEV double csnd_re(double rho, double &eps, double ye) const {
    const double lr = log(crho(rho));
    const double lt = logtemp_re(rho, eps, ye);
    return sqrt(interp(CS2, lr, lt, ye));
  }
  ASX_DEV double temp_re(double rho, double &eps, double ye) const {
    return exp(logtemp_re(rho, eps, ye));
  }
  // press_re, temp_re and kappa_re at one (rho, eps, Ye) from one
  // temperature solve.  Called in turn, the reference's functions solve
  // three times, the second and third time at the eps the first clamped;
  // where that clamp applied, the later solves may land an ulp away from
  // the table edge, which is the only difference
  ASX_DEV void state_re(double rho, double &eps, double ye, double &press, double &temp,
                        double &kap, Cell &c) const {
    double lr, lt;
    solve_re(rho, eps, c, lr, lt, press);
    temp = exp(lt);
    kap = entropy_rt(rho, temp, ye);
  }
  // entropy_from_valid_rho_temp_ye (:320-329)
  ASX_DEV double entropy_rt(double rho, double temp, double ye) const {
    return interp(ENT, log(crho(rho)), log(ctemp(temp)), ye);
  }
  // kappa_from_valid_rho_eps_ye (:331-336): the entropy at T(rho, eps, Ye)
  ASX_DEV double kappa_re(double rho, double &eps, double ye) const {
    return entropy_rt(rho, temp_re(rho, eps, ye), ye);
  }
  // the same where the temperature is known to lie near `temp`
  ASX_DEV double kappa_near(double rho, double &eps, double ye, double temp) const {
    Cell c;
    start_cell(c, ye, temp);
    double press, t, kap;
    state_re(rho, eps, ye, press, t, kap, c);
    return kap;
  }
  // eps_from_valid_rho_press_ye is refused by the reference for tables;
  // the callers that reach it (pressure atmosphere, use_temperature = no)
  // are refused at the C ABI
  ASX_DEV double eps_rp(double, double, double) const { return __builtin_nan(""); }
  // p and eps from (rho, kappa): refused by the reference for tables
  // (eos_3p_tabulated3d.hxx:315-333), and at the C ABI here
  ASX_DEV double press_rk(double, double, double) const { return __builtin_nan(""); }
  ASX_DEV double eps_rk(double, double, double) const { return __builtin_nan(""); }
};

} // namespace asx
