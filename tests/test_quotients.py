"""The device code's quotients (asx_quotient.hpp), compiled for the host with
the two hardware instructions restated, against the host's division over the
whole range of doubles."""
import ctypes as C
import os
import subprocess

import numpy as np

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "asterx_amd", "csrc")
SHIM = r"""
#include <cmath>
#include <cstdint>
#include <cstring>
#define ASX_DEV inline
// v_rcp_f64: an estimate good to 2^-23 or better, here 1/x with the low bits cut
static double est(double x) {
  double r = 1.0 / x;
  if (!std::isfinite(r) || r == 0.0) return r;
  uint64_t u;
  std::memcpy(&u, &r, 8);
  u &= ~((uint64_t(1) << 28) - 1);
  std::memcpy(&r, &u, 8);
  return r;
}
// v_div_fixup_f64 of a quotient q of n / d: special operands give what a
// division gives, the others q
static double fixup(double q, double d, double n) {
  return std::isnan(d) || std::isnan(n) || d == 0.0 || std::isinf(d) || std::isinf(n) ? n / d : q;
}
#define __builtin_amdgcn_rcp est
#define __builtin_amdgcn_div_fixup fixup
#include "asx_quotient.hpp"
extern "C" void quotients(int64_t n, const double *x, const double *d, double *q, double *want,
                          double *rn, double *ra, double *rwant) {
  for (int64_t i = 0; i < n; ++i) {
    const asx::Divisor v(d[i]);
    q[i] = v.holds() ? x[i] / v : x[i] / v.d;
    want[i] = x[i] / d[i];
    rn[i] = asx::rcp_normal(d[i]);
    ra[i] = asx::rcp_any(d[i]);
    rwant[i] = 1.0 / d[i];
  }
}
"""


def _run(tmp_path, x, d):
    src, so = str(tmp_path / "q.cpp"), str(tmp_path / "q.so")
    with open(src, "w") as f:
        f.write(SHIM)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-march=x86-64-v3", "-ffp-contract=off",
                           "-fPIC", "-shared", "-I", CSRC, "-o", so, src])
    out = [np.zeros(len(x)) for _ in range(5)]
    p = lambda a: C.c_void_p(a.ctypes.data)
    C.CDLL(so).quotients(C.c_int64(len(x)), p(x), p(d), *[p(a) for a in out])
    return out


def test_quotients_and_reciprocals(tmp_path):
    rng = np.random.default_rng(0)
    ends = [0.0, 5e-324, 1e-320, 1e-315, 3e-309, 1e-308, 2.2250738585072014e-308, 1e-300, 1e-160,
            0.1, 1.0, 3.0, 1e160, 1e300, 8.9e307, 1.7976931348623157e308, np.inf, np.nan]
    ends = np.array(ends + [-e for e in ends])
    # every pair of ends, and every end against mantissas of one binade
    x, d = (a.ravel() for a in np.meshgrid(ends, ends))
    m = rng.uniform(1, 2, 64)
    a, b = (t.ravel() for t in np.meshgrid(ends, m))
    n = 10 ** 6
    u = np.ldexp(rng.uniform(1, 2, (2, n)), rng.integers(-1073, 1024, (2, n)))
    w = rng.uniform(1, 2, (2, n)) * 10.0 ** rng.uniform(-40, 40, (2, n))
    x = np.concatenate([x, a, b, u[0], w[0]])
    d = np.concatenate([d, b, a, u[1], w[1]])
    q, want, rn, ra, rwant = _run(tmp_path, x, d)
    same = (q == want) | (np.isnan(q) & np.isnan(want))
    # the remainder x - d q is below 2^-52 x, the quotient's last bit lies at
    # 2^-52 of it: either may be subnormal, as 1/d may be, and the last bit
    # then off by one
    tiny = (np.abs(x) < 2.0 ** -969) | (np.abs(want) < 2.0 ** -1021) | (np.abs(d) > 2.0 ** 1021)
    bad = ~(same | tiny)
    assert not bad.any(), (x[bad][:3], d[bad][:3], q[bad][:3])
    assert (np.abs(q[~same] - want[~same]) <= np.spacing(np.abs(want[~same]))).all()
    # reciprocals: a unit in the last place where x and 1/x are normal ...
    ok = (np.abs(d) >= 2.0 ** -1021) & (np.abs(d) <= 2.0 ** 1021)
    for r in (rn, ra):
        assert (np.abs(r[ok] - rwant[ok]) <= np.spacing(np.abs(rwant[ok]))).all()
    # ... and what a division gives at a zero, an infinity and NaN
    sp = (d == 0) | ~np.isfinite(d)
    assert np.array_equal(ra[sp], rwant[sp], equal_nan=True)
    assert np.array_equal(np.signbit(ra[d == 0]), np.signbit(d[d == 0]))
