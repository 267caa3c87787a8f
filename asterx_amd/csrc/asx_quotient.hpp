// Quotients and reciprocals in fewer instructions than a division.  No HIP
// header is needed, so the sequences are checked on the host as well.
#pragma once

#ifndef ASX_DEV
#define ASX_DEV __device__ __forceinline__
#endif

namespace asx {

// Quotients by one divisor: x / d from d's correctly rounded reciprocal with
// the remainder of the first product added back (Markstein's sequence): the
// rounded quotient, the same bits as a division, in six instructions instead
// of about a dozen with a quarter-rate one among them.  Where the remainder is
// no finite number -- a zero, an infinity or a NaN in x or d, or a quotient
// that overflows -- the product itself is what a division gives.  What may
// differ from a division: the sign of a zero, the last bit where the remainder
// or 1/d is subnormal, and an overflow that is an ulp away.  Not for a
// subnormal divisor, whose reciprocal overflows: where holds() is false, divide
// (a factor that brings the divisor into range instead costs each quotient a
// multiplication, 3 % of an independent zone's con2prim).
struct Divisor {
  double d, r;
  ASX_DEV explicit Divisor(double x) : d(x), r(1.0 / x) {}
  ASX_DEV bool holds() const { return !(__builtin_fabs(d) < 0x1p-1022); }
};
ASX_DEV double operator/(double x, const Divisor &v) {
  const double q = x * v.r, e = __builtin_fma(-v.d, q, x);
  return __builtin_isfinite(e) ? __builtin_fma(e, v.r, q) : q;
}
ASX_DEV double &operator/=(double &x, const Divisor &v) { return x = x / v; }

// 1 / x for a normal x whose reciprocal is normal too, within about one unit
// in the last place: the hardware estimate and two Newton steps, without the
// scaling and the fix-ups of a division that works over the whole range.
ASX_DEV double rcp_normal(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
  return __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
}
// The same with a zero, an infinity and NaN as a division takes them: the
// Newton steps turn the estimate for a zero or an infinity into NaN, which the
// division's own last instruction puts right.
ASX_DEV double rcp_any(double x) { return __builtin_amdgcn_div_fixup(rcp_normal(x), x, 1.0); }

} // namespace asx
