// fdiv.hpp -- correctly rounded FP64 division with a shared reciprocal.
//
// For a / b the compiler emits the gfx9 IEEE division sequence
//
//   s_b = v_div_scale(b, b, a);  s_a = v_div_scale(a, b, a)   (range scaling)
//   y   = v_rcp_f64(s_b)
//   e   = fma(-s_b, y, 1);  y = fma(y, e, y)                   (Newton, twice)
//   e   = fma(-s_b, y, 1);  y = fma(y, e, y)
//   q   = s_a * y;  r = fma(-s_b, q, s_a)
//   d   = v_div_fmas(r, y, q)       = fma(r, y, q) unless scaled
//   res = v_div_fixup(d, b, a)      = d unless an operand or the result is
//                                     zero, infinite, NaN or out of range
//
// When |a| and |b| lie in [2^-390, 2^390] (or a is zero), the scaling steps
// return their operands unchanged: the exponent difference stays below 768,
// neither operand nor the quotient is denormal, the numerator's exponent is
// far above the near-underflow threshold and 1/b is normal.  In that case the
// fixup only matters for a zero numerator (signed zero).  Then the
// sequence without those steps yields the same bits.  y depends on b alone, so one
// refined reciprocal serves every quotient with that denominator: each
// further quotient costs a multiply and two FMAs instead of the whole
// sequence.
//
// Signed zeros: with the remainder taken as r' = fma(b, q, -a) = -r (exact)
// and the result fma(-r', y, q), a zero numerator yields the zero the fixup
// would return (sign of a times sign of b) for every b > 0.  All callers
// divide by positive quantities.
//
// Callers check the range condition (usually once for a group of
// divisions) and fall back to plain `/` when it fails.
#pragma once
#ifndef HYPE_KNS
#define HYPE_KNS hype  // kernel namespace; the contracted build uses its own
#endif
#include <hip/hip_runtime.h>

namespace HYPE_KNS {

// high word of 2^388: a positive double is below 2^388 if and only if its
// high word is below this one
constexpr unsigned FDIV_TOP_WORD = (1023u + 388u) << 20;
__device__ __forceinline__ unsigned hi_word(double x) { return (unsigned)__double2hiint(x); }

// refined reciprocal of b.  One third-order step, y0 (1 + e + e^2) with
// e = 1 - b y0, in place of the sequence's two Newton steps: three fused
// operations instead of four.  |e| <= 2^-23 (the hardware's bound for
// v_rcp_f64), so the step's own error is below 2^-68 and the result is the
// rounded reciprocal up to 2^-15 of an ulp in the halfway cases.  The sequence's
// is so up to 2^-39: that the quotient and remainder step below round correctly
// from either is an observation.  On the device none of 5.4e8 quotients and as
// many reciprocals differed from the compiler's (a quarter of them at random, the
// others with an operand within 2^-28 of a power of two), nor any of the 2^18
// reciprocals of the numbers below 2, which lie closest to halfway
__device__ __forceinline__ double recip_nr(double b) {
  const double y = __builtin_amdgcn_rcp(b);
  const double e = fma(-b, y, 1.0);
  return fma(y, fma(e, e, e), y);
}

// a / b for b > 0 in range, given y = recip_nr(b); bitwise equal to a / b
__device__ __forceinline__ double div_y(double a, double b, double y) {
  const double q = a * y;
  const double rn = fma(b, q, -a);
  return fma(-rn, y, q);
}

// 1 / b for b > 0 in range, given y = recip_nr(b); bitwise equal to 1.0 / b
__device__ __forceinline__ double inv_y(double b, double y) {
  const double rn = fma(b, y, -1.0);
  return fma(-rn, y, y);
}

// a / b for a b that is the same for every cell, given y = recip_nr(b): the
// quotient step and the sequence's fixup, 4 instructions instead of 11.  The
// fixup handles zeros, infinities and NaN.  b is a product of (gamma - 1)
// factors, so 0 or at least 2^-105 in magnitude; a is a sum of products of
// pressures, zero or far above 2^-960, where the remainder would no longer be
// exact.  Nor does a finite quotient overflow: it is an energy no larger than the
// cells' that the pressure was reconstructed from (Kapila's squared sound speed,
// a product of two pressures, overflows long before).
__device__ __forceinline__ double div_const(double a, double b, double y) {
  return __builtin_amdgcn_div_fixup(div_y(a, b, y), b, a);
}

// sqrt(x) for x >= 2^-767, and for zero, infinity, NaN and negative x: one step of
// Goldschmidt's coupled iteration for the root g and its half reciprocal h (error
// below 2^-44), then two corrections with the exact remainder x - g^2, the second of
// which rounds correctly.  Without the rescaling of tiny arguments it takes 13
// instructions instead of 18.  Arguments are squared sound speeds, at least
// 1e-12 or already reported as inadmissible.
__device__ __forceinline__ double sqrt_adm(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y;
  double h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  double d = fma(-g, g, x);
  g = fma(d, h, g);
  d = fma(-g, g, x);
  g = fma(d, h, g);
  return __builtin_amdgcn_class(x, 0x260) ? x : g;  // +inf, +0 and -0
}

// a / b for any operands: the whole sequence, with recip_nr's step in place of
// its two Newton steps (10 instructions instead of 11).  Written out, the
// compiler also schedules across the divisions' chains, which hides the wait
// after each reciprocal.  With one inlined copy of the row sweep per kernel:
// Kapila 1024x512, 10 steps, 4247 -> 4130 us; Baer-Nunziato 2048x1024, 3 steps,
// 8191 -> 8053 us.
__device__ __forceinline__ double fdiv(double a, double b) {
  bool scaled_b, scaled;
  const double sb = __builtin_amdgcn_div_scale(a, b, false, &scaled_b);
  const double sa = __builtin_amdgcn_div_scale(a, b, true, &scaled);
  const double y = recip_nr(sb);
  const double q = sa * y;
  const double r = fma(-sb, q, sa);
  return __builtin_amdgcn_div_fixup(__builtin_amdgcn_div_fmas(r, y, q, scaled), b, a);
}

}  // namespace HYPE_KNS
