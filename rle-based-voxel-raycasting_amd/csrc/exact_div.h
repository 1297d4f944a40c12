// Correctly rounded fp32 quotients by a divisor whose reciprocal is shared
// (plain C++ so a host check can run the same code: the includer defines
// RLEVOX_HD as the function qualifiers it needs).
//
// Markstein's theorems (IBM J. Res. Dev. 34, 1990): an estimate of 1/b within
// one ulp, corrected once by its exact residual, is 1/b rounded to nearest
// unless b's significand is all ones; and with that reciprocal a*r, corrected
// once by its residual, is a/b rounded to nearest (one product and two fused
// multiply-adds: Brisebarre, Muller, Raina, IEEE Trans. Comput. 53, 2004, who
// start from this).  That holds while nothing over- or underflows, which the
// ranges of div_safe and div_dividend_safe see to.
#pragma once

#include <math.h>
#include <stdint.h>
#include <string.h>

namespace rlevox {

// 1/b rounded to nearest from an estimate y within one ulp.
RLEVOX_HD inline float recip_exact(float b, float y) { return fmaf(fmaf(-b, y, 1.0f), y, y); }

// a/b rounded to nearest, r = recip_exact of b.
RLEVOX_HD inline float div_exact(float a, float b, float r) {
  const float q = a * r;
  return fmaf(fmaf(-b, q, a), r, q);
}

// A divisor in [2^-30, 2^30) in magnitude, its significand not all ones.
RLEVOX_HD inline bool div_safe(float b) {
  uint32_t u;
  memcpy(&u, &b, 4);
  const float m = fabsf(b);
  return (m >= 9.313225746154785e-10f) & (m < 1073741824.0f) & ((u & 0x7fffffu) != 0x7fffffu);
}

// A dividend for such a divisor: zero, or in [2^-60, 2^60) in magnitude.
// (Below, the quotient may be off in its last place.)
RLEVOX_HD inline bool div_dividend_safe(float a) {
  const float m = fabsf(a);
  return (a == 0.0f) | ((m >= 8.673617379884035e-19f) & (m < 1152921504606846976.0f));
}

}  // namespace rlevox
