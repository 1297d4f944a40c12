// The quotients from shared reciprocals (csrc/exact_div.h) against fp32
// division: the reciprocal for every significand from estimates at most one
// ulp off, and quotients of random and of hard operands (dividends next to
// multiples of the divisor's halves, so that the quotient lies next to a
// rounding boundary) over the ranges div_safe and div_dividend_safe accept.
// Built and run by tests/test_exact_div.py; EXACT_DIV_PLANT=1 accepts every
// significand, =2 leaves the quotient's correction out, mistakes the check
// must catch.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

#define RLEVOX_HD
#include "../../rle-based-voxel-raycasting_amd/csrc/exact_div.h"

using namespace rlevox;

#ifndef EXACT_DIV_PLANT
#define EXACT_DIV_PLANT 0
#endif

static float bits(uint32_t u) {
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}
static uint32_t word(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  return u;
}

static bool accept(float b) { return div_safe(b) || (EXACT_DIV_PLANT == 1 && div_safe(bits(word(b) & ~1u))); }
static float quotient(float a, float b, float r) { return EXACT_DIV_PLANT == 2 ? a * r : div_exact(a, b, r); }

int main() {
  long recips = 0, quots = 0, bad_r = 0, bad_q = 0;
  for (uint32_t m = 0; m < (1u << 23); m++) {
    for (int e : {127, 100, 150}) {
      const float b = bits((uint32_t)e << 23 | m);
      if (!accept(b)) continue;
      const float want = 1.0f / b;
      const double ulp = std::ldexp(1.0, std::ilogb(want) - 23);
      for (int k = -1; k <= 1; k++) {
        const float y = bits(word(want) + k);
        if (std::fabs((double)y - 1.0 / (double)b) > ulp) continue;
        recips++;
        if (word(recip_exact(b, y)) != word(want)) bad_r++;
      }
    }
  }
  std::mt19937_64 rng(3);
  auto mant = [&] { return (uint32_t)rng() & 0x7fffffu; };
  for (long i = 0; i < 40000000; i++) {
    const uint32_t sb = (uint32_t)(rng() & 1) << 31, sa = (uint32_t)(rng() & 1) << 31;
    float b = bits(sb | (uint32_t)(97 + rng() % 60) << 23 | mant());
    float a = bits(sa | (uint32_t)(67 + rng() % 120) << 23 | mant());
    if (i % 16 == 1) b = bits((word(b) & 0xff800000u) | (0x7fffffu - (uint32_t)(rng() % 4)));
    if (i % 16 == 2) b = bits((word(b) & 0xff800000u) | (uint32_t)(rng() % 4));
    if (i % 16 == 3) a = 0.0f;
    if (i % 4 == 0) {  // a quotient next to a midpoint: a = b * (q + half an ulp), rounded
      const double q = (double)bits(127u << 23 | mant()) + std::ldexp(1.0, -24);
      a = (float)((double)b * q);
      if (rng() & 1) a = std::nextafterf(a, 0.0f);
    }
    if (!accept(b) || !div_dividend_safe(a)) continue;
    const float y = 1.0f / b;
    float est = bits(word(y) + (uint32_t)(rng() % 3) - 1u);
    if (std::fabs((double)est - 1.0 / (double)b) > std::ldexp(1.0, std::ilogb(y) - 23)) est = y;
    quots++;
    if (word(quotient(a, b, recip_exact(b, est))) != word(a / b)) {
      if (bad_q++ < 5) std::printf("%a / %a: %a, division %a\n", a, b, quotient(a, b, recip_exact(b, est)), a / b);
    }
  }
  std::printf("exact_div reciprocals %ld, quotients %ld, mismatches %ld %ld\n", recips, quots, bad_r, bad_q);
  return bad_r || bad_q ? 1 : 0;
}
