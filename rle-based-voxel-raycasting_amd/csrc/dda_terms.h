// Closed form of the DDA's crossing sequences (plain C++ so a host check can
// run the same code: the includer defines RLEVOX_HD as the function
// qualifiers it needs).
//
// A line's walk (Cuda_Render.h:398-414) adds a constant g to a sum s again and
// again in fp32, s_{k+1} = fl(s_k + g), and the kernels need the terms of a
// chunk of steps at once.  While the sum stays in one binade, every term is
// a multiple of the binade's ulp u and each addition rounds s_k + g to that
// grid, so it moves the sum by the same multiple G of u each time.  Only a
// tie (g halfway between two multiples) depends on the sum's parity; the
// first tie leaves an even multiple and from there each tie takes the same
// side again, so two equal steps in a row show that G holds.  Then
// s_k = s + k*G, which is representable, and one fused multiply-add gives it
// exactly.  Where the sum leaves its binade once within the chunk, a second
// pair (c2, G2) covers the terms past the crossing.
#pragma once

#include <math.h>
#include <stdint.h>
#include <string.h>

namespace rlevox {

RLEVOX_HD inline uint32_t dda_bits(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  return u;
}
RLEVOX_HD inline float dda_float(uint32_t u) {
  float f;
  memcpy(&f, &u, 4);
  return f;
}

// True when every value between a and b lies in a's binade, on a's side of
// zero, with |b| >= |a|, and both are finite.
RLEVOX_HD inline bool dda_same_binade(float a, float b) {
  const uint32_t x = dda_bits(a), y = dda_bits(b);
  return (((x ^ y) >> 23) == 0) & (y >= x) & (((x >> 23) & 0xffu) != 0xffu);
}

// A sequence at its next term s: terms 0..rem are s + k*G (rem < 0: none
// known).
struct DdaSeq {
  float s, G, rem;
};

// Fits the sequence from s by g.  rcp: any reciprocal good to a few ulps
// (the count it gives is checked).
template <class Rcp>
RLEVOX_HD inline DdaSeq dda_fit(float s, float g, Rcp rcp) {
  const float s1 = s + g, s2 = s1 + g;
  const float G = s1 - s;
  // the terms below the next power of two
  const float lim = dda_float((dda_bits(s) & 0xff800000u) + 0x00800000u);
  float k = floorf((lim - s) * rcp(G));
  k = fminf(fmaxf(k, 0.0f), 4194304.0f);
  if (!dda_same_binade(s, fmaf(k, G, s))) k = fmaxf(k - 1.0f, 0.0f);
  if (!dda_same_binade(s, fmaf(k, G, s))) k = 0.0f;
  if (s2 - s1 != G) k = fminf(k, 1.0f);
  // not finite, or a negative zero (which a product with k loses)
  if (!dda_same_binade(s, s) | (dda_bits(s) == 0x80000000u)) k = -1.0f;
  return DdaSeq{s, G, k};
}

// The terms of a chunk, over at most two binades.
struct DdaTerms {
  float s, G;    // term k = s + k*G for k <= K
  float c2, G2;  // term k = c2 + k*G2 for k > K
  float K;
  float last;    // up to this term
};

// Terms past q.rem: the first by its own addition, the others from a fit of
// their own.
template <class Rcp>
RLEVOX_HD inline DdaTerms dda_terms(const DdaSeq& q, float g, Rcp rcp) {
  const float m = q.rem + 1.0f;
  const DdaSeq r = dda_fit(fmaf(q.rem, q.G, q.s) + g, g, rcp);
  const float c2 = fmaf(-m, r.G, r.s);
  const bool ok = (q.rem >= 0.0f) & (r.rem >= 0.0f) & (fmaf(m, r.G, c2) == r.s);
  return DdaTerms{q.s, q.G, c2, r.G, q.rem, ok ? m + r.rem : q.rem};
}

RLEVOX_HD inline float dda_term(const DdaTerms& q, float k) {
  return k <= q.K ? fmaf(k, q.G, q.s) : fmaf(k, q.G2, q.c2);
}

// The sequence k terms on (k <= t.last).
RLEVOX_HD inline DdaSeq dda_advance(const DdaTerms& t, float k) {
  const bool hi = k > t.K;
  return DdaSeq{dda_term(t, k), hi ? t.G2 : t.G, (hi ? t.last : t.K) - k};
}

}  // namespace rlevox
