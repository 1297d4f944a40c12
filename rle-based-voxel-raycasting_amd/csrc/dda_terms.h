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
  return ((x ^ y) >> 23) == 0 && y >= x && ((x >> 23) & 0xffu) != 0xffu;
}

struct DdaTerms {
  float s, G;    // term k = s + k*G for k <= K
  float c2, G2;  // term k = c2 + k*G2 for k > K
  float K;
};

// One binade: true when terms 0..n of the sequence from s by g are s + k*G.
RLEVOX_HD inline bool dda_fit_one(float s, float g, float n, DdaTerms& q) {
  const float s1 = s + g, s2 = s1 + g;
  q.s = s;
  q.G = s2 - s1;
  q.c2 = s;
  q.G2 = q.G;
  q.K = n;
  return s1 - s == q.G && dda_same_binade(s, fmaf(n, q.G, s));
}

// At most one crossing into another binade within terms 0..n.  rcp: any
// reciprocal good to a few ulps (the count it gives is checked).
template <class Rcp>
RLEVOX_HD inline bool dda_fit_two(float s, float g, float n, DdaTerms& q, Rcp rcp) {
  const float s1 = s + g, s2 = s1 + g;
  const float G = s1 - s;
  // K: the last term in s's binade, i.e. below the next power of two
  const float lim = dda_float((dda_bits(s) & 0xff800000u) + 0x00800000u);
  float K = floorf((lim - s) * rcp(G));
  K = fminf(fmaxf(K, 0.0f), n);
  if (!dda_same_binade(s, fmaf(K, G, s))) K -= 1.0f;
  if (dda_same_binade(s, fmaf(K + 1.0f, G, s))) K += 1.0f;
  const float sK = fmaf(K, G, s);
  const bool ok1 = K >= 0.0f && dda_same_binade(s, sK) &&
                   !dda_same_binade(s, fmaf(K + 1.0f, G, s)) && (K < 2.0f || s2 - s1 == G);
  // past the crossing: the first term by its own addition, then steps of G2
  const float t0 = sK + g, t1 = t0 + g, t2 = t1 + g;
  const float G2 = t2 - t1, m = K + 1.0f;
  const float c2 = fmaf(-m, G2, t0);
  const bool ok2 = t1 - t0 == G2 && dda_same_binade(t0, fmaf(n - m, G2, t0)) &&
                   fmaf(m, G2, c2) == t0;
  q.s = s;
  q.G = G;
  q.c2 = c2;
  q.G2 = G2;
  q.K = K;
  return ok1 && ok2 && K < n;
}

RLEVOX_HD inline float dda_term(const DdaTerms& q, float k) {
  return k <= q.K ? fmaf(k, q.G, q.s) : fmaf(k, q.G2, q.c2);
}

}  // namespace rlevox
