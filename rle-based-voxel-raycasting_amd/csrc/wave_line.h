// Wavefront-per-line raycast: the 64 lanes of one wavefront walk one ray
// line together and produce results bit-identical to render_line().
//
//  1. DDA chunk: up to 64 DDA steps per pass, lane k taking step k.  The
//     crossing distances and positions are repeated fp32 additions
//     (Cuda_Render.h:398-414) of six independent sequences, whose terms
//     the lanes take from a closed form (dda_terms.h) that gives the same
//     values; the x/z order is the merge order of the two distance
//     sequences (ties go to x: the walk takes z only when strictly closer).
//  2. Gather: each lane loads its cell's pointer-map entry, one round trip
//     for the whole chunk, issued one chunk ahead (software pipeline).
//  3. Stateless projection per lane: clip-top inputs and F, the projected
//     top of the first drawn element in front of the eye.
//  4. Run cache: each step that may act copies the head of its column
//     (header, runs, colours) into LDS; it then precomputes, in parallel,
//     the span parameters of that first element and F2, the projected top
//     of the next element the loop would test.
//  5. Ordered replay: with the current floating horizon ymin, a step whose
//     clip-top test culls it or whose F <= ymin changes no line state (the
//     element loop breaks first, Cuda_Render.h:467,543).  A ballot finds the
//     next step that acts; only those steps are replayed, in order, using
//     the precomputed values, and the loop over further elements runs only
//     when F2 > ymin.
//     Runs of acting steps of the simple kind (a span drawn from the
//     horizon up, the top clip untouched, the next element not drawn) are
//     applied at once by a horizon sweep: the horizon before each step is
//     a prefix maximum across the lanes (DPP lane moves), and each lane
//     draws one row of the swept rows.
//  6. Spans are drawn 64 pixels per pass: lane k applies the per-pixel
//     increments k times from the span start, exactly as the pixel loop
//     does (Cuda_Render.h:687), and the line's LDS bitmap is updated from a
//     ballot of the drawn pixels.
//  7. The walk ends once no later step can draw (walk_end.h), and steps over
//     stretches that cannot (walk_skip.h), leaving the line as the full walk
//     to the far distance does.
//  8. Two-wavefront form (k_raycast_wave2): one wavefront walks the DDA and
//     gathers (1-2), the other projects, caches and draws (3-7); chunks pass
//     between them through a three-slot LDS ring with one workgroup barrier
//     per chunk.
//  9. Three-wavefront form (k_raycast_wave3): one wavefront walks (1-2), one
//     prepares (3-4), one draws (5-7), each as far ahead of the next as two
//     rings in LDS allow.
#pragma once

#include <type_traits>

#include "device.h"

#include "dda_terms.h"

namespace rlevox {

__device__ inline float readlane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ inline int readlane_i(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

// Marks a value that is the same in every lane as uniform, so the compiler
// keeps it in a scalar register and branches on it with scalar branches
// instead of exec masks (only for values that really are uniform).
__device__ inline int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline float uni_f(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ inline uint64_t uni64(uint64_t v) {
  return ((uint64_t)(uint32_t)uni((int)(v >> 32)) << 32) | (uint32_t)uni((int)(uint32_t)v);
}

__device__ inline bool lds_bit(const uint32_t* bits, int y) { return (bits[y >> 5] >> (y & 31)) & 1u; }

// LDS hand-off between the lanes of one wavefront, on LDS that only this
// wavefront uses.  (Between the two wavefronts of a line ChunkRing and its
// workgroup barrier hand over, between three LineRings and its counters, with
// this point on either side of a counter.)  A wavefront's LDS instructions
// execute in program order, so a write by one lane is seen by a later read
// of another lane once the compiler keeps both on their side of this point.
// Unlike a workgroup barrier, this emits no s_barrier and does not wait for
// the wavefront's outstanding global loads (the prefetches stay in flight).
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Slab words cached per step (from the 16-byte boundary at or below the
// column header): covers header, elements and colours of typical columns.
// The counting walk's depth; the other kernels are built for 24, 40 and 56
// words (a tuning choice).
constexpr int kRunCache = 40;
// The cache holds 16-byte words of 8 slab words, word i of all 64 lanes'
// columns side by side: the layout in which the loads write LDS themselves
// (global_load_lds_dwordx4: lane l's 16 bytes go to the base + 16*l), so no
// register holds them on the way.  20 to 28 registers did, across the next
// chunk's DDA, and the batch kernel spilled.
// Slab word j (from the 16-byte boundary) of a lane's column:
__device__ inline int rc_index(int lane, int j) { return ((j & ~7) << 6) + (lane << 3) + (j & 7); }

// The cache as LDS (the loads into it need the address space).
typedef __attribute__((address_space(3))) uint16_t lds_u16;

// One column of the cache: word i from the column header on.
struct RcColumn {
  const lds_u16* rc;
  int lane, delta;
  __device__ int index(int i) const { return rc_index(lane, delta + i); }
  __device__ uint16_t operator[](int i) const { return rc[index(i)]; }
};

// LDS floats per wavefront used by the DDA chunk.
constexpr int kDdaLds = 6 * 68 + 64;

// First y in [from, to) whose bit is clear, or `to` (from <= to).
__device__ inline int first_clear(const uint32_t* bits, int from, int to, int lane) {
  for (int base = from; base < to; base += 64) {
    const int y = base + lane;
    const uint64_t m = uni64(ballot(y < to && !lds_bit(bits, y)));
    if (m) return uni(base + __builtin_ctzll(m));
  }
  return to;
}

// Number of entries of the increasing 64-array `arr` that precede value v:
// (LE ? arr[l] <= v : arr[l] < v).  `guess` is an estimate of the answer.
template <bool LE>
__device__ inline int rank_in(const float* arr, float v, int guess) {
  int j = min(max(guess, 0), 64);
  auto before = [&](int l) { return LE ? !(v < arr[l]) : (arr[l] < v); };
  while (j > 0 && !before(j - 1)) j--;
  while (j < 64 && before(j)) j++;
  return j;
}

// Wavefront scans with DPP lane moves (register reads across lanes, no LDS
// round trip): row_shr:n (0x110 + n) inside each 16-lane row, then
// row_bcast:15 (0x142, into rows 1 and 3) and row_bcast:31 (0x143, into
// rows 2 and 3) across rows, wave_shr:1 (0x138) for the exclusive form.  A
// lane whose source lies outside keeps `old`, the operation's identity.
// Call with every lane of the wavefront active.
template <int CTRL, int ROW_MASK = 0xf>
__device__ inline int dpp_move(int old, int v) {
  return __builtin_amdgcn_update_dpp(old, v, CTRL, ROW_MASK, 0xf, false);
}

// Exclusive prefix maximum over the lanes of the wavefront (lane 0 gets
// `init`).
__device__ inline int prefix_max_excl(int v, int init, int lane) {
  v = max(v, dpp_move<0x111>(INT32_MIN, v));
  v = max(v, dpp_move<0x112>(INT32_MIN, v));
  v = max(v, dpp_move<0x114>(INT32_MIN, v));
  v = max(v, dpp_move<0x118>(INT32_MIN, v));
  v = max(v, dpp_move<0x142, 0xa>(INT32_MIN, v));
  v = max(v, dpp_move<0x143, 0xc>(INT32_MIN, v));
  const int prev = dpp_move<0x138>(INT32_MIN, v);
  return lane == 0 ? init : max(init, prev);
}

// Inclusive prefix sum of v over lanes 0..lane.
__device__ inline int prefix_sum_incl(int v, int lane) {
  (void)lane;
  v += dpp_move<0x111>(0, v);
  v += dpp_move<0x112>(0, v);
  v += dpp_move<0x114>(0, v);
  v += dpp_move<0x118>(0, v);
  v += dpp_move<0x142, 0xa>(0, v);
  v += dpp_move<0x143, 0xc>(0, v);
  return v;
}

// ------------------------------------------------------------ span pixels

// Sets the bitmap bits of rows base..base+63 given by mask m.  Lane 0 issues
// LDS atomic ORs whose results nobody waits for.  Only rows below the span
// end (< rs) are ever in m, so the words stay inside the bitmap.
__device__ inline void bits_or(uint32_t* bits, int base, uint64_t m, int lane) {
  if (m && lane == 0) {
    const int w0 = base >> 5, off = base & 31;
    const uint32_t lo = (uint32_t)(m << off);
    if (lo) atomicOr(&bits[w0], lo);
    const uint32_t mid = off ? (uint32_t)(m >> (32 - off)) : (uint32_t)(m >> 32);
    if (mid) atomicOr(&bits[w0 + 1], mid);
    const uint32_t hi = off ? (uint32_t)(m >> (64 - off)) : 0u;
    if (hi) atomicOr(&bits[w0 + 2], hi);
  }
}

// Slab word of a column: from the run cache (at rc[index]) where it holds the
// word, else from memory.  Nearly always it holds every lane's, and that way
// is kept apart, uniformly, until the word has arrived (the empty asm reads
// it): joined earlier, it would wait for the memory load's counter, and with
// it for every store the wavefront has in flight (one counter for both).
__device__ inline uint32_t column_word(bool cached, const lds_u16* rc, int index, g_u16* mem) {
  uint32_t w;
  if (ballot(!cached) == 0) {
    w = rc[index];
    asm volatile("" : "+v"(w));
  } else {
    if (cached) w = rc[index];
    else w = *mem;
    asm volatile("" : "+v"(w));
  }
  return w;
}

// Sets the bitmap bits of rows [from, to), to <= from + 64: lane l < 3 ORs
// word l of the range.
__device__ inline void bits_set_range(uint32_t* bits, int from, int to, int lane) {
  const int w = (from >> 5) + lane;
  const int lo = max(from - 32 * w, 0), hi = min(to - 32 * w, 32);
  if (lane < 3 && lo < hi) atomicOr(&bits[w], (~0u << lo) & (~0u >> (32 - hi)));
}

// The n-th of a span's per-pixel increments from (uz, oz) on
// (Cuda_Render.h:687): n additions each, the last ones of a multiple of four
// without a test between them.
__device__ inline void span_steps(float& uz, float& oz, float u2dz, float onedz2, int n) {
  if (n & 1) {
    uz += u2dz;
    oz += onedz2;
  }
  if (n & 2) {
    uz += u2dz;
    oz += onedz2;
    uz += u2dz;
    oz += onedz2;
  }
  for (n >>= 2; n > 0; n--) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      uz += u2dz;
      oz += onedz2;
    }
  }
}

// A pixel's colour index and depth (Cuda_Render.h:690-723) from its u/z and
// 1/z.  tlo and thi are integers below 2^24, so the index needs no clamp.
__device__ inline void span_texel(float uz, float oz, float tlo, float thi, uint32_t& u,
                                  uint32_t& depth) {
  float z, v;
  const bool safe = div_safe(oz) & div_dividend_safe(uz);
  if (ballot(!safe) == 0) {  // both quotients from one reciprocal
    z = recip_exact(oz, __builtin_amdgcn_rcpf(oz));
    v = div_exact(uz, oz, z);
  } else {
    z = 1.0f / oz;
    v = uz / oz;
  }
  u = (uint32_t)d_f2i(fminf(fmaxf(v, tlo), thi));
  depth = (uint32_t)d_f2i(z) & 0xfffeu;
}

// Draws pixels [y0, s2) of one span (uniform arguments; Cuda_Render.h:
// 678-733).  Pixel y0+k has had k per-pixel increments.
__device__ inline int draw_span(int y0, int s2, float uzb, float ozb, float u2dz, float onedz2,
                                float tlo, float thi, RcColumn cached, int ccap,
                                g_u16* colours, int cofs, g_u32_out* row,
                                uint32_t* bits, int lane) {
  int drawn = 0;
  for (int base = y0; base < s2; base += 64) {
    float uz = uzb, oz = ozb;
    span_steps(uz, oz, u2dz, onedz2, max(min(lane, s2 - 1 - base), 0));
    const int y = base + lane;
    const bool draw = y < s2 && !lds_bit(bits, y);
    if (draw) {
      uint32_t u, depth;
      span_texel(uz, oz, tlo, thi, u, depth);
      const int cw = cofs + (int)u;
      row[y] = column_word(cw < ccap, cached.rc, cached.index(cw), colours + u) + (depth << 16);
    }
    const uint64_t dm = ballot(draw);
    drawn += (int)__popcll(dm);
    bits_or(bits, base, dm, lane);  // pixel base+i is bit i of dm
    wave_sync();
    if (base + 64 < s2) {
      uzb = readlane_f(uz, 63) + u2dz;
      ozb = readlane_f(oz, 63) + onedz2;
    }
  }
  return drawn;
}

// The clear rows of a span [s1, e2): for spans of at most 64 rows one LDS
// read and one ballot give both the first clear row y0 (which fixes the
// span's start value, Cuda_Render.h:678-680) and the rows to draw.
struct SpanWindow {
  int y0;      // first clear row, or e2
  uint64_t m;  // fused: clear rows, bit j = row s1 + j
  bool fused;
};

__device__ inline SpanWindow span_window(const uint32_t* bits, int s1, int e2, int lane) {
  SpanWindow w;
  if (e2 - s1 <= 64) {
    const bool clear = lane < e2 - s1 && !lds_bit(bits, s1 + lane);
    w.m = uni64(ballot(clear));
    w.y0 = uni(w.m ? s1 + (int)__builtin_ctzll(w.m) : e2);
    w.fused = true;
  } else {
    w.y0 = first_clear(bits, s1, e2, lane);
    w.m = 0;
    w.fused = false;
  }
  return w;
}

// Draws the clear rows of [w.y0, e2) (Cuda_Render.h:687-733): pixel y0+k has
// had k per-pixel increments.
__device__ inline int span_draw(const SpanWindow& w, int s1, int e2, float uzb, float ozb,
                                float u2dz, float onedz2, float tlo, float thi,
                                RcColumn cached, int ccap, g_u16* colours,
                                int cofs, g_u32_out* row, uint32_t* bits, int lane) {
  if (!w.fused)
    return draw_span(w.y0, e2, uzb, ozb, u2dz, onedz2, tlo, thi, cached, ccap, colours, cofs, row,
                     bits, lane);
  if ((w.m >> lane) & 1) {
    float uz = uzb, oz = ozb;
    span_steps(uz, oz, u2dz, onedz2, lane - (w.y0 - s1));  // row y0 or later
    uint32_t u, depth;
    span_texel(uz, oz, tlo, thi, u, depth);
    const int cw = cofs + (int)u;
    row[s1 + lane] =
        column_word(cw < ccap, cached.rc, cached.index(cw), colours + u) + (depth << 16);
  }
  bits_or(bits, s1, w.m, lane);
  wave_sync();
  return (int)__popcll(w.m);
}

// DDA walk state of one line (Cuda_Render.h:270-367); uniform but for s, g.
struct DdaWalk {
  // Lane j < 6 holds sequence j, its next term and fit q and its increment g:
  // the next crossing distances dd0, dd1 (0, 1) and the positions i0x, i0y,
  // i1x, i1y of the x and z crossings (2-5); 0, 2, 3 belong to the x
  // crossings.
  DdaSeq q;
  float g;
  float px, py, dnow;                  // last step taken
  int idx;
  int mip, gridx, gridz, mapswitch, shift;
  int dzlog;  // dz = 2^dzlog
  // The window of steps the walk has looked ahead over: lane g holds the
  // bound of its steps 8g..8g+7 (walk_skip.h); the walk's next step in it
  // (negative: still before it), its length.
  float bound;
  int ofs, end;
  float dz, z, yswitch;
  g_entry* map;
  g_u16* slab;
};

// One chunk of up to 64 DDA steps: lane k holds step k and its gathered
// pointer-map entry.  The mip level is constant within a chunk.
struct DdaChunk {
  int L, mip, shift;
  int first;  // lanes below hold no step of the line's own
  g_u16* slab;
  float db, dn, pbx, pby;  // per lane: distances and position before the step
  int ib;
  uint2 ent;
};

// One chunk of the walk from the closed form of its six sequences (lane j < 6
// passes sequence j's in q).  The walk's order of x and z steps is the merge
// of the two distance sequences (ties go to x: the walk takes z only when
// strictly closer).  Lane t guesses i, the x crossings among its t earlier
// steps, as floor(e0 + e1*t); its own step then says what lane t+1 must hold.
// While some lane disagrees with its predecessor all take the predecessor's
// word: the lanes that agree from lane 0 on are the sequential walk's, and
// each pass adds at least one, so the loop ends with the walk's order.
// The chunk may begin T steps on: lane 0 then settles i against the terms
// before it.  What came before lane 0's step is not made out (c.first = 1):
// the caller lets the chunk begin one step early, on one that cannot draw.
// False (the walk unchanged) when the chunk needs terms beyond those fitted.
//
// Bound by its own dependent instructions (about 100 in place of the 64
// chained additions and LDS stores of dda_chain, which took 3.1 K cycles of
// a walking wavefront's chunk).  The sequences' constants go through LDS and
// come back as broadcasts: scalar registers for all 30 of them spilled.
__device__ inline bool dda_merge(DdaWalk& w, DdaChunk& c, const DdaTerms& q, int T, int L, float e0,
                                 float e1, bool xseq, float* dl, int lane) {
  float4* row = reinterpret_cast<float4*>(dl);  // {s, G, c2, G2} of each sequence
  float* rowK = dl + 24;
  if (lane < 6) {
    row[lane] = make_float4(q.s, q.G, q.c2, q.G2);
    rowK[lane] = q.K;
  }
  wave_sync();
  auto term = [](float4 v, float K, float k) {
    const bool hi = k > K;
    return __builtin_fmaf(k, hi ? v.w : v.y, hi ? v.z : v.x);
  };
  const float tf = (float)(T + lane);
  float fi = fminf(fmaxf(floorf(e0 + e1 * tf), 0.0f), tf);
  float dn, next;
  bool z;
  {
    const float4 A = row[0], B = row[1];
    const float KA = rowK[0], KB = rowK[1];
    for (;;) {
      const float a = term(A, KA, fi), b = term(B, KB, tf - fi);
      z = b < a;
      dn = z ? b : a;
      next = z ? fi : fi + 1.0f;
      float own = fi;  // lane 0's: 0 at T = 0
      if (T > 0) {
        const bool few = tf > fi && !(term(B, KB, tf - fi - 1.0f) < a);
        const bool many = fi > 0.0f && b < term(A, KA, fi - 1.0f);
        own += few ? 1.0f : (many ? -1.0f : 0.0f);
      }
      const float told = __int_as_float(dpp_move<0x138>(__float_as_int(own), __float_as_int(next)));
      if (!(ballot(told != fi) & (~0ull >> (64 - L)))) break;
      fi = told;
    }
  }
  // the terms after the chunk's last step must still be within the fits
  const float nx = readlane_f(next, L - 1);
  const float n = xseq ? nx : (float)(T + L) - nx;
  if (ballot(n > q.last) & 0x3f) return false;
  const float k = z ? tf - fi : fi;
  const int sx = z ? 4 : 2;
  const float x = term(row[sx], rowK[sx], k);
  const float y = term(row[sx + 1], rowK[sx + 1], k);
  // a step's cell follows from the position before it: the previous lane's
  c.dn = dn;
  c.db = __int_as_float(dpp_move<0x138>(__float_as_int(w.dnow), __float_as_int(dn)));
  c.pbx = __int_as_float(dpp_move<0x138>(__float_as_int(w.px), __float_as_int(x)));
  c.pby = __int_as_float(dpp_move<0x138>(__float_as_int(w.py), __float_as_int(y)));
  c.ib = dpp_move<0x138>(w.idx, z ? 1 : 0);
  c.first = T > 0 ? 1 : 0;
  w.dnow = readlane_f(dn, L - 1);
  w.px = readlane_f(x, L - 1);
  w.py = readlane_f(y, L - 1);
  w.idx = readlane_i(z ? 1 : 0, L - 1);
  w.q = dda_advance(q, n);
  wave_sync();
  return true;
}

// One chunk of the walk by its own additions, for chunks whose sequences
// cross more than one binade (a line's first chunk, mostly) or are not
// finite (rays along an axis).  Lane j < 6 walks sequence j, storing every
// term to LDS (one add and one store per term for all six sequences at
// once); each term is made by the same additions the sequential walk makes
// (the k-th x-crossing term has seen k additions whatever the
// interleaving).  Lane k then reads term k and finds its merge rank.
// Layout: six sequences of 65 terms at a stride of 68 floats (the writers,
// lanes 0..5, hit different LDS banks), then 64 merge slots.
__device__ inline void dda_chain(DdaWalk& w, DdaChunk& c, int L, float* dl, int lane) {
  c.db = c.dn = c.pbx = c.pby = 0;
  c.ib = 0;
  c.first = 0;
  constexpr int kSeq = 68;
  float* sA = dl;
  float* sB = dl + kSeq;
  float* sX0 = dl + 2 * kSeq;
  float* sY0 = dl + 3 * kSeq;
  float* sX1 = dl + 4 * kSeq;
  float* sY1 = dl + 5 * kSeq;
  int* slot = reinterpret_cast<int*>(dl + 6 * kSeq);
  const float dd0 = readlane_f(w.q.s, 0), dd1 = readlane_f(w.q.s, 1);
  const float gd0 = readlane_f(w.g, 0), gd1 = readlane_f(w.g, 1);
  if (lane < 6) {
    float t = w.q.s;
    float* dst = dl + lane * kSeq;
    dst[0] = t;
#pragma unroll
    for (int k = 1; k <= 64; k++) {  // term 64 is the state after a full chunk
      t = t + w.g;
      dst[k] = t;
    }
  }
  wave_sync();
  const float ak = sA[lane], bk = sB[lane];
  // Merge ranks: rx = lane + #{j : sB[j] < ak}, rz = lane + #{j : sA[j] <= bk}.
  // The sequences grow by about gd per term, so a guess g is off by at most
  // one in practice; three probes around it settle the rank exactly
  // (the sequences are sorted), else the lane searches.
  const float qx = (ak - dd1) * __builtin_amdgcn_rcpf(gd1);
  const float qz = (bk - dd0) * __builtin_amdgcn_rcpf(gd0);
  const int gx = (int)fminf(fmaxf(ceilf(qx), 0.0f), 64.0f);
  const int gz = (int)fminf(fmaxf(ceilf(qz), 0.0f), 64.0f);
  const float bm = sB[max(gx - 1, 0)], b0 = sB[gx], bp = sB[min(gx + 1, 64)];
  const float am = sA[max(gz - 1, 0)], a0 = sA[gz], ap = sA[min(gz + 1, 64)];
  const bool okx = (gx == 0 || bm < ak) && (gx >= 63 || !(bp < ak));
  const bool okz = (gz == 0 || !(bk < am)) && (gz >= 63 || bk < ap);
  int cx = gx + ((gx < 64 && b0 < ak) ? 1 : 0);
  int cz = gz + ((gz < 64 && !(bk < a0)) ? 1 : 0);
  if (!okx) cx = rank_in<false>(sB, ak, gx);
  if (!okz) cz = rank_in<true>(sA, bk, gz);
  const int rx = lane + cx;
  const int rz = lane + cz;
  if (rx < L) slot[rx] = lane;
  if (rz < L) slot[rz] = 64 + lane;
  const int nx = uni((int)__popcll(ballot(rx < L)));
  const int nz = L - nx;
  // The walk's state after the chunk, read in one round trip: the next
  // terms (index nx of the x sequences, nz of the z sequences) and the last
  // step, which is the later of x-term nx-1 and z-term nz-1 (a z-term
  // follows an equal x-term).
  const float ns = lane < 6 ? dl[lane * kSeq + (((0x0d >> lane) & 1) ? nx : nz)] : 0.0f;
  const float lA = sA[max(nx - 1, 0)], lX0 = sX0[max(nx - 1, 0)], lY0 = sY0[max(nx - 1, 0)];
  const float lB = sB[max(nz - 1, 0)], lX1 = sX1[max(nz - 1, 0)], lY1 = sY1[max(nz - 1, 0)];
  wave_sync();
  const int cc = lane < L ? slot[lane] : 0;
  const int p = (lane < L && lane > 0) ? slot[lane - 1] : 0;
  if (lane < L) {
    c.dn = cc < 64 ? sA[cc] : sB[cc - 64];
    if (lane == 0) {
      c.db = w.dnow;
      c.pbx = w.px;
      c.pby = w.py;
      c.ib = w.idx;
    } else {
      c.db = p < 64 ? sA[p] : sB[p - 64];
      c.pbx = p < 64 ? sX0[p] : sX1[p - 64];
      c.pby = p < 64 ? sY0[p] : sY1[p - 64];
      c.ib = p < 64 ? 0 : 1;
    }
  }
  const bool last_z = nz > 0 && (nx == 0 || !(lB < lA));
  w.dnow = uni_f(last_z ? lB : lA);
  w.px = uni_f(last_z ? lX1 : lX0);
  w.py = uni_f(last_z ? lY1 : lY0);
  w.idx = last_z ? 1 : 0;
  w.q.s = ns;
  w.q.rem = -1.0f;
  wave_sync();
}

// The line's constants, held in LDS: in registers across the walk they cost
// wavefronts.
struct LineConsts {
  WalkEnd end;
  SkipLine line;
};
constexpr int kLineConstWords = (int)(sizeof(LineConsts) / 4);

// The bounds of the window that begins `ahead` steps on, n steps before the
// next mip switch or the far distance.  HOLD: the line's constants may stay in
// registers around the calls; else each call reads them again (held, the batch
// kernel spills 16 bytes: 64 views 5.07 against 4.97 ms).
template <bool HOLD, class Scene>
__device__ inline void dda_look_ahead(DdaWalk& w, const Scene& sc, const LineConsts& lc,
                                      int ahead, int n, int lane) {
  if (!HOLD) asm volatile("" ::: "memory");
  const float sA = readlane_f(w.q.s, 0), sB = readlane_f(w.q.s, 1);
  const float gA = readlane_f(w.g, 0), gB = readlane_f(w.g, 1);
  const int other = w.idx ? 2 : 4;  // the sequences of the other kind's positions
  const SkipBase b = SkipBase::of(lc.line, w.px, w.py, w.dnow, sA, sB, gA, gB, w.idx ? sA : sB,
                                  readlane_f(w.q.s, other), readlane_f(w.q.s, other + 1),
                                  __builtin_amdgcn_rcpf(gA + gB));
  const SkipLevel v{w.mip, w.gridx, w.gridz, (skip_tops*)sc.mip[uni(w.mip)].tops, sc.mip[uni(w.mip)].top};
  const int t0 = ahead + lane * kSkipSteps;
  const float bound = skip_bound(lc.end, lc.line, b, v, sc.sy, t0, t0 + kSkipSteps);
  w.bound = t0 < n ? bound : -__builtin_inff();
  w.ofs = -ahead;
  w.end = min(kSkipWindow, n - ahead);
}

// Steps that cannot draw are looked for up to this far ahead (the chunk's
// steps are counted in floats, and its terms come from two binades).
constexpr int kSkipReach = 2048;

// Advances the walk by one chunk of up to 64 steps.  SKIP: steps that cannot
// draw above the horizon row ymin (a row the line has reached or passed) are
// stepped over on the way.  HOLD: see dda_look_ahead.  Returns false when the
// line has reached the far distance.
template <bool SKIP, bool HOLD, class Scene>
__device__ inline bool dda_next_chunk(DdaWalk& w, DdaChunk& c, const Scene& sc,
                                      const LineConsts& lc, int zfar, int ymin, float* dl,
                                      int lane) {
  for (;;) {
    // distance mip switch (Cuda_Render.h:343-365), uniform
    while (w.z > (float)w.mapswitch || w.yswitch > 512.0f) {
      w.yswitch = w.yswitch * 0.5f;
      if (w.mip < sc.nmips - 1) {
        w.mip = uni(w.mip + 1);
        w.gridx >>= 1;
        w.gridz >>= 1;
        w.map = (g_entry*)sc.mip[w.mip].map;
        w.slab = (g_u16*)sc.mip[w.mip].slabs;
        w.shift = sc.mip[w.mip].shift;
      }
      w.g *= 2;
      w.mapswitch *= 2;
      w.dz *= 2;
      w.dzlog++;
      w.ofs = w.end = 0;
      w.q.rem = -1.0f;
    }
    // Iterations left before the next mip switch and before z passes z_far.
    // z, dz = 2^dzlog and mapswitch are exact integers below 2^31, and
    // z <= mapswitch here; a negative distance to z_far ends the line either
    // way, so the shifts decide exactly as the divisions would.
    const int zi = (int)w.z;
    const int n_mip = ((w.mapswitch - zi) >> w.dzlog) + 1;
    const int n_far = (zfar - zi) >> w.dzlog;
    if (n_far <= 0) return false;
    const int n = min(n_mip, n_far);
    // steps ahead that cannot draw (at least; n when none of the level's can)
    int hidden = 0;
    if (SKIP) {
      bool look = w.ofs >= w.end;
      for (;;) {
        if (look) dda_look_ahead<HOLD>(w, sc, lc, hidden, n, lane);
        const int at = max(w.ofs, 0) / kSkipSteps;  // the group of the next step
        const uint64_t vis = uni64(ballot(!skip_hidden(w.bound, ymin))) >> at;
        if (vis) {
          hidden = max((at + (int)__builtin_ctzll(vis)) * kSkipSteps - w.ofs, 0);
          break;
        }
        hidden = w.end - w.ofs;  // to the window's end: look on from there
        if (hidden >= n || hidden > kSkipReach) break;
        look = true;
      }
    }
    // The chunk: L steps from T steps on, which begin one step before the
    // first that may draw.  emit = false: none of them may.
    int T = max(hidden - 1, 0), L = min(64, n - T);
    bool emit = true;
    if (hidden >= n || hidden > kSkipReach) {
      T = max(min(hidden, n) - 64, 0);
      L = min(64, min(hidden, n) - T);
      emit = false;
    }
    // Closed form (dda_terms.h): past a line's first chunk, where every
    // sequence crosses many binades, nearly every chunk's sequences stay in
    // one or cross into the next one once.
    const bool xseq = (0x0d >> lane) & 1;  // lanes 0, 2, 3
    bool ok = false;
    if (w.dnow > 0.0f) {
      const float sA = readlane_f(w.q.s, 0), sB = readlane_f(w.q.s, 1);
      const float gA = readlane_f(w.g, 0), gB = readlane_f(w.g, 1);
      // x crossings among the first t steps: the merge of sA + i*gA and
      // sB + j*gB, i + j = t, wants A's term i-1 <= B's term j and B's
      // term j-1 < A's term i, so i = floor((sB - sA + gA + t*gB) / (gA + gB))
      const float gr = __builtin_amdgcn_rcpf(gA + gB);
      const float e0 = (sB - sA + gA) * gr, e1 = gB * gr;
      if (ballot(w.q.rem < 0.0f) & 0x3f) w.q = dda_fit(w.q.s, w.g, HwRcp());
      for (;;) {
        // terms the chunk may need of either kind (checked afterwards)
        const float n_steps = (float)(T + L);
        const float ex = floorf(fminf(fmaxf(e0 + e1 * n_steps, 0.0f), n_steps));
        const float nv = (xseq ? ex : n_steps - ex) + 1.0f;
        DdaTerms q{w.q.s, w.q.G, w.q.s, w.q.G, w.q.rem, w.q.rem};
        if (ballot(nv > w.q.rem) & 0x3f) q = dda_terms(w.q, w.g, HwRcp());
        ok = !(ballot(nv > q.last) & 0x3f) && dda_merge(w, c, q, T, L, e0, e1, xseq, dl, lane);
        if (!SKIP || ok || T == 0) break;
        // too many binades on the way: half of it, or one chunk from here
        if (T >= 128) {
          T >>= 1;
          L = 64;
          emit = false;
        } else {
          T = 0;
          L = min(64, n);
          emit = hidden < L;
        }
      }
    } else {
      T = 0;
      L = min(64, n);
      emit = hidden < L;
    }
    if (!ok) dda_chain(w, c, L, dl, lane);
    w.z += (float)(T + L) * w.dz;
    if (SKIP) w.ofs += T + L;
    if (emit) {
      c.L = L;
      c.mip = w.mip;
      c.shift = w.shift;
      c.slab = w.slab;
      return true;
    }
  }
}

// Cell of each step of the chunk just walked (Cuda_Render.h:416-442) and the
// load of its pointer-map entry (left in flight).  fix_x, fix_z: what the fix-up
// adds to the cell of an x, a z crossing (0 or -1; as floats: integer selects
// made 320x240 2%, 1280x720 1% slower).
__device__ inline void dda_gather(const DdaWalk& w, DdaChunk& c, float vpx, float vpz,
                                  float fix_x, float fix_z, int lane) {
  const int voxel_x = d_f2i(vpx + c.pbx) + (int)((float)(1 - c.ib) * fix_x);
  const int voxel_z = d_f2i(vpz + c.pby) + (int)((float)c.ib * fix_z);
  const int vx = (voxel_x >> w.mip) & (w.gridx - 1);
  const int vz = (voxel_z >> w.mip) & (w.gridz - 1);
  c.ent = make_uint2(0u, 0u);
  if (lane < c.L && lane >= c.first) {
    const v2u32 e = w.map[vx + vz * w.gridx];
    c.ent = make_uint2(e.x, e.y);
  }
}

// Chunks handed from the producer wavefront (DDA + pointer gather) to the
// consumer wavefront (projection, run cache, replay) of a two-wavefront
// line: three slots used round robin.
struct ChunkRing {
  float db[3][64], dn[3][64];
  uint2 ent[3][64];
  g_u16* slab[3];
  int L[3], mip[3], shift[3], have[3];
  // written by the consumer in the round that uses the slot
  int stop[3], horizon[3];
  LineConsts lc;  // the producer's
};

// The fields the consumer reads: distances, level and the gathered entry.
__device__ inline void ring_put_dda(ChunkRing& r, int s, const DdaChunk& c, bool have, int lane) {
  if (have) {
    r.db[s][lane] = c.db;
    r.dn[s][lane] = c.dn;
  }
  if (lane == 0) {
    r.slab[s] = c.slab;
    r.L[s] = have ? c.L : 0;
    r.mip[s] = c.mip;
    r.shift[s] = c.shift;
    r.have[s] = have ? 1 : 0;
  }
}

__device__ inline void ring_get(const ChunkRing& r, int s, DdaChunk& c, int lane) {
  c.L = uni(r.L[s]);
  c.mip = uni(r.mip[s]);
  c.shift = uni(r.shift[s]);
  c.slab = (g_u16*)uni64((uint64_t)r.slab[s]);
  c.db = r.db[s][lane];
  c.dn = r.dn[s][lane];
  c.ent = r.ent[s][lane];
}

// A step's stateless projection (Cuda_Render.h:444-466).
struct StepProj {
  float pz, py3, czz, cyy, top;
};

// A chunk as the replay needs it: per lane the step's distances and column,
// its first drawn element in front of the eye (F: projected top) and the top
// F2 of the next element the loop tests.
struct DdaPrepared {
  int L, mip, shift;
  g_u16* slab;
  float db, dn;
  uint2 ent;
  int F, F2, kF, ygF, textureF, s1F;
  bool cand, drawF;
  float texF, s1rF, u1zF, u2dzF, onez1F, onedz2F;
  uint32_t nel;  // elements looked at (counted by the counting walk only)
};
constexpr int kPreparedWords = 16;  // per lane: all but L, mip, shift, slab, nel

// A three-wavefront line's hand-offs: walked chunks through one ring,
// prepared ones (and their run caches) through another.  A wavefront waits
// only where a slot is missing, on a counter in LDS: a chunk without
// candidates is prepared in a third of the time of one with, a walk over a
// hidden stretch takes twice a plain one, and a barrier per chunk would
// charge every round the longest of the three.  The waits sleep 256 or 512
// cycles a turn: polling every 64 cost the other lines' wavefronts issue slots
// (1366x768 400 us against 394).  More walked chunks ahead are walked with an
// older horizon and hold LDS (3 / 4 / 6 slots: 1280x720 727 / 715 / 718 us).
constexpr int kWalkSlots = 4, kPrepSlots = 2;
struct LineRings {
  float db[kWalkSlots][64], dn[kWalkSlots][64];
  uint2 ent[kWalkSlots][64];
  uint32_t prep[kPrepSlots][kPreparedWords][64];
  g_u16 *slab[kWalkSlots], *pslab[kPrepSlots];
  int L[kWalkSlots], mip[kWalkSlots], shift[kWalkSlots];
  int pL[kPrepSlots], pmip[kPrepSlots], pshift[kPrepSlots];
  // chunks complete in either ring so far, and the line's chunks (INT32_MAX
  // until the walk, the preparation has ended)
  int walked, walk_total, prepared, prep_total;
  int taken;  // walked chunks read from their slots
  // prepared chunks replayed, whether the line has ended, its horizon
  int replayed, stop, horizon;
  LineConsts lc;  // the walker's
};

// The counters above, each written by one wavefront and read by others.  A
// wavefront's LDS instructions execute in program order, so one that reads a
// counter finds what its writer had written or read in the rings before it;
// wave_sync keeps the compiler to that order.  All wavefronts of a block are
// resident, and each wait ends with another's next chunk or its end.
__device__ inline int ring_read(const int& v) {
  return uni(__hip_atomic_load(&v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
}
__device__ inline void ring_write(int& at, int v, int lane) {
  wave_sync();
  if (lane == 0) __hip_atomic_store(&at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ inline void prep_put(LineRings& r, int s, const DdaPrepared& p, int lane) {
  auto put = [&](int i, uint32_t v) { r.prep[s][i][lane] = v; };
  auto putf = [&](int i, float v) { put(i, __float_as_uint(v)); };
  put(0, p.ent.x);
  put(1, p.ent.y);
  putf(2, p.db);
  putf(3, p.dn);
  put(4, (uint32_t)p.F);
  put(5, (uint32_t)p.F2);
  put(6, (uint32_t)p.kF);
  put(7, (uint32_t)p.ygF);
  put(8, (uint32_t)p.textureF | (p.cand ? 1u << 30 : 0u) | (p.drawF ? 1u << 31 : 0u));
  put(9, (uint32_t)p.s1F);
  putf(10, p.texF);
  putf(11, p.s1rF);
  putf(12, p.u1zF);
  putf(13, p.u2dzF);
  putf(14, p.onez1F);
  putf(15, p.onedz2F);
  if (lane == 0) {
    r.pslab[s] = p.slab;
    r.pL[s] = p.L;
    r.pmip[s] = p.mip;
    r.pshift[s] = p.shift;
  }
}

__device__ inline void prep_get(const LineRings& r, int s, DdaPrepared& p, int lane) {
  auto get = [&](int i) { return r.prep[s][i][lane]; };
  auto getf = [&](int i) { return __uint_as_float(get(i)); };
  p.L = uni(r.pL[s]);
  p.mip = uni(r.pmip[s]);
  p.shift = uni(r.pshift[s]);
  p.slab = (g_u16*)uni64((uint64_t)r.pslab[s]);
  p.ent = make_uint2(get(0), get(1));
  p.db = getf(2);
  p.dn = getf(3);
  p.F = (int)get(4);
  p.F2 = (int)get(5);
  p.kF = (int)get(6);
  p.ygF = (int)get(7);
  p.cand = (get(8) >> 30) & 1u;  // textureF: 0 to 2^24
  p.drawF = get(8) >> 31;
  p.textureF = (int)(get(8) & 0x3fffffffu);
  p.s1F = (int)get(9);
  p.texF = getf(10);
  p.s1rF = getf(11);
  p.u1zF = getf(12);
  p.u2dzF = getf(13);
  p.onez1F = getf(14);
  p.onedz2F = getf(15);
}

// WAVES: wavefronts of the line's block.  Of two, wavefront 0 produces the
// DDA chunks (and their pointer gathers) two chunks ahead of wavefront 1,
// which consumes them; the two halves of the work overlap.  Of three, the
// second prepares chunks for the third (LineRings).  One wavefront does both,
// software-pipelined.  PAR_ELEMS: the ordered replay
// precomputes a column's remaining elements across the lanes (pays where
// steps often show several elements, as in grazing views of caved terrain;
// the persistent batch kernel leaves it off, where its registers spill).
// HOLD: see dda_look_ahead.
// LDS arguments: bits = the line's bitmap, dl = DDA scratch, rc = run cache
// (kPrepSlots of them for three wavefronts), sweep_lds = 64 ints for the
// horizon sweep followed by kLineConstWords words for the line's constants.
// Scene, Map: SceneDev and rlevox_raymap as kernel arguments or in constant
// memory.
template <bool COUNT, int WAVES = 1, bool PAR_ELEMS = true, int RC = kRunCache, bool HOLD = false,
          class Scene, class Map>
__device__ inline void render_line_wave(int x, const Scene& sc, const Map& rm,
                                        uint32_t* __restrict__ row_, int32_t* __restrict__ clip_,
                                        uint32_t* bits, float* dl, lds_u16* rc, int* sweep_lds,
                                        unsigned long long* counts, ChunkRing* ring = nullptr,
                                        LineRings* rings = nullptr) {
  static_assert(!(COUNT && WAVES > 1), "the counting variant walks with one wavefront");
  constexpr bool TWO = WAVES == 2;
  const int lane = threadIdx.x & 63;
  // wavefront 0 of several walks; the last one draws
  const bool producer = WAVES > 1 && threadIdx.x < 64;
  const bool drawer = WAVES == 1 || (int)threadIdx.x >= 64 * (WAVES - 1);
  g_u32_out* row = (g_u32_out*)row_;
  typedef __attribute__((address_space(1))) int32_t g_i32_out;
  g_i32_out* clip = (g_i32_out*)clip_;
  const int rs = uni(rm.rs);
  const float half = uni_f((float)(rs / 2));
  if (lane == 0 && drawer) {
    clip[0] = 0;
    clip[1] = -1;
  }

  // ---- line plane (Cuda_Render.h:128-172), uniform
  const int r0 = rm.res[0], r1 = r0 + rm.res[1], r2 = r1 + rm.res[2];
  int q = 0;
  if (x >= r2) q = 3;
  else if (x >= r1) q = 2;
  else if (x >= r0) q = 1;
  float qofs = (float)x;
  if (q == 1) qofs -= (float)r0;
  if (q == 2) qofs -= (float)r1;
  if (q == 3) qofs -= (float)r2;
  const float a = qofs / (float)rm.res[q];
  F3 p1 = f3ld(rm.p_2d[5]);
  const F3 e0 = f3ld(rm.p_no[2 * q]);
  F3 p2 = e0 + (f3ld(rm.p_no[2 * q + 1]) - e0) * a;
  {
    const float s2 = line_scale(p1, p2, rm.clip_max, rm.clip_min);
    const F3 c2 = p1 + (p2 - p1) * s2;
    const float s1 = line_scale(p2, p1, rm.clip_max, rm.clip_min);
    const F3 c1 = p2 + (p1 - p2) * s1;
    p1 = c1;
    p2 = c2;
  }
  const F3 p1_3d = mat_apply(rm.to3d, p1 * 4.0f);
  const F3 p2_3d = mat_apply(rm.to3d, p2 * 4.0f);
  F3 dir = (p1_3d + p2_3d) * 0.5f - f3ld(rm.p4);
  dir.y = 0;
  {
    const float d = dir.x * dir.x + dir.y * dir.y + dir.z * dir.z;
    const float inv = 1.0f / sqrtf(d);
    dir = dir * inv;
  }
  const float ray_x = uni_f(rm.cos_myaw * dir.x + rm.sin_myaw * dir.z);
  const float ray_z = uni_f(rm.cos_myaw * dir.z - rm.sin_myaw * dir.x);
  const bool vertical = q < 2;
  const float sin_x = uni_f(rm.sin_x), cos_x = uni_f(rm.cos_x);
  bool reverse = false;
  if (vertical && ray_z <= 0) reverse = true;
  if (!vertical && ray_x <= 0 && sin_x > 0) reverse = true;
  if (!vertical && ray_x > 0 && sin_x < 0) reverse = true;
  float hmul = reverse ? -half : half;
  if (vertical) hmul = -hmul;
  hmul = uni_f(hmul);
  const int p_add = reverse ? 1 : -2;
  int p1x = uni(d_f2i((float)rs * p1.x)) + p_add;
  int p1y = uni(d_f2i((float)rs * p1.y)) + p_add;
  int p2x = uni(d_f2i((float)rs * p2.x)) - p_add;
  int p2y = uni(d_f2i((float)rs * p2.y)) - p_add;
  p1x = min(max(p1x, 0), rs - 1);
  p1y = min(max(p1y, 0), rs - 1);
  p2x = min(max(p2x, 0), rs - 1);
  p2y = min(max(p2y, 0), rs - 1);
  if (p1y == p2y) return;
  int ymin, ymax;
  if (vertical) {
    ymin = rs - 1 - p1y;
    ymax = rs - 1 - p2y;
  } else {
    ymin = rs - 1 - p1x;
    ymax = rs - 1 - p2x;
  }
  if (reverse) {
    ymin = rs - 1 - ymin;
    ymax = rs - 1 - ymax;
  }
  if (ymin > ymax) {
    const int t = ymin;
    ymin = ymax;
    ymax = t;
  }
  if (ymin >= ymax) return;

  // ---- clear the range and the bitmap (Cuda_Render.h:255-264), coalesced
  if (drawer) {
    for (int n = ymin + lane; n <= ymax; n += 64) row[n] = RLEVOX_CLEAR_TEXEL;
    const int words = bitmap_words(rs);
    for (int w = lane; w < words; w += 64) bits[w] = 0;
    if (lane == 0) {
      clip[0] = ymin;
      clip[1] = ymax;
    }
    wave_sync();
  }
  LineCounts cnt;
  if (COUNT) cnt.cleared = (uint64_t)(ymax - ymin + 1);

  // ---- DDA setup (Cuda_Render.h:270-304), uniform
  const float vpx = uni_f(rm.position[0]), vpy = uni_f(rm.position[1]), vpz = uni_f(rm.position[2]);
  const float ddx = ray_x * rm.cos_y + ray_z * rm.sin_y;
  const float ddy = ray_x * rm.sin_y - ray_z * rm.cos_y;
  float sign_x = -1, sign_y = -1;
  float frac_x = vpx - (float)uni(d_f2i(vpx));
  float frac_y = vpz - (float)uni(d_f2i(vpz));
  if (ddx >= 0) {
    sign_x = 1;
    frac_x = 1 - frac_x;
  }
  if (ddy >= 0) {
    sign_y = 1;
    frac_y = 1 - frac_y;
  }
  const float fix_x = uni_f(ddx >= 0 ? 0.0f : -1.0f), fix_z = uni_f(ddy >= 0 ? 0.0f : -1.0f);
  DdaWalk wk;
  {
    const float g0y = ddy / fabsf(ddx), g1x = ddx / fabsf(ddy);
    const float g0x = sign_x, g1y = sign_y;
    const float i0x = g0x * frac_x, i0y = g0y * frac_x, i1x = g1x * frac_y, i1y = g1y * frac_y;
    const float gv[6] = {sqrtf(g0x * g0x + g0y * g0y), sqrtf(g1x * g1x + g1y * g1y), g0x, g0y, g1x, g1y};
    const float sv[6] = {sqrtf(i0x * i0x + i0y * i0y), sqrtf(i1x * i1x + i1y * i1y), i0x, i0y, i1x, i1y};
    wk.q = DdaSeq{0.0f, 0.0f, -1.0f};
    wk.g = 0;
#pragma unroll
    for (int j = 0; j < 6; j++) {
      wk.q.s = lane == j ? sv[j] : wk.q.s;
      wk.g = lane == j ? gv[j] : wk.g;
    }
  }
  wk.px = wk.py = wk.dnow = 0;
  wk.idx = 0;
  wk.mip = 0;
  wk.gridx = sc.mip[0].sx;
  wk.gridz = sc.mip[0].sz;
  wk.map = (g_entry*)sc.mip[0].map;
  wk.slab = (g_u16*)sc.mip[0].slabs;
  wk.shift = sc.mip[0].shift;
  wk.mapswitch = rm.mapswitch;
  wk.dz = 1;
  wk.dzlog = 0;
  wk.z = 0;
  wk.yswitch = vpy;
  const float z_add = sin_x;
  const float y_add = uni_f((vertical ? cos_x : 0.0f) * hmul);
  const int zfar = uni(rm.far_distance);
  const float mountain = vpy;
  wk.bound = 0;
  wk.ofs = wk.end = 0;
  // the line's constants, in LDS behind the sweep marks (the producer of a
  // two-wavefront line has its own)
  LineConsts* lc = reinterpret_cast<LineConsts*>(sweep_lds + 64);
  if (TWO && producer) lc = &ring->lc;
  if (WAVES == 3 && producer) lc = &rings->lc;
  const WalkEnd* wend = &lc->end;
  if (lane == 0 && (producer || drawer)) {
    lc->end.init(cos_x, sin_x, hmul, ray_x, ray_z, vertical, mountain, half);
    lc->line.init(ddx, ddy, vpx, vpz);
  }
  wave_sync();
  const float wfloor = uni_f(wend->floor_());  // held in a scalar register across the walk

  // Software pipeline: while chunk c's run-cache loads are in flight the DDA
  // of chunk c+1 runs, and while chunk c is replayed the pointer-map gather
  // of chunk c+1 is in flight.  The walk does
  // not depend on the replay (only the line's end does), so a chunk
  // computed past the end of the line is simply dropped.  The step's code
  // appears once (unrolled over two register sets it took 40 KB of the 64 KB
  // instruction cache that two compute units share).
  auto project = [&](float db, float dn) {
    const float ddelta = dn - db;
    const float vs_x = ray_x * db;
    const float vs_z = ray_z * db;
    const float corr_x = ray_x * ddelta;
    const float corr_z = ray_z * ddelta;
    StepProj p;
    p.pz = cos_x * vs_z + sin_x * mountain;
    p.py3 = vertical ? cos_x * mountain - sin_x * vs_z : vs_x;
    p.py3 *= hmul;
    p.czz = cos_x * corr_z;
    p.cyy = vertical ? -sin_x * corr_z : corr_x;
    p.cyy *= hmul;
    p.top = p.pz * half + p.py3;
    return p;
  };
  auto prepare = [&](auto produce, const DdaChunk& cur, DdaChunk& nxt, bool& have_next,
                     lds_u16* rc, DdaPrepared& out) {
    const int L = cur.L, mip = cur.mip, shift = cur.shift;
    g_u16* slab = cur.slab;
    const uint2 ent = cur.ent;
    const uint64_t wofs = (uint64_t)ent.x << shift;  // column's slab word offset

    // ---- per-lane stateless projection (Cuda_Render.h:444-466)
    const bool valid = lane < L;
    const StepProj sp = project(cur.db, cur.dn);
    const float pz = sp.pz, py3 = sp.py3, czz = sp.czz, cyy = sp.cyy, top = sp.top;
    const uint32_t slen = ent.y & 0xffffu;
    g_u16* runs = slab + 2 + wofs;

    // F: projected top of the first drawn element in front of the eye.  A
    // step whose cell top is already below the horizon with pz > 0 stays
    // culled as the horizon rises (the replay's clip-top test, monotone in
    // ymin for pz > 0): it can never act, and its F is not needed.
    const bool culled0 = pz > 0.0f && top <= pz * (float)ymin;
    int F = INT32_MIN, kF = -1, ygF = 0;
    uint32_t nel = 0;
    float texF = 0;
    int textureF = 0;
    float ytopF = 0, ybotF = 0;
    if (!culled0) {
      uint32_t w = ent.y >> 16;
      int yg = 0;
      float tex = 0;
      for (uint32_t k = 0; k < slen; k++) {
        if (k > 0) w = runs[k];
        nel++;
        int dr = (int)(w >> 10);
        yg += (int)(w & 1023u) << mip;
        if (dr == 0) continue;
        const int texture = (int)tex;
        tex += (float)dr;
        dr <<= mip;
        const float ytop = (float)yg;
        yg += dr;
        float zz1 = pz, yy1 = py3;
        if (mountain + ytop >= 0) {
          zz1 += czz;
          yy1 += cyy;
        }
        const float pz1 = zz1 + z_add * ytop;
        if (pz1 <= 0) continue;
        const float py1 = yy1 + y_add * ytop;
        F = d_f2i(half + py1 / pz1);
        kF = (int)k;
        ygF = yg;
        texF = tex;
        textureF = texture;
        ytopF = ytop;
        ybotF = (float)yg;
        break;
      }
    }

    // ---- run cache: the head of each candidate column.  The horizon only rises, so F > ymin now is necessary for
    // acting; the clip-top test is monotone in ymin only for pz > 0.
    const bool cand = valid && F > ymin && !culled0;
    const uint64_t rc_base = wofs & ~(uint64_t)7;  // 16-byte aligned start
    const int rc_delta = (int)(wofs - rc_base);
    const RcColumn cached{rc, lane, rc_delta};
    const int ccap = cand ? RC - rc_delta : 0;
    static_assert(RC % 8 == 0 && RC >= 24, "the run cache is fetched in 16-byte words");
    constexpr int kWords = RC / 8;
    // ---- next chunk's DDA, before the cache's loads go out: an LDS access
    // waits for every load that writes LDS
    if constexpr (decltype(produce)::value) have_next = dda_next_chunk<!COUNT, HOLD>(wk, nxt, sc, *lc, zfar, ymin, dl, lane);

    // A wait for this wavefront's LDS reads (the last chunk's, of the cache)
    // before the loads may write it, and for the loads before it is read.
    constexpr int kWaitLds = 0xc07f, kWaitLoads = 0x0f70;  // lgkmcnt(0), vmcnt(0)
    if (cand) {
      typedef __attribute__((address_space(1))) const void g_void;
      typedef __attribute__((address_space(3))) void l_void;
      __builtin_amdgcn_s_waitcnt(kWaitLds);
      g_u16* src = slab + rc_base;
#pragma unroll
      for (int i = 0; i < kWords; i++)
        __builtin_amdgcn_global_load_lds((g_void*)(src + 8 * i), (l_void*)(rc + 512 * i), 16, 0, 0);
    }

    // first element's lower end and span parameters (Cuda_Render.h:554-660)
    int s1F = 0;
    bool drawF = false;
    float s1rF = 0, u1zF = 0, u2dzF = 0, onez1F = 0, onedz2F = 0;
    int F2 = INT32_MIN;
    if (cand) {
      float zz2 = pz, yy2 = py3;
      if (mountain + ybotF < 0) {
        zz2 += czz;
        yy2 += cyy;
      }
      const float pz2 = zz2 + z_add * ybotF;
      if (pz2 > 0) {
        drawF = true;
        const float py2 = yy2 + y_add * ybotF;
        const float pz1r = pz + z_add * ytopF;
        const float py1r = py3 + y_add * ytopF;
        const float pz2r = pz + z_add * ybotF;
        const float py2r = py3 + y_add * ybotF;
        // The quotients by pz1r, pz2r and the span's length share their
        // divisors' reciprocals (exact_div.h): 43 instructions in place of 99
        // for the nine.  |py| below 2^-60 is fine, next to half >= 8.
        const bool safe = div_safe(pz1r) & div_safe(pz2r) &
                          (fmaxf(fabsf(py1r), fabsf(py2r)) < 1152921504606846976.0f);
        if (ballot(!safe) == 0) {
          onez1F = recip_exact(pz2r, __builtin_amdgcn_rcpf(pz2r));
          const float onez2 = recip_exact(pz1r, __builtin_amdgcn_rcpf(pz1r));
          const float q2 = div_exact(py2r, pz2r, onez1F);
          const float len = (half + div_exact(py1r, pz1r, onez2)) - (half + q2);
          s1rF = half + q2;
          u1zF = div_exact(texF, pz2r, onez1F);
          u2dzF = div_exact((float)textureF, pz1r, onez2) - u1zF;
          onedz2F = onez2 - onez1F;
          // the bottom edge itself, unless the near-edge correction moved it
          s1F = d_f2i(half + q2 - 1.0f);
          const bool moved = mountain + ybotF < 0;
          if (ballot(moved) != 0 && moved) s1F = d_f2i(half + py2 / pz2 - 1.0f);
          const bool safe_len = div_safe(len) & div_dividend_safe(u2dzF) & div_dividend_safe(onedz2F);
          if (ballot(!safe_len) == 0) {
            const float r = recip_exact(len, __builtin_amdgcn_rcpf(len));
            u2dzF = div_exact(u2dzF, len, r);
            onedz2F = div_exact(onedz2F, len, r);
          } else {
            u2dzF /= len;
            onedz2F /= len;
          }
        } else {
          s1F = d_f2i(half + py2 / pz2 - 1.0f);
          const float s2r = half + py1r / pz1r;
          s1rF = half + py2r / pz2r;
          u1zF = texF / pz2r;
          u2dzF = (float)textureF / pz1r - u1zF;
          onez1F = 1.0f / pz2r;
          onedz2F = 1.0f / pz1r - onez1F;
          u2dzF /= s2r - s1rF;
          onedz2F /= s2r - s1rF;
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(kWaitLoads);
    // ---- next chunk's pointer gather: in flight during this chunk's replay
    if constexpr (decltype(produce)::value) {
      if (have_next) dda_gather(wk, nxt, vpx, vpz, fix_x, fix_z, lane);
    }
    wave_sync();  // run cache filled
    if (cand) {  // F2: projected top of the next element the loop tests
      int yg = ygF;
      for (uint32_t k = (uint32_t)kF + 1; k < slen; k++) {
        const int ci = (int)k + 2;
        const uint32_t w = column_word(ci < ccap, rc, cached.index(ci), runs + k);
        int dr = (int)(w >> 10);
        yg += (int)(w & 1023u) << mip;
        if (dr == 0) continue;
        dr <<= mip;
        const float ytop = (float)yg;
        yg += dr;
        float zz1 = pz, yy1 = py3;
        if (mountain + ytop >= 0) {
          zz1 += czz;
          yy1 += cyy;
        }
        const float pz1 = zz1 + z_add * ytop;
        if (pz1 <= 0) continue;
        const float py1 = yy1 + y_add * ytop;
        F2 = d_f2i(half + py1 / pz1);
        break;
      }
    }

    out.L = L;
    out.mip = mip;
    out.shift = shift;
    out.slab = slab;
    out.db = cur.db;
    out.dn = cur.dn;
    out.ent = ent;
    out.F = F;
    out.F2 = F2;
    out.kF = kF;
    out.ygF = ygF;
    out.textureF = textureF;
    out.s1F = s1F;
    out.cand = cand;
    out.drawF = drawF;
    out.texF = texF;
    out.s1rF = s1rF;
    out.u1zF = u1zF;
    out.u2dzF = u2dzF;
    out.onez1F = onez1F;
    out.onedz2F = onedz2F;
    out.nel = nel;
  };
  // ---- ordered replay of the steps that act; false when the line has ended
  auto replay = [&](const DdaPrepared& in, lds_u16* rc) -> bool {
    const int L = in.L, mip = in.mip, shift = in.shift;
    g_u16* slab = in.slab;
    const uint2 ent = in.ent;
    const bool valid = lane < L;
    // Made again rather than held: the drawing wavefront of three gets db and
    // dn, and the batch kernel has registers to spare that way (64 views 5.32
    // -> 5.20 ms).
    const StepProj sp = project(in.db, in.dn);
    const float pz = sp.pz, py3 = sp.py3, czz = sp.czz, cyy = sp.cyy, top = sp.top;
    const int F = in.F, F2 = in.F2, kF = in.kF, ygF = in.ygF, textureF = in.textureF;
    const int s1F = in.s1F;
    const bool cand = in.cand, drawF = in.drawF;
    const float texF = in.texF, s1rF = in.s1rF, u1zF = in.u1zF, u2dzF = in.u2dzF;
    const float onez1F = in.onez1F, onedz2F = in.onedz2F;
    const uint32_t nel = in.nel;
    int cur_step = 0;
    bool done = false;
    for (;;) {
      ymin = uni(ymin);
      ymax = uni(ymax);
      if (ymin >= ymax) {
        done = true;
        break;
      }
      const bool culled = top <= pz * (float)ymin;
      const bool act = valid && lane >= cur_step && !culled && F > ymin;
      const uint64_t am = uni64(ballot(act));
      if (!COUNT && (am & (am - 1))) {
        // ---- horizon sweep: a run of acting steps applied at once.  The
        // typical step draws its first element's span from the horizon up
        // (s1 <= ymin), leaves the top clip alone (F < ymax) and breaks at
        // its next element (F2 <= F): its only effects are ymin = F and the
        // rows [ymin, F) drawn.  The horizon before step t is then the prefix
        // maximum M_t of the earlier actors' F.  Each lane checks that, under
        // M_t, it acts exactly when the speculation says it does and that
        // its step is of that simple kind; the steps before the first lane
        // failing a check, whose spans together stay within 64 rows that are
        // all clear in the bitmap (row F included, where the horizon stops),
        // are applied here exactly as the ordered replay would apply them.
        const int Fs = act ? F : INT32_MIN;
        const int M = prefix_max_excl(Fs, ymin, lane);
        const bool spec_actor = act && F > M;
        const bool true_actor = valid && lane >= cur_step && !(top <= pz * (float)M) && F > M;
        const bool simple = cand && drawF && s1F <= M && F < ymax && F2 <= F && F - ymin <= 63;
        const bool ok = spec_actor == true_actor && (!spec_actor || simple);
        const uint64_t bad = uni64(ballot(lane >= cur_step && !ok));
        const int limit = uni(bad ? (int)__builtin_ctzll(bad) : 64);
        const uint64_t acc = uni64(ballot(spec_actor && lane < limit));
        if (acc) {
          const int last = 63 - (int)__builtin_clzll(acc);
          const int fend = uni(readlane_i(F, last));
          // rows ymin..fend (fend < ymin + 64) must all be clear
          const bool rclear = lane > fend - ymin || !lds_bit(bits, ymin + lane);
          if (uni64(ballot(rclear)) == ~0ull) {
            // row r = ymin + j belongs to the accepted step with the highest
            // start row <= j (starts are marked in LDS)
            sweep_lds[lane] = -1;
            wave_sync();
            if ((acc >> lane) & 1) sweep_lds[M - ymin] = lane;
            wave_sync();
            const int mark = sweep_lds[lane];
            const uint64_t smask = uni64(ballot(mark >= 0));
            const int nrows = fend - ymin;
            const bool mine = lane < nrows;
            const uint64_t upto = lane >= 63 ? ~0ull : ((2ull << lane) - 1ull);
            const int srow = 63 - (int)__builtin_clzll((smask & upto) | 1ull);
            const int a0 = __shfl(mark, srow);
            const int a = mine ? a0 : 0;
            const float s1r = __shfl(s1rF, a), u1z = __shfl(u1zF, a), u2dz = __shfl(u2dzF, a);
            const float onez1 = __shfl(onez1F, a), onedz2 = __shfl(onedz2F, a);
            const float thi = __shfl(texF, a) - 1.0f;
            const float tlo = (float)__shfl(textureF, a);
            const uint32_t aofs = (uint32_t)__shfl((int)ent.x, a);
            const uint32_t alen = (uint32_t)__shfl((int)ent.y, a) & 0xffffu;
            if (mine) {
              const int y0 = ymin + srow;
              const float mult = (float)(y0 + 1) - s1r;
              float uz = u1z + u2dz * mult, oz = onez1 + onedz2 * mult;
              span_steps(uz, oz, u2dz, onedz2, lane - srow);
              uint32_t u, depth;
              span_texel(uz, oz, tlo, thi, u, depth);
              const uint64_t wofs = (uint64_t)aofs << shift;
              const int tdelta = (int)((aofs << shift) & 7u);
              const int cw = 2 + (int)alen + tdelta + (int)u;
              row[ymin + lane] =
                  column_word(cw < RC, rc, rc_index(a, cw), slab + 2 + wofs + alen + u) +
                  (depth << 16);
            }
            bits_set_range(bits, ymin, fend, lane);
            wave_sync();
            ymin = fend;
            cur_step = limit;
            continue;
          }
        }
      }
      const int t = uni(am ? (int)__builtin_ctzll(am) : L);
      if (COUNT) {
        // no-op steps [cur_step, t): pointer loads and elements walked to the break
        const bool noop_loaded = valid && lane >= cur_step && lane < t && !culled;
        cnt.steps += (uint64_t)(t - cur_step);
        cnt.ptr += (uint64_t)__popcll(ballot(noop_loaded));
        unsigned long long e = noop_loaded ? nel : 0, r = (noop_loaded && nel) ? nel - 1 : 0;
        for (int o = 32; o > 0; o >>= 1) {
          e += __shfl_xor(e, o);
          r += __shfl_xor(r, o);
        }
        cnt.elems += e;
        cnt.rle += r;
      }
      if (!am) break;
      if (COUNT) {
        cnt.steps++;
        cnt.ptr++;
      }

      const uint64_t tofs = (uint64_t)(uint32_t)readlane_i((int)ent.x, t) << shift;
      const uint32_t tlf = (uint32_t)readlane_i((int)ent.y, t);
      const uint32_t tslen = tlf & 0xffffu;
      g_u16* truns = slab + 2 + tofs;
      g_u16* tcol = truns + tslen;
      const bool tcached = readlane_i((int)cand, t) != 0;
      const int tdelta = (int)(tofs & 7u);
      const RcColumn tcache{rc, t, tdelta};
      const int tcap = tcached ? RC - tdelta : 0;
      const float tpz = readlane_f(pz, t), tpy = readlane_f(py3, t);
      const float tczz = readlane_f(czz, t), tcyy = readlane_f(cyy, t);

      // element loop state after the first drawn element in front
      uint32_t k0;
      int ygen;
      float tex;
      const bool fast = !COUNT && tcached;
      if (fast) {
        // ---- first drawn element: precomputed (Cuda_Render.h:540-733)
        const int s2 = readlane_i(F, t);  // > ymin by the ballot
        const bool tdraw = readlane_i((int)drawF, t) != 0;
        int s1 = readlane_i(s1F, t);
        if (tdraw && s1 < ymax) {
          int e2 = s2;
          if (e2 >= ymax) {
            e2 = ymax;
            ymax = s1;
          }
          if (s1 <= ymin) {
            s1 = ymin;
            ymin = e2;
            if (ymax > ymin) ymin = first_clear(bits, ymin, ymax, lane);
          }
          const SpanWindow sw = span_window(bits, s1, e2, lane);
          if (sw.y0 < e2) {
            const float s1r = readlane_f(s1rF, t);
            const float u1z = readlane_f(u1zF, t), u2dz = readlane_f(u2dzF, t);
            const float onez1 = readlane_f(onez1F, t), onedz2 = readlane_f(onedz2F, t);
            const float mult = (float)(sw.y0 + 1) - s1r;
            const float uzb = u1z + u2dz * mult;
            const float ozb = onez1 + onedz2 * mult;
            const float thi = readlane_f(texF, t) - 1.0f;
            const float tlo = (float)readlane_i(textureF, t);
            span_draw(sw, s1, e2, uzb, ozb, u2dz, onedz2, tlo, thi, tcache, tcap, tcol,
                      2 + (int)tslen, row, bits, lane);
          }
        }
        // the next element tested breaks unless it reaches above ymin
        if (readlane_i(F2, t) <= ymin) {
          cur_step = t + 1;
          continue;
        }
        k0 = (uint32_t)readlane_i(kF, t) + 1;
        ygen = readlane_i(ygF, t);
        tex = readlane_f(texF, t);
      } else {
        k0 = 0;
        ygen = 0;
        tex = 0;
      }

      // ---- remaining elements (Cuda_Render.h:511-734)
      if constexpr (!COUNT && PAR_ELEMS) {
        // Lane j precomputes element k0 + base + j of the column: its run
        // word, its rows and texture range from prefix sums over the lanes
        // (integers, so equal to the sequential sums; tex holds integers
        // below 2^24, so its float sums are exact too), and every projection
        // and span parameter the sequential loop would compute for it, with
        // the same operations in the same order.  The uniform loop below
        // then applies the horizon clip, the bitmap and the drawing to one
        // element after another, reading those values by lane.
        bool stop = false;
        for (uint32_t base = k0; base < tslen && !stop; base += 64) {
          const uint32_t k = base + (uint32_t)lane;
          const bool in = k < tslen;
          const bool first = k == 0 || !in;
          uint32_t w = column_word(first || (int)k + 2 < tcap, rc,
                                   tcache.index(first ? 2 : (int)k + 2), truns + k);
          w = in ? (k == 0 ? tlf >> 16 : w) : 0;
          const int edrawn = (int)(w >> 10);
          const int eskip = (int)(w & 1023u) << mip;
          const int yinc = prefix_sum_incl(eskip + (edrawn << mip), lane);
          const int tinc = prefix_sum_incl(edrawn, lane);
          const int ytop_i = ygen + yinc - (edrawn << mip);  // after this element's skip
          const int texture = (int)(tex + (float)(tinc - edrawn));
          const float etex = tex + (float)tinc;  // tex after this element
          const float ytop = (float)ytop_i;
          const float ybot = (float)(ytop_i + (edrawn << mip));
          float zz1 = tpz, yy1 = tpy;
          if (mountain + ytop >= 0) {
            zz1 += tczz;
            yy1 += tcyy;
          }
          const float pz1 = zz1 + z_add * ytop;
          const float py1 = yy1 + y_add * ytop;
          const int es2 = d_f2i(half + py1 / pz1);
          float zz2 = tpz, yy2 = tpy;
          if (mountain + ybot < 0) {
            zz2 += tczz;
            yy2 += tcyy;
          }
          const float pz2 = zz2 + z_add * ybot;
          const float py2 = yy2 + y_add * ybot;
          const int es1 = d_f2i(half + py2 / pz2 - 1.0f);
          const float pz1r = tpz + z_add * ytop;
          const float py1r = tpy + y_add * ytop;
          const float pz2r = tpz + z_add * ybot;
          const float py2r = tpy + y_add * ybot;
          const float s2r = half + py1r / pz1r;
          const float es1r = half + py2r / pz2r;
          const float eu1z = etex / pz2r;
          float eu2dz = (float)texture / pz1r - eu1z;
          const float eonez1 = 1.0f / pz2r;
          float eonedz2 = 1.0f / pz1r - eonez1;
          eu2dz /= s2r - es1r;
          eonedz2 /= s2r - es1r;
          // flags: drawn, in front at the top, in front at the bottom
          const int eflags = (in && edrawn != 0 ? 1 : 0) | (pz1 > 0 ? 2 : 0) | (pz2 > 0 ? 4 : 0);
          const int nb = (int)min(64u, tslen - base);
          // Only elements that can act are visited.  Within the loop ymax
          // only falls and ymin never rises above the ymax of this point,
          // so an element that can neither draw (needs bottom row s1 <
          // ymax) nor stop the column (needs top row s2 <= ymin) from here
          // on stays inert: the loop below would reach one of its
          // `continue`s for it.
          const bool can_act = lane < nb && (eflags & 3) == 3 &&
                               (es2 <= ymax || ((eflags & 4) && es1 < ymax));
          for (uint64_t act = ballot(can_act); act != 0; act &= act - 1) {
            const int j = (int)__builtin_ctzll(act);
            const int f = readlane_i(eflags, j);
            if (!(f & 1) || !(f & 2)) continue;
            int s2 = readlane_i(es2, j);
            if (s2 <= ymin) {
              stop = true;
              break;
            }
            if (!(f & 4)) continue;
            int s1 = readlane_i(es1, j);
            if (s1 >= ymax) continue;
            if (s2 >= ymax) {
              s2 = ymax;
              ymax = s1;
            }
            if (s1 <= ymin) {
              s1 = ymin;
              ymin = s2;
              if (ymax > ymin) ymin = first_clear(bits, ymin, ymax, lane);
            }
            const SpanWindow sw = span_window(bits, s1, s2, lane);
            if (sw.y0 >= s2) continue;
            const float s1r = readlane_f(es1r, j);
            const float u2dz = readlane_f(eu2dz, j), onedz2 = readlane_f(eonedz2, j);
            const float mult = (float)(sw.y0 + 1) - s1r;
            const float uzb = readlane_f(eu1z, j) + u2dz * mult;
            const float ozb = readlane_f(eonez1, j) + onedz2 * mult;
            span_draw(sw, s1, s2, uzb, ozb, u2dz, onedz2, (float)readlane_i(texture, j),
                      readlane_f(etex, j) - 1.0f, tcache, tcap, tcol, 2 + (int)tslen, row, bits,
                      lane);
          }
          ygen += readlane_i(yinc, 63);
          tex += (float)readlane_i(tinc, 63);
        }
        cur_step = t + 1;
        continue;
      }
      // ---- remaining elements (Cuda_Render.h:511-734), uniform
      for (uint32_t k = k0; k < tslen; k++) {
        uint32_t w;
        if (k == 0) w = tlf >> 16;
        else w = column_word((int)k + 2 < tcap, rc, tcache.index((int)k + 2), truns + k);
        if (COUNT) {
          cnt.elems++;
          if (k > 0) cnt.rle++;
        }
        int drawn = (int)(w >> 10);
        ygen += (int)(w & 1023u) << mip;
        if (drawn == 0) continue;
        const int texture = (int)tex;
        tex += (float)drawn;
        drawn <<= mip;
        const float ytop = (float)ygen;
        ygen += drawn;
        const float ybot = (float)ygen;
        float zz1 = tpz, yy1 = tpy;
        if (mountain + ytop >= 0) {
          zz1 += tczz;
          yy1 += tcyy;
        }
        const float pz1 = zz1 + z_add * ytop;
        if (pz1 <= 0) continue;
        const float py1 = yy1 + y_add * ytop;
        int s2 = uni(d_f2i(half + py1 / pz1));
        if (s2 <= ymin) break;
        float zz2 = tpz, yy2 = tpy;
        if (mountain + ybot < 0) {
          zz2 += tczz;
          yy2 += tcyy;
        }
        const float pz2 = zz2 + z_add * ybot;
        if (pz2 <= 0) continue;
        const float py2 = yy2 + y_add * ybot;
        int s1 = uni(d_f2i(half + py2 / pz2 - 1.0f));
        if (s1 >= ymax) continue;
        if (s2 >= ymax) {
          s2 = ymax;
          ymax = s1;
        }
        if (s1 <= ymin) {
          s1 = ymin;
          ymin = s2;
          if (ymax > ymin) ymin = first_clear(bits, ymin, ymax, lane);
        }
        const SpanWindow sw = span_window(bits, s1, s2, lane);
        if (sw.y0 >= s2) continue;
        const int y0 = sw.y0;
        const float pz1r = tpz + z_add * ytop;
        const float py1r = tpy + y_add * ytop;
        const float pz2r = tpz + z_add * ybot;
        const float py2r = tpy + y_add * ybot;
        const float s2r = half + py1r / pz1r;
        const float s1r = half + py2r / pz2r;
        const float u1z = tex / pz2r;
        float u2dz = (float)texture / pz1r - u1z;
        const float onez1 = 1.0f / pz2r;
        float onedz2 = 1.0f / pz1r - onez1;
        u2dz /= s2r - s1r;
        onedz2 /= s2r - s1r;
        const float mult = (float)(y0 + 1) - s1r;
        const float uzb = u1z + u2dz * mult;
        const float ozb = onez1 + onedz2 * mult;
        if (COUNT) cnt.spans++;
        const int d = span_draw(sw, s1, s2, uzb, ozb, u2dz, onedz2, (float)texture, tex - 1.0f,
                                tcache, tcap, tcol, 2 + (int)tslen, row, bits, lane);
        if (COUNT) cnt.col += (uint64_t)d;
      }
      cur_step = t + 1;
    }
    // ---- early end of the walk (WalkEnd): later steps lie beyond this
    // chunk's last crossing distance
    if (!done && L > 0 && !cnt.ended && wfloor < (float)ymin + (1.0f - WalkEnd::kAbs) &&
        wend->done(readlane_f(in.dn, L - 1), ymin, sc.mip[uni(mip)].top, sc.sy)) {
      if (COUNT) cnt.end_walk();  // the counting variant walks on to count the reference's work
      else done = true;
    }
    return !done;
  };
  // a chunk prepared and replayed by one wavefront
  auto chunk_step = [&](auto produce, const DdaChunk& cur, DdaChunk& nxt, bool& have_next) {
    if (ymin >= ymax) return false;
    DdaPrepared p;
    prepare(produce, cur, nxt, have_next, rc, p);
    return replay(p, rc);
  };
  if constexpr (WAVES == 1) {
    // the first step has no chunk of its own (L = 0) and only walks ahead
    DdaChunk cur, nxt;
    cur.L = 0;
    cur.mip = 0;
    cur.shift = 0;
    cur.slab = wk.slab;
    cur.db = cur.dn = 0.0f;
    cur.ent = make_uint2(0u, 0u);
    bool have = true;
    const std::true_type yes;
    while (have && chunk_step(yes, cur, nxt, have)) {
      // the copy waits for the gather, whose entries the next step starts with
      cur.L = nxt.L;
      cur.mip = nxt.mip;
      cur.shift = nxt.shift;
      cur.slab = nxt.slab;
      cur.db = nxt.db;
      cur.dn = nxt.dn;
      cur.ent = nxt.ent;
    }
  } else if constexpr (WAVES == 3) {
    LineRings& r = *rings;
    if (producer && lane == 0) {
      r.walked = r.prepared = r.taken = r.replayed = r.stop = 0;
      r.walk_total = r.prep_total = INT32_MAX;
      r.horizon = ymin;
    }
    __syncthreads();
    if (producer) {
      // chunk n is walked, then chunk n-1 (whose gather ran meanwhile)
      // completed and chunk n's gather issued
      uint2 ent = make_uint2(0u, 0u);
      int s = 0, before = 0;  // slots of chunks n, n-1
      for (int n = 0;; n++) {
        int stop;
        for (;;) {
          const int taken = ring_read(r.taken);
          stop = ring_read(r.stop);
          ymin = ring_read(r.horizon);
          if (stop || n - taken < kWalkSlots) break;
          __builtin_amdgcn_s_sleep(8);
        }
        if (stop) break;
        wave_sync();
        DdaChunk c;
        const bool more = dda_next_chunk<true, HOLD>(wk, c, sc, *lc, zfar, ymin, dl, lane);
        if (n > 0) {
          r.ent[before][lane] = ent;  // waits for the gather
          ring_write(r.walked, n, lane);
        }
        if (!more) {
          ring_write(r.walk_total, n, lane);
          break;
        }
        dda_gather(wk, c, vpx, vpz, fix_x, fix_z, lane);
        ent = c.ent;
        r.db[s][lane] = c.db;
        r.dn[s][lane] = c.dn;
        if (lane == 0) {
          r.slab[s] = c.slab;
          r.L[s] = c.L;
          r.mip[s] = c.mip;
          r.shift[s] = c.shift;
        }
        before = s;
        s = s == kWalkSlots - 1 ? 0 : s + 1;
      }
    } else if (!drawer) {
      const std::false_type no;
      DdaChunk cur, unused;
      bool hu = false;
      int s = 0, n = 0;
      for (;; n++) {
        int stop, walked;
        for (;;) {
          walked = ring_read(r.walked);
          const int total = ring_read(r.walk_total);
          stop = ring_read(r.stop);
          const int replayed = ring_read(r.replayed);
          ymin = ring_read(r.horizon);
          if (stop || total <= n || (walked > n && n - replayed < kPrepSlots)) break;
          __builtin_amdgcn_s_sleep(4);
        }
        if (stop || walked <= n) break;
        wave_sync();
        cur.L = uni(r.L[s]);
        cur.mip = uni(r.mip[s]);
        cur.shift = uni(r.shift[s]);
        cur.slab = (g_u16*)uni64((uint64_t)r.slab[s]);
        cur.db = r.db[s][lane];
        cur.dn = r.dn[s][lane];
        cur.ent = r.ent[s][lane];
        ring_write(r.taken, n + 1, lane);
        DdaPrepared p;
        prepare(no, cur, unused, hu, rc + (n & 1) * (64 * RC), p);
        prep_put(r, n & 1, p, lane);
        ring_write(r.prepared, n + 1, lane);
        s = s == kWalkSlots - 1 ? 0 : s + 1;
      }
      ring_write(r.prep_total, n, lane);
    } else {
      for (int n = 0;; n++) {
        int prepared;
        for (;;) {
          prepared = ring_read(r.prepared);
          const int total = ring_read(r.prep_total);
          if (prepared > n || total <= n) break;
          __builtin_amdgcn_s_sleep(4);
        }
        if (prepared <= n) break;
        wave_sync();
        DdaPrepared p;
        prep_get(r, n & 1, p, lane);
        p.nel = 0;
        if (!replay(p, rc + (n & 1) * (64 * RC))) break;
        ring_write(r.horizon, ymin, lane);
        ring_write(r.replayed, n + 1, lane);
      }
      ring_write(r.stop, 1, lane);
    }
  } else {
    // Round i: slot i%3 holds chunk i complete, slot (i+1)%3 chunk i+1's DDA
    // (its gather in flight in the producer).  The producer walks chunk i+2
    // and stores chunk i+1's entries while the consumer processes chunk i;
    // a block barrier ends the round.  Both wavefronts read the same flags
    // after each barrier (have[i%3] last written two rounds before, stop[i%3]
    // in this round), so they run the same rounds and the same barriers.
    ChunkRing& r = *ring;
    if (producer) {
      // chunk n is walked, then chunk n-1's entries stored and chunk n's
      // gather issued; the barriers after n = 1, 2, ... end the rounds
      DdaChunk p;
      uint2 ent = make_uint2(0u, 0u);  // of the gather in flight
      bool pend = false, more = true;
      int s = 0, s1 = 2, s2 = 1;  // slots of chunks n, n-1, n-2
      for (int n = 0;; n++) {
        if (n >= 2 && !uni(r.have[s2])) break;
        more = more && dda_next_chunk<true, HOLD>(wk, p, sc, *lc, zfar, ymin, dl, lane);
        ring_put_dda(r, s, p, more, lane);
        if (pend) r.ent[s1][lane] = ent;  // waits for the gather
        if (more) {
          dda_gather(wk, p, vpx, vpz, fix_x, fix_z, lane);
          ent = p.ent;
        }
        pend = more;
        if (n >= 1) __syncthreads();
        if (n >= 2) {
          if (uni(r.stop[s2])) break;
          ymin = uni(r.horizon[s2]);
        }
        s2 = s1;
        s1 = s;
        s = s == 2 ? 0 : s + 1;
      }
    } else {
      __syncthreads();
      const std::false_type no;
      DdaChunk cur, unused;
      bool hu = false;
      int s = 0;
      for (;;) {
        if (!uni(r.have[s])) break;
        ring_get(r, s, cur, lane);
        const bool more = chunk_step(no, cur, unused, hu);
        // A slot's flag is read after this round's barrier and rewritten
        // three rounds later, so no wavefront can see a later round's value.
        if (lane == 0) {
          r.stop[s] = more ? 0 : 1;
          r.horizon[s] = ymin;
        }
        __syncthreads();
        if (uni(r.stop[s])) break;
        s = s == 2 ? 0 : s + 1;
      }
    }
  }
  if (COUNT && lane == 0) cnt.flush(counts);
}

}  // namespace rlevox
