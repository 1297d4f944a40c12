// Stretches of a line's walk that cannot draw (shared by the raycast kernels;
// plain C++ so a host check can run the same code: the includer defines
// RLEVOX_HD as the function qualifiers it needs).
//
// The end of a walk (walk_end.h) asks whether anything from here to the far
// distance can rise above the floating horizon, with the highest run of
// whole levels.  Most of a line's steps lie behind hills that already cover
// them long before that holds.  Here the same bound is taken over groups of
// kSkipSteps consecutive steps, with the highest run of the blocks of
// kSkipBlock x kSkipBlock cells that the group's steps can touch: a group
// whose bound stays at or below the horizon changes nothing (its first
// drawn element in front of the eye breaks the element loop, Cuda_Render.h:
// 540-543), now or at any later, higher horizon.
//
// A group's distances come from the two crossing sequences in real numbers:
// after t steps from the last step taken, i = floor(e0 + e1*t) of them crossed
// in x (dda_merge in wave_line.h has the same formula), j = t - i in z, and
// the last lies at the larger of sA + (i-1)*gA and sB + (j-1)*gB.  Rounding
// in the walk's sums drifts from that by at most half an ulp a step (6e-8 of
// the distance); twice that is allowed for, as the positions' sums drift by as
// much of their own.
//
// Its cells come from straight lines along the ray, one for either kind of
// crossing.  The walk's six sums have each been rounding since the start of
// the line, by an amount that is the same at every step within a binade, so
// the x crossings, the z crossings and the distances drift apart with the
// length of the whole walk: by hundredths of a cell after 1000 steps at one
// level, by several cells after 60000.  The line of the last step's kind goes
// through that step, that of the other kind through its next crossing, whose
// position and distance the walk holds (SkipBase::of).  The group's cells are
// those between the two.
#pragma once

#include <math.h>
#include <stdint.h>

#include "walk_end.h"

namespace rlevox {

constexpr int kSkipSteps = 8;           // steps per group
constexpr int kSkipBlockLog = 4;        // cells per block side: 16
constexpr int kSkipWindow = 64 * kSkipSteps;

// Blocks along a grid side of n cells.
RLEVOX_HD inline int skip_blocks(int n) {
  return n >> kSkipBlockLog > 0 ? n >> kSkipBlockLog : 1;
}

struct SkipLine {  // the line: ground direction and eye column
  float dirx, dirz;
  float x0, x1, z0, z1;  // the eye's coordinates less, plus a margin
  RLEVOX_HD void init(float dx, float dz, float px, float pz) {
    dirx = dx;
    dirz = dz;
    // From an eye at a negative coordinate the reference's crossings do not
    // lie on the ray (the fraction of the coordinate is negative,
    // Cuda_Render.h:283-296): nothing is claimed there.
    const bool on = (px >= 0.0f) & (pz >= 0.0f);
    // the rounding of positions' sums with the eye's coordinates
    const float m = on ? 0.02f + 2e-6f * (px + pz) : __builtin_nanf("");
    x0 = px - m;
    x1 = px + m;
    z0 = pz - m;
    z1 = pz + m;
  }
};
struct SkipBase {  // the last step taken, and what follows it
  float px, pz, dnow;
  float sA, sB, gA, gB;  // next crossing distances and their spacings
  float e0, e1;
  // where the line of the other kind's crossings is at distance 0 (NaN: on
  // the last step's)
  float ox = __builtin_nanf(""), oz = __builtin_nanf("");

  // (od, nx, nz): distance and position of the next crossing of the other kind
  // than the last step's; r: the reciprocal of gA + gB, to a few ulps.
  RLEVOX_HD static SkipBase of(const SkipLine& l, float px, float pz, float dnow, float sA, float sB,
                               float gA, float gB, float od, float nx, float nz, float r) {
    return SkipBase{px, pz, dnow, sA, sB, gA, gB, (sB - sA + gA) * r, gB * r,
                    fmaf(-l.dirx, od, nx), fmaf(-l.dirz, od, nz)};
  }
  // Bounds of the distance of the t-th step from here (t = 0: of the base).
  // They hold for any split t = i + j, as the guess may be off: for rays near
  // an axis e1*t rounds by more than the share of the rarer crossings.  The
  // t-th crossing is not beyond both x's i-th and z's j-th.  Either i of the
  // first t are x's, and it is not before x's i-th, or j + 1 are z's, and it is
  // not before z's j+1-st; likewise with x and z exchanged.
  RLEVOX_HD float split(float t) const { return fminf(fmaxf(floorf(fmaf(e1, t, e0)), 0.0f), t); }
  RLEVOX_HD float far_(float t) const {
    const float i = split(t), j = t - i;
    return fmaxf(fmaxf(fmaf(i - 1.0f, gA, sA), fmaf(j - 1.0f, gB, sB)), dnow);
  }
  RLEVOX_HD float near_(float t) const {
    // a kind's 0-th crossing is at or before the base: a spacing before its
    // next one, less the rounding of that sum
    constexpr float kBelow = 0.99999988f;
    const float i = split(t), j = t - i;
    const float a = fminf(fmaf(i - 1.0f, gA, sA * kBelow), fmaf(j, gB, sB));
    const float b = fminf(fmaf(j - 1.0f, gB, sB * kBelow), fmaf(i, gA, sA));
    return fmaxf(fmaxf(a, b), dnow);
  }
};
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(1))) const int32_t skip_tops;  // read as global memory
#else
typedef const int32_t skip_tops;
#endif
struct SkipLevel {
  int mip, gridx, gridz;
  skip_tops* tops;  // per block: highest run top (world row), x fastest
  int top;              // highest run top of the level and all coarser ones
};

// x towards zero (device: saturating, NaN to 0, in one instruction; host: of x
// within range).
RLEVOX_HD inline int skip_trunc(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  int r;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(x));
  return r;
#else
  return x > -2e9f && x < 2e9f ? (int)x : 0;
#endif
}

// What steps t0..t1-1 after the base can touch: crossing distances lo..hi and
// blocks cx0..cx1, cz0..cz1 (before the grid's wrap) at a level whose blocks
// have 2^sh cells of level 0 a side.  sane = false: not known.
struct SkipRange {
  float lo, hi;
  int cx0, cx1, cz0, cz1;
  bool sane;
};

RLEVOX_HD inline SkipRange skip_range(const SkipLine& l, const SkipBase& b, int sh, int t0, int t1) {
  SkipRange r;
  // a step uses the distances and the position of its ends: steps t0..t1-1
  // those of t0..t1
  const float f0 = (float)t0, f1 = f0 + (float)(t1 - t0);
  const float lo0 = b.near_(f0), hi0 = b.far_(f1);
  const float drift = fmaf(1.2e-7f, f1, 2e-6f) * hi0;
  r.lo = fmaxf(lo0 - drift, 0.0f);
  r.hi = hi0 + drift;
  // the two lines at distance 0; drift also holds what the positions' sums
  // drift within the group's window
  const float px = fmaf(-l.dirx, b.dnow, b.px), pz = fmaf(-l.dirz, b.dnow, b.pz);
  const float ax = l.dirx * r.lo, bx = l.dirx * r.hi, az = l.dirz * r.lo, bz = l.dirz * r.hi;
  const float x0 = fminf(ax, bx) + (fminf(px, b.ox) + l.x0), x1 = fmaxf(ax, bx) + (fmaxf(px, b.ox) + l.x1);
  const float z0 = fminf(az, bz) + (fminf(pz, b.oz) + l.z0), z1 = fmaxf(az, bz) + (fmaxf(pz, b.oz) + l.z1);
  r.sane = (x0 > -1e9f) & (x1 < 1e9f) & (z0 > -1e9f) & (z1 < 1e9f);
  // a position's voxel is its truncation, or one less (the cell fix-up)
  r.cx0 = (skip_trunc(x0) - 1) >> sh;
  r.cx1 = skip_trunc(x1) >> sh;
  r.cz0 = (skip_trunc(z0) - 1) >> sh;
  r.cz1 = skip_trunc(z1) >> sh;
  return r;
}

// Upper bound (with WalkEnd's margins) of the rows that steps t0..t1-1 after
// the base can project a run top to; infinite where none can be given.
RLEVOX_HD inline float skip_bound(const WalkEnd& e, const SkipLine& l, const SkipBase& b,
                                  const SkipLevel& v, int sy, int t0, int t1) {
  const SkipRange g = skip_range(l, b, v.mip + kSkipBlockLog, t0, t1);
  const int nx = skip_blocks(v.gridx), nz = skip_blocks(v.gridz);  // powers of two
  const int ix0 = g.cx0 & (nx - 1), ix1 = g.cx1 & (nx - 1);
  const int iz0 = (g.cz0 & (nz - 1)) * nx, iz1 = (g.cz1 & (nz - 1)) * nx;
  const int t00 = v.tops[iz0 + ix0], t01 = v.tops[iz0 + ix1];
  const int t10 = v.tops[iz1 + ix0], t11 = v.tops[iz1 + ix1];
  const int p = t00 < t01 ? t00 : t01, q = t10 < t11 ? t10 : t11;
  // steps that span more blocks (a level coarser than the grids go, or sums
  // far apart) take the whole level's top
  const int top = ((g.cx1 - g.cx0 <= 1) & (g.cz1 - g.cz0 <= 1)) ? (p < q ? p : q) : v.top;
  // pz is affine in distance and height: positive at the four corners, it is
  // positive throughout, and the projection's supremum is at a corner
  bool ok = g.sane;
  const WalkEnd::D dl = e.at_d(g.lo), dh = e.at_d(g.hi);
  const WalkEnd::D yt = e.at_y(e.m + (float)top), yb = e.at_y(e.m + (float)sy);
  const float c0 = e.corner(dl, yt, ok), c1 = e.corner(dh, yt, ok);
  const float c2 = e.corner(dl, yb, ok), c3 = e.corner(dh, yb, ok);
  return ok ? fmaxf(fmaxf(c0, c1), fmaxf(c2, c3)) : __builtin_inff();
}

// The bound truncates to at most ymin.
RLEVOX_HD inline bool skip_hidden(float bound, int ymin) {
  return bound < (float)ymin + (1.0f - WalkEnd::kAbs);
}

}  // namespace rlevox
