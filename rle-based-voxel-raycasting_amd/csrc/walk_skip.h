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
// A group's distances and cells come from the walk in real numbers: after t
// steps from the last step taken, i = floor(e0 + e1*t) of them crossed in x
// (dda_merge in wave_line.h has the same formula) and the last lies at the
// larger of sA + (i-1)*gA and sB + (t-i-1)*gB, on a straight line from the
// base.  Rounding in the walk's sums drifts from that by at most half an ulp
// a step (6e-8 of the distance); twice that is allowed for.
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
  float dirx, dirz, vpx, vpz;
  RLEVOX_HD void init(float dx, float dz, float px, float pz) {
    dirx = dx;
    dirz = dz;
    // From an eye at a negative coordinate the reference's crossings do not
    // lie on the ray (the fraction of the coordinate is negative,
    // Cuda_Render.h:283-296): nothing is claimed there.
    vpx = px >= 0.0f ? px : __builtin_nanf("");
    vpz = pz >= 0.0f ? pz : __builtin_nanf("");
  }
};
struct SkipBase {  // the last step taken, and what follows it
  float px, pz, dnow;
  float sA, sB, gA, gB;  // next crossing distances and their spacings
  float e0, e1;
  // Distance of the t-th step from here (t = 0: of the base).
  RLEVOX_HD float dist(float t) const {
    const float i = fminf(fmaxf(floorf(e0 + e1 * t), 0.0f), t), j = t - i;
    const float a = i > 0.0f ? sA + (i - 1.0f) * gA : dnow;
    const float b = j > 0.0f ? sB + (j - 1.0f) * gB : dnow;
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

// Upper bound (with WalkEnd's margins) of the rows that steps t0..t1-1 after
// the base can project a run top to; infinite where none can be given.
RLEVOX_HD inline float skip_bound(const WalkEnd& e, const SkipLine& l, const SkipBase& b,
                                  const SkipLevel& v, int sy, int t0, int t1) {
  // a step uses the distances and the position of its ends: steps t0..t1-1
  // those of t0..t1
  const float lo0 = b.dist((float)t0), hi0 = b.dist((float)t1);
  const float drift = (2e-6f + 1.2e-7f * (float)t1) * hi0;
  const float lo = fmaxf(lo0 - drift, 0.0f), hi = hi0 + drift;
  const float ax = l.vpx + b.px + l.dirx * (lo - b.dnow), bx = l.vpx + b.px + l.dirx * (hi - b.dnow);
  const float az = l.vpz + b.pz + l.dirz * (lo - b.dnow), bz = l.vpz + b.pz + l.dirz * (hi - b.dnow);
  // a position's voxel is its truncation, or one less (the cell fix-up), so
  // down to one below, and up to one above where it is negative
  const float m = 0.02f + 1e-6f * (fabsf(ax) + fabsf(bx) + fabsf(az) + fabsf(bz));
  const float xa = fminf(ax, bx), za = fminf(az, bz);
  const float x0 = xa - 1.0f - m, x1 = fmaxf(ax, bx) + (xa < 1.0f ? 1.0f : 0.0f) + m;
  const float z0 = za - 1.0f - m, z1 = fmaxf(az, bz) + (za < 1.0f ? 1.0f : 0.0f) + m;
  const bool sane = (x0 > -1e9f) & (x1 < 1e9f) & (z0 > -1e9f) & (z1 < 1e9f);
  const int sh = v.mip + kSkipBlockLog;
  const int cx0 = (int)floorf(sane ? x0 : 0.0f) >> sh, cx1 = (int)floorf(sane ? x1 : 0.0f) >> sh;
  const int cz0 = (int)floorf(sane ? z0 : 0.0f) >> sh, cz1 = (int)floorf(sane ? z1 : 0.0f) >> sh;
  const int nx = skip_blocks(v.gridx), nz = skip_blocks(v.gridz);  // powers of two
  const int ix0 = cx0 & (nx - 1), ix1 = cx1 & (nx - 1);
  const int iz0 = (cz0 & (nz - 1)) * nx, iz1 = (cz1 & (nz - 1)) * nx;
  const int t00 = v.tops[iz0 + ix0], t01 = v.tops[iz0 + ix1];
  const int t10 = v.tops[iz1 + ix0], t11 = v.tops[iz1 + ix1];
  const int p = t00 < t01 ? t00 : t01, q = t10 < t11 ? t10 : t11;
  // steps that span more blocks (a level coarser than the grids go) take
  // the whole level's top
  const int top = ((cx1 - cx0 <= 1) & (cz1 - cz0 <= 1)) ? (p < q ? p : q) : v.top;
  // pz is affine in distance and height: positive at the four corners, it is
  // positive throughout, and the projection's supremum is at a corner
  bool ok = sane;
  const WalkEnd::D dl = e.at_d(lo), dh = e.at_d(hi);
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
