// Checks what a group of steps can touch (skip_range of csrc/walk_skip.h)
// against the walk itself (Cuda_Render.h:270-304,376-442): the fp32 sums of
// random lines are walked step by step, and for groups of every window from a
// base, up to the kernels' reach ahead of it, each step must lie at distances
// within lo..hi and in a block within cx0..cx1, cz0..cz1.  Rays in all
// directions, some within 1e-1 to 1e-7 of an axis, from eyes at 0 to 1e5; the
// distance at which a level ends is the argument.  Built and run by
// tests/test_walk_range.py; WALK_RANGE_PLANT=1 takes both kinds' crossings
// for one line, a mistake the check must catch.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#define RLEVOX_HD
#include "../../rle-based-voxel-raycasting_amd/csrc/walk_skip.h"

#ifndef WALK_RANGE_PLANT
#define WALK_RANGE_PLANT 0
#endif

constexpr int kReach = 2048;  // kSkipReach of wave_line.h

struct Step {  // before the step
  float px, pz, d, sA, sB, ax, az, bx, bz;
  int ib;
};

int main(int argc, char** argv) {
  const int mipd = argc > 1 ? std::atoi(argv[1]) : 1024;
  const long budget = argc > 2 ? std::atol(argv[2]) : 20000000;
  std::mt19937 rng(5);
  std::uniform_real_distribution<float> u(0.0f, 1.0f);
  long steps = 0, groups = 0, near = 0, below = 0, above = 0, outside = 0;
  for (int line = 0; steps < budget; line++) {
    float a = 6.2831853f * u(rng);
    if (line % 4 == 3) {
      const float off = std::pow(10.0f, -1.0f - 6.0f * u(rng));
      a = 1.5707963f * (float)(rng() % 4) + (u(rng) < 0.5f ? off : -off);
    }
    const float dx = std::cos(a), dz = std::sin(a);
    const float span = line % 3 == 0 ? 100000.0f : 4096.0f;
    const float vpx = span * u(rng), vpz = span * u(rng);
    float fx = vpx - std::floor(vpx), fz = vpz - std::floor(vpz);
    const float signx = dx >= 0 ? 1.0f : -1.0f, signz = dz >= 0 ? 1.0f : -1.0f;
    if (dx >= 0) fx = 1 - fx;
    if (dz >= 0) fz = 1 - fz;
    float g0x = signx, g0z = dz / std::fabs(dx), g1x = dx / std::fabs(dz), g1z = signz;
    float ax = g0x * fx, az = g0z * fx, bx = g1x * fz, bz = g1z * fz;
    float gA = std::sqrt(g0x * g0x + g0z * g0z), gB = std::sqrt(g1x * g1x + g1z * g1z);
    float sA = std::sqrt(ax * ax + az * az), sB = std::sqrt(bx * bx + bz * bz);
    rlevox::SkipLine sl;
    sl.init(dx, dz, vpx, vpz);
    const int fix_x = dx >= 0 ? 0 : -1, fix_z = dz >= 0 ? 0 : -1;
    float px = 0, pz = 0, d = 0;
    int ib = 0, mip = 0;
    // levels of mipd, mipd, mipd steps, at twice the stride each
    for (int level = 0; level < 3 && steps < budget; level++) {
      const int n = mipd;
      std::vector<Step> s((size_t)n + 1);
      for (int k = 0;; k++) {
        s[k] = Step{px, pz, d, sA, sB, ax, az, bx, bz, ib};
        if (k == n) break;
        if (sB < sA) {
          d = sB, sB += gB, px = bx, pz = bz, bx += g1x, bz += g1z, ib = 1;
        } else {
          d = sA, sA += gA, px = ax, pz = az, ax += g0x, az += g0z, ib = 0;
        }
      }
      steps += n;
      const int sh = mip + rlevox::kSkipBlockLog;
      for (int base = 0; base < n; base += 1 + (int)(600 * u(rng))) {
        const Step& b0 = s[base];
        const float r = 1.0f / (gA + gB);
        rlevox::SkipBase b = rlevox::SkipBase::of(
            sl, b0.px, b0.pz, b0.d, b0.sA, b0.sB, gA, gB, b0.ib ? b0.sA : b0.sB, b0.ib ? b0.ax : b0.bx,
            b0.ib ? b0.az : b0.bz, r);
        if (WALK_RANGE_PLANT) b.ox = b.oz = NAN;
        const int ahead = rng() % 2 ? 0 : (int)(kReach * u(rng));
        for (int g = 0; g < 64; g += 1 + (int)(rng() % 8)) {
          const int t0 = ahead + g * rlevox::kSkipSteps, t1 = t0 + rlevox::kSkipSteps;
          if (base + t1 > n) break;
          const rlevox::SkipRange q = rlevox::skip_range(sl, b, sh, t0, t1);
          if (!q.sane) continue;
          groups++;
          // two blocks a side: what the bound looks up (else the level's top)
          const bool fits = q.cx1 - q.cx0 <= 1 && q.cz1 - q.cz0 <= 1;
          near += fits;
          for (int t = t0; t < t1; t++) {
            const Step& p = s[base + t];
            if (p.d < q.lo) below++;
            if (s[base + t + 1].d > q.hi) above++;
            const int vx = (int)(vpx + p.px) + (p.ib ? 0 : fix_x);
            const int vz = (int)(vpz + p.pz) + (p.ib ? fix_z : 0);
            const int cx = vx >> sh, cz = vz >> sh;
            if (fits && (cx < q.cx0 || cx > q.cx1 || cz < q.cz0 || cz > q.cz1)) outside++;
          }
        }
      }
      mip++;
      g0x *= 2, g0z *= 2, g1x *= 2, g1z *= 2, gA *= 2, gB *= 2;
    }
  }
  std::printf("steps %ld, groups %ld, of two blocks a side %ld, below lo %ld, above hi %ld, outside %ld\n",
              steps, groups, near, below, above, outside);
  return 0;
}
