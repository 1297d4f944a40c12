// Checks the skipped stretches of a line's walk (csrc/walk_skip.h) against
// the oracle's full walk (Cuda_Render.h:96-736 restated in
// oracle/oracle.cpp): the oracle is included with hooks that evaluate, before
// every DDA step, the bound of the group the step belongs to, from a window
// begun as the kernels begin theirs (a mip switch or kSkipWindow steps after
// the last).  A step that still draws or moves the line's window although its
// group was hidden is a violation.  Seeded terrains of two sizes (one smaller
// than a block at its last level), random poses (also at
// negative coordinates, and with headings along and between the axes) with eye heights from -10 to
// 2000 voxels above the surface, pitches from -1.3 to 1.45 rad, resolutions
// from 160x120 to 1280x720 and mip distances from 40 to 4096.  Built and run
// by tests/test_walk_skip.py; WALK_SKIP_PLANT=n lowers every block's top by n
// rows, a mistake the check must catch.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#define RLEVOX_HD
#include "../../rle-based-voxel-raycasting_amd/csrc/walk_skip.h"

#ifndef WALK_SKIP_PLANT
#define WALK_SKIP_PLANT 0
#endif

struct Trace {
  rlevox::WalkEnd we;
  rlevox::SkipLine line;
  rlevox::SkipBase base;
  long base_step, group, steps, hidden, wrong, chunks, chunk_end, ended;
  float gd0, gd1, bound;
  bool hide;
};
static Trace* g_tr = nullptr;
static int g_top[16];
static int g_sx[16], g_sz[16];
static std::vector<int32_t> g_blocks[16];
static int g_sy = 0;

static void step_hook(Trace& t, long step, float px, float pz, float dnow, float s0, float s1, float g0,
                      float g1, int mip, int ymin, int ymax) {
  if (t.base_step < 0 || t.gd0 != g0 || t.gd1 != g1 || step - t.base_step >= rlevox::kSkipWindow) {
    const float r = 1.0f / (g0 + g1);
    t.base = {px, pz, dnow, s0, s1, g0, g1, (s1 - s0 + g0) * r, g1 * r};
    t.base_step = step;
    t.gd0 = g0;
    t.gd1 = g1;
    t.group = -1;
  }
  const long g = (step - t.base_step) / rlevox::kSkipSteps;
  if (g != t.group) {
    t.group = g;
    const rlevox::SkipLevel v{mip, g_sx[mip], g_sz[mip], g_blocks[mip].data(), g_top[mip]};
    t.bound = rlevox::skip_bound(t.we, t.line, t.base, v, g_sy, (int)g * rlevox::kSkipSteps,
                                 ((int)g + 1) * rlevox::kSkipSteps);
  }
  t.hide = rlevox::skip_hidden(t.bound, ymin);
  if (t.we.done(dnow, ymin, g_top[mip], g_sy)) t.ended = 1;
  if (t.ended || ymin >= ymax) return;
  t.steps++;
  t.hidden += t.hide ? 1 : 0;
  if (step >= t.chunk_end && !t.hide) {
    t.chunks++;
    t.chunk_end = step + 64;
  }
}

#define ORC_HOOK_LINE_BEGIN                                                                  \
  Trace& tr_ = g_tr[x];                                                                      \
  tr_.we.init(cos_x, sin_x, res_x2_mul_reverse, ray_x, ray_z, vertical, vpy, res_y2);        \
  tr_.line.init(dx, dy, vpx, vpz);
#define ORC_HOOK_STEP                                                                        \
  step_hook(tr_, (long)c_steps, pos_x, pos_y, dds_dist_now, dds_dist0, dds_dist1,           \
            grad_dist0, grad_dist1, mip_lvl, y_clip_min, y_clip_max);
#define ORC_HOOK_ACT                                                                         \
  if (tr_.hide) tr_.wrong++;
#define ORC_HOOK_LINE_END
#include "../../oracle/oracle.cpp"

// Highest run top (world row) of each level and all coarser ones.
static void level_tops(const std::vector<rlevox_mip>& mips) {
  int t = mips[0].sy;
  for (int m = (int)mips.size() - 1; m >= 0; m--) {
    const rlevox_mip& mp = mips[m];
    const int nx = rlevox::skip_blocks(mp.sx), nz = rlevox::skip_blocks(mp.sz);
    g_sx[m] = mp.sx;
    g_sz[m] = mp.sz;
    g_blocks[m].assign((size_t)nx * nz, mips[0].sy);
    for (int64_t c = 0; c < (int64_t)mp.sx * mp.sz; c++) {
      const uint32_t ofs = mp.ptrmap[2 * c], lf = mp.ptrmap[2 * c + 1];
      const uint16_t* runs = mp.slabs + ((uint64_t)ofs << mp.offset_shift) + 2;
      uint32_t w = lf >> 16;
      int y = 0;
      for (uint32_t k = 0; k < (lf & 0xffffu); k++) {
        if (k > 0) w = runs[k];
        y += (int)(w & 1023u) << m;
        if (w >> 10) {
          if (y < t) t = y;
          const int bx = (int)(c % mp.sx) >> rlevox::kSkipBlockLog, bz = (int)(c / mp.sx) >> rlevox::kSkipBlockLog;
          int32_t& bt = g_blocks[m][(size_t)bz * nx + bx];
          if (y + WALK_SKIP_PLANT < bt) bt = y + WALK_SKIP_PLANT;
          break;
        }
      }
    }
    g_top[m] = t;
  }
  g_sy = mips[0].sy;
}

static int surface_row(const rlevox_mip& m0, int x, int z) {
  const int64_t c = (int64_t)(z & (m0.sz - 1)) * m0.sx + (x & (m0.sx - 1));
  const uint32_t ofs = m0.ptrmap[2 * c];
  const uint16_t* col = m0.slabs + ((uint64_t)ofs << m0.offset_shift);
  int y = 0;
  for (int e = 0; e < col[0]; e++) {
    const uint16_t w = col[2 + e];
    y += w & 1023;
    if (w >> 10) return y;
  }
  return m0.sy;
}

int main(int argc, char** argv) {
  const int views = argc > 1 ? std::atoi(argv[1]) : 40;
  long violations = 0, steps = 0, hidden = 0, chunks = 0;
  const int big = argc > 2 ? std::atoi(argv[2]) : 0;
  const int sizes[][2] = {{160, 120}, {320, 240}, {640, 480}, {512, 512}, {1280, 720}};
  for (int scene = 0; scene < 2; scene++) {
    rlevox_gen_params gp{};
    gp.size_xz = scene == 0 ? (big ? big : 512) : 64;
    gp.size_y = scene == 0 ? (big ? 1024 : 256) : 64;
    gp.nmips = scene == 0 ? (big ? 6 : 4) : 3;
    gp.octaves = scene == 0 ? (big ? 8 : 6) : 4;
    gp.seed = 3 + scene;
    gp.persistence = 0.5f;
    gp.hmin = scene == 0 ? gp.size_y / 8 : 8;
    gp.hmax = scene == 0 ? gp.size_y - gp.size_y / 8 : 48;
    gp.cave_layers = 1.0f;
    gp.cave_max_layers = scene == 0 ? 31 : 8;
    rlevox_hscene* hs = nullptr;
    if (rlevox_gen_scene(&gp, &hs) != RLEVOX_OK) {
      std::printf("generator failed: %s\n", rlevox_last_error());
      return 1;
    }
    std::vector<rlevox_mip> mips(rlevox_hscene_nmips(hs));
    for (int i = 0; i < (int)mips.size(); i++) rlevox_hscene_mip(hs, i, &mips[i]);
    level_tops(mips);
    std::mt19937 rng(11 + scene);
    std::uniform_real_distribution<float> u(0.0f, 1.0f);
    for (int v = 0; v < views; v++) {
      const int W = sizes[v % 5][0], H = sizes[v % 5][1];
      const float x = u(rng) * gp.size_xz, z = u(rng) * gp.size_xz;
      const int kind = v % 4;
      const float alt = kind == 0 ? -10 + 30 * u(rng) : (kind == 1 ? 20 + 280 * u(rng) : 300 + 1700 * u(rng));
      float pitch = (v / 4) % 4 == 0 ? -1.3f + 1.29f * u(rng)
                    : (v / 4) % 4 == 1 ? 0.01f + 0.59f * u(rng)
                    : (v / 4) % 4 == 2 ? 0.6f + 0.85f * u(rng) : -0.1f + 0.2f * u(rng);
      if (std::fabs(pitch) < 0.01f) pitch = 0.01f;
      rlevox_pose p{};
      p.pos[0] = x + gp.size_xz * (v % 7 == 3 ? -3 : 1);
      p.pos[1] = alt - (float)surface_row(mips[0], (int)x, (int)z);
      p.pos[2] = z + gp.size_xz * (v % 7 == 3 || v % 7 == 5 ? -1 : 1);
      p.rot[0] = pitch;
      p.rot[1] = v % 6 == 2 ? 0.78539816f * (float)(int)(8 * u(rng)) : 6.2831853f * u(rng);
      rlevox_raymap rm;
      const int mipd[] = {0, 0, 40, 4096, 300};
      if (orc_raymap(&p, W, H, mipd[(v / 5) % 5], 0, &rm) != 0) continue;
      const int lines = rm.map_line_count;
      if (lines <= 0) continue;
      std::vector<Trace> tr(lines);
      for (Trace& t : tr) {
        t.base_step = -1;
        t.steps = t.hidden = t.wrong = t.chunks = t.chunk_end = t.ended = 0;
        t.gd0 = t.gd1 = 0;
        t.hide = false;
      }
      g_tr = tr.data();
      std::vector<uint32_t> raybuf((size_t)lines * rm.rs);
      std::vector<int32_t> clip((size_t)lines * 2);
      rlevox_counters ctr;
      orc_raycast(mips.data(), (int)mips.size(), &rm, raybuf.data(), clip.data(), &ctr, 0);
      for (const Trace& t : tr) {
        violations += t.wrong;
        steps += t.steps;
        hidden += t.hidden;
        chunks += t.chunks;
      }
    }
    rlevox_hscene_free(hs);
  }
  std::printf("steps %ld, hidden %ld, chunks of 64 walked %ld, violations %ld\n", steps, hidden, chunks,
              violations);
  return 0;
}
