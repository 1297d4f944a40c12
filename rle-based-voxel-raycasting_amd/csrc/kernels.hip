// HIP kernels for gfx950: plain per-view raycast, compose, gap-fill, and the
// batched persistent raycast over a device work queue.
#include <hip/hip_runtime.h>

#include "device.h"
#include "kernels.h"
#include "wave_line.h"

namespace rlevox {

// ------------------------------------------------------------------ plain
// One lane per ray line (cudaRender, Cuda_Main.cu:150-181); each lane keeps
// its line bitmap in LDS, word w of lane l at lds[w*blockDim + l] so lanes
// reading the same word index hit distinct banks.
template <bool COUNT>
__global__ __launch_bounds__(256) void k_raycast_plain(SceneDev sc, rlevox_raymap rm,
                                                       uint32_t* __restrict__ raybuf,
                                                       int32_t* __restrict__ clip,
                                                       unsigned long long* counts) {
  extern __shared__ uint32_t lds[];
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= rm.map_line_count) return;
  const LineBits bits{lds + threadIdx.x, (int)blockDim.x};
  render_line<COUNT>(x, sc, rm, raybuf + (size_t)x * (size_t)rm.rs, clip + 2 * x, bits, counts);
}

// Blocks take the ray lines from the last to the first: the lines of the
// last segments of the ray map start first, which for views looking down
// puts the long lines (those reaching the sky, walked to the far distance)
// at the head of the launch.  Measured 1-6% faster than index order on
// 1080p and 4K flythroughs and random views, equal on grazing views.
//
// One wavefront (= one block) per ray line.  Registers are capped for five
// wavefronts per SIMD (5120 resident lines on 256 CUs), four with the
// lane-parallel element replay (PAR), whose walk would spill.  It pays where
// columns hold many runs: four 4K frames over terrain of 5.9 runs a column
// 926 us with it, 905 without; four grazing ones over 7.6 runs 820 and 850.
// Without it the walk's constants stay in registers (read again, a product of
// each chunk's projection spills: 976 against 963 us).
template <bool COUNT, bool PAR, int RC>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(PAR ? 4 : 5))) void k_raycast_wave(SceneDev sc, rlevox_raymap rm,
                                                     uint32_t* __restrict__ raybuf,
                                                     int32_t* __restrict__ clip,
                                                     unsigned long long* counts) {
  __shared__ uint4 rcache[64 * RC / 8];
  __shared__ int sweep[64 + kLineConstWords];
  __shared__ __align__(16) float dda[kDdaLds];
  extern __shared__ uint32_t lds[];
  if ((int)blockIdx.x >= rm.map_line_count) return;
  const int x = rm.map_line_count - 1 - (int)blockIdx.x;  // last line first
  render_line_wave<COUNT, 1, PAR, RC, !PAR>(x, sc, rm, raybuf + (size_t)x * (size_t)rm.rs,
                                           clip + 2 * x, lds, dda,
                                           (lds_u16*)rcache, sweep, counts);
}

// Two wavefronts (= one block) per ray line: wavefront 0 walks the DDA and
// gathers the pointer map, wavefront 1 projects, caches and draws.  Six
// wavefronts per SIMD (80 registers): it takes 77 as it is, 82 to 84 with the
// line's constants held across the walk.
template <int RC>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(6))) void k_raycast_wave2(SceneDev sc, rlevox_raymap rm,
                                                       uint32_t* __restrict__ raybuf,
                                                       int32_t* __restrict__ clip) {
  __shared__ uint4 rcache[64 * RC / 8];
  __shared__ int sweep[64 + kLineConstWords];
  __shared__ __align__(16) float dda[kDdaLds];
  __shared__ ChunkRing ring;
  extern __shared__ uint32_t lds[];
  if ((int)blockIdx.x >= rm.map_line_count) return;
  const int x = rm.map_line_count - 1 - (int)blockIdx.x;  // last line first
  render_line_wave<false, 2, true, RC>(x, sc, rm, raybuf + (size_t)x * (size_t)rm.rs,
                                          clip + 2 * x, lds, dda,
                                          (lds_u16*)rcache, sweep, nullptr,
                                          &ring);
}

// Three wavefronts per ray line: one walks, one projects and fetches the
// columns, one draws.  A frame of few lines takes as long as its longest one
// (320x240: 45 chunks at 3.7 K cycles), and that line's round was the longer
// of its walk (2.6 K cycles) and its step (1.4 K to prepare, 1.4 K to draw).
template <int RC>
__global__ __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(5))) void k_raycast_wave3(SceneDev sc, rlevox_raymap rm,
                                                       uint32_t* __restrict__ raybuf,
                                                       int32_t* __restrict__ clip) {
  __shared__ uint4 rcache[kPrepSlots * 64 * RC / 8];
  __shared__ int sweep[64 + kLineConstWords];
  __shared__ __align__(16) float dda[kDdaLds];
  __shared__ LineRings rings;
  extern __shared__ uint32_t lds[];
  if ((int)blockIdx.x >= rm.map_line_count) return;
  const int x = rm.map_line_count - 1 - (int)blockIdx.x;  // last line first
  render_line_wave<false, 3, true, RC>(x, sc, rm, raybuf + (size_t)x * (size_t)rm.rs,
                                          clip + 2 * x, lds, dda,
                                          (lds_u16*)rcache, sweep, nullptr,
                                          nullptr, &rings);
}

int raycast_wave3_lds(int run_cache, int rs) {
  const int rc = run_cache ? run_cache : kRunCacheDefault;
  return kPrepSlots * 64 * rc * 2 + (64 + kLineConstWords) * 4 + kDdaLds * 4 + (int)sizeof(LineRings) +
         bitmap_words(rs) * 4;
}

// Tiles of 32x8 pixels, one pixel per thread: a tile's quotients and its loads
// are one chain, hidden by other workgroups (64x16 tiles of four pixels per
// thread: 640x480 5.0 against 4.9 us, 1366x768 7.4 against 6.5).
__global__ __launch_bounds__(256) void k_compose(rlevox_raymap rm, const uint32_t* __restrict__ raybuf,
                                                 const int32_t* __restrict__ clip,
                                                 uint16_t* __restrict__ col,
                                                 int32_t* __restrict__ dep) {
  __shared__ ComposeTile<32, 8> ct;
  const int x0 = blockIdx.x * 32, y0 = blockIdx.y * 8;
  compose_tile_stage(rm, x0, y0, ct);
  __syncthreads();
  compose_tile(rm, raybuf, clip, x0, y0, ct, [&](int px, int row, uint16_t c, int32_t d) {
    col[(size_t)row * rm.W + px] = c;
    dep[(size_t)row * rm.W + px] = d;
  });
}

// Tile of block b of a grid of n tiles, gx per row: blocks are dispatched
// round robin over the 8 XCDs, and each XCD takes groups of 32
// pixel rows, the groups dealt round robin, so the border rows that the
// tiles of a group share come through the same L2 (1080p gap-fill HBM fetch
// 99 -> 27 MB at the same speed; contiguous eighths of the image per XCD
// fetched 15 MB but ran 2% slower, the eighths differing in work).
template <int ROWS>
__device__ inline int xcd_tile(int b, int n, int gx) {
  const int G = 32 / ROWS * gx, full = n / (8 * G) * (8 * G);
  if (b >= full) return b;  // the last partial round in dispatch order
  const int x = b & 7, k = b >> 3;
  return ((k / G) * 8 + x) * G + (k % G);
}

template <int ROWS>
__global__ __launch_bounds__(256) void k_gapfill(int W, int H, const uint16_t* __restrict__ cin,
                                                 const int32_t* __restrict__ dep,
                                                 uint16_t* __restrict__ cout) {
  __shared__ GapTile<ROWS> tile;
  const int gx = (int)gridDim.x;
  const int t = xcd_tile<ROWS>((int)(blockIdx.y * gridDim.x + blockIdx.x),
                               (int)(gridDim.x * gridDim.y), gx);
  const int ty = t / gx;
  gapfill_tile(W, H, cin, dep, cout, (t - ty * gx) * 64, ty * ROWS, tile);
}

template <int RC>
static void launch_waves(const SceneDev& sc, const rlevox_raymap& rm, uint32_t* raybuf,
                         int32_t* clip, int waves, bool par, hipStream_t s) {
  const size_t lds = (size_t)bitmap_words(rm.rs) * sizeof(uint32_t);
  if (waves == 3)
    hipLaunchKernelGGL(k_raycast_wave3<RC>, dim3(rm.map_line_count), dim3(192), lds, s, sc, rm,
                       raybuf, clip);
  else if (waves == 2)
    hipLaunchKernelGGL(k_raycast_wave2<RC>, dim3(rm.map_line_count), dim3(128), lds, s, sc, rm,
                       raybuf, clip);
  else if (par)
    hipLaunchKernelGGL((k_raycast_wave<false, true, RC>), dim3(rm.map_line_count), dim3(64), lds, s,
                       sc, rm, raybuf, clip, nullptr);
  else
    hipLaunchKernelGGL((k_raycast_wave<false, false, RC>), dim3(rm.map_line_count), dim3(64), lds, s,
                       sc, rm, raybuf, clip, nullptr);
}

hipError_t launch_raycast_plain(const SceneDev& sc, const rlevox_raymap& rm, uint32_t* raybuf,
                                int32_t* clip, int block, int run_cache, bool par, hipStream_t s,
                                unsigned long long* counts) {
  const int lines = rm.map_line_count;
  if (lines <= 0) return hipSuccess;
  if (block >= 1 && block <= 3) {  // wavefront kernels
    if (run_cache == 0) run_cache = kRunCacheDefault;
    if (counts) {  // counting walks with one wavefront and the default run cache
      const size_t lds = (size_t)bitmap_words(rm.rs) * sizeof(uint32_t);
      hipLaunchKernelGGL((k_raycast_wave<true, true, kRunCache>), dim3(lines), dim3(64), lds, s, sc, rm,
                         raybuf, clip, counts);
    } else if (run_cache == 24) {
      launch_waves<24>(sc, rm, raybuf, clip, block, par, s);
    } else if (run_cache == 56) {
      launch_waves<56>(sc, rm, raybuf, clip, block, par, s);
    } else {
      launch_waves<kRunCache>(sc, rm, raybuf, clip, block, par, s);
    }
    return hipGetLastError();
  }
  const int grid = (lines + block - 1) / block;
  const size_t lds = (size_t)bitmap_words(rm.rs) * block * sizeof(uint32_t);
  if (counts)
    hipLaunchKernelGGL(k_raycast_plain<true>, dim3(grid), dim3(block), lds, s, sc, rm, raybuf,
                       clip, counts);
  else
    hipLaunchKernelGGL(k_raycast_plain<false>, dim3(grid), dim3(block), lds, s, sc, rm, raybuf,
                       clip, counts);
  return hipGetLastError();
}

// The world row of each column's first drawn run (the element walk of
// Cuda_Render.h:511-524 up to the first element with drawn voxels), reduced
// to the minimum over one block of columns per workgroup and over the level.
// Columns are validated at upload, so the walk stays inside the slab array.
constexpr int kTopSide = 1 << kSkipBlockLog;
__global__ __launch_bounds__(kTopSide * kTopSide) void k_column_tops(
    const uint2* __restrict__ map, const uint16_t* __restrict__ slabs, int shift, int level, int sx,
    int sz, int32_t empty, int32_t* __restrict__ tops, int32_t* out) {
  __shared__ int32_t wave_best[kTopSide * kTopSide / 64];
  const int nx = skip_blocks(sx);
  const int bz = (int)blockIdx.x / nx, bx = (int)blockIdx.x - bz * nx;
  const int x = bx * kTopSide + (threadIdx.x & (kTopSide - 1));
  const int z = bz * kTopSide + (threadIdx.x >> kSkipBlockLog);
  int best = INT32_MAX;
  if (x < sx && z < sz) {
    const uint2 e = map[(size_t)z * sx + x];
    const uint32_t n = e.y & 0xffffu;
    const uint16_t* runs = slabs + 2 + ((uint64_t)e.x << shift);
    uint32_t w = e.y >> 16;
    int y = 0;
    for (uint32_t k = 0; k < n; k++) {
      if (k > 0) w = runs[k];
      y += (int)(w & 1023u) << level;
      if (w >> 10) {
        best = y;
        break;
      }
    }
  }
  for (int o = 32; o > 0; o >>= 1) best = min(best, __shfl_xor(best, o));
  if ((threadIdx.x & 63) == 0) wave_best[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < kTopSide * kTopSide / 64; i++) best = min(best, wave_best[i]);
    tops[blockIdx.x] = min(best, empty);
    if (best != INT32_MAX) atomicMin(out, best);
  }
}

hipError_t launch_column_tops(const MipDev& m, int level, int32_t empty, int32_t* tops,
                              int32_t* out, hipStream_t s) {
  const int64_t blocks = (int64_t)skip_blocks(m.sx) * skip_blocks(m.sz);
  hipLaunchKernelGGL(k_column_tops, dim3((unsigned)blocks), dim3(kTopSide * kTopSide), 0, s, m.map,
                     m.slabs, m.shift, level, m.sx, m.sz, empty, tops, out);
  return hipGetLastError();
}

template <int ROWS>
static void launch_gapfill_rows(int W, int H, const uint16_t* cin, const int32_t* dep,
                                uint16_t* cout, hipStream_t s) {
  hipLaunchKernelGGL(k_gapfill<ROWS>, dim3((W + 63) / 64, (H + ROWS - 1) / ROWS), dim3(256), 0, s, W,
                     H, cin, dep, cout);
}

hipError_t launch_compose(const rlevox_raymap& rm, const uint32_t* raybuf, const int32_t* clip,
                          uint16_t* col, int32_t* dep, hipStream_t s) {
  hipLaunchKernelGGL(k_compose, dim3((rm.W + 31) / 32, (rm.H + 7) / 8), dim3(256), 0, s, rm, raybuf,
                     clip, col, dep);
  return hipGetLastError();
}

hipError_t launch_gapfill(int W, int H, const uint16_t* cin, const int32_t* dep, uint16_t* cout,
                          hipStream_t s) {
  // Taller tiles stage less border per pixel (64x4: 9.6 staged pixels for
  // each of its own, 64x8: 5.5, 64x16: 3.4) but leave fewer workgroups, and a
  // tile's staging and taps overlap only with other tiles.  Measured in us,
  // 4 / 8 / 16 rows: 640x480 4.8 / 5.5 / 7.7, 1280x720 9.5 / 8.9 / 9.8,
  // 1366x768 16.5 / 17.0 / 19.4, 1920x1080 13.7 / 12.3 / 13.2, 3840x2160
  // 52.8 / 43.6 / 42.6.
  const int64_t pixels = (int64_t)W * H;
  if (pixels >= 4 << 20)
    launch_gapfill_rows<16>(W, H, cin, dep, cout, s);
  else if (pixels >= 3 << 18)
    launch_gapfill_rows<8>(W, H, cin, dep, cout, s);
  else
    launch_gapfill_rows<4>(W, H, cin, dep, cout, s);
  return hipGetLastError();
}

}  // namespace rlevox

namespace rlevox {

// Fills count uint32 words; used instead of hipMemset so the same code can
// be captured into a graph.
__global__ __launch_bounds__(256) void k_fill_u32(uint32_t* __restrict__ p, uint32_t v, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

// Copies n 16-byte words: a plain streaming kernel of known traffic, used to
// calibrate hardware byte counters against an exact read+write volume.
__global__ __launch_bounds__(256) void k_copy_u128(uint4* __restrict__ dst,
                                                  const uint4* __restrict__ src, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    dst[i] = src[i];
}

hipError_t launch_copy_u128(void* dst, const void* src, uint64_t n16, hipStream_t s) {
  if (n16 == 0) return hipSuccess;
  uint64_t blocks = (n16 + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_copy_u128, dim3((unsigned)blocks), dim3(256), 0, s, (uint4*)dst,
                     (const uint4*)src, n16);
  return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, uint32_t value, uint64_t count, hipStream_t s) {
  if (count == 0) return hipSuccess;
  uint64_t blocks = (count + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, s, p, value, count);
  return hipGetLastError();
}

}  // namespace rlevox
