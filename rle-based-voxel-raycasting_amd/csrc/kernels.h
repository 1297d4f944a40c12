// Host-side launchers of the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "device.h"

namespace rlevox {

// Default run-cache depth of the wavefront kernels, in words.  With the cache
// loaded straight into LDS the deeper ones save no time and hold LDS (us with
// 24 / 40 / 56: four 1080p frames 572 / 574 / -, four at 4K 1120 / 1125 /
// 1127, four grazing ones 969 / 971 / 976; 640x480 with three wavefronts 325 /
// 327 / -).
constexpr int kRunCacheDefault = 24;

// block: 1, 2 or 3 = wavefronts per line, else lanes per block of the
// lane-per-line kernel.  run_cache: LDS run-cache words of the wavefront
// kernels (24, 40 or 56; 0 = kRunCacheDefault; the counting variant always uses 40).  par:
// lane-parallel element replay where one wavefront walks a line.
hipError_t launch_raycast_plain(const SceneDev& sc, const rlevox_raymap& rm, uint32_t* raybuf,
                                int32_t* clip, int block, int run_cache, bool par, hipStream_t s,
                                unsigned long long* counts = nullptr);
// LDS bytes of a line of the kernel with three wavefronts per line.
int raycast_wave3_lds(int run_cache, int rs);
hipError_t launch_compose(const rlevox_raymap& rm, const uint32_t* raybuf, const int32_t* clip,
                          uint16_t* col, int32_t* dep, hipStream_t s);
// Smallest world row of a drawn run's top over the columns of each block of
// one level (walk_skip.h) into tops, `empty` where a block draws nothing, and
// over all of them atomically min-ed into *out (which must hold INT32_MAX or
// a larger row).
hipError_t launch_column_tops(const MipDev& m, int level, int32_t empty, int32_t* tops,
                              int32_t* out, hipStream_t s);
hipError_t launch_gapfill(int W, int H, const uint16_t* cin, const int32_t* dep, uint16_t* cout,
                          hipStream_t s);

}  // namespace rlevox
