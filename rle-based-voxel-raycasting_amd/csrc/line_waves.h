// Wavefronts per ray line of a single render (plain C++ so a host check can
// run the same code).
#pragma once

namespace rlevox {

// Widest ray-buffer line (screen width) up to which the automatic choice
// walks each line with several wavefronts, one on the DDA and one drawing.
// Whole frames over a flythrough of the 4096^2 terrain, us with two
// wavefronts / one: 1920x1080 133 / 150, 2560x1440 161 / 170, 3200x1800
// 221 / 198, 3840x2160 252 / 225.
constexpr int kTwoWaveMaxWidth = 2560;
// Lines up to which a line of that width is walked by three wavefronts: the
// lines whose LDS the compute units hold at once (line_lds a line, rounded up
// to the unit that LDS is given out in).  With them all resident a frame takes
// as long as its longest line, which three wavefronts walk faster; beyond,
// lines wait for LDS.  On 256 compute units of 160 KB that is 1792 lines with
// a run cache of 24 words, 1536 with 40 and 1280 with 56 (us per frame, three
// / two: 320x240, 441 lines, 83 / 91; 640x480, 882-1125 lines, 79 / 88;
// 1366x768, 1532-1654 lines, 98 / 99; 1280x720, 1626-1891 lines, 88 / 94;
// 1920x1080, 2048-3050 lines, 170 / 132.  Three over two, the raycast alone,
// 1024x768 to 1600x900, 1408-1536 / 1536-1664 / 1664-1792 lines: with 24 words
// 0.94 / 0.98 / 0.95, with 40 0.93 / 0.97 / 1.02, with 56 1.04 / 1.15 / 1.16).
constexpr int kLdsUnit = 1280;

inline int three_wave_max_lines(int num_cus, int lds_per_cu, int line_lds) {
  return num_cus * (lds_per_cu / ((line_lds + kLdsUnit - 1) / kLdsUnit * kLdsUnit));
}

// By the tuning's waves_per_block: 1 is one, 2 and 3 are two, 4 is three up to
// three_max lines and two beyond, 0 as 4 up to that width and one beyond.
inline int line_waves(int waves_per_block, int lines, int rs, int three_max) {
  const bool wide = rs > kTwoWaveMaxWidth;
  if (waves_per_block == 1 || (waves_per_block == 0 && wide)) return 1;
  if (waves_per_block == 0 || waves_per_block == 4) return !wide && lines <= three_max ? 3 : 2;
  return 2;
}

}  // namespace rlevox
