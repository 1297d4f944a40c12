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
// lines whose LDS (21 KB each) the 256 compute units hold at once.  With
// them all resident a frame takes as long as its longest line, which three
// wavefronts walk faster; beyond, lines wait for LDS (us per frame, three
// / two: 320x240, 441 lines, 83 / 91; 640x480, 882-1125 lines, 79 / 88;
// 1366x768, 1532-1654 lines, 98 / 99; 1280x720, 1626-1891 lines, 88 / 94;
// 1920x1080, 2048-3050 lines, 170 / 132).
constexpr int kThreeWaveMaxLines = 1792;

// By the tuning's waves_per_block: 1 is one, 2 and 3 are two, 4 is three up to
// those lines and two beyond, 0 as 4 up to that width and one beyond.
inline int line_waves(int waves_per_block, int lines, int rs) {
  const bool wide = rs > kTwoWaveMaxWidth;
  if (waves_per_block == 1 || (waves_per_block == 0 && wide)) return 1;
  if (waves_per_block == 0 || waves_per_block == 4)
    return !wide && lines <= kThreeWaveMaxLines ? 3 : 2;
  return 2;
}

}  // namespace rlevox
