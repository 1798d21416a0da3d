// kf_icp_grid.hpp — blocks and pixels of the tracking kernels by image size (host side).
#pragma once

namespace kf {

constexpr int kStepThreads = 512;  // tracking step: 8 waves per block

// Pixels of a tracking step's 512-thread block by the level's size, so that a block per CU
// (256) covers the level and no SIMD has more pixels than it must: half a block's waves
// take one pixel per thread up to 65,536 pixels (level 2 of 640x480: 75 blocks, one wave
// per SIMD), all of them up to 131,072 (level 1: 150), two and a half pixels per thread up
// to 327,680 (level 0: 240), three beyond (the fewest slots; a step's block sums them all;
// from 393,217 pixels on some CUs hold two blocks: 800x600 10/5/4 iterations 177 us, plain
// 168, with room for one 216 and 212).
// A step inside the kernel: levels 2 and 1 of 640x480 4.0 us, level 0 6.3 us (7.75 with
// 200 blocks of three pixels a thread and the per-thread sums, 5.6 below); 1024-thread
// blocks 5.9 us at level 0 but 4.5 below.
constexpr int kShapes = 4;
constexpr int kShapePixels[kShapes] = {kStepThreads / 2, kStepThreads, 5 * kStepThreads / 2, 3 * kStepThreads};

inline int step_shape(int pixels) {
  int k = 0;
  while (k + 1 < kShapes && pixels > 256 * kShapePixels[k]) ++k;
  return k;
}

// Blocks of a step (one slot each); `most`: the tracker's slots.
inline int step_blocks(int pixels, int most) {
  const int p = kShapePixels[step_shape(pixels)], b = pixels / p + (pixels % p != 0);
  return b < most ? b : most;
}

// Blocks that the single-launch form takes for a level.  The grid barrier needs all of a
// call's blocks on the chip at once, one to a CU, so that calls on several streams have to
// share the CUs.  Up to 196,608 pixels at the finest level two or more calls fit 256 CUs
// with a block per three pixels a thread there (one pixel at the others), and a block makes
// several slots: 320x240 takes 50 blocks, not its step's 150.  10/5/4 iterations: 319x241
// 169 us (a block per slot 156), 480x360 202 (175).  Beyond that a second such call would
// not fit, and a block per slot is the faster: 640x480 180 us (200 blocks 211).
inline int chain_blocks(int pixels, int level, int most) {
  const int p = kStepThreads * (level == 0 ? 3 : 1), few = pixels / p + (pixels % p != 0);
  const int own = step_blocks(pixels, most);
  return few <= 128 && few < own ? few : own;
}

}  // namespace kf
