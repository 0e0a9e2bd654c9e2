// jne_segments.h -- the mixed pass's segments of a walk and the rule by which a
// batch of few waves is split over them.  Plain C++: the host test of the rule
// builds it without HIP.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace jne {

constexpr int kSegSteps = 64;  // steps per FP64 segment and per RNG round
constexpr uint32_t segment_count(uint32_t T) { return (T + kSegSteps - 1) / kSegSteps; }

// Split batches: a segment's Gram as FP32 values, as the MFMA leaves them, and
// its FP64 eps, in memory: per wave and segment kSegFloats floats
//   c columns: rows 0..23 (accumulator v of half h of column j at v 24 + 12 h + j),
//   z columns: rows 12..23 at 288 + 12 (row - 12) + j,
//   rows 24..26 at 432 + 24 (row - 24) + j of the c, + 12 + j of the z columns,
// then 12 doubles.
constexpr int kSegFloats = 504;
constexpr int kSegDoubles = kSegFloats / 2 + 12;
constexpr int kSplitSegs = 4;  // segments per wave: a carry period (4 CALLS is a multiple of 64)
constexpr uint32_t split_chunks(uint32_t T) { return (segment_count(T) + kSplitSegs - 1) / kSplitSegs; }

// fp16x2 batches by seed whose waves leave the GPU mostly idle are split over
// their walks' segments: a segment then also writes and reads its 2.1 KB, as
// long as its share of a full GPU's time, so the line lies where the two forms
// meet (waves; in turn / split, ms): dim 12, T = 1,000: 400 0.039 / 0.026, 800
// 0.040 / 0.043; T = 10^4: 1 0.307 / 0.06, 400 0.325 / 0.161, 800 0.330 / 0.267,
// 1,200 0.387 / 0.417; dim 7, T = 400: 400 0.0196 / 0.0188, 800 0.0204 / 0.0218.
#ifndef JNE_MFMA_SPLIT_WAVES
#define JNE_MFMA_SPLIT_WAVES 700
#endif
// The segments' sums grow with T (700 waves: 0.23 GB at T = 10^4, 23 GB at T =
// 10^6) and stay with the context: a batch that needs more than this is not
// split.  700 waves reach it at T = 11,585, one at T = 8.13 million.
constexpr size_t kMaxSplitBytes = size_t(1) << 28;
// A launch's chunks are its grid's y dimension, of which 65,535 are counted on.
static_assert(kMaxSplitBytes / sizeof(double) / kSegDoubles / kSplitSegs < 65535, "one wave's chunks fit the grid");

// Doubles of the segments' sums of a batch of `waves` waves (0: not split).
constexpr size_t segment_split_doubles(uint32_t waves, uint32_t T) {
  if (waves > JNE_MFMA_SPLIT_WAVES || segment_count(T) <= (uint32_t)kSplitSegs) return 0;
  const size_t doubles = (size_t)waves * segment_count(T) * kSegDoubles;
  return doubles <= kMaxSplitBytes / sizeof(double) ? doubles : 0;
}

}  // namespace jne
