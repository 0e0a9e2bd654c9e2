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
// their walks' segments.  A segment then also writes and reads its 2.1 KB, as
// long as its share of a full GPU's time, and the launch has a second kernel, the
// time of some segments: the line lies where the two forms meet, at fewer waves
// the fewer segments a walk has.  Split over in turn, whole calls of dim 12: 5
// segments 100 waves 1.00, 700 1.03; 8 segments 400 0.99, 700 1.05; 16 segments 600
// 0.96, 800 1.03; 157 segments 1 0.33, 700 0.76, 900 0.97, 1,000 1.04; of dim 5: 5
// segments 100 1.00, 700 1.04; 8 segments 700 0.98; 157 segments 1,000 0.80.
#ifndef JNE_MFMA_SPLIT_WAVES
#define JNE_MFMA_SPLIT_WAVES 950u
#define JNE_MFMA_SPLIT_WAVES_LESS 4000u
#endif
constexpr uint32_t split_waves(uint32_t segments) {
  const uint32_t less = JNE_MFMA_SPLIT_WAVES_LESS / segments;
  return segments > (uint32_t)kSplitSegs && JNE_MFMA_SPLIT_WAVES > less ? JNE_MFMA_SPLIT_WAVES - less : 0;
}

// The segments' sums grow with T (700 waves: 0.23 GB at T = 10^4, 23 GB at T =
// 10^6) and stay with the context: a batch that needs more than this is not
// split.  700 waves reach it at T = 11,585, one at T = 8.13 million.
constexpr size_t kMaxSplitBytes = size_t(1) << 28;
// A launch's chunks are its grid's y dimension, of which 65,535 are counted on.
static_assert(kMaxSplitBytes / sizeof(double) / kSegDoubles / kSplitSegs < 65535, "one wave's chunks fit the grid");

// Doubles of the segments' sums of a batch of `waves` waves (0: not split).
constexpr size_t segment_split_doubles(uint32_t waves, uint32_t T) {
  if (waves > split_waves(segment_count(T))) return 0;
  const size_t doubles = (size_t)waves * segment_count(T) * kSegDoubles;
  return doubles <= kMaxSplitBytes / sizeof(double) ? doubles : 0;
}

}  // namespace jne
