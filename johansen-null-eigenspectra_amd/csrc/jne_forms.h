// jne_forms.h -- the shapes and forms of the FP64 moment passes: a walk's blocks of
// steps, lanes per walk and waves by dim, and the rules by which a launch is
// split.  Plain C++: the host tests of the rules build it without HIP.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

namespace jne {

// Steps per block: 240 (whole Philox calls and whole batches of every dim),
// and at most 16 blocks per walk.
constexpr uint32_t kBlockUnit = 240, kMaxBlocks = 16;
constexpr uint32_t block_steps(uint32_t T) {
  return kBlockUnit * ((T + kBlockUnit * kMaxBlocks - 1) / (kBlockUnit * kMaxBlocks));
}
constexpr uint32_t block_count(uint32_t T) { return (T + block_steps(T) - 1) / block_steps(T); }

// Per-dim shape of the FP64 moment kernel: lanes per walk (L) and target
// waves per SIMD (the register cap).  Measured on MI355X at T = 4,000 to 10^4.
// Dims with L = 1 run the register-only kernel (its own wave targets): at
// dim 7 its 105 sums fit two waves per SIMD (131,072 walks at T = 10^4: 11.0
// ms against 14.4 with seven lanes per walk); dim 8's 132 would not.
// Alternatives within 2%: (2, 3) at dim 8, (3, 2) at dim 9; slower: (2, 2) at
// dim 10 by 35%, (3, 2) at dims 11 and 12 by 8-11%.
struct Fp64Shape {
  int lanes, waves;
};
#ifndef JNE_FP64_SHAPES
#define JNE_FP64_SHAPES \
  {1, 2}, {1, 2}, {1, 2}, {1, 2}, {1, 2}, {1, 2}, {1, 2}, {2, 2}, {9, 4}, {5, 3}, {4, 2}, {4, 2}
#endif
constexpr Fp64Shape kFp64Shapes[12] = {JNE_FP64_SHAPES};
constexpr int lanes_for_dim(int d) { return kFp64Shapes[d - 1].lanes; }
constexpr int waves_for_dim(int d) { return kFp64Shapes[d - 1].waves; }

// target waves per SIMD of the register-only kernel by dim (the register cap:
// 512 / waves VGPRs per lane); it runs the dims whose shape has one lane per walk.
// One wave per SIMD reaches 88% of two waves' rate; 4 waves at dim 3 and 3 at
// dim 4 are 3 and 4% faster than 3 and 2.
#ifndef JNE_FP64_REG_WAVES
#define JNE_FP64_REG_WAVES 4, 4, 4, 3, 2, 2, 2, 2, 2, 2, 2, 2
#endif
constexpr int kFp64RegWaves[12] = {JNE_FP64_REG_WAVES};

// The forms of a moment launch.  One lane group per walk fills the GPU (the
// waves resident at the kernel's occupancy) in whole rounds only; the walks of
// the last, partial round are split over their blocks, as are all walks of a
// batch too small for one lane group each.  A split costs a second launch and
// the sums' way through memory, the time of some steps of the walk.  So the
// split walks run, with units = their blocks (a last, short one counted by its
// steps, a walk of one block as one),
//   one wave per block          up to wave (1 - wave_t / T) units,
//   one lane per component      up to row (1 - row_t / T) units (walk_moments_fp64, L = dim),
//   the dim's own lane group    above.
// The lines are fitted to the calls' times in every form at 18 lengths from 10
// to 10^4 steps and 15 batches from 1 to 100,000 walks of each dim: the chosen
// form is 0.2% slower than the fastest on average and 2 to 20% at its worst
// place by dim.  us of whole calls of model 4, in turn / own group / row / wave:
//   dim 3:  T = 100, 3,000 walks 46 / 54 / 38 / 34, 12,000 49 / 56 / 43 / 67,
//           22,000 52 / 60 / 58 / 103; T = 1,000, 2,000 walks 250 / 90 / 58 / 68
//   dim 7:  T = 240, 1,000 walks (in groups of seven lanes) 86 / 197 / 88 / 73,
//           2,000 87 / 195 / 87 / 85; T = 1,000, 500 walks 221 / 211 / 104 / 102, 22,000
//           403 / 345 / 350
//   dim 12: T = 120, 1,000 walks 149 / 160 / 133 / 127, 12,000 154 / 173 / 163; T =
//           1,000, 500 walks 462 / 233 / 164 / 170, 3,000 481 / 269 / 273
constexpr uint32_t kSimds = 1024;
struct FormLines {
  uint32_t wave, wave_t, row, row_t;
};
#ifndef JNE_FORM_LINES
#define JNE_FORM_LINES                                                                                     \
  {3500, 80, 0, 0}, {4000, 30, 32000, 80}, {5000, 10, 29000, 30}, {4000, 10, 48000, 20},                  \
      {5000, 10, 47000, 30}, {4500, 10, 40000, 10}, {2250, 40, 54000, 10}, {2250, 10, 24000, 10},          \
      {3000, 45, 0, 0}, {1500, 10, 11500, 30}, {1500, 10, 13000, 10}, {1250, 10, 11000, 10}
#endif
constexpr FormLines kFormLines[12] = {JNE_FORM_LINES};

enum class SplitForm { wave, row, own };
inline double split_units(uint32_t T, uint32_t m) { return m * std::max(1.0, (double)T / block_steps(T)); }
inline double wave_line(int d, uint32_t T) { return kFormLines[d - 1].wave * (1.0 - kFormLines[d - 1].wave_t / (double)T); }
inline double row_line(int d, uint32_t T) { return kFormLines[d - 1].row * (1.0 - kFormLines[d - 1].row_t / (double)T); }
inline SplitForm split_form(int d, uint32_t T, uint32_t m) {
  const double units = split_units(T, m);
  return units <= wave_line(d, T) ? SplitForm::wave : units <= row_line(d, T) ? SplitForm::row : SplitForm::own;
}
// m walks' part of what the row and wave forms take
inline double form_load(int d, uint32_t T, uint32_t m) {
  return split_units(T, m) / std::max(wave_line(d, T), row_line(d, T));
}

// Lanes per walk of a launch of n walks that is not split.  A lane per walk is
// the better form at dim 7 once a wave per SIMD is nearly full, and again when
// two are; fewer walks leave their chains exposed and run in groups of seven
// lanes (ms in one lane / seven): T = 1,000: 1 walk 0.712 / 0.209, 12,000 0.736 /
// 0.311, 55,000 0.796 / 0.700, 60,000 0.798 / 0.793, 65,000 0.802 / 0.871, 70,000
// 1.209 / 0.909, 100,000 1.236 / 1.212; T = 240: 55,000 0.219 / 0.218, 70,000 0.336
// / 0.278, 100,000 0.345 / 0.359.
inline int fp64_turn_lanes(int d, uint32_t n) {
  if (d == 7 && (n <= 55000 || (n > 64 * kSimds && n <= 95000))) return 7;
  return lanes_for_dim(d);
}

// Walks of n whose blocks one lane group takes in turn (the rest are split).
// Walks of one block have nothing to split but the lanes' work.  Whole rounds of
// the GPU's waves are taken in turn, and a rest of 90% of one with them.  For the
// others both times are estimated, in steps of a SIMD with all its waves (one
// alone reaches 0.84 of that rate): in turn, the deepest SIMD's waves of T steps
// (less what starts while the rounds before end); split, the rest's steps spread
// evenly, but no less than the deepest SIMD's whole blocks, and the sums' way
// through memory with their launches (130 steps behind whole rounds; else 40 of
// the short steps below dim 7, 35 at dim 7, 20 above).  The rates and steps are fitted to the
// times.  Split and in turn, ms: dim 6, T = 248 (blocks of 240 and 8 steps): 65,536
// walks 0.168 and 0.162, 170,000 0.409 and 0.365; T = 333: 65,536 0.179 and 0.207,
// 170,000 0.491 and 0.477; T = 1,000: 65,536 0.485 and 0.593, 170,000 1.324 and
// 1.399; dim 2, T = 248, 90,000 0.075 and 0.067; dim 9, T = 264, 12,000 0.143 and
// 0.135; dim 10, T = 241, 30,000 0.274 and 0.255; dim 12, T = 1,000, 16,384 0.368 and
// 0.481, 50,001 1.226 and 1.378; dim 7 (in turn in groups of seven lanes), T = 480,
// 36,000 0.329 and 0.273, 50,000 0.337 and 0.363.
// A rest small enough for the row or wave form is split up to dim 8; at dims 9-12,
// whose own groups need fewer walks to fill the GPU, it is split where the form's
// time, which grows with its units, is under the time in turn (split and in turn,
// ms: dim 11, T = 241, 45,000 walks 0.452 and 0.418, 67,236 0.571 and 0.594; dim 10, T
// = 300, 45,000 0.400 and 0.382; dim 12, T = 1,000, 100,000 2.41 and 2.60).
inline uint32_t fp64_turns(int d, uint32_t T, uint32_t n) {
  const uint32_t L = lanes_for_dim(d), wave = 64 / L;  // walks per wave
  const uint32_t round = wave * kSimds * (L == 1 ? kFp64RegWaves[d - 1] : waves_for_dim(d));
  const uint32_t rest = n % round, bn = block_steps(T);
  // dim 7 in turn has a lane group per walk (fp64_turn_lanes), what the row form is
  // without its second launch, so its walks of one block and a little more are
  // split for the wave form only (T = 241, 12,000 walks: 0.114 ms in turn, 0.121 row;
  // T = 300: 0.127 and 0.121)
  if (d == 7 && T <= 270 && n < round) return split_form(d, T, n) == SplitForm::wave ? 0 : n;
  if (block_count(T) == 1) return split_form(d, T, n) == SplitForm::own ? n : 0;
  const bool first = rest == n;
  const SplitForm form = split_form(d, T, rest);
  if (form != SplitForm::own && (first || rest == 0 || d <= 8)) return n - rest;
  if ((uint64_t)rest * 100 >= (uint64_t)round * 90) return n;
  const double full = L == 1 ? kFp64RegWaves[d - 1] : waves_for_dim(d);
  const auto deep = [full](double w) {  // time of ceil(w) waves: 0.84 of the full rate with one, linear between
    const double k = std::max(1.0, std::ceil(w));
    return k >= full ? k : k / (1.0 - 0.16 * (full - k) / (full - 1.0));
  };
  const double w = (double)((rest + wave - 1) / wave) / kSimds, t = (double)T;
  // dim 7's groups of seven lanes: nine walks per wave, four waves per SIMD
  const double in_turn = first && d == 7 && fp64_turn_lanes(d, n) == 7 ? t * (0.2 + 0.147 * std::ceil(n / (9.0 * kSimds)))
                         : first ? t * deep(w)
                                 : t * ((full > 2.0 ? deep(w) : std::ceil(w)) - 0.145);
  const double split =
      form != SplitForm::own
          ? bn * (full > 2.0 ? 0.5 + 0.8 * form_load(d, T, rest) : 0.1 + 0.5 * form_load(d, T, rest)) + 115.0
          : std::max(t * w, bn * deep(w * (T / bn))) + (!first ? 130.0 : d < 7 ? 40.0 : d == 7 ? 35.0 : 20.0);
  return split < in_turn ? n - rest : n;
}

}  // namespace jne
