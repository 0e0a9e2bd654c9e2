// jne_walk_fp64.hip -- FP64 walk path: one-pass moments + FP64 eigen epilogue.
//
// Replaces, per walk, the reference's
//   brownian_motion_matrix      src/rng_matrix.rs:57-141
//   calculate_eigenvalues       src/johansen_statistics.rs:59-85
//   construct_f_matrix          src/johansen_statistics.rs:102-197
//   sum_of_outer_products       src/matrix_utils.rs:67-85
//   GeneralizedEigen (dggev)    src/johansen_statistics.rs:35-45
// without materialising B, dB or F.  Kernel 1 streams the walk once and keeps
// the moments of x_t = [b_t, 1, u_t, u_t^2, e_t] (b_t = B_t before step t,
// e_t = B_{t+1} - B_t, u_t = (t+1)/T) in FP64; kernel 2 forms S11 and S01 of
// the requested model from those moments (demeaning and detrending are Schur
// complements on the {1, u} columns) and solves the eigenproblem -- as one
// kernel, or for the larger dims as two (algebra up to M = W^T W, then Jacobi).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "jne_blocks.h"
#include "jne_internal.h"
#include "jne_rng.h"
#include "jne_tridiag.h"

// The smallest dim whose eigenvalues come from the tridiagonal QL solve
// (jne_tridiag.h) instead of cyclic Jacobi: 1.2x (dim 7) to 1.55x (dim 12)
// faster there; below dim 7 the two time alike (dim 5) or Jacobi leads, and
// Jacobi keeps the higher relative accuracy of the smallest eigenvalues of
// M = W^T W (QL's error is absolute, a few ulp of |M|, as with dggev).
#ifndef JNE_EIGEN_QL_MIN_DIM
#define JNE_EIGEN_QL_MIN_DIM 7
#endif
// Tuning: unroll the steps of a round (rolled and unrolled time alike).
#ifndef JNE_FP64_UNROLL_STEPS
#define JNE_FP64_UNROLL_STEPS 0
#endif
// The Philox calls of a lane in a round are unrolled, so their chains
// overlap: +3-6% at dims 8, 10, 11 and 12, with the same waves per SIMD (at
// dims 7 and 9 a lane draws one call per round).
#ifndef JNE_FP64_UNROLL_CALLS
#define JNE_FP64_UNROLL_CALLS 1
#endif

namespace jne {

// ---------------------------------------------------------------------------
// Kernel 1: moments (jne_blocks.h: block sums, added up with the walk's state).
//
// A walk is owned by a group of L lanes.  Every lane keeps the block's whole
// path state c (dim doubles, in a lane-specific rotated order) and
// accumulates its share of the block's sums:
//   rows k < R of  sum z c^T               (R = DP/L, DP = dim padded to L)
//   rows k < R, cyclic offsets 0..DP/2 of  sum c c^T
//   rows k < R of  S, A1, A2
// Lane r's row k is component (r*R + k) mod DP, so the L lanes cover every
// entry; register indices are compile-time constants.
//
// The walk advances in rounds of S steps.  The S*dim normals of a round are
// S*dim/4 Philox calls, dealt round-robin to the group's lanes and stored to
// LDS as doubles, twice per step row (row = [z_0..z_{dim-1}, 0.., z_0..z_{dim-1},
// 0..], 2*DP entries) so that a lane's rotated read of DP entries is one base
// address plus immediates.  The walk index is the fastest LDS dimension (odd
// pitch) so that the lanes of a wave read from different banks.
//
// SPLIT = false: the group takes its walk's blocks in turn and adds each to
// the sums in acc (its own entries, written by the block before); the last
// block scales them into the canonical layout.  SPLIT = true: block blockIdx.y
// alone, its sums to acc[(blockIdx.y * block_moment_count + entry) * ld + walk]
// for walk_blocks_add.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void keep_order() { asm volatile("" ::: "memory"); }

// waves per SIMD (the register cap) of a lane group of LW lanes: the dim's
// own shape, or one row of the sums per lane (LW = D, at most 96 registers)
constexpr int group_waves(int d, int lw) { return lw == lanes_for_dim(d) ? waves_for_dim(d) : 4; }

// A lane's sums over the blocks it takes in turn, between blocks: the first
// NR of its slots in registers, the next NL in LDS, the rest in acc (at x,
// where their last value goes).  The slots are compile-time constants once
// the loops are unrolled.
template <int NR, int NL>
struct Totals {
  double reg[NR > 0 ? NR : 1];
  double (*lds)[64];
  __device__ __forceinline__ double add(int slot, bool first, bool last, double* x, double t) {
    if (slot < NR) return reg[slot] = (first ? 0.0 : reg[slot]) + t;
    if (slot < NR + NL) {
      double& y = lds[slot - NR][threadIdx.x];
      return y = (first ? 0.0 : y) + t;
    }
    const double v = (first ? 0.0 : *x) + t;
    if (!last) *x = v;
    return v;
  }
};
// by dim: the slots that fit beside the block's sums without spills, and the
// LDS that leaves the kernel's waves resident.  With every slot in acc all the
// waves of a round write at once, which cost 10% at dim 5 (35 us per block of
// 131,072 walks); with all 60 slots on chip it does not show.
#ifndef JNE_FP64_TOTALS
#define JNE_FP64_TOTALS \
  {8, 0}, {15, 0}, {5, 17}, {3, 21}, {25, 35}, {0, 34}, {0, 33}, {24, 0}, {8, 10}, {0, 6}, {0, 10}, {12, 10}
#endif
struct Fp64Totals {
  int regs, lds;
};
constexpr Fp64Totals kFp64Totals[12] = {JNE_FP64_TOTALS};
// of a lane group of LW lanes: the dim's own, or (a row of the sums per lane,
// LW = D) all its slots in registers
constexpr Fp64Totals group_totals(int d, int lw) {
  return lw == lanes_for_dim(d) ? kFp64Totals[d - 1] : Fp64Totals{d + d / 2 + 4, 0};
}

template <int D, int LW, bool FROM_NORMALS, bool SPLIT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(group_waves(D, LW), group_waves(D, LW))))
void walk_moments_fp64(const uint32_t* __restrict__ seeds, const double* __restrict__ zin, uint32_t rng_stream,
                       uint32_t T, uint32_t n_walks, double* __restrict__ acc, size_t ld) {
  using Sh = WalkShape<D, LW>;
  constexpr int L = Sh::L;
  constexpr int DP = Sh::DP;
  constexpr int R = DP / L;
  constexpr int H = DP / 2;
  constexpr int GPW = Sh::GPW;
  constexpr int S = Sh::S;
  constexpr int C = Sh::C;
  constexpr int IT = (C + L - 1) / L;
  constexpr int RW = 2 * DP;        // LDS row width per step
  constexpr int GP = GPW | 1;       // odd walk pitch: a wave's reads spread over the banks
  static_assert(kBlockUnit % S == 0, "a block must be whole rounds");
  __shared__ double ws[S][RW][GP];
  __shared__ double bs[DP][GP];  // the state at the block's start
  constexpr int NR = SPLIT ? 0 : group_totals(D, LW).regs, NL = SPLIT ? 0 : group_totals(D, LW).lds;
  __shared__ double tot_lds[NL > 0 ? NL : 1][64];
  Totals<NR, NL> tot;
  tot.lds = tot_lds;

  const int lane = threadIdx.x;
  // walk fastest across the lanes (lane = r * GPW + g): the 16 lanes of a
  // 64-bit LDS access group read the same row of 16 different walks (odd walk
  // pitch: distinct banks), and the output stores of a lane row go to
  // consecutive walks.
  const int r = lane / GPW;
  const int g = lane - r * GPW;
  const bool in_group = r < L;
  const int gs = in_group ? g : 0;
  const size_t walk = (size_t)blockIdx.x * GPW + gs;
  const bool valid = in_group && walk < n_walks;
  const size_t wc = walk < n_walks ? walk : (size_t)(n_walks - 1);
  uint32_t seed = 0;
  if constexpr (!FROM_NORMALS) seed = seeds[wc];
  const double* zw = FROM_NORMALS ? zin + wc * (size_t)T * D : nullptr;
  const int rot = r * R;
  const CallPos<D> pos0(r);  // normals of this lane's first Philox call in a round

  if (in_group) {
    if constexpr (DP != D) {  // zero the padding columns once
      for (int s = 0; s < S; ++s)
        for (int i = D + r; i < DP; i += L) {
          ws[s][i][gs] = 0.0;
          ws[s][DP + i][gs] = 0.0;
        }
    }
    for (int i = r; i < DP; i += L) bs[i][gs] = 0.0;
  }

  const uint32_t bn = block_steps(T);
  uint32_t ts = SPLIT ? blockIdx.y * bn : 0;
  do {
    const uint32_t n = T - ts < bn ? T - ts : bn;
    double c[DP], ge[R][DP], gc[R][H + 1], s0[R], a1[R], a2[R];
#pragma unroll
    for (int m = 0; m < DP; ++m) c[m] = 0.0;
#pragma unroll
    for (int k = 0; k < R; ++k) {
#pragma unroll
      for (int m = 0; m < DP; ++m) ge[k][m] = 0.0;
#pragma unroll
      for (int m = 0; m <= H; ++m) gc[k][m] = 0.0;
      s0[k] = a1[k] = a2[k] = 0.0;
    }

    for (uint32_t t0 = ts; t0 < ts + n; t0 += S) {
      // produce: this round's increments
      if (in_group) {
        const uint32_t q0 = (uint32_t)((uint64_t)t0 * D / 4);  // < 2^32: dim <= kMaxDim, steps <= kMaxSteps
        CallPos<D> pos = pos0;
#if JNE_FP64_UNROLL_CALLS
#pragma unroll
#else
#pragma unroll 1
#endif
        for (int it = 0; it < IT; ++it) {
          const int call = it * L + r;
          if (IT * L == C || call < C) {
            int sj[4], ij[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) pos.at(j, sj[j], ij[j]);
            double wv[4];
            if constexpr (!FROM_NORMALS) {
              float v[4];
              normals4(q0 + call, seed, rng_stream, v);
#pragma unroll
              for (int j = 0; j < 4; ++j) wv[j] = (double)v[j];
            } else {
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                const uint32_t t = t0 + sj[j];
                wv[j] = t < T ? zw[(size_t)t * D + ij[j]] : 0.0;
              }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              ws[sj[j]][ij[j]][gs] = wv[j];
              ws[sj[j]][DP + ij[j]][gs] = wv[j];
            }
          }
          pos.template advance<L>();
        }
      }
      __syncthreads();
      // consume: advance the block's path S steps
      const int ns = (ts + n - t0) < (uint32_t)S ? (int)(ts + n - t0) : S;
#if JNE_FP64_UNROLL_STEPS
#pragma unroll
#else
#pragma unroll 1
#endif
      for (int s = 0; s < S; ++s) {
        if (s >= ns) break;
        const double* w = &ws[s][rot][gs];
#pragma unroll
        for (int k = 0; k < R; ++k) {
          const double wk = w[k * GP];
#pragma unroll
          for (int m = 0; m < DP; ++m) ge[k][m] = fma(wk, c[m], ge[k][m]);
#pragma unroll
          for (int dl = 0; dl <= H; ++dl) gc[k][dl] = fma(c[k], c[(k + dl) % DP], gc[k][dl]);
          a2[k] += a1[k];
          a1[k] += s0[k];
          s0[k] += c[k];
        }
#pragma unroll
        for (int m = 0; m < DP; ++m) c[m] += w[m * GP];
      }
      __syncthreads();
    }

    if constexpr (SPLIT) {
      if (!valid) return;
      double* const o = acc + (size_t)blockIdx.y * block_moment_count(D) * ld + walk;
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const int ci = (rot + k) % DP;
        if (ci >= D) continue;
#pragma unroll
        for (int m = 0; m < DP; ++m) {
          const int cj = (rot + m) % DP;
          if (cj < D) o[(size_t)blk_ge(D, ci, cj) * ld] = ge[k][m];
        }
#pragma unroll
        for (int dl = 0; dl <= H; ++dl) {
          const int cj = (rot + k + dl) % DP;
          if (cj < D) o[(size_t)(ci < cj ? blk_gc(D, ci, cj) : blk_gc(D, cj, ci)) * ld] = gc[k][dl];
        }
        o[(size_t)blk_vec(D, 0, ci) * ld] = s0[k];
        o[(size_t)blk_vec(D, 1, ci) * ld] = a1[k];
        o[(size_t)blk_vec(D, 2, ci) * ld] = a2[k];
        o[(size_t)blk_vec(D, 3, ci) * ld] = c[k];
      }
      return;
    } else {
      // add the block to the walk's sums: the S of the other lanes' rows go
      // through the round's LDS (its last reads came before the barrier above)
      double(*const ss)[GP] = ws[0];
      if (in_group) {
#pragma unroll
        for (int k = 0; k < R; ++k) ss[(rot + k) % DP][gs] = s0[k];
      }
      __syncthreads();
      const bool first = ts == 0, last = ts + n >= T;
      if (valid) {
        const BlockConst bc = block_const(ts, n);
        const MomentScale sc = moment_scale(T);
        // opaque copies: the entries' addresses are formed here, not kept in
        // registers across the block (keep_order bounds the loads in flight)
        double* o = acc + walk;
        size_t ld_ = ld;
        int rot_ = rot;
        asm volatile("" : "+v"(o), "+s"(ld_), "+v"(rot_));
        int slot = 0;
#pragma unroll
        for (int k = 0; k < R; ++k) {
          const int ci = (rot_ + k) % DP;
          const bool has_i = DP == D || ci < D;
          const double bi = bs[ci][gs];
#pragma unroll
          for (int m = 0; m < DP; ++m, ++slot) {
            const int cj = (rot_ + m) % DP;
            if (m % 4 == 0) keep_order();
            if (!has_i || (DP != D && cj >= D)) continue;
            double* const x = o + (size_t)(D * D + ci * D + cj) * ld_;
            const double v = tot.add(slot, first, last, x, block_zb(c[k], bs[cj][gs], ge[k][m]));
            if (last) *x = v * sc.dt;
          }
#pragma unroll
          for (int dl = 0; dl <= H; ++dl, ++slot) {
            const int cj = (rot_ + k + dl) % DP;
            if (dl % 4 == 0) keep_order();
            if (!has_i || (DP != D && cj >= D)) continue;
            // at an even DP both owners of a pair at distance DP/2 hold it: the
            // lower component's adds it
            if (DP % 2 == 0 && dl == H && cj < ci) continue;
            const bool up = ci < cj;
            const double bj = bs[cj][gs], sj = ss[cj][gs];
            double* const x = o + (size_t)(up ? ci * D + cj : cj * D + ci) * ld_;
            const double v = tot.add(slot, first, last, x,
                                     block_bb(bc, up ? bi : bj, up ? bj : bi, up ? s0[k] : sj, up ? sj : s0[k], gc[k][dl]));
            if (last) {
              *x = v * sc.dt;
              o[(size_t)(up ? cj * D + ci : ci * D + cj) * ld_] = v * sc.dt;
            }
          }
          if (has_i) {
            double* const x = o + (size_t)(2 * D * D + ci) * ld_;
            const double m0 = tot.add(slot, first, last, x, block_m0(bc, bi, s0[k]));
            const double m1 = tot.add(slot + 1, first, last, x + (size_t)D * ld_, block_m1(bc, bi, s0[k], a1[k]));
            const double m2 =
                tot.add(slot + 2, first, last, x + (size_t)(2 * D) * ld_, block_m2(bc, bi, s0[k], a1[k], a2[k]));
            if (last) store_vector_moments(sc, m0, m1, m2, bi + c[k], o, D, ci, ld_, 0);
          }
          slot += 3;
        }
      }
      __syncthreads();
      if (in_group) {
#pragma unroll
        for (int k = 0; k < R; ++k) bs[(rot + k) % DP][gs] += c[k];
      }
      if constexpr (DP != D) {  // the padding columns that held S
        if (in_group)
          for (int i = D + r; i < DP; i += L) ss[i][gs] = 0.0;
      }
      __syncthreads();
      ts += n;
    }
  } while (!SPLIT && ts < T);
}

// ---------------------------------------------------------------------------
// Kernel 1, one lane per walk (the dims whose shape has L = 1): the same sums
// as walk_moments_fp64 with L = 1, with the increments kept in registers
// instead of LDS.  A lane draws its walk's Philox calls in batches of NB calls
// (kFp64RegCalls: three independent calls in flight at dims 1-4 and 6, the
// five of a whole-step group at dim 5, seven at dim 7) and consumes the batch's
// G = 4 NB / dim steps from registers: no LDS, no barriers inside a block.
//
// Bound by VALU issue: at dim 5 a wave-step issues 235 instructions in 722
// cycles, 65 of them FP64 at 3.9 and 1.25 Philox calls of 357 cycles.  The
// increments' moments, the powers of u and the scaling of each normal left the
// step with the block sums.  262,144 walks at T = 10^4, before (every term
// per step) and after: dim 1 2.86 and 2.12 ms, dim 3 8.94 and 7.4, dim 5 16.2
// and 14.4, dim 6 20.1 and 17.4; dim 7 34.6 ms with seven lanes per walk
// through LDS, 28.4 with the block sums there, 22 here.
// ---------------------------------------------------------------------------
// Philox calls per batch by dim (a multiple of the calls of one whole-step
// group: 1, 1, 3, 1, 5, 3 at dims 1..6)
#ifndef JNE_FP64_REG_CALLS
#define JNE_FP64_REG_CALLS 3, 3, 3, 3, 5, 3, 7, 6, 9, 5, 11, 3
#endif
constexpr int kFp64RegCalls[12] = {JNE_FP64_REG_CALLS};

template <int D>
struct RegBatch {
  static constexpr int NC = (4 / gcd_int(D, 4)) * D / 4;  // calls per whole-step group
  static constexpr int NB = kFp64RegCalls[D - 1];         // calls per batch
  static constexpr int G = 4 * NB / D;                     // steps per batch
  static_assert(NB % NC == 0, "a batch must be whole steps");
  static_assert(kBlockUnit % G == 0, "a block must be whole batches");
};

template <int D, bool FROM_NORMALS, bool SPLIT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kFp64RegWaves[D - 1], kFp64RegWaves[D - 1])))
void walk_moments_fp64_reg(const uint32_t* __restrict__ seeds, const double* __restrict__ zin, uint32_t rng_stream,
                           uint32_t T, uint32_t n_walks, double* __restrict__ acc, size_t ld) {
  constexpr int G = RegBatch<D>::G;
  // dim 7: a step's calls are drawn just before it (a whole batch's normals
  // beside the 105 sums would spill)
  constexpr bool kLazy = D >= 7 && !FROM_NORMALS;
  const size_t walk = (size_t)blockIdx.x * 64 + threadIdx.x;
  const bool valid = walk < n_walks;
  const size_t wc = valid ? walk : (size_t)(n_walks - 1);
  uint32_t seed = 0;
  if constexpr (!FROM_NORMALS) seed = seeds[wc];
  const double* zw = FROM_NORMALS ? zin + wc * (size_t)T * D : nullptr;

  const uint32_t bn = block_steps(T);
  uint32_t ts = SPLIT ? blockIdx.y * bn : 0;
  constexpr int NR = SPLIT ? 0 : kFp64Totals[D - 1].regs, NL = SPLIT ? 0 : kFp64Totals[D - 1].lds;
  __shared__ double tot_lds[NL > 0 ? NL : 1][64];
  Totals<NR, NL> tot;
  tot.lds = tot_lds;
  // the state at the block's start: needed between blocks only
  __shared__ double bs_lds[SPLIT ? 1 : D][64];
  auto bs = [&](int m) -> double& { return bs_lds[m][threadIdx.x]; };
  if constexpr (!SPLIT) {
#pragma unroll
    for (int m = 0; m < D; ++m) bs(m) = 0.0;
  }
  do {
    const uint32_t n = T - ts < bn ? T - ts : bn;
    double c[D], ge[D][D], gc[D * (D + 1) / 2], s0[D], a1[D], a2[D];
#pragma unroll
    for (int k = 0; k < D; ++k) {
      c[k] = s0[k] = a1[k] = a2[k] = 0.0;
#pragma unroll
      for (int m = 0; m < D; ++m) ge[k][m] = 0.0;
    }
#pragma unroll
    for (int e = 0; e < D * (D + 1) / 2; ++e) gc[e] = 0.0;

    // one step of the block's path from its increments w[0..D)
    auto step = [&](const double* w) {
      int e = 0;
#pragma unroll
      for (int k = 0; k < D; ++k) {
#pragma unroll
        for (int m = 0; m < D; ++m) ge[k][m] = fma(w[k], c[m], ge[k][m]);
#pragma unroll
        for (int m = k; m < D; ++m, ++e) gc[e] = fma(c[k], c[m], gc[e]);
        a2[k] += a1[k];
        a1[k] += s0[k];
        s0[k] += c[k];
      }
#pragma unroll
      for (int k = 0; k < D; ++k) c[k] += w[k];
    };
    // a batch: G steps from t0; the tail batch masks the steps past the block
    auto batch = [&](uint32_t t0, auto tail_tag) {
      constexpr bool tail = decltype(tail_tag)::value;
      double w[G * D];
      const uint32_t q0 = (uint32_t)((uint64_t)t0 * D / 4);  // < 2^32: dim <= kMaxDim, steps <= kMaxSteps
      // the calls that steps s < s1 still need, of the first `have`
      auto draw = [&](int have, int s1) {
#pragma unroll
        for (int q = have; q < (s1 * D + 3) / 4; ++q) {
          float v[4];
          normals4(q0 + q, seed, rng_stream, v);
#pragma unroll
          for (int j = 0; j < 4; ++j) w[4 * q + j] = (double)v[j];
        }
      };
      if constexpr (FROM_NORMALS) {
#pragma unroll
        for (int e = 0; e < G * D; ++e) {
          const uint32_t t = t0 + (uint32_t)(e / D);
          w[e] = (!tail || t < T) ? zw[(size_t)t0 * D + e] : 0.0;
        }
      } else if constexpr (!kLazy) {
        draw(0, G);
      }
#pragma unroll
      for (int s = 0; s < G; ++s) {
        if constexpr (kLazy) {
          draw((s * D + 3) / 4, s + 1);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (tail && t0 + s >= T) break;
        step(&w[s * D]);
      }
    };
    const uint32_t full = n / G;
    for (uint32_t q = 0; q < full; ++q) batch(ts + q * G, BoolTag<false>{});
    if (full * G < n) batch(ts + full * G, BoolTag<true>{});  // the walk's last block only

    if constexpr (SPLIT) {
      if (!valid) return;
      double* const o = acc + (size_t)blockIdx.y * block_moment_count(D) * ld + walk;
#pragma unroll
      for (int k = 0; k < D; ++k) {
#pragma unroll
        for (int m = 0; m < D; ++m) o[(size_t)blk_ge(D, k, m) * ld] = ge[k][m];
        o[(size_t)blk_vec(D, 0, k) * ld] = s0[k];
        o[(size_t)blk_vec(D, 1, k) * ld] = a1[k];
        o[(size_t)blk_vec(D, 2, k) * ld] = a2[k];
        o[(size_t)blk_vec(D, 3, k) * ld] = c[k];
      }
#pragma unroll
      for (int e = 0; e < D * (D + 1) / 2; ++e) o[(size_t)(D * D + e) * ld] = gc[e];
      return;
    } else {
      const bool first = ts == 0, last = ts + n >= T;
      if (valid) {
        const BlockConst bc = block_const(ts, n);
        const MomentScale sc = moment_scale(T);
        double* o = acc + walk;  // opaque copies, as in walk_moments_fp64
        size_t ld_ = ld;
        asm volatile("" : "+v"(o), "+s"(ld_));
        int e = 0, slot = 0;
#pragma unroll
        for (int k = 0; k < D; ++k) {
          keep_order();
#pragma unroll
          for (int m = 0; m < D; ++m, ++slot) {
            if (D >= 7 && m % 2 == 0) keep_order();
            double* const x = o + (size_t)(D * D + k * D + m) * ld_;
            const double v = tot.add(slot, first, last, x, block_zb(c[k], bs(m), ge[k][m]));
            if (last) *x = v * sc.dt;
          }
          keep_order();
#pragma unroll
          for (int m = k; m < D; ++m, ++e, ++slot) {
            if (D >= 7 && m % 2 == 0) keep_order();
            double* const x = o + (size_t)(k * D + m) * ld_;
            const double v = tot.add(slot, first, last, x, block_bb(bc, bs(k), bs(m), s0[k], s0[m], gc[e]));
            if (last) {
              *x = v * sc.dt;
              o[(size_t)(m * D + k) * ld_] = v * sc.dt;
            }
          }
          double* const x = o + (size_t)(2 * D * D + k) * ld_;
          const double m0 = tot.add(slot, first, last, x, block_m0(bc, bs(k), s0[k]));
          const double m1 = tot.add(slot + 1, first, last, x + (size_t)D * ld_, block_m1(bc, bs(k), s0[k], a1[k]));
          const double m2 =
              tot.add(slot + 2, first, last, x + (size_t)(2 * D) * ld_, block_m2(bc, bs(k), s0[k], a1[k], a2[k]));
          slot += 3;
          if (last) store_vector_moments(sc, m0, m1, m2, bs(k) + c[k], o, D, k, ld_, 0);
        }
      }
#pragma unroll
      for (int k = 0; k < D; ++k) bs(k) += c[k];
      ts += n;
    }
  } while (!SPLIT && ts < T);
}

// ---------------------------------------------------------------------------
// Kernel 1, one wave per block of a walk (blockIdx.x: the walk, blockIdx.y:
// the block): the batches of a few walks, where latency counts.  Rounds of
// kWaveRound steps: the wave draws the round's normals, lanes 0..dim-1 run
// their component's path and S, A1, A2, and every lane adds its entries of
// sum z c^T and of the upper triangle of sum c c^T over the round's steps.
// Each sum takes its terms in the order of the other forms (the same bits).
// ---------------------------------------------------------------------------
constexpr int kWaveRound = 64;

template <int D, bool FROM_NORMALS>
__global__ __launch_bounds__(64) void walk_moments_fp64_wave(const uint32_t* __restrict__ seeds,
                                                             const double* __restrict__ zin, uint32_t rng_stream,
                                                             uint32_t T, double* __restrict__ part, size_t ld) {
  constexpr int R = kWaveRound, NE = D * D + D * (D + 1) / 2, NQ = (NE + 63) / 64;
  constexpr int C = R * D / 4;  // Philox calls per round
  __shared__ __align__(16) double zs[R * D], cs[R * D];  // t-major
  const int l = threadIdx.x;
  const size_t walk = xcd_walk(blockIdx.x, gridDim.x);
  uint32_t seed = 0;
  if constexpr (!FROM_NORMALS) seed = seeds[walk];
  const double* zw = FROM_NORMALS ? zin + walk * (size_t)T * D : nullptr;
  const uint32_t bn = block_steps(T), ts = blockIdx.y * bn, n = T - ts < bn ? T - ts : bn;
  // entry e = l + 64 q: the product of the components x[q], y[q] of z or c and c
  const double* px[NQ];
  const double* py[NQ];
  double acc[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    int e = l + 64 * q;
    if (e >= NE) e = 0;
    int i = e / D, j = e - (e / D) * D;
    px[q] = zs + i;
    if (e >= D * D) {
      e -= D * D;
      for (i = 0; e >= D - i; ++i) e -= D - i;
      j = i + e;
      px[q] = cs + i;
    }
    py[q] = cs + j;
    acc[q] = 0.0;
  }
  double c = 0.0, s0 = 0.0, a1 = 0.0, a2 = 0.0;
  for (uint32_t t0 = 0; t0 < n; t0 += R) {
    const int ns = n - t0 < (uint32_t)R ? (int)(n - t0) : R;
    if constexpr (FROM_NORMALS) {
      for (int e = l; e < ns * D; e += 64) zs[e] = zw[(size_t)(ts + t0) * D + e];
    } else {
      const uint32_t q0 = (uint32_t)((uint64_t)(ts + t0) * D / 4);
      for (int q = l; q < C && 4 * q < ns * D; q += 64) {
        float v[4];
        normals4(q0 + q, seed, rng_stream, v);
#pragma unroll
        for (int j = 0; j < 4; ++j) zs[4 * q + j] = (double)v[j];
      }
    }
    __syncthreads();
    if (l < D) {
#pragma unroll 8
      for (int t = 0; t < ns; ++t) {
        cs[t * D + l] = c;
        a2 += a1;
        a1 += s0;
        s0 += c;
        c += zs[t * D + l];
      }
    }
    __syncthreads();
#pragma unroll 4
    for (int t = 0; t < ns; ++t) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) acc[q] = fma(px[q][t * D], py[q][t * D], acc[q]);
    }
    __syncthreads();
  }
  double* const o = part + (size_t)blockIdx.y * block_moment_count(D) * ld + walk;
#pragma unroll
  for (int q = 0; q < NQ; ++q)
    if (l + 64 * q < NE) o[(size_t)(l + 64 * q) * ld] = acc[q];
  if (l < D) {
    o[(size_t)blk_vec(D, 0, l) * ld] = s0;
    o[(size_t)blk_vec(D, 1, l) * ld] = a1;
    o[(size_t)blk_vec(D, 2, l) * ld] = a2;
    o[(size_t)blk_vec(D, 3, l) * ld] = c;
  }
}

// The walks' moments from their blocks' sums (part: n_walks per entry): a
// workgroup takes 64 walks, its wave k row k of sum z c^T, the upper
// triangle's row k of sum c c^T and component k's vector sums, adding the
// blocks in order with the operations of the kernels that take them in turn.
// Bound by its reads; the waves share the S and E they all read through L1.
// Above dim 6 blockIdx.y halves the columns (no spills).
template <int D>
struct AddShape {
  static constexpr int NH = D > 6 ? 2 : 1, JW = (D + NH - 1) / NH;
};
template <int D>
__global__ __launch_bounds__(64 * D) void walk_blocks_add(uint32_t T, uint32_t n_walks, const double* __restrict__ part,
                                                          double* __restrict__ acc, size_t ld) {
  constexpr int JW = AddShape<D>::JW;
  const int k = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j0 = blockIdx.y * JW;
  const size_t walk = (size_t)blockIdx.x * 64 + (threadIdx.x & 63);
  if (walk >= n_walks) return;
  const uint32_t bn = block_steps(T);
  const MomentScale sc = moment_scale(T);
  const double* p = part + walk;
  double b[JW], ge[JW], gc[JW], m0 = 0.0, m1 = 0.0, m2 = 0.0, bk = 0.0;
#pragma unroll
  for (int q = 0; q < JW; ++q) b[q] = ge[q] = gc[q] = 0.0;
  for (uint32_t ts = 0; ts < T; ts += bn, p += (size_t)block_moment_count(D) * n_walks) {
    auto at = [&](int e) { return p[(size_t)e * n_walks]; };
    const BlockConst bc = block_const(ts, T - ts < bn ? T - ts : bn);
    const double sk = at(blk_vec(D, 0, k)), ek = at(blk_vec(D, 3, k));
#pragma unroll
    for (int q = 0; q < JW; ++q) {
      const int j = j0 + q;
      if (j >= D) break;
      const double bj = b[q];
      ge[q] += block_zb(ek, bj, at(blk_ge(D, k, j)));
      if (j >= k) gc[q] += block_bb(bc, bk, bj, sk, at(blk_vec(D, 0, j)), at(blk_gc(D, k, j)));
      b[q] = bj + at(blk_vec(D, 3, j));
    }
    if (j0 == 0) {
      const double a1 = at(blk_vec(D, 1, k)), a2 = at(blk_vec(D, 2, k));
      m0 += block_m0(bc, bk, sk);
      m1 += block_m1(bc, bk, sk, a1);
      m2 += block_m2(bc, bk, sk, a1, a2);
    }
    bk += ek;
  }
  double* const o = acc + walk;
#pragma unroll
  for (int q = 0; q < JW; ++q) {
    const int j = j0 + q;
    if (j >= D) break;
    o[(size_t)(D * D + k * D + j) * ld] = ge[q] * sc.dt;
    if (j >= k) {
      o[(size_t)(k * D + j) * ld] = gc[q] * sc.dt;
      o[(size_t)(j * D + k) * ld] = gc[q] * sc.dt;
    }
  }
  if (j0 == 0) store_vector_moments(sc, m0, m1, m2, bk, o, D, k, ld, 0);
}

// ---------------------------------------------------------------------------
// Kernel 2: per-walk model algebra + generalized eigen solve (one thread per
// walk; split in two kernels where the fused one would fit too few waves).  F_t = X_t - P Z_t with P = (sum X Z^T)(sum Z Z^T)^-1 applied to the
// projected rows of X:
//   model 0: X = b,            no Z
//   model 1: X = [b; 1],       no Z
//   model 2: X = [b_0..b_{d-2}; y], Z = [1], y = u - 1/2 not projected
//   model 3: X = [b; y],       Z = [1], y not projected
//   model 4: X = [b_0..b_{d-2}; u^2], Z = [1; u], all rows projected
// S11 = dt (XX - sum_{projected} XZ ZZ^-1 ZX),  S01raw = eX - eZ ZZ^-1 ZX.
// The eigenvalues of S11^-1 S10 S01 are those of M = W^T W, W = L^-1 S10
// (S11 = L L^T), plus nF - dim structural zeros (models 1 and 3).
// ---------------------------------------------------------------------------
template <int N>
struct SymReg {
  // upper triangle (i <= j) of an N x N symmetric matrix in registers
  double v[N * (N + 1) / 2];
  __device__ __forceinline__ static constexpr int idx(int i, int j) {
    return i <= j ? i * N - i * (i - 1) / 2 + (j - i) : j * N - j * (j - 1) / 2 + (i - j);
  }
  __device__ __forceinline__ double& operator()(int i, int j) { return v[idx(i, j)]; }
};

// 1/x and 1/sqrt(x) in FP64: the hardware estimate and one Newton step
// (error a few ulp; a rotation needs orthogonality, not correct rounding)
__device__ __forceinline__ double rcp_nr(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  return fma(r, fma(-x, r, 1.0), r);
}
__device__ __forceinline__ double rsq_nr(double x) {
  const double r = __builtin_amdgcn_rsq(x);
  return r * fma(-0.5 * x * r, r, 1.5);
}

template <int N>
__device__ __forceinline__ void jacobi_rotate(SymReg<N>& a, int p, int q) {
  const double apq = a(p, q);
  const double app = a(p, p), aqq = a(q, q);
  // threshold Jacobi: below 1e-18 sqrt(|app aqq|), zeroing a_pq moves the
  // eigenvalues by at most ~1e-18 of themselves (a(p, q) = 0 is such a case)
  if (apq * apq <= 1e-36 * fabs(app * aqq)) {
    a(p, q) = 0.0;
    return;
  }
  // theta clamped so theta^2 stays finite (t ~ 1/(2 theta) there anyway)
  const double theta = fmin(fmax((aqq - app) * rcp_nr(2.0 * apq), -1e150), 1e150);
  const double h = fma(theta, theta, 1.0);
  double t = rcp_nr(fabs(theta) + h * rsq_nr(h));
  if (theta < 0.0) t = -t;
  const double c = rsq_nr(fma(t, t, 1.0));
  const double s = t * c;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    if (k == p || k == q) continue;
    const double akp = a(k, p), akq = a(k, q);
    a(k, p) = c * akp - s * akq;
    a(k, q) = s * akp + c * akq;
  }
  a(p, p) = app - t * apq;
  a(q, q) = aqq + t * apq;
  a(p, q) = 0.0;
}

template <int N>
__device__ __forceinline__ void jacobi_eigvals(SymReg<N>& a) {
  for (int sweep = 0; sweep < 40; ++sweep) {
    double off = 0.0, dia = 0.0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      dia = fma(a(i, i), a(i, i), dia);
#pragma unroll
      for (int j = i + 1; j < N; ++j) off = fma(a(i, j), a(i, j), off);
    }
    if (!(off > 1e-34 * dia)) break;
#pragma unroll
    for (int p = 0; p < N - 1; ++p) {
#pragma unroll
      for (int q = p + 1; q < N; ++q) jacobi_rotate<N>(a, p, q);
    }
  }
}

template <int MODEL, int D>
struct EigenShape {
  static constexpr int NX = (MODEL == 1 || MODEL == 3) ? D + 1 : D;  // nF
  static constexpr int NB = (MODEL == 2 || MODEL == 4) ? D - 1 : D;  // b rows in X
  static constexpr int NZ = MODEL == 4 ? 2 : ((MODEL == 2 || MODEL == 3) ? 1 : 0);
  // one workgroup's W in LDS: NX*D doubles per walk.  Above 20 KiB fewer than
  // 8 workgroups (2 waves per SIMD) fit a CU, and the solve runs as two
  // kernels: the algebra up to M = W^T W, then Jacobi on M without LDS.
  static constexpr bool kSplit = NX * D * 64 * 8 > 20 * 1024;
};

// Model algebra, Cholesky of S11 and M = W^T W for walk wc (the prefix of the
// solve; W goes through the workgroup's LDS buffer wsh).
template <int MODEL, int D>
__device__ __forceinline__ void eigen_prep(const double* __restrict__ acc, size_t ld, uint32_t T, size_t wc,
                                           int tid, double (*wsh)[64], SymReg<D>& M, bool& pd_out) {
  constexpr int NX = EigenShape<MODEL, D>::NX;
  constexpr int NB = EigenShape<MODEL, D>::NB;
  constexpr int NZ = EigenShape<MODEL, D>::NZ;
  auto A = [&](int e) -> double { return acc[(size_t)e * ld + wc]; };
  auto GBB = [&](int i, int j) { return A(i * D + j); };
  auto GEB = [&](int k, int j) { return A(D * D + k * D + j); };
  auto MB = [&](int p, int i) { return A(2 * D * D + p * D + i); };
  auto ME = [&](int p, int k) { return A(2 * D * D + (3 + p) * D + k); };

  const double Tn = (double)T;
  const double dt = 1.0 / Tn;
  // closed forms of sum_t u_t^p, u_t = (t+1)/T, t = 0..T-1
  const double c1 = (Tn + 1.0) * 0.5;
  const double c2 = (Tn + 1.0) * (2.0 * Tn + 1.0) / (6.0 * Tn);
  const double c3 = (Tn + 1.0) * (Tn + 1.0) / (4.0 * Tn);
  const double c4 = (Tn + 1.0) * (2.0 * Tn + 1.0) * (3.0 * Tn * Tn + 3.0 * Tn - 1.0) / (30.0 * Tn * Tn * Tn);

  // XZ row x, column z (z = 0: 1, z = 1: u)
  auto XZ = [&](int x, int z) -> double {
    if (x < NB) return MB(z, x);
    if constexpr (MODEL == 2 || MODEL == 3) return c1 - 0.5 * Tn;  // sum y
    else if constexpr (MODEL == 4) return z == 0 ? c2 : c3;        // sum u^2, sum u^3
    else return 0.0;
  };
  auto projected = [&](int x) -> bool {
    if constexpr (MODEL == 4) return true;
    else if constexpr (MODEL == 2 || MODEL == 3) return x < NB;
    else return false;
  };
  auto XX = [&](int i, int j) -> double {
    if (i < NB && j < NB) return GBB(i, j);
    if (i >= NB && j >= NB) {
      if constexpr (MODEL == 1) return Tn;
      else if constexpr (MODEL == 2 || MODEL == 3) return c2 - c1 + 0.25 * Tn;  // sum (u - 1/2)^2
      else return c4;
    }
    const int bi = i < NB ? i : j;
    if constexpr (MODEL == 1) return MB(0, bi);
    else if constexpr (MODEL == 2 || MODEL == 3) return MB(1, bi) - 0.5 * MB(0, bi);  // sum b y
    else return MB(2, bi);                                                            // sum b u^2
  };
  auto EX = [&](int k, int j) -> double {
    if (j < NB) return GEB(k, j);
    if constexpr (MODEL == 1) return ME(0, k);
    else if constexpr (MODEL == 2 || MODEL == 3) return ME(1, k) - 0.5 * ME(0, k);
    else return ME(2, k);
  };

  // ZZ^-1 (closed form): model 4: [[T, c1], [c1, c2]]^-1, det = (T^2 - 1)/12
  double zi00 = 0.0, zi01 = 0.0, zi11 = 0.0;
  if constexpr (NZ == 1) zi00 = dt;
  if constexpr (NZ == 2) {
    const double det = (Tn * Tn - 1.0) / 12.0;
    zi00 = c2 / det;
    zi01 = -c1 / det;
    zi11 = Tn / det;
  }
  // P_x = XZ_x ZZ^-1 for every X row
  double P0[NX], P1[NX];
#pragma unroll
  for (int x = 0; x < NX; ++x) {
    P0[x] = 0.0;
    P1[x] = 0.0;
    if constexpr (NZ == 1) P0[x] = XZ(x, 0) * zi00;
    if constexpr (NZ == 2) {
      const double a0 = XZ(x, 0), a1 = XZ(x, 1);
      P0[x] = a0 * zi00 + a1 * zi01;
      P1[x] = a0 * zi01 + a1 * zi11;
    }
  }
  auto proj = [&](int i, int j) -> double {  // XZ_i ZZ^-1 ZX_j with projection mask
    if constexpr (NZ == 0) return 0.0;
    else {
      if (projected(i)) return NZ == 2 ? P0[i] * XZ(j, 0) + P1[i] * XZ(j, 1) : P0[i] * XZ(j, 0);
      if (projected(j)) return NZ == 2 ? P0[j] * XZ(i, 0) + P1[j] * XZ(i, 1) : P0[j] * XZ(i, 0);
      return 0.0;
    }
  };

  // S11 (lower triangle in SymReg form) and its Cholesky factor in place;
  // dinv[j] = 1 / L(j, j), which the substitutions below multiply by
  SymReg<NX> Lf;
  double dinv[NX];
  bool pd = true;
#pragma unroll
  for (int i = 0; i < NX; ++i) {
#pragma unroll
    for (int j = 0; j <= i; ++j) Lf(i, j) = (XX(i, j) - proj(i, j)) * dt;
  }
#pragma unroll
  for (int j = 0; j < NX; ++j) {
    double s = Lf(j, j);
#pragma unroll
    for (int k = 0; k < j; ++k) s -= Lf(j, k) * Lf(j, k);
    pd = pd && (s > 0.0);
    const double ljj = sqrt(s > 0.0 ? s : 1.0);
    const double inv = 1.0 / ljj;
    Lf(j, j) = ljj;
    dinv[j] = inv;
#pragma unroll
    for (int i = j + 1; i < NX; ++i) {
      double v = Lf(i, j);
#pragma unroll
      for (int k = 0; k < j; ++k) v -= Lf(i, k) * Lf(j, k);
      Lf(i, j) = v * inv;
    }
  }

  // W column k = L^-1 (row k of S01raw), stored to LDS
#pragma unroll 1
  for (int k = 0; k < D; ++k) {
    double wv[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      double v = EX(k, i);
      if constexpr (NZ > 0) {
        if (projected(i)) {
          const double ez0 = ME(0, k);
          v -= NZ == 2 ? P0[i] * ez0 + P1[i] * ME(1, k) : P0[i] * ez0;
        }
      }
#pragma unroll
      for (int j = 0; j < i; ++j) v -= Lf(i, j) * wv[j];
      wv[i] = v * dinv[i];
      wsh[i * D + k][tid] = wv[i];
    }
  }

  // M = W^T W (D x D)
#pragma unroll
  for (int k = 0; k < D * (D + 1) / 2; ++k) M.v[k] = 0.0;
#pragma unroll 1
  for (int i = 0; i < NX; ++i) {
    double row[D];
#pragma unroll
    for (int k = 0; k < D; ++k) row[k] = wsh[i * D + k][tid];
#pragma unroll
    for (int k = 0; k < D; ++k) {
#pragma unroll
      for (int l = k; l < D; ++l) M(k, l) = fma(row[k], row[l], M(k, l));
    }
  }
  pd_out = pd;
}

// sqrt, 1/x and 1/sqrt(x) for jne_tridiag.h: the hardware estimates and one
// Newton step
struct TriMath {
  __device__ __forceinline__ static double sqrt(double x) { return x > 0.0 ? x * rsq_nr(x) : 0.0; }
  __device__ __forceinline__ static double rcp(double x) { return rcp_nr(x); }
  __device__ __forceinline__ static double rsqrt(double x) { return rsq_nr(x); }
};

// The eigenvalues of M (tridiagonal reduction + implicit QL from dim
// JNE_EIGEN_QL_MIN_DIM, cyclic Jacobi below it), |lambda| sorted descending,
// NX - D structural zeros; NaN rows for a walk whose S11 was not positive
// definite.
template <int D, int NX>
__device__ __forceinline__ void eigen_finish(SymReg<D>& M, bool pd, double* __restrict__ o) {
  double ev[D];
  if constexpr (D >= JNE_EIGEN_QL_MIN_DIM) {
    tridiag_eigvals<D, TriMath>(M.v, ev);
#pragma unroll
    for (int k = 0; k < D; ++k) ev[k] = fabs(ev[k]);
  } else {
    jacobi_eigvals<D>(M);
#pragma unroll
    for (int k = 0; k < D; ++k) ev[k] = fabs(M(k, k));
  }
  // sort descending (odd-even transposition, fixed network)
#pragma unroll
  for (int pass = 0; pass < D; ++pass) {
#pragma unroll
    for (int k = pass & 1; k + 1 < D; k += 2) {
      const double hi = fmax(ev[k], ev[k + 1]);
      const double lo = fmin(ev[k], ev[k + 1]);
      ev[k] = hi;
      ev[k + 1] = lo;
    }
  }
  const double nan = __longlong_as_double(0x7FF8000000000000LL);
#pragma unroll
  for (int k = 0; k < D; ++k) o[k] = pd ? ev[k] : nan;
  if constexpr (NX > D) o[D] = pd ? 0.0 : nan;
}

// One thread per walk: the whole solve in one kernel (small D).
template <int MODEL, int D>
__global__ __launch_bounds__(64) void walk_eigen_fp64(const double* __restrict__ acc, size_t ld, uint32_t T,
                                                      uint32_t n_walks, double* __restrict__ out) {
  constexpr int NX = EigenShape<MODEL, D>::NX;
  __shared__ double wsh[NX * D][64];
  const int tid = threadIdx.x;
  const size_t w = (size_t)blockIdx.x * 64 + tid;
  const bool valid = w < n_walks;
  const size_t wc = valid ? w : (size_t)(n_walks - 1);
  SymReg<D> M;
  bool pd;
  eigen_prep<MODEL, D>(acc, ld, T, wc, tid, wsh, M, pd);
  if (!valid) return;
  eigen_finish<D, NX>(M, pd, out + w * NX);
}

// Split form, first kernel: M and the definiteness flag, entry-major
// (m[e * ld + walk], e < D(D+1)/2; e = D(D+1)/2 holds 1 or 0).
template <int MODEL, int D>
__global__ __launch_bounds__(64) void walk_eigen_prep(const double* __restrict__ acc, size_t ld, uint32_t T,
                                                      uint32_t n_walks, double* __restrict__ m) {
  constexpr int NX = EigenShape<MODEL, D>::NX;
  __shared__ double wsh[NX * D][64];
  const int tid = threadIdx.x;
  const size_t w = (size_t)blockIdx.x * 64 + tid;
  const bool valid = w < n_walks;
  const size_t wc = valid ? w : (size_t)(n_walks - 1);
  SymReg<D> M;
  bool pd;
  eigen_prep<MODEL, D>(acc, ld, T, wc, tid, wsh, M, pd);
  if (!valid) return;
#pragma unroll
  for (int e = 0; e < D * (D + 1) / 2; ++e) m[(size_t)e * ld + w] = M.v[e];
  m[(size_t)(D * (D + 1) / 2) * ld + w] = pd ? 1.0 : 0.0;
}

// Split form, second kernel: the eigenvalues of M in registers, no LDS
// (eigen_finish: tridiagonal QL from dim JNE_EIGEN_QL_MIN_DIM, Jacobi below).
template <int D, int NX>
__global__ __launch_bounds__(64) void walk_eigen_jacobi(const double* __restrict__ m, size_t ld, uint32_t n_walks,
                                                        double* __restrict__ out) {
  const size_t w = (size_t)blockIdx.x * 64 + threadIdx.x;
  if (w >= n_walks) return;
  SymReg<D> M;
#pragma unroll
  for (int e = 0; e < D * (D + 1) / 2; ++e) M.v[e] = m[(size_t)e * ld + w];
  const bool pd = m[(size_t)(D * (D + 1) / 2) * ld + w] != 0.0;
  eigen_finish<D, NX>(M, pd, out + w * NX);
}


// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
size_t fp64_part_doubles(int d, uint32_t T, uint32_t n) {
  return (size_t)block_count(T) * block_moment_count(d) * (n - fp64_turns(d, T, n));
}

template <int D>
static hipError_t launch_moments_d(const uint32_t* seeds, const double* zin, uint32_t rng_stream, uint32_t T,
                                   uint32_t n, double* acc, size_t ld, double* part, size_t part_doubles,
                                   hipStream_t st) {
  constexpr int L = WalkShape<D>::L;
  // LW lanes per walk (0: one wave) for m walks into out
  auto go = [&](auto lw_tag, auto split_tag, const uint32_t* s, const double* z, uint32_t m, double* out, size_t ldo) {
    constexpr int LW = decltype(lw_tag)::value;
    constexpr bool SPLIT = decltype(split_tag)::value;
    const dim3 grid(LW == 0 ? m : (m + 64 / (LW ? LW : 1) - 1) / (64 / (LW ? LW : 1)), SPLIT ? block_count(T) : 1);
    if constexpr (LW == 0) {
      if (z)
        hipLaunchKernelGGL((walk_moments_fp64_wave<D, true>), grid, dim3(64), 0, st, s, z, rng_stream, T, out, ldo);
      else
        hipLaunchKernelGGL((walk_moments_fp64_wave<D, false>), grid, dim3(64), 0, st, s, z, rng_stream, T, out, ldo);
    } else if constexpr (LW == 1) {
      if (z)
        hipLaunchKernelGGL((walk_moments_fp64_reg<D, true, SPLIT>), grid, dim3(64), 0, st, s, z, rng_stream, T, m, out,
                           ldo);
      else
        hipLaunchKernelGGL((walk_moments_fp64_reg<D, false, SPLIT>), grid, dim3(64), 0, st, s, z, rng_stream, T, m, out,
                           ldo);
    } else {
      if (z)
        hipLaunchKernelGGL((walk_moments_fp64<D, LW, true, SPLIT>), grid, dim3(64), 0, st, s, z, rng_stream, T, m, out,
                           ldo);
      else
        hipLaunchKernelGGL((walk_moments_fp64<D, LW, false, SPLIT>), grid, dim3(64), 0, st, s, z, rng_stream, T, m, out,
                           ldo);
    }
    return hipGetLastError();
  };
  uint32_t turns = fp64_turns(D, T, n);
  if (part == nullptr || part_doubles < fp64_part_doubles(D, T, n)) turns = n;
  if constexpr (D == 7) {
    if (turns == n && fp64_turn_lanes(D, n) == 7) return go(IntTag<7>{}, BoolTag<false>{}, seeds, zin, n, acc, ld);
  }
  hipError_t e = hipSuccess;
  if (turns > 0) e = go(IntTag<L>{}, BoolTag<false>{}, seeds, zin, turns, acc, ld);
  if (e != hipSuccess || turns == n) return e;
  // the split rest
  const uint32_t m = n - turns;
  const uint32_t* s = seeds ? seeds + turns : nullptr;
  const double* z = zin ? zin + (size_t)turns * T * D : nullptr;
  switch (split_form(D, T, m)) {
    case SplitForm::wave: e = go(IntTag<0>{}, BoolTag<true>{}, s, z, m, part, m); break;
    case SplitForm::row: e = go(IntTag<D>{}, BoolTag<true>{}, s, z, m, part, m); break;
    case SplitForm::own: e = go(IntTag<L>{}, BoolTag<true>{}, s, z, m, part, m); break;
  }
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(walk_blocks_add<D>, dim3((m + 63) / 64, AddShape<D>::NH), dim3(64 * D), 0, st, T, m, part,
                     acc + turns, ld);
  return hipGetLastError();
}

template <int MODEL, int D>
static hipError_t launch_eigen_md(const double* acc, size_t ld, uint32_t T, uint32_t n, double* out, double* mbuf,
                                  hipStream_t st) {
  const unsigned grid = (unsigned)((n + 63) / 64);
  if constexpr (EigenShape<MODEL, D>::kSplit) {
    if (mbuf == nullptr) return hipErrorInvalidValue;
    hipLaunchKernelGGL((walk_eigen_prep<MODEL, D>), dim3(grid), dim3(64), 0, st, acc, ld, T, n, mbuf);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((walk_eigen_jacobi<D, EigenShape<MODEL, D>::NX>), dim3(grid), dim3(64), 0, st, mbuf, ld, n,
                       out);
  } else {
    hipLaunchKernelGGL((walk_eigen_fp64<MODEL, D>), dim3(grid), dim3(64), 0, st, acc, ld, T, n, out);
  }
  return hipGetLastError();
}

hipError_t launch_walk_moments_fp64(int d, const uint32_t* seeds, const double* zin, uint32_t rng_stream, uint32_t T,
                                    uint32_t n, double* acc, size_t ld, double* part, size_t part_doubles,
                                    hipStream_t st) {
  switch (d) {
#define JNE_CASE(DD) \
  case DD:           \
    return launch_moments_d<DD>(seeds, zin, rng_stream, T, n, acc, ld, part, part_doubles, st);
    JNE_CASE(1) JNE_CASE(2) JNE_CASE(3) JNE_CASE(4) JNE_CASE(5) JNE_CASE(6)
    JNE_CASE(7) JNE_CASE(8) JNE_CASE(9) JNE_CASE(10) JNE_CASE(11) JNE_CASE(12)
#undef JNE_CASE
    default:
      return hipErrorInvalidValue;
  }
}

template <int MODEL>
static hipError_t launch_eigen_m(int d, const double* acc, size_t ld, uint32_t T, uint32_t n, double* out,
                                 double* mbuf, hipStream_t st) {
  switch (d) {
#define JNE_CASE(DD) \
  case DD:           \
    return launch_eigen_md<MODEL, DD>(acc, ld, T, n, out, mbuf, st);
    JNE_CASE(1) JNE_CASE(2) JNE_CASE(3) JNE_CASE(4) JNE_CASE(5) JNE_CASE(6)
    JNE_CASE(7) JNE_CASE(8) JNE_CASE(9) JNE_CASE(10) JNE_CASE(11) JNE_CASE(12)
#undef JNE_CASE
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_walk_eigen_fp64(int model, int d, const double* acc, size_t ld, uint32_t T, uint32_t n,
                                  double* out, double* mbuf, hipStream_t st) {
  switch (model) {
    case 0: return launch_eigen_m<0>(d, acc, ld, T, n, out, mbuf, st);
    case 1: return launch_eigen_m<1>(d, acc, ld, T, n, out, mbuf, st);
    case 2: return launch_eigen_m<2>(d, acc, ld, T, n, out, mbuf, st);
    case 3: return launch_eigen_m<3>(d, acc, ld, T, n, out, mbuf, st);
    case 4: return launch_eigen_m<4>(d, acc, ld, T, n, out, mbuf, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace jne
