// jne_blocks.h -- the FP64 moment passes' sums over blocks of steps.
//
// A walk's moments are formed block by block: inside a block that starts at
// step ts with the unscaled state B = sum_{r < ts} z_r, the kernels accumulate
// moments of the block's own path c_t = sum_{ts <= r < t} z_r (which starts at
// zero) and of its normals z_t, and the block is then added to the walk's sums
// with B.  With b = B + c, te = ts + n the end of the block and the sums over
// its steps:
//
//   sum b b^T       += n B B^T + B S^T + S B^T + GC        S = sum c, GC = sum c c^T
//   sum z b^T       += E B^T + GE                          E = sum z, GE = sum z c^T
//   sum b           += n B + S
//   sum (t+1) b     += B sum (t+1)   + te S - A1
//   sum (t+1)^2 b   += B sum (t+1)^2 + te^2 S - 2 te A1 + 2 A2 + A1
//   B               += E
//
// A1 = sum m c and A2 = sum m (m - 1)/2 c with m = te - (t+1).  The kernels of dims
// 1..12 form them as the running sums of S and A1 (each added before its source is
// advanced), with no powers of t; those of the wide dims, whose lanes take every
// fourth step, with the weights m and m (m - 1)/2.  The moments of the increments follow from the
// others by summation by parts: sum (t+1) z = T B_T - sum b and
// sum (t+1)^2 z = T^2 B_T - 2 sum (t+1) b + sum b.  Everything is unscaled
// until the end, where e = s z and b scale by s = sqrt(1/T).
//
// The blocks depend on T alone, and a block's sums run over its steps in
// order, so a walk's results are the same bits whether one lane takes the
// blocks in turn (large batches) or every block has lanes of its own and a
// second kernel adds them up (batches that would leave the GPU idle).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "jne_forms.h"

namespace jne {

// Doubles of one block's sums: GE (d*d), GC (upper triangle), S, A1, A2, E.
constexpr int block_moment_count(int d) { return d * d + d * (d + 1) / 2 + 4 * d; }
__host__ __device__ constexpr int blk_ge(int d, int k, int j) { return k * d + j; }
__host__ __device__ constexpr int blk_gc(int d, int i, int j) { return d * d + i * d - i * (i - 1) / 2 + (j - i); }  // i <= j
__host__ __device__ constexpr int blk_vec(int d, int p, int i) { return d * d + d * (d + 1) / 2 + p * d + i; }  // S, A1, A2, E

// Per-block constants: n, sum (t+1), sum (t+1)^2 over the block's steps and te.
struct BlockConst {
  double n, u1, u2, te;
};
__device__ __forceinline__ BlockConst block_const(uint32_t ts, uint32_t n) {
  BlockConst c;
  const double nd = (double)n, a = (double)ts + 1.0, h = nd - 1.0;
  c.n = nd;
  c.te = (double)(ts + n);
  c.u1 = fma(nd, a, 0.5 * (nd * h));
  c.u2 = fma(nd * a, a, fma(a, nd * h, nd * h * (2.0 * nd - 1.0) * (1.0 / 6.0)));
  return c;
}

// A block's terms of the walk's sums (lo <= hi in sum b b^T).
__device__ __forceinline__ double block_bb(const BlockConst& c, double b_lo, double b_hi, double s_lo, double s_hi, double gc) {
  return fma(b_lo, fma(c.n, b_hi, s_hi), fma(s_lo, b_hi, gc));
}
__device__ __forceinline__ double block_zb(double e_k, double b_j, double ge) { return fma(e_k, b_j, ge); }
__device__ __forceinline__ double block_m0(const BlockConst& c, double b, double s) { return fma(c.n, b, s); }
__device__ __forceinline__ double block_m1(const BlockConst& c, double b, double s, double a1) {
  return fma(b, c.u1, fma(c.te, s, -a1));
}
__device__ __forceinline__ double block_m2(const BlockConst& c, double b, double s, double a1, double a2) {
  return fma(b, c.u2, fma(c.te * c.te, s, fma(-2.0 * c.te, a1, fma(2.0, a2, a1))));
}

// The canonical moments (see moment_count) of a walk from its unscaled sums.
struct MomentScale {
  double dt, s, T;
};
__device__ __forceinline__ MomentScale moment_scale(uint32_t T) {
  MomentScale m;
  m.T = (double)T;
  m.dt = 1.0 / m.T;
  m.s = sqrt(m.dt);
  return m;
}
// the six vector moments of component i: m0, m1, m2 the sums of b, (t+1) b and
// (t+1)^2 b, bT the state after the last step
__device__ __forceinline__ void store_vector_moments(const MomentScale& k, double m0, double m1, double m2, double bT,
                                                     double* __restrict__ acc, int d, int i, size_t ld, size_t walk) {
  double* const o = acc + (size_t)(2 * d * d + i) * ld + walk;
  const size_t p = (size_t)d * ld;
  o[0] = k.s * m0;
  o[p] = (k.s * k.dt) * m1;
  o[2 * p] = (k.s * (k.dt * k.dt)) * m2;
  o[3 * p] = k.s * bT;
  o[4 * p] = k.s * fma(-k.dt, m0, bT);
  o[5 * p] = k.s * fma(k.dt * k.dt, fma(-2.0, m1, m0), bT);
}

}  // namespace jne
