// jne_walk_wide.hip -- FP64 walk path for dims 13..32 (runtime dim).
//
// The reference's per-walk operator takes any dim
// (calculate_eigenvalues, src/johansen_statistics.rs:59-85; the CLI checks
// only dim > 0, src/cli.rs:201-225).  The register-resident kernels of
// jne_walk_fp64.hip cover dims 1..12; above that a walk's Gram and its
// eigenproblem no longer fit one lane's registers, so here one wave owns one
// walk and keeps both in registers spread over its lanes and in LDS:
//
//   walk_moments_wide  the block sums of jne_blocks.h (the canonical entry-major
//                      layout of jne_internal.h): per round of R steps the wave
//                      draws the R*dim normals (Philox calls dealt over the
//                      lanes, the stream of jne_rng.h), lanes 0..dim-1 run their
//                      component's path c, and the sums of [c; z] c^T over the
//                      round go through the FP64 matrix instructions, 4 steps at
//                      a time;
//   walk_eigen_wide    model algebra (S11 and S01 as Schur complements on the
//                      moments), Cholesky of S11, W = L^-1 S10, M = W^T W,
//                      with lanes working on matrix entries, rows or columns
//                      in parallel; then the Householder reduction of M to
//                      tridiagonal form (lane i holding row i in registers)
//                      and eigenvalue k by a group of lanes, by multisection
//                      on Sturm counts (jne_tridiag.h).
//
// The arithmetic is FP64 throughout, as in walk_moments_fp64 /
// walk_eigen_fp64, so the results meet the same 1e-9 parity with the
// reference's dggev solve.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "jne_blocks.h"
#include "jne_internal.h"
#include "jne_rng.h"
#include "jne_tridiag.h"

namespace jne {

namespace {

// Steps per round: a multiple of 4 that divides kBlockUnit, with at most 128
// Philox calls; of those the one that fills the 64-lane call iterations best,
// the longer on a tie (dim 13..16: 16, 17..19: 24, 20..25: 20 to 24, 26..32: 16).
__host__ __device__ constexpr int wide_round_steps(int d) {
  int best = 4;
  for (int r = 8; r <= 24; r += 4) {
    const int calls = r * d / 4, old = best * d / 4;
    if (calls > 128 || kBlockUnit % r != 0) continue;
    // calls / lanes drawn against old / lanes drawn
    if (calls * ((old + 63) / 64) >= old * ((calls + 63) / 64)) best = r;
  }
  return best;
}

typedef double d64x4 __attribute__((ext_vector_type(4)));

}  // namespace

// The operand rows of a walk, 16 to a tile: positions 0..DB-1 the path c of the
// components (zero from dim on), DB..2 DB-1 their normals z, DB = 4 NB.  A lane's
// operand of tile q is X[position 16 q + l % 16][step 4 g + l / 16], as A (rows)
// and B (columns) alike.
template <int NB>
struct WideShape {
  static constexpr int DB = 4 * NB;
  static constexpr int NT = (2 * NB + 3) / 4;               // tiles
  static constexpr int NR = NB == 8 ? 2 : 1;                // row tiles taken by 16x16x4 products
  static constexpr int NU = NB == 8 ? 0 : NB - 4;           // 4-row blocks past them: 4x4x4 products
  static constexpr int NC = NB == 4 ? 1 : 2;                // tiles that hold path components
  static constexpr int N16 = NB == 8 ? 2 * NT - 1 : NT;     // 16x16 accumulators
  static constexpr int N4 = NU * (NT - 1);                  // 4x4 accumulators (4 blocks each)
  static constexpr int ND = 4 * N16 + N4;                   // accumulator doubles per lane
  static constexpr int waves = NB <= 6 ? 4 : 3;
  // accumulator entry x of lane l: its row (a component) and column (a position)
  static __device__ __forceinline__ void entry(int x, int l, int& row, int& col) {
    if (x < 4 * N16) {
      const int t = x / 4, r = x % 4;
      row = l / 16 + 4 * r + (t >= NT ? 16 : 0);
      col = 16 * (t >= NT ? t - NT + 1 : t) + l % 16;
    } else {
      const int y = x - 4 * N16;
      row = 16 + 4 * (y / (NT - 1)) + l / 16;
      col = 16 * (1 + y % (NT - 1)) + l % 16;
    }
  }
};

// One wave per walk, taking its blocks in turn with the totals in registers, or
// (SPLIT) per block blockIdx.y of a walk, its sums to acc for wide_blocks_add.
//
// Bound by the FP64 matrix instructions and the normals, which share the SIMD:
// a 16x16x4 product takes 65 cycles (15.8 FMAs per cycle against 14.2 from
// v_fma_f64) and 4x4x4 ones fill the rows past 16 where a 16-row tile would be
// mostly padding.  Operands are read once per 4 steps (2 to 8 LDS reads per
// lane); the VALU tiles that stood here read 8 to 13 doubles per lane and step
// for 8 to 32 FMAs and were bound by LDS.  At dim 32 a step costs 218 cycles of
// its SIMD, 112 of them in matrix instructions and 78 in the 25 VALU ones, most
// of those the normals'.  Before and now, ms: 16,384 walks at T = 10^4, dim 32
// 22.7 and 15.8 (eigen solve included); 12,288 walks at T = 4,000, dim 16 3.16
// and 1.79, dim 20 4.36 and 2.90, dim 24 4.72 and 3.03; 500 walks there (split
// over their blocks), dim 16 0.484 and 0.129, dim 32 0.879 and 0.251.  The
// symmetric tile as three 4x4x4 products (50 cycles for 65) gained nothing:
// its operands are two more LDS reads.
template <int NB, bool FROM_NORMALS, bool SPLIT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WideShape<NB>::waves)))
void walk_moments_wide(const uint32_t* __restrict__ seeds, const double* __restrict__ zin, uint32_t rng_stream,
                       uint32_t T, uint32_t n_walks, int D, double* __restrict__ acc, size_t ld) {
  using Sh = WideShape<NB>;
  constexpr int DB = Sh::DB, NT = Sh::NT, ND = Sh::ND;
  extern __shared__ double wide_x[];  // X[tile][step][16], R steps (wide_moments_lds_bytes)
  __shared__ double qv[16 * NT], bv[16 * NT], sv[32], a1v[32], a2v[32];
  const int l = threadIdx.x;
  if (blockIdx.x >= n_walks) return;  // whole wave exits together
  const size_t walk = xcd_walk(blockIdx.x, n_walks);
  const int R = wide_round_steps(D);
  const int calls = R * D / 4;
  uint32_t seed = 0;
  if constexpr (!FROM_NORMALS) seed = seeds[walk];
  const double* zw = FROM_NORMALS ? zin + walk * (size_t)T * D : nullptr;
  auto at = [&](int pos, int t) { return ((pos >> 4) * R + t) * 16 + (pos & 15); };

  for (int e = l; e < NT * R * 16; e += 64) wide_x[e] = 0.0;  // the padding stays zero
  // where the normals of this lane's calls l and l + 64 of a round go
  int zo[2][4], zt[2];
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int n0 = 4 * (l + 64 * it);
    int t = n0 / D, i = n0 - t * D;
    zt[it] = t;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      zo[it][j] = at(DB + i, t);
      if (++i == D) {
        i = 0;
        ++t;
      }
    }
  }
  __syncthreads();

  double tot[SPLIT ? 1 : ND], m0 = 0.0, m1 = 0.0, m2 = 0.0, base = 0.0;  // base: the state at the block's start
  if constexpr (!SPLIT) {
#pragma unroll
    for (int x = 0; x < ND; ++x) tot[x] = 0.0;
  }
  const uint32_t bn = block_steps(T);
  uint32_t ts = SPLIT ? blockIdx.y * bn : 0;
  do {
    const uint32_t n = T - ts < bn ? T - ts : bn;
    d64x4 g16[Sh::N16];
    double g4[Sh::N4 > 0 ? Sh::N4 : 1], s[Sh::NC], a1[Sh::NC], a2[Sh::NC];
#pragma unroll
    for (int x = 0; x < Sh::N16; ++x) g16[x] = d64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int x = 0; x < Sh::N4; ++x) g4[x] = 0.0;
#pragma unroll
    for (int q = 0; q < Sh::NC; ++q) s[q] = a1[q] = a2[q] = 0.0;
    double c = 0.0;                                  // the path of component l (lanes l < D)
    double mk = (double)n - 1.0 - (double)(l >> 4);  // te - (t + 1) of this lane's step

    for (uint32_t t0 = 0; t0 < n; t0 += R) {
      const int ns = n - t0 < (uint32_t)R ? (int)(n - t0) : R;
      // the round's normals
#pragma unroll
      for (int it = 0; it < 2; ++it) {
        const int q = l + 64 * it;
        if (q < calls) {
          float v[4];
          if constexpr (!FROM_NORMALS) normals4((uint64_t)(ts + t0) * D / 4 + q, seed, rng_stream, v);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            double z;
            if constexpr (FROM_NORMALS)
              z = 4 * q + j < ns * D ? zw[(size_t)(ts + t0) * D + 4 * q + j] : 0.0;
            else
              z = (double)v[j];
            wide_x[zo[it][j]] = z;
          }
        }
      }
      __syncthreads();
      // component l's path; the steps past the walk's end (its last round) are zeroed
      if (l < D) {
        double* const xc = wide_x + at(l, 0);
        double* const xz = wide_x + at(DB + l, 0);
        for (int t = ns; t < R; ++t) xz[t * 16] = 0.0;
        for (int t = 0; t < R; t += 4) {
          double z[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) z[j] = xz[(t + j) * 16];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            xc[(t + j) * 16] = c;
            c += z[j];
          }
        }
        for (int t = ns; t < R; ++t) xc[t * 16] = 0.0;
      }
      __syncthreads();
      const int groups = (ns + 3) / 4;
      for (int g = 0; g < groups; ++g) {
        double x[NT];
#pragma unroll
        for (int q = 0; q < NT; ++q) x[q] = wide_x[(q * R + 4 * g) * 16 + l];
        const double h = 0.5 * mk, w2 = fma(h, mk, -h);  // m and m (m - 1)/2
#pragma unroll
        for (int q = 0; q < Sh::NC; ++q) {
          s[q] += x[q];
          a1[q] = fma(mk, x[q], a1[q]);
          a2[q] = fma(w2, x[q], a2[q]);
        }
        mk -= 4.0;
#pragma unroll
        for (int q = 0; q < NT; ++q) g16[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[0], x[q], g16[q], 0, 0, 0);
        if constexpr (NB == 8) {
#pragma unroll
          for (int q = 1; q < NT; ++q)
            g16[NT + q - 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[1], x[q], g16[NT + q - 1], 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < Sh::NU; ++u) {
          // components 16 + 4 u .. + 3 in each of the four 4-row slots
          const double xu = wide_x[(R + 4 * g) * 16 + (l & 48) + 4 * u + (l & 3)];
#pragma unroll
          for (int q = 1; q < NT; ++q)
            g4[u * (NT - 1) + q - 1] =
                __builtin_amdgcn_mfma_f64_4x4x4f64(xu, x[q], g4[u * (NT - 1) + q - 1], 0, 0, 0);
        }
      }
      __syncthreads();
    }

    // S, A1, A2 of position 16 q + l % 16: the four step groups' shares
#pragma unroll
    for (int q = 0; q < Sh::NC; ++q) {
#pragma unroll
      for (int o = 16; o <= 32; o <<= 1) {
        s[q] += __shfl_xor(s[q], o);
        a1[q] += __shfl_xor(a1[q], o);
        a2[q] += __shfl_xor(a2[q], o);
      }
      if (l < 16) {
        sv[16 * q + l] = s[q];
        a1v[16 * q + l] = a1[q];
        a2v[16 * q + l] = a2[q];
      }
    }
    __syncthreads();
    auto grams = [&](int x) { return x < 4 * Sh::N16 ? g16[x / 4][x % 4] : g4[x - 4 * Sh::N16]; };
    if constexpr (SPLIT) {
      double* const o = acc + (size_t)blockIdx.y * block_moment_count(D) * ld + walk;
#pragma unroll
      for (int x = 0; x < ND; ++x) {
        int i, p;
        Sh::entry(x, l, i, p);
        if (p < DB) {
          if (i <= p && p < D) o[(size_t)blk_gc(D, i, p) * ld] = grams(x);
        } else if (i < D && p - DB < D) {
          o[(size_t)blk_ge(D, p - DB, i) * ld] = grams(x);
        }
      }
      if (l < D) {
        o[(size_t)blk_vec(D, 0, l) * ld] = sv[l];
        o[(size_t)blk_vec(D, 1, l) * ld] = a1v[l];
        o[(size_t)blk_vec(D, 2, l) * ld] = a2v[l];
        o[(size_t)blk_vec(D, 3, l) * ld] = c;
      }
      return;
    } else {
      // the block's terms: for row i and column j both are B_i q_j + (S_i b_j +
      // sum), with q, b = n B + S, B on a path column and E, 0 on a normals'
      const BlockConst bc = block_const(ts, n);
      if (l < D) {
        const double sl = sv[l];
        bv[l] = base;
        qv[l] = fma(bc.n, base, sl);
        bv[DB + l] = 0.0;
        qv[DB + l] = c;
        m0 += block_m0(bc, base, sl);
        m1 += block_m1(bc, base, sl, a1v[l]);
        m2 += block_m2(bc, base, sl, a1v[l], a2v[l]);
        base += c;
      }
      __syncthreads();
      // an opaque copy: the entries' indices are formed here, not kept in
      // registers across the block
      int lf = l;
      asm volatile("" : "+v"(lf));
#pragma unroll
      for (int x = 0; x < ND; ++x) {
        int i, p;
        Sh::entry(x, lf, i, p);
        if (i < D && (p < DB ? p < D : p - DB < D)) tot[x] += fma(bv[i], qv[p], fma(sv[i], bv[p], grams(x)));
      }
      __syncthreads();
      ts += n;
    }
  } while (!SPLIT && ts < T);

  if constexpr (!SPLIT) {
    const MomentScale sc = moment_scale(T);
    double* const o = acc + walk;
    int lf = l;
    asm volatile("" : "+v"(lf));
#pragma unroll
    for (int x = 0; x < ND; ++x) {
      int i, p;
      Sh::entry(x, lf, i, p);
      const double v = tot[x] * sc.dt;
      if (p < DB) {
        if (i <= p && p < D) {
          o[(size_t)(i * D + p) * ld] = v;
          o[(size_t)(p * D + i) * ld] = v;
        }
      } else if (i < D && p - DB < D) {
        o[(size_t)(D * D + (p - DB) * D + i) * ld] = v;
      }
    }
    if (l < D) store_vector_moments(sc, m0, m1, m2, base, o, D, l, ld, 0);
  }
}

// The walks' moments from their blocks' sums (part: n_walks per entry), in the
// order and with the operations of the kernel that takes the blocks in turn:
// 64 walks per workgroup, wave w of it row 4 blockIdx.y + w, columns
// 8 blockIdx.z .. + 7 of sum z c^T and sum c c^T.
__global__ __launch_bounds__(256) void wide_blocks_add(int D, uint32_t T, uint32_t n_walks,
                                                       const double* __restrict__ part, double* __restrict__ acc,
                                                       size_t ld) {
  constexpr int JW = 8;
  const int k = __builtin_amdgcn_readfirstlane(4 * blockIdx.y + (threadIdx.x >> 6)), j0 = JW * blockIdx.z;
  const size_t walk = (size_t)blockIdx.x * 64 + (threadIdx.x & 63);
  if (walk >= n_walks || k >= D) return;
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
      ge[q] += fma(bj, ek, fma(at(blk_vec(D, 0, j)), 0.0, at(blk_ge(D, k, j))));
      if (j >= k) gc[q] += block_bb(bc, bk, bj, sk, at(blk_vec(D, 0, j)), at(blk_gc(D, k, j)));
      b[q] = bj + at(blk_vec(D, 3, j));
    }
    if (j0 == 0) {
      const double x1 = at(blk_vec(D, 1, k)), x2 = at(blk_vec(D, 2, k));
      m0 += block_m0(bc, bk, sk);
      m1 += block_m1(bc, bk, sk, x1);
      m2 += block_m2(bc, bk, sk, x1, x2);
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

// A row-major matrix in LDS with a runtime pitch: m[i][j].
struct LdsMat {
  double* p;
  int pitch;
  __device__ __forceinline__ double* operator[](int i) const { return p + i * pitch; }
};

// LDS bytes of walk_eigen_wide for (model, dim): S11 (NX x (NX + 1)), S10 (NX x
// (D + 1)), P0, P1 (NX each) and the vector moments (6 D), NX = D + 1 for models
// 1 and 3, else D.
size_t wide_eigen_lds_bytes(int model, int D) {
  const size_t nx = (model == 1 || model == 3) ? (size_t)D + 1 : (size_t)D;
  return sizeof(double) * (nx * (nx + 1) + nx * ((size_t)D + 1) + 2 * nx + 6 * (size_t)D);
}

// Lane `from`'s value of x (from is wave-uniform).
__device__ __forceinline__ double lane_f64(double x, int from) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), from),
                          __builtin_amdgcn_readlane(__double2loint(x), from));
}

// One wave per walk: the model algebra of walk_eigen_fp64 (F = X - P Z with
// P = (sum X Z^T)(sum Z Z^T)^-1 on the projected rows; models 0..4 as in
// construct_f_matrix, src/johansen_statistics.rs:102-197), then the
// generalized eigenproblem of src/johansen_statistics.rs:24-47 as the
// symmetric one of M = W^T W, W = L^-1 S10, S11 = L L^T.  16,384 walks at dims
// 16, 24 and 32: 0.38, 0.77 and 1.47 ms with the walks dealt over the XCDs, the
// algebra in LDS and ratio counts; now 0.28, 0.55 and 1.01 ms.
template <int DP>
__global__ __launch_bounds__(64) void walk_eigen_wide(int model, int D, const double* __restrict__ acc, size_t ld,
                                                      uint32_t T, uint32_t n_walks, double* __restrict__ out) {
  // LDS sized by the launch for this (model, dim) (wide_eigen_lds_bytes):
  // sum b b^T and from it S11 (NX x NX, pitch NX + 1); sum e b^T and from it S10
  // (NX x D, pitch D + 1); the projections P0, P1; the vector moments.  Once the
  // rows of S11 and S10 are in registers, M (D x D, pitch D + 1) takes the
  // bytes of S11 and the broadcast vectors those of S10.
  extern __shared__ __align__(16) double wide_lds[];
  const int NX = (model == 1 || model == 3) ? D + 1 : D;
  const LdsMat Ls{wide_lds, NX + 1};
  const LdsMat Ws{wide_lds + NX * (NX + 1), D + 1};
  const LdsMat Ms{wide_lds, D + 1};
  double* const P0 = wide_lds + NX * (NX + 1) + NX * (D + 1);
  double* const P1 = P0 + NX;
  double* const V = P1 + NX;
  const int l = threadIdx.x;
  if (blockIdx.x >= n_walks) return;
  const size_t walk = xcd_walk(blockIdx.x, n_walks);
  const int NB = (model == 2 || model == 4) ? D - 1 : D;
  const int NZ = model == 4 ? 2 : ((model == 2 || model == 3) ? 1 : 0);
  auto A = [&](int e) -> double { return acc[(size_t)e * ld + walk]; };
  // the walk's moments to LDS, many loads in flight (one after the other, as the
  // algebra asks for them, they took 23 us of a walk's latency at dim 32)
  const int hr = l >> 5, lc = l & 31;  // row (of two at a time) and column of this lane
#pragma unroll
  for (int q = 0; q < 3; ++q)
    if (l + 64 * q < 6 * D) V[l + 64 * q] = A(2 * D * D + l + 64 * q);
  if (lc < D) {
#pragma unroll 8
    for (int i = hr; i < D; i += 2) {
      Ws[lc][i] = A(D * D + i * D + lc);
      if (lc <= i) Ls[i][lc] = A(i * D + lc);
    }
  }
  __syncthreads();
  auto GBB = [&](int i, int j) { return Ls[i][j]; };  // j <= i
  auto GEB = [&](int k, int j) { return Ws[j][k]; };
  auto MB = [&](int p, int i) { return V[p * D + i]; };
  auto ME = [&](int p, int k) { return V[(3 + p) * D + k]; };

  const double Tn = (double)T;
  const double dt = 1.0 / Tn;
  // closed forms of sum_t u_t^p, u_t = (t+1)/T, t = 0..T-1
  const double c1 = (Tn + 1.0) * 0.5;
  const double c2 = (Tn + 1.0) * (2.0 * Tn + 1.0) / (6.0 * Tn);
  const double c3 = (Tn + 1.0) * (Tn + 1.0) / (4.0 * Tn);
  const double c4 = (Tn + 1.0) * (2.0 * Tn + 1.0) * (3.0 * Tn * Tn + 3.0 * Tn - 1.0) / (30.0 * Tn * Tn * Tn);
  auto XZ = [&](int x, int z) -> double {
    if (x < NB) return MB(z, x);
    if (model == 2 || model == 3) return c1 - 0.5 * Tn;  // sum y, y = u - 1/2
    if (model == 4) return z == 0 ? c2 : c3;             // sum u^2, sum u^3
    return 0.0;
  };
  auto projected = [&](int x) -> bool { return model == 4 || ((model == 2 || model == 3) && x < NB); };
  auto XX = [&](int i, int j) -> double {
    if (i < NB && j < NB) return GBB(i, j);
    if (i >= NB && j >= NB) {
      if (model == 1) return Tn;
      if (model == 2 || model == 3) return c2 - c1 + 0.25 * Tn;  // sum (u - 1/2)^2
      return c4;
    }
    const int bi = i < NB ? i : j;
    if (model == 1) return MB(0, bi);
    if (model == 2 || model == 3) return MB(1, bi) - 0.5 * MB(0, bi);  // sum b y
    return MB(2, bi);                                                  // sum b u^2
  };
  auto EX = [&](int k, int j) -> double {
    if (j < NB) return GEB(k, j);
    if (model == 1) return ME(0, k);
    if (model == 2 || model == 3) return ME(1, k) - 0.5 * ME(0, k);
    return ME(2, k);
  };
  // ZZ^-1 in closed form: model 4: [[T, c1], [c1, c2]]^-1, det = (T^2 - 1)/12
  double zi00 = 0.0, zi01 = 0.0, zi11 = 0.0;
  if (NZ == 1) zi00 = dt;
  if (NZ == 2) {
    const double det = (Tn * Tn - 1.0) / 12.0;
    zi00 = c2 / det;
    zi01 = -c1 / det;
    zi11 = Tn / det;
  }
  if (l < NX) {
    double p0 = 0.0, p1 = 0.0;
    if (NZ == 1) p0 = XZ(l, 0) * zi00;
    if (NZ == 2) {
      const double a0 = XZ(l, 0), a1 = XZ(l, 1);
      p0 = a0 * zi00 + a1 * zi01;
      p1 = a0 * zi01 + a1 * zi11;
    }
    P0[l] = p0;
    P1[l] = p1;
  }
  __syncthreads();
  auto proj = [&](int i, int j) -> double {  // XZ_i ZZ^-1 ZX_j on the projected rows
    if (NZ == 0) return 0.0;
    if (projected(i)) return NZ == 2 ? P0[i] * XZ(j, 0) + P1[i] * XZ(j, 1) : P0[i] * XZ(j, 0);
    if (projected(j)) return NZ == 2 ? P0[j] * XZ(i, 0) + P1[j] * XZ(i, 1) : P0[j] * XZ(i, 0);
    return 0.0;
  };
  // S11 (lower triangle) and S10 = S01raw^T: S01raw = eX - eZ ZZ^-1 ZX
  for (int i = hr; i < NX; i += 2) {
    if (lc <= i) Ls[i][lc] = (XX(i, lc) - proj(i, lc)) * dt;
    if (i == 32 && lc == 0) Ls[32][32] = (XX(32, 32) - proj(32, 32)) * dt;
    if (lc < D) {
      double v = EX(lc, i);
      if (NZ > 0 && projected(i)) v -= NZ == 2 ? P0[i] * ME(0, lc) + P1[i] * ME(1, lc) : P0[i] * ME(0, lc);
      Ws[i][lc] = v;
    }
  }
  __syncthreads();

  // S11 = L L^T, W = L^-1 S10 and M = W^T W in one pass over L's columns: lane i
  // < NX keeps row i of S11 (a, from the current column on) and of S10 (b), lane
  // 63 - k row k of M (b).  Step j: lane j's pivot gives L_jj and W_j = S10_j /
  // L_jj; the column L_ij and W_j are broadcast through LDS; then
  //   S11_ik -= L_ij L_kj,   S10_i -= L_ij W_j,   M_k += W_j[k] W_j,
  // the last two one FMA of every lane.  At dim 32 with NX = 33 the last row of
  // S10 takes the lane of the last row of M: that row is the others' last
  // column, its diagonal entry summed by every lane.  Bound by the LDS reads of
  // the broadcasts (33 of 16 bytes per lane and step at dim 32).  In LDS, one
  // triangular loop after the other, the three took 50 us of a walk's latency at
  // dim 32 and now take 33; with the loads above, 16,384 walks 0.72 to 0.63 ms.
  bool pd = true;
  {
    double a[DP + 1], b[DP];
    const int lr = l < NX ? l : 0;
#pragma unroll
    for (int m = 0; m <= DP; ++m) {
      const double x = Ls[lr][m < NX ? m : 0];
      a[m] = l < NX && m <= l ? x : 0.0;
    }
#pragma unroll
    for (int m = 0; m < DP; ++m) {
      const double x = Ws[lr][m < D ? m : 0];
      b[m] = l < NX && m < D ? x : 0.0;
    }
    __syncthreads();
    double* const Wj = wide_lds + NX * (NX + 1);  // W_j, DP entries
    double* const Lj = Wj + DP;                      // column j from the diagonal on, 64 entries
    const bool last = D + NX > 64;                   // a row of M has no lane
    const int mk = 63 - l;                           // this lane's row of M
    const bool m_lane = l >= NX && mk < D;
    double dlast = 0.0;
    for (int j = 0; j < NX; ++j) {
      const double s = lane_f64(a[0], j);
      pd = pd && (s > 0.0);
      const double ljj = sqrt(s > 0.0 ? s : 1.0);
      const double inv = 1.0 / ljj;
      const double lij = l > j && l < NX ? a[0] * inv : 0.0;
      if (l >= j) Lj[l - j] = lij;
      if (l == j) {
#pragma unroll
        for (int m = 0; m < DP; ++m) Wj[m] = b[m] * inv;
      }
      __syncthreads();
      const double cb = l < NX ? -lij : (m_lane ? Wj[m_lane ? mk : 0] : 0.0);
      if (last) dlast = fma(Wj[D - 1], Wj[D - 1], dlast);
#pragma unroll
      for (int m = 0; m < DP; ++m) b[m] = fma(cb, Wj[m], b[m]);
#pragma unroll
      for (int m = 1; m <= DP; ++m) a[m - 1] = fma(-lij, Lj[m], a[m]);
      __syncthreads();  // every lane has read the column before the next step writes its own
    }
    if (m_lane) {
#pragma unroll
      for (int m = 0; m < DP; ++m)
        if (m < D) Ms[mk][m] = b[m];
      if (last) Ms[D - 1][mk] = b[DP - 1];  // D = DP = 32
    }
    if (last && l == 0) Ms[D - 1][D - 1] = dlast;
    __syncthreads();
  }

  // ---- Householder reduction of M to tridiagonal form: lane i keeps row i
  // of M in registers (columns padded to DP with zeros).  Step k broadcasts
  // column k below the diagonal (x) through LDS, every lane forms the same
  // reflector v = x - alpha e_{k+1}, tau = 2 / |v|^2 from it, lane i its entry
  // of p = tau M v, which is broadcast in turn; then w = p - (tau/2)(p.v) v and
  // lane i updates its row, M -= v w^T + w v^T on the trailing block.  d_k is
  // final once step k starts and e_k = alpha.  The scratch vectors (5 DP
  // doubles) use the bytes of W and P0, P1, at least D (D + 3) >= 5 DP doubles
  // since DP <= D + 7.
  double* const Xs = wide_lds + NX * (NX + 1);
  double* const Ps = Xs + DP;
  double* const Dg = Ps + DP;
  double* const Eg = Dg + DP;
  double* const EVs = Eg + DP;
  double row[DP];
  if (l < D) {
#pragma unroll
    for (int j = 0; j < DP; ++j) row[j] = j < D ? Ms[l][j < D ? j : 0] : 0.0;
  } else {
#pragma unroll
    for (int j = 0; j < DP; ++j) row[j] = 0.0;
  }
  if (l >= D && l < DP) {  // padding entries of the broadcast vectors stay 0
    Xs[l] = 0.0;
    Ps[l] = 0.0;
  }
#pragma unroll
  for (int k = 0; k < DP - 2; ++k) {
    if (k < D - 2) {
      const double xi = l > k ? row[k] : 0.0;
      if (l > k && l < D) Xs[l] = xi;
      __syncthreads();
      double v[DP];
      double sigma = 0.0;
#pragma unroll
      for (int j = k + 2; j < DP; ++j) {
        v[j] = Xs[j];
        sigma = fma(v[j], v[j], sigma);
      }
      const double x0 = Xs[k + 1];
      const double nrm = sqrt(fma(x0, x0, sigma));
      const double alpha = x0 > 0.0 ? -nrm : nrm;
      const double v0 = x0 - alpha;
      const double vn = fma(v0, v0, sigma);
      // tau = 0 when x = 0: the reflection is the identity, e_k = 0
      const double tau = vn > 0.0 ? 2.0 / vn : 0.0;
      v[k + 1] = v0;
      const double vi = l == k + 1 ? v0 : xi;
      double s = 0.0;
#pragma unroll
      for (int j = k + 1; j < DP; ++j) s = fma(row[j], v[j], s);
      const double pi = l > k ? tau * s : 0.0;
      if (l > k && l < D) Ps[l] = pi;
      __syncthreads();
      double pj[DP];
      double pv = 0.0;
#pragma unroll
      for (int j = k + 1; j < DP; ++j) {
        pj[j] = Ps[j];
        pv = fma(pj[j], v[j], pv);
      }
      const double K = 0.5 * tau * pv;
      const double wi = fma(-K, vi, pi);
#pragma unroll
      for (int j = k + 1; j < DP; ++j) {
        const double wj = fma(-K, v[j], pj[j]);
        row[j] = fma(-vi, wj, fma(-wi, v[j], row[j]));
      }
      if (l == 0) Eg[k] = tau > 0.0 ? alpha : x0;
      if (l == k) Dg[k] = row[k];
    }
  }
  // the last 2 x 2 block: d_{D-2}, d_{D-1} and e_{D-2} = M[D-1][D-2]
  double dii = 0.0, sub = 0.0;
#pragma unroll
  for (int j = 0; j < DP; ++j) {
    if (l == j) dii = row[j];
    if (l == j + 1) sub = row[j];
  }
  if (l == D - 2 || l == D - 1) Dg[l] = dii;
  if (l == D - 1) Eg[D - 2] = sub;
  __syncthreads();

  // ---- eigenvalue g (ascending) of the tridiagonal matrix by the P = 64 / D
  // lanes g, g + D, .., g + (P - 1) D: from the Gershgorin interval, each round
  // lane g + jD takes the Sturm count at the (j+1)-th of P equally spaced
  // interior points, the counts meet in a ballot, and every lane of the group
  // keeps the sub-interval whose upper point is the first count past g: (P + 1)-fold
  // per round, where bisection halves (P = 2 at D = 22..32, 4 at D <= 16).  Bound
  // by the counts' FP64 operations: with a reciprocal per term (16,384 walks at
  // dim 32) the rounds took 0.56 ms, with the minors themselves 0.24; one walk at
  // dim 32: 64 to 24 us.
  double dg[DP], e2[DP];
#pragma unroll
  for (int j = 0; j < DP; ++j) {
    dg[j] = j < D ? Dg[j < D ? j : 0] : 0.0;
    const double e = j < D - 1 ? Eg[j < D - 1 ? j : 0] : 0.0;
    e2[j] = e * e;
  }
  double lo, hi, pivmin;
  sturm_bounds<DP>(dg, e2, D, lo, hi, pivmin);
  const double scale = sturm_scale<DP>(dg, e2, D, lo, hi);
  const int P = 64 / D;  // >= 2 (D <= 32)
  const int grp = l % D, jp = l / D;  // lanes with jp >= P follow their group
  const double inv_sections = 1.0 / (double)(P + 1);
  int rounds = 0;  // (P + 1)^rounds >= 2^54: at most the width 54 halvings leave
  for (double w = 1.0; w > 0x1p-54; w *= inv_sections) ++rounds;
  for (int it = 0; it < rounds; ++it) {
    const double step = (hi - lo) * inv_sections;
    bool past = false;
    if (jp < P) past = sturm_count<DP>(dg, e2, D, lo + (double)(jp + 1) * step) > grp;
    const unsigned long long mask = __ballot(past) >> grp;  // bit q D: the group's point q
    int first = P;
#pragma unroll
    for (int q = 64 / (DP - (DP > 16 ? 7 : 3)) - 1; q >= 0; --q) first = (mask >> (q * D)) & 1ull ? q : first;
    if (first < P) hi = lo + (double)(first + 1) * step;
    if (first > 0) lo = lo + (double)first * step;
  }
  const double lam = 0.5 * (lo + hi) / scale;

  // |lambda| sorted descending (rank of each by lane), NX - D structural zeros
  if (l < D) EVs[l] = fabs(lam);
  __syncthreads();
  const double nan = __longlong_as_double(0x7FF8000000000000LL);
  double* o = out + walk * (size_t)NX;
  if (l < D) {
    const double ev = EVs[l];
    int rank = 0;
    for (int j = 0; j < D; ++j) {
      const double x = EVs[j];
      rank += (x > ev || (x == ev && j < l)) ? 1 : 0;
    }
    o[pd ? rank : l] = pd ? ev : nan;
  }
  if (l == 0 && NX > D) o[D] = pd ? 0.0 : nan;
}

// One wave per walk in whole rounds of the GPU's resident waves; the walks of
// the last, partial round get a wave per block, as in the kernels of dims
// 1..12 (a rest of 90% of a round is not split, for its sums' way through memory).
static uint32_t wide_turns(int d, uint32_t T, uint32_t n) {
  const int nb = (d + 3) / 4;
  const uint32_t round = 1024u * (nb <= 6 ? 4 : 3), rest = n % round;
  if (block_count(T) == 1) return n;
  return (uint64_t)rest * 100 >= (uint64_t)round * 90 ? n : n - rest;
}

size_t wide_part_doubles(int d, uint32_t T, uint32_t n) {
  return (size_t)block_count(T) * block_moment_count(d) * (n - wide_turns(d, T, n));
}

hipError_t launch_walk_moments_wide(int d, const uint32_t* seeds, const double* zin, uint32_t rng_stream, uint32_t T,
                                    uint32_t n, double* acc, size_t ld, double* part, size_t part_doubles,
                                    hipStream_t st) {
  if (d <= kMaxDim || d > kMaxWideDim) return hipErrorInvalidValue;
  auto go = [&](auto nb_tag, auto split_tag, const uint32_t* s, const double* z, uint32_t m, double* out, size_t ldo) {
    constexpr int NB = decltype(nb_tag)::value;
    constexpr bool SPLIT = decltype(split_tag)::value;
    const dim3 grid(m, SPLIT ? block_count(T) : 1);
    const size_t lds = sizeof(double) * WideShape<NB>::NT * 16 * (size_t)wide_round_steps(d);
    if (z)
      hipLaunchKernelGGL((walk_moments_wide<NB, true, SPLIT>), grid, dim3(64), lds, st, s, z, rng_stream, T, m, d, out,
                         ldo);
    else
      hipLaunchKernelGGL((walk_moments_wide<NB, false, SPLIT>), grid, dim3(64), lds, st, s, z, rng_stream, T, m, d, out,
                         ldo);
    return hipGetLastError();
  };
  auto go_d = [&](auto split_tag, const uint32_t* s, const double* z, uint32_t m, double* out, size_t ldo) {
    switch ((d + 3) / 4) {
      case 4: return go(IntTag<4>{}, split_tag, s, z, m, out, ldo);
      case 5: return go(IntTag<5>{}, split_tag, s, z, m, out, ldo);
      case 6: return go(IntTag<6>{}, split_tag, s, z, m, out, ldo);
      case 7: return go(IntTag<7>{}, split_tag, s, z, m, out, ldo);
      default: return go(IntTag<8>{}, split_tag, s, z, m, out, ldo);
    }
  };
  uint32_t turns = wide_turns(d, T, n);
  if (part == nullptr || part_doubles < wide_part_doubles(d, T, n)) turns = n;
  hipError_t e = hipSuccess;
  if (turns > 0) e = go_d(BoolTag<false>{}, seeds, zin, turns, acc, ld);
  if (e != hipSuccess || turns == n) return e;
  const uint32_t m = n - turns;
  if ((e = go_d(BoolTag<true>{}, seeds ? seeds + turns : nullptr, zin ? zin + (size_t)turns * T * d : nullptr, m, part,
                m)) != hipSuccess)
    return e;
  hipLaunchKernelGGL(wide_blocks_add, dim3((m + 63) / 64, (d + 3) / 4, (d + 7) / 8), dim3(256), 0, st, d, T, m, part,
                     acc + turns, ld);
  return hipGetLastError();
}

hipError_t launch_walk_eigen_wide(int model, int d, const double* acc, size_t ld, uint32_t T, uint32_t n, double* out,
                                  hipStream_t st) {
  if (d <= kMaxDim || d > kMaxWideDim || model < 0 || model > 4) return hipErrorInvalidValue;
  const size_t lds = wide_eigen_lds_bytes(model, d);
  if (d <= 16)
    hipLaunchKernelGGL(walk_eigen_wide<16>, dim3(n), dim3(64), lds, st, model, d, acc, ld, T, n, out);
  else if (d <= 24)
    hipLaunchKernelGGL(walk_eigen_wide<24>, dim3(n), dim3(64), lds, st, model, d, acc, ld, T, n, out);
  else
    hipLaunchKernelGGL(walk_eigen_wide<32>, dim3(n), dim3(64), lds, st, model, d, acc, ld, T, n, out);
  return hipGetLastError();
}

}  // namespace jne
