// jne_walk_mfma.hip -- mixed-precision moment pass on the matrix cores.
//
// Same output as walk_moments_fp64 (the canonical per-walk moments consumed by
// walk_eigen_fp64), computed as a split between FP64 per-segment terms and an
// MFMA Gram of small within-segment quantities.  With s = sqrt(1/T), z_t the
// unscaled normals, a segment of n <= 64 steps [ts, ts + n) starting at the
// FP64 state B0 = B_ts, k = t - ts and c_t = sum_{ts <= r < t} z_r - m with
// m = eps/2 (so b_t = B0 + s m + s c_t and e_t = s z_t):
//
//   sum b b^T   = sum_seg [n B0' B0'^T + s (B0' sig^T + sig B0'^T)] + s^2 sum c c^T
//   sum e b^T   = sum_seg [s eps B0'^T]                            + s^2 sum z c^T
//   sum u^p b   = sum_seg [B0' sum_seg u^p]                        + s   sum u^p c
//   sum u^p e   =                                                    s   sum u^p z
//
// (eps = sum_seg z, sig = sum_seg c, B0' = B0 + s m).  The bracketed terms are FP64, once per
// segment.  The rest comes from the Gram of the 32 rows
//
//   X = [z_0..z_{D-1}, 0.., c_0..c_{D-1} (from row 12), 0.., 1, k, k(k-1)/2, 0..]
//
// (the last three from row 24) over the segment's steps, accumulated by
// v_mfma_f32_32x32x16_{f16,bf16} on hi/lo (or hi/mid/lo) splits, or by
// v_mfma_f32_32x32x2f32 on FP32 values.  The rows 1, k, k(k-1)/2 are small
// integers, exact in every operand format, so sum u^p x with u_t = (ts+1+k)/T
// is formed without rounding u: the MFMA gives sum x, sum k x and
// sum k(k-1)/2 x per segment and the FP64 flush weights them by the segment's
// start ts.  The FP32 accumulators are flushed into FP64 once per segment, so
// FP32 rounding never spans more than 64 steps; the segment sums of z that
// drive the state B0 are formed in FP64 from the stored normals.
//
// One wave per walk.  A segment runs in three phases: the wave draws its
// normals into LDS rows (64 Philox calls per iteration; where a segment's
// calls are not whole iterations, the last one's spare lanes draw the next
// segment's first calls, and the calls are stored whole, for the scan to lay
// the rows from them); a scan lays the c rows beside them (lane (i, p)
// takes a block of steps of component i, sums it in FP64 for eps and writes
// each c_t as the FP32 rounding of an FP64 running sum); then lane l feeds
// row l%32 of X for 8 of every 16 steps (half l/32), read straight from its
// LDS row, as both the A and the B operand of X X^T.  Each lane keeps its
// share of the FP64 Gram in registers; it goes to LDS once, after the last
// segment, for the output.
//
// At dims 1, 2, 3, 4 and 6 one walk would leave most of the 32 x 32 tile and
// of the lanes idle, so a wave carries W = 12 / dim walks as the 12
// components of one walk of the kernel: walk w's components are rows
// w dim .. w dim + dim - 1 of each block, drawn from its own Philox stream,
// and the output keeps only the blocks on the diagonal (the products across
// walks are formed and dropped).  Every quantity a walk's output depends on is
// formed from that walk's own rows, so its results are those of a wave of its
// own.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/jne.h"
#include "jne_internal.h"
#include "jne_rng.h"
#include "jne_segments.h"

// Tuning: how many of a lane's Philox calls of a segment to unroll
// (independent chains for the scheduler, at the cost of registers: 2 is the
// most that fits beside the FP64 Gram without spills at dim 12, and runs
// 0.4% faster than 1); target waves per SIMD.
#ifndef JNE_MFMA_UNROLL_CALLS
#define JNE_MFMA_UNROLL_CALLS 2
#endif
#ifndef JNE_MFMA_UNROLL_CALLS_FP16X2
#define JNE_MFMA_UNROLL_CALLS_FP16X2 3
#endif
#ifndef JNE_MFMA_WAVES
#define JNE_MFMA_WAVES 4
#endif
// fp16 split: round-to-nearest hi (else truncated hi); add the lo*lo product
#ifndef JNE_MFMA_SPLIT_ROUND
#define JNE_MFMA_SPLIT_ROUND 1
#endif
#ifndef JNE_MFMA_LOLO
#define JNE_MFMA_LOLO 0
#endif
// unroll of the loop over a segment's 4 MFMA chunks
#ifndef JNE_MFMA_CHUNK_UNROLL
#define JNE_MFMA_CHUNK_UNROLL 4
#endif
// dims 1, 2, 3, 4 and 6: 12 / dim walks per wave, as the components of one
// 12-component walk of the kernel (0: one walk per wave at every dim)
#ifndef JNE_MFMA_PACK
#define JNE_MFMA_PACK 1
#endif

namespace jne {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __fp16 fp16x2 __attribute__((ext_vector_type(2)));

constexpr int kChunks = 4;     // 16-step MFMA chunks per segment
constexpr int kRowC = 12;      // first row of the c block
constexpr int kRowDet = 24;    // rows 24, 25, 26: 1, k, k(k-1)/2

// The FP64 Gram entries the output needs, compact in LDS:
//   column c in [12, 24) (the c block): rows 0..26  at (c - 12) * 28 + r
//   column c < 12 (the z block):        rows 24..26 at 336 + 3 c + (r - 24)
// The c-block pitch of 28 keeps every group of 4 rows 16-byte aligned.
//   symmetric form only, column c < 12: rows 12..23 at 372 + 12 c + (r - 12)
constexpr int kGramPitch = 28;
constexpr int kGramZ = 12 * kGramPitch;
constexpr int kGramT = kGramZ + 12 * 3;
constexpr int kGramSize = kGramT + 12 * 12;

template <int D>
struct MfmaShape {
  static constexpr int CALLS = kSegSteps * D / 4;       // Philox calls per segment
  static constexpr int IT = (CALLS + 63) / 64;          // call iterations per lane
  // By-seed form, when a segment's calls are not whole 64-call iterations:
  // the spare lanes of a segment's last iteration draw the next segment's
  // first calls (the same Philox counters), which wait in an LDS buffer of
  // at most OVF calls, so the segments draw CALLS calls each on average
  // instead of 64 IT.
  static constexpr bool CARRY = CALLS > 64 && CALLS % 64 != 0;
  static constexpr int OVF = CARRY ? 64 - gcd_int(CALLS, 64) : 1;
  static constexpr int ZP = kSegSteps + 4;              // LDS pitch of one row (floats)
  static constexpr int NG = (D * D + 63) / 64;          // (i, j) grid entries per lane
  // scan: SP lanes per component, BS steps each (the last BL): as many lanes as
  // the wave has for D components, up to 8 (a lane's offset takes SP - 1
  // additions, so more lanes of fewer steps gain nothing).  Against four lanes
  // of 16 steps, 100,000 walks at T = 10,000: dim 9 14.0 to 13.4 ms, dim 10
  // 14.5 to 14.1, dim 11 15.3 to 15.2; five lanes of 13 steps at dim 12 gain
  // nothing over four whose steps are whole 16-byte units (15.5 and 15.5 ms).
  static constexpr int BS = D == 12 ? 16 : 64 / D < 8 ? (kSegSteps + 64 / D - 1) / (64 / D) : kSegSteps / 8;
  static constexpr int SP = (kSegSteps + BS - 1) / BS;
  static constexpr int BL = kSegSteps - (SP - 1) * BS;
  static_assert(SP * D <= 64 && BL >= 1 && BL <= BS, "the scan lanes cover a segment");
  // LDS rows, each at its row index of X: z (0..D-1), c (12..12+D-1), 1, k,
  // k(k-1)/2 (24..26); the compact FP64 Gram takes the same bytes after the
  // last segment
  static constexpr int ROW_BYTES = (kRowDet + 3) * ZP * 4;
  static constexpr int RAW_BYTES = ROW_BYTES > kGramSize * 8 ? ROW_BYTES : kGramSize * 8;
  static_assert(D <= kRowC, "dim must fit the z block");
};

// Per-component FP64 values of a segment (see the kernel).
struct alignas(16) SegVec {
  double P, b, Q, E;
};

// hi/lo splits by truncation: hi keeps the leading bits (exact in the narrow
// format), lo = x - hi is exact in FP32 and rounded once to the narrow format.
__device__ __forceinline__ float trunc_bits(float x, uint32_t mask) {
  return __uint_as_float(__float_as_uint(x) & mask);
}

// A wave-uniform double in scalar registers (VALU instructions read them as
// operands), keeping two vector registers free.
__device__ __forceinline__ double uniform_f64(double x) {
  const uint64_t b = (uint64_t)__double_as_longlong(x);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// MFMA of one 16-step chunk.  x[8] are this lane's 8 row values (steps 8h + k,
// or 2k + h for the interleaved FP32 form).
//
// Symmetric form (kSymmetric): of the cross products of the split pieces only
// one of each transposed pair is formed -- acc2 gets hi lo^T but not
// lo hi^T = (hi lo^T)^T -- and the wave's FP64 Gram accumulates
// F = acc + 2 acc2 for rows 0..23.  The Gram is then (F + F^T) / 2, formed once
// per walk from the two transposed entries, which restores
// hi hi^T + hi lo^T + lo hi^T: one MFMA per chunk fewer.  Rows 24..26 (the
// constants 1, k, k(k-1)/2 with k < 64, at most 1,953) are exact in fp16, so
// their lo is zero, acc + acc2 is already their full product and the
// per-segment sums read it directly.  In bf16 (8 significant bits) k(k-1)/2 is
// not exact, so the bf16 forms keep both cross products.
#ifndef JNE_MFMA_SYM
#define JNE_MFMA_SYM 1
#endif
template <int PREC>
struct ChunkMfma;

template <>
struct ChunkMfma<JNE_PREC_MFMA_FP16X2> {
  static constexpr bool kInterleaved = false;
  static constexpr bool kSymmetric = JNE_MFMA_SYM;
  __device__ __forceinline__ static void run(const float (&x)[8], floatx16& acc, floatx16& acc2) {
    half8 hi, lo;
#if JNE_MFMA_SPLIT_ROUND
    // hi = x rounded to fp16 (packed pairs); x - hi is exact in fp32, and
    // v_dot2_f32_f16 forms it from the packed pair directly: (hi0, hi1).(-1, 0) + x0
    const fp16x2 m0 = {(__fp16)-1.0f, (__fp16)0.0f}, m1 = {(__fp16)0.0f, (__fp16)-1.0f};
#pragma unroll
    for (int k = 0; k < 8; k += 2) {
      fp16x2 hp;
      hp[0] = (__fp16)x[k];
      hp[1] = (__fp16)x[k + 1];
      hi[k] = (_Float16)hp[0];
      hi[k + 1] = (_Float16)hp[1];
      lo[k] = (_Float16)__builtin_amdgcn_fdot2(hp, m0, x[k], false);
      lo[k + 1] = (_Float16)__builtin_amdgcn_fdot2(hp, m1, x[k + 1], false);
    }
#else
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float h = trunc_bits(x[k], 0xFFFFE000u);  // 11 significant bits
      hi[k] = (_Float16)h;
      lo[k] = (_Float16)(x[k] - h);
    }
#endif
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, hi, acc, 0, 0, 0);
    acc2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, lo, acc2, 0, 0, 0);
    if constexpr (!kSymmetric) acc2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, hi, acc2, 0, 0, 0);
#if JNE_MFMA_LOLO
    // lo lo^T is symmetric: in the symmetric form it joins hi hi^T
    if constexpr (kSymmetric)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, lo, acc, 0, 0, 0);
    else
      acc2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, lo, acc2, 0, 0, 0);
#endif
  }
};

template <>
struct ChunkMfma<JNE_PREC_MFMA_BF16X2> {
  static constexpr bool kInterleaved = false;
  static constexpr bool kSymmetric = false;
  __device__ __forceinline__ static void run(const float (&x)[8], floatx16& acc, floatx16& acc2) {
    bf16x8 hi, lo;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float h = trunc_bits(x[k], 0xFFFF0000u);  // 8 significant bits
      hi[k] = (__bf16)h;
      lo[k] = (__bf16)(x[k] - h);
    }
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, hi, acc, 0, 0, 0);
    acc2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, lo, acc2, 0, 0, 0);
    acc2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, hi, acc2, 0, 0, 0);
  }
};

template <>
struct ChunkMfma<JNE_PREC_MFMA_BF16X3> {
  static constexpr bool kInterleaved = false;
  static constexpr bool kSymmetric = false;
  __device__ __forceinline__ static void run(const float (&x)[8], floatx16& acc, floatx16& acc2) {
    bf16x8 hi, mi, lo;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float h = trunc_bits(x[k], 0xFFFF0000u);
      const float r1 = x[k] - h;
      const float m = trunc_bits(r1, 0xFFFF0000u);
      hi[k] = (__bf16)h;
      mi[k] = (__bf16)m;
      lo[k] = (__bf16)(r1 - m);
    }
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, hi, acc, 0, 0, 0);
    acc2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, mi, acc2, 0, 0, 0);
    acc2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(mi, hi, acc2, 0, 0, 0);
    acc2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, lo, acc2, 0, 0, 0);
    acc2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, hi, acc2, 0, 0, 0);
    acc2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(mi, mi, acc2, 0, 0, 0);
  }
};

template <>
struct ChunkMfma<JNE_PREC_MFMA_FP32> {
  static constexpr bool kInterleaved = true;
  static constexpr bool kSymmetric = false;
  __device__ __forceinline__ static void run(const float (&x)[8], floatx16& acc, floatx16&) {
#pragma unroll
    for (int m = 0; m < 8; ++m) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[m], x[m], acc, 0, 0, 0);
  }
};

// The compensated FP32 VALU check (JNE_PREC_FP32_KAHAN) runs the same
// segment split with the MFMA Gram replaced by FP32 products of the same X
// rows (z, c, 1, k, k(k-1)/2) added into Kahan-compensated FP32 sums, one
// per Gram entry the flush reads: for each c column the z, c and constant
// rows, for each z column the rows k and k(k-1)/2.  Lane l owns entries
// l, l + 64, ...; each segment's sums go to an LDS tile of doubles
// (sum - compensation, formed in FP64) that every lane reads in the MFMA
// output layout, so the flush is shared with the MFMA precisions.
template <int D>
struct KahanShape {
  static constexpr int PER_C = 2 * D + 3;            // rows per c column
  static constexpr int NE = D * PER_C + 2 * D;       // entries per segment
  static constexpr int NQ = (NE + 63) / 64;          // entries per lane
  static constexpr int COLS = kRowC + D;             // tile columns (X rows 0..11+D)
};

// X rows (i, j) of entry e of the compensated Gram (see KahanShape).
template <int D>
__device__ __forceinline__ void kahan_entry(int e, int& i, int& j) {
  using K = KahanShape<D>;
  if (e < D * K::PER_C) {
    const int jc = e / K::PER_C, r = e - jc * K::PER_C;
    j = kRowC + jc;
    i = r < D ? r : r < 2 * D ? kRowC + (r - D) : kRowDet + (r - 2 * D);
  } else {
    const int ez = e - D * K::PER_C;
    j = ez >> 1;
    i = kRowDet + 1 + (ez & 1);
  }
}

__device__ __forceinline__ void kahan_add(float& s, float& c, float x) {
#pragma clang fp contract(off)
  const float y = x - c;
  const float t = s + y;
  c = (t - s) - y;
  s = t;
}

// Philox calls of a segment unrolled: by-seed form only (the from-normals
// form has no Philox chains to overlap), whole iterations only, and not with
// the three-way bf16 split, whose operands leave no registers for it.  The
// fp16x2 pass keeps three calls in flight, all of a dim-12 segment's three
// iterations: within its 128 VGPRs with one walk per wave; packed waves spill 6
// registers at dims 3 and 6 and are still 24 and 12% faster than with two
// (65,536 walks at T = 5,000: 1.74 to 1.33 ms and 2.97 to 2.61), whose third
// iteration is a loop of its own.  The other operand splits hold more
// registers and keep two.
template <int D, int PREC, bool FROM_NORMALS>
struct CallUnroll {
  static constexpr int U =
      PREC == JNE_PREC_MFMA_FP16X2 ? JNE_MFMA_UNROLL_CALLS_FP16X2 : JNE_MFMA_UNROLL_CALLS;
  static constexpr int value = (U > 1 && !FROM_NORMALS && PREC != JNE_PREC_MFMA_BF16X3 && MfmaShape<D>::CALLS % 64 == 0)
                                   ? (MfmaShape<D>::IT < U ? MfmaShape<D>::IT : U)
                                   : 1;
};

// The per-segment FP64 terms, shared by the kernel that takes a walk's segments
// in turn and the one that adds them up from memory (mfma_segments_add), so that
// both perform the same operations.
struct SegLen {
  double n, a, s1, s2;  // steps, ts + 1, sum u, sum u^2 over the segment
};
__device__ __forceinline__ SegLen seg_len(uint32_t ts, uint32_t n, double dt, double dt2) {
  // sum over the segment of u^p, u = (t+1)/T, in closed form:
  // sum_{k<n} (A + k)^p with A = ts + 1, n <= 64:
  // n A^p + p A^(p-1) n(n-1)/2 (+ n(n-1)(2n-1)/6 for p = 2).  Positive
  // terms and exact integers: no division and no cancellation, unlike the
  // difference of the two cubic prefix sums
  SegLen v;
  v.n = (double)n;
  v.a = (double)ts + 1.0;
  const double k1 = (double)(n * (n - 1) / 2), k2 = (double)(n * (n - 1) * (2 * n - 1) / 6);
  v.s1 = (v.n * v.a + k1) * dt;
  v.s2 = ((v.n * v.a) * v.a + (2.0 * v.a) * k1 + k2) * dt2;
  return v;
}
__device__ __forceinline__ double seg_state(double b0, double s, double eps, float& m) {
  m = (float)(0.5 * eps);
  return b0 + s * (double)m;
}
__device__ __forceinline__ void seg_pq(SegVec& v, double n, double s, double sig) {
  v.P = n * v.b + s * sig;
  v.Q = s * sig;
}
// rows 24..26 hold sum x, sum k x, sum k(k-1)/2 x: added as sum x, sum u x,
// sum u^2 x with u = (a + k)/T
__device__ __forceinline__ void seg_det(double* g, double a, double dt, double dt2, double P0, double P1, double P2) {
  g[0] += P0;
  g[1] += (a * P0 + P1) * dt;
  g[2] += ((a * a) * P0 + (2.0 * a + 1.0) * P1 + 2.0 * P2) * dt2;
}

// Target waves per SIMD, at least and at most.  At most JNE_MFMA_WAVES for fp32 at
// the small dims with a wave per walk, whose registers and LDS leave room for a 17th
// wave per CU: one SIMD of four then ran five, and the others waited for it (8,000
// walks of 1,000 x 5: 242 us so, 225 with four).
constexpr int min_waves(int prec) { return prec == JNE_PREC_FP32_KAHAN ? 2 : JNE_MFMA_WAVES; }
constexpr int max_waves(int d, int prec) { return prec == JNE_PREC_MFMA_FP32 && d <= 8 ? JNE_MFMA_WAVES : 8; }

// D: components of the wave (W walks of D / W each).  SPLIT: segments
// kSplitSegs blockIdx.y .. + 3 of the wave's walks, to acc (the layout at kSegFloats).
template <int D, int PREC, bool FROM_NORMALS, int W = 1, bool SPLIT = false>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(min_waves(PREC), max_waves(D, PREC))))
void walk_moments_mfma(const uint32_t* __restrict__ seeds, const double* __restrict__ zin, uint32_t rng_stream,
                       uint32_t T, uint32_t n_walks, double* __restrict__ acc, size_t ld) {
  constexpr int DW = D / W;  // components of one walk
  static_assert(D % W == 0 && (W == 1 || MfmaShape<D>::CALLS % 64 == 0), "packed walks need whole iterations");
  using Sh = MfmaShape<D>;
  constexpr int ZP = Sh::ZP, NG = Sh::NG, SP = Sh::SP, BS = Sh::BS;
  constexpr bool kKahan = PREC == JNE_PREC_FP32_KAHAN;
  using Op = ChunkMfma<kKahan ? JNE_PREC_MFMA_FP32 : PREC>;
  constexpr bool kSym = !kKahan && Op::kSymmetric;
  using KS = KahanShape<D>;

  // Row r of X lives in LDS row r: the segment's normals z (rows 0..D-1), its
  // c rows (12..12+D-1) and the constant rows 1, k, k(k-1)/2 (24..26), written
  // once.  With a pitch of 17 16-byte units, the 8 lanes of a 128-bit read
  // group (8 consecutive rows) fall in distinct banks.  After the last
  // segment the same bytes hold the FP64 Gram.
  __shared__ __align__(16) unsigned char rows_raw[Sh::RAW_BYTES];
  float(*const xs)[ZP] = reinterpret_cast<float(*)[ZP]>(rows_raw);
  float(*const zbuf)[ZP] = xs;
  float(*const cbuf)[ZP] = xs + kRowC;
  double* const gram = reinterpret_cast<double*>(rows_raw);
  // sums of the scan blocks, block p of component i at [EP + p][i].  With fewer than
  // eight scan lanes the EP = SP - 1 rows before a lane's own are those of the
  // blocks before it and zeros, read again as its offset.  With eight (dims 5, 7
  // and 8) a lane selects from the sums it has read: seven more LDS reads cost a
  // wave alone 3-5% and the batches of up to a wave or two per SIMD with it (dim 8,
  // T = 1,000, bf16x3: 5,000 walks 158 to 149 us, 1 walk 72 to 70; dim 5, fp16x2: 701
  // walks 61.5 to 59, 100,000 walks 1.232 to 1.202 ms).
  constexpr int EP = SP < 8 ? SP - 1 : 0;
  __shared__ __align__(16) double vecs[(SP + EP + 11) * D];  // one array: no padding between its parts
  double(*const eps_part)[D] = reinterpret_cast<double(*)[D]>(vecs);
  // (not with the three-way bf16 split, whose operands leave no registers for it)
  constexpr bool kCarry = Sh::CARRY && !FROM_NORMALS && PREC != JNE_PREC_MFMA_BF16X3 && PREC != JNE_PREC_FP32_KAHAN;
  __shared__ float4 ovf[kCarry ? Sh::OVF : 1];  // calls drawn ahead for the next segment
  // the segment's calls in the order drawn (step-major: component i of step t at
  // t D + i), in the c rows' bytes until the scan lays the z rows from it: one
  // 16-byte store per call, where a call's four rows and steps, which change
  // from call to call at these dims, took 112 of its 590 issue cycles (100,000
  // walks at T = 10,000, dim 9: 14.7 to 14.0 ms)
  static_assert(!kCarry || Sh::CALLS * 4 <= D * ZP, "a segment's calls fit the c rows");
  float4* const zcall = reinterpret_cast<float4*>(&xs[kRowC][0]);
  double* const seg_eps = vecs + (SP + EP) * D;
  double* const b0s = seg_eps + D;  // B at the segment start (FP64)
  // per component j of a segment: b = B0 + s m (the state the centred c rows
  // are relative to), P = n b + s sig, Q = s sig, E = s eps, so that the
  // segment adds b_i P_j + Q_i b_j to sum b b^T and E_i b_j to sum e b^T
  __shared__ SegVec seg[D];
  double* const mb = b0s + D;  // 3 D: sum over segments of B0' sum_seg u^p (lanes l < 3D)
  // 2 D: Gram rows 24..26 of the c columns, then of the z columns
  double(*const gd)[3] = reinterpret_cast<double(*)[3]>(mb + 3 * D);
  // the compensated check's per-segment Gram entries, [X row][X column]
  __shared__ double gk[kKahan ? kRowDet + 3 : 1][kKahan ? KS::COLS : 1];

  const int l = threadIdx.x;
  const int row = l & 31;  // also the accumulator column
  const int h = l >> 5;
  const uint32_t n_groups = (n_walks + W - 1) / W;
  if (blockIdx.x >= n_groups) return;  // whole wave exits together
  // the wave's first walk
  const size_t walk = (size_t)(SPLIT ? blockIdx.x : xcd_walk(blockIdx.x, n_groups)) * W;
  uint32_t seed = 0;
  if constexpr (!FROM_NORMALS && W == 1) seed = seeds[walk];
  const double* zw = FROM_NORMALS ? zin + walk * (size_t)T * DW : nullptr;
  // packed walks: a segment's Philox call c belongs to walk c / (16 DW) (a
  // walk draws 16 DW calls per segment); the walks' seeds, in LDS
  __shared__ uint32_t wseed[W];
  if constexpr (W > 1 && !FROM_NORMALS) {
    if (l < W) wseed[l] = seeds[walk + l < n_walks ? walk + l : n_walks - 1];
    __syncthreads();
  }

  const bool is_z = row < D;
  const bool is_c = row >= kRowC && row < kRowC + D;
  // LDS row feeding this lane's row of X: its own; rows 27..31 read rows
  // 19..23 (distinct banks from rows 24..26 in their read group).  Their Gram
  // entries, and those of the rows of unused components (dim < 12, zero), are
  // never read.
  const float* const xrow = xs[row < kRowDet + 3 ? row : row - 8];

  // the rows of unused components (dim < 12) zero, then the constant rows,
  // exact small integers (k(k-1)/2 <= 2016)
  if constexpr (D < kRowC) {
    for (int r = D; r < kRowC; ++r)
      for (int t = l; t < ZP; t += 64) {
        xs[r][t] = 0.0f;
        xs[kRowC + r][t] = 0.0f;
      }
  }
  for (int t = l; t < ZP; t += 64) {
    const float kf = (float)t;
    xs[kRowDet][t] = 1.0f;
    xs[kRowDet + 1][t] = kf;
    xs[kRowDet + 2][t] = kf * (kf - 1.0f) * 0.5f;
  }

  // FP64 Gram in registers: g[v] sums accumulator v of every segment, Gram
  // element [8(v/4) + 4h + v%4][l%32].  The output needs, on a c column, rows
  // 0..23 (v = 0..11 on both halves) and rows 24..26 (v = 12..14 on the
  // lower half), and on a z column rows 24..26; rows 24..26 are summed in LDS.
  double g[12];
#pragma unroll
  for (int v = 0; v < 12; ++v) g[v] = 0.0;
  // rows 24..26 (v = 12..14 on the lower half) of the c and z columns: in LDS
  const bool det_lane = h == 0 && (is_c || is_z);
  double* const gdl = gd[is_c ? row - kRowC : D + (row < D ? row : 0)];
  for (int e = l; e < 6 * D; e += 64) gd[e / 3][e % 3] = 0.0;

  // (i, j) grid entries of this lane: e = l + 64 g
  int gi[NG], gj[NG];
#pragma unroll
  for (int q = 0; q < NG; ++q) {
    const int e = l + 64 * q;
    gi[q] = e < D * D ? e / D : 0;
    gj[q] = e < D * D ? e % D : 0;
  }
  double bbA[NG], ebA[NG];
#pragma unroll
  for (int q = 0; q < NG; ++q) bbA[q] = ebA[q] = 0.0;
  // the compensated check: this lane's Gram entries as LDS row offsets; the
  // entries no lane computes (rows of unused components) stay zero
  int kei[kKahan ? KS::NQ : 1], kej[kKahan ? KS::NQ : 1];
  if constexpr (kKahan) {
    for (int e = l; e < (kRowDet + 3) * KS::COLS; e += 64) (&gk[0][0])[e] = 0.0;
#pragma unroll
    for (int q = 0; q < KS::NQ; ++q) {
      int i = 0, j = 0;
      if (l + 64 * q < KS::NE) kahan_entry<D>(l + 64 * q, i, j);
      kei[q] = i;
      kej[q] = j;
    }
  }
  const int mp = l / D, mi = l % D;  // moment vector entry (power mp, component mi) for l < 3D
  const CallPos<D> pos0(l);          // normals of this lane's first Philox call in a segment
  // scan lane (component si, block sp): steps [sp BS, sp BS + BS) of a segment
  const int si = l % D, sp = l / D;
  const bool scan_lane = l < SP * D;

  for (int e = l; e < EP * D; e += 64) eps_part[e / D][e % D] = 0.0;
  if (l < D) b0s[l] = 0.0;
  if (l < 3 * D) mb[l] = 0.0;
  // walk constants: uniform, held in scalar registers
  const double dt = uniform_f64(1.0 / (double)T);
  const double s = uniform_f64(sqrt(dt));
  const double dt2 = uniform_f64(dt * dt);
  const uint32_t rounds = segment_count(T);
  const uint32_t r0 = SPLIT ? blockIdx.y * kSplitSegs : 0;
  uint32_t drawn = r0 * (uint32_t)Sh::CALLS;  // calls drawn so far (carry form): a multiple of 64

  // one segment; the partial last segment (T not a multiple of 64) runs a copy
  // with the step masks, so the loop over full segments carries none of them
  auto segment = [&](uint32_t r, auto tail_tag) {
    constexpr bool tail = decltype(tail_tag)::value;
    const uint32_t ts = r * kSegSteps;
    // ---- normals of the segment -> LDS
    // Wave priority: low while drawing (long runs of independent VALU work),
    // high from the scan to the flush, whose LDS round trips and MFMA
    // dependences leave gaps that the other waves' drawing then fills.
    __builtin_amdgcn_s_setprio(0);
    if constexpr (kCarry) {
      // calls [r CALLS, drawn) came with the previous segment's last iteration
      const int pending = (int)(drawn - r * (uint32_t)Sh::CALLS);
      if (l < pending) zcall[l] = ovf[l];
      // the rest, 64 calls per iteration; calls past the segment (spare lanes
      // of the last iteration) wait in ovf for the next one
      const uint32_t need = (r + 1) * (uint32_t)Sh::CALLS - drawn;
      const int nit = (int)((need + 63) / 64);
      int c = pending + l;  // this lane's call, counted from the segment's first
      for (int j = 0; j < nit; ++j) {
        float v[4];
        normals4(drawn + 64u * j + l, seed, rng_stream, v);  // 32-bit counter (kMaxSteps)
        float4* const dst = c < Sh::CALLS ? zcall + c : ovf + (c - Sh::CALLS);
        *dst = make_float4(v[0], v[1], v[2], v[3]);
        c += 64;
      }
      drawn += 64u * (uint32_t)nit;
    } else if constexpr (W > 1) {
      // call c: local call cl of walk w, whose normals 4 cl .. 4 cl + 3 are
      // (step, component) of that walk, component i -> row w DW + i
#pragma unroll CallUnroll<D, PREC, FROM_NORMALS>::value
      for (int j = 0; j < Sh::IT; ++j) {
        const int c = l + 64 * j;
        const int w = c / (16 * DW), cl = c - w * (16 * DW);
        float v[4];
        if constexpr (!FROM_NORMALS) normals4((uint32_t)((uint64_t)ts * DW / 4) + cl, wseed[w], rng_stream, v);
        const CallPos<DW> p(cl);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          int tl, i;
          p.at(jj, tl, i);
          const uint32_t t = ts + tl;
          float z;
          if constexpr (FROM_NORMALS) {
            const size_t wk = walk + w < n_walks ? (size_t)w : 0;
            z = t < T ? (float)zw[wk * (size_t)T * DW + (size_t)t * DW + i] : 0.0f;
          } else {
            z = (!tail || t < T) ? v[jj] : 0.0f;
          }
          zbuf[w * DW + i][tl] = z;
        }
      }
    } else {
    CallPos<D> pos = pos0;
#pragma unroll CallUnroll<D, PREC, FROM_NORMALS>::value
    for (int j = 0; j < Sh::IT; ++j) {
      const int c = l + 64 * j;
      if (Sh::IT * 64 != Sh::CALLS && c >= Sh::CALLS) break;
      float v[4];
      if constexpr (!FROM_NORMALS) normals4((uint32_t)((uint64_t)ts * D / 4) + c, seed, rng_stream, v);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        int tl, i;
        pos.at(jj, tl, i);
        const uint32_t t = ts + tl;
        float z;
        if constexpr (FROM_NORMALS)
          z = t < T ? (float)zw[(size_t)t * D + i] : 0.0f;
        else
          z = (!tail || t < T) ? v[jj] : 0.0f;
        zbuf[i][tl] = z;
      }
      pos.template advance<64>();
    }
    }
    __syncthreads();

    __builtin_amdgcn_s_setprio(2);
    // ---- scan, part 1: lane (si, sp) sums its block of component si in FP64:
    // the partial sums give the segment's eps, which drives the FP64 state,
    // and the offsets of the c rows in the blocks after it
    const auto block = [&](auto step) {  // step(j) for the steps sp BS + j of the lane's block
#pragma unroll
      for (int j = 0; j < Sh::BL; ++j) step(j);
      if constexpr (Sh::BL < BS) {
        if (sp < SP - 1) {
#pragma unroll
          for (int j = Sh::BL; j < BS; ++j) step(j);
        }
      }
    };
    float zb[BS];
    if (scan_lane) {
      float* const zrow = &zbuf[si][sp * BS];
      const float* const drawn_z = reinterpret_cast<const float*>(zcall) + sp * (BS * D) + si;
      double e = 0.0;
      block([&](int j) {
        if constexpr (kCarry) {
          const float z = drawn_z[j * D];
          zb[j] = (!tail || ts + (uint32_t)(sp * BS + j) < T) ? z : 0.0f;
          zrow[j] = zb[j];
        } else {
          zb[j] = zrow[j];
        }
        e = j ? e + (double)zb[j] : (double)zb[j];  // (no 0.0 + first term: one add fewer)
      });
      eps_part[EP + sp][si] = e;
    }
    __syncthreads();

    // ---- scan, part 2: eps of component si; the c rows are centred on m =
    // eps/2 (an FP32 value): c_t = sum_{ts <= q < t} z_q - m halves their mean
    // square, so the FP32 accumulation rounds less, and b_t = (B0 + s m) + s c_t.
    // Steps at or beyond T get c = 0 (their z are 0), so they add nothing.
    if (scan_lane) {
      double ep[SP];
#pragma unroll
      for (int p = 0; p < SP; ++p) ep[p] = eps_part[EP + p][si];
      double e = ep[0];
#pragma unroll
      for (int p = 1; p < SP; ++p) e += ep[p];
      float m;
      const double bm = seg_state(SPLIT ? 0.0 : b0s[si], s, e, m);
      // running sum in FP64 (exact but for FP64 rounding): each c_t is then
      // rounded to FP32 once
      double c = -(double)m;
#pragma unroll
      for (int p = 0; p < SP - 1; ++p) {
        if constexpr (EP > 0)
          c += eps_part[sp + p][si];
        else
          c += p < sp ? ep[p] : 0.0;
      }
      float* const crow = &cbuf[si][sp * BS];
      block([&](int j) {
        crow[j] = (!tail || ts + (uint32_t)(sp * BS + j) < T) ? (float)c : 0.0f;
        c += (double)zb[j];
      });
      if (sp == 0) {
        seg_eps[si] = e;
        if constexpr (!SPLIT) {
          seg[si].b = bm;
          seg[si].E = s * e;
        }
      }
    }
    __syncthreads();

    // ---- the segment's Gram of X: f[v] is element [8(v/4) + 4h + v%4][l%32]
    // (the 32x32 MFMA output layout)
    using F = typename std::conditional<SPLIT, float, double>::type;
    F f[16];
    if constexpr (kKahan) {
      // FP32 products in Kahan-compensated FP32 sums, then to LDS
      float ks[KS::NQ], kc[KS::NQ];
#pragma unroll
      for (int q = 0; q < KS::NQ; ++q) ks[q] = kc[q] = 0.0f;
#pragma unroll 2
      for (int k4 = 0; k4 < kSegSteps / 4; ++k4) {
#pragma unroll
        for (int q = 0; q < KS::NQ; ++q) {
          const float4 a = *reinterpret_cast<const float4*>(&xs[kei[q]][4 * k4]);
          const float4 b = *reinterpret_cast<const float4*>(&xs[kej[q]][4 * k4]);
          kahan_add(ks[q], kc[q], a.x * b.x);
          kahan_add(ks[q], kc[q], a.y * b.y);
          kahan_add(ks[q], kc[q], a.z * b.z);
          kahan_add(ks[q], kc[q], a.w * b.w);
        }
      }
#pragma unroll
      for (int q = 0; q < KS::NQ; ++q)
        if (l + 64 * q < KS::NE) gk[kei[q]][kej[q]] = (double)ks[q] - (double)kc[q];
      __syncthreads();
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int i = 8 * (v / 4) + 4 * h + v % 4;
        f[v] = (i < kRowDet + 3 && row < KS::COLS) ? gk[i][row] : 0.0;
      }
    } else {
      // 4 chunks of 16 steps on the matrix cores
      floatx16 accm = {}, accc = {};
#pragma unroll JNE_MFMA_CHUNK_UNROLL
      for (int ch = 0; ch < kChunks; ++ch) {
        const int off = 16 * ch;
        float x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = xrow[off + (Op::kInterleaved ? 2 * k + h : 8 * h + k)];
        Op::run(x, accm, accc);
      }
#pragma unroll
      for (int v = 0; v < 16; ++v)
        f[v] = (F)((kSym && v < 12) ? __builtin_fmaf(2.0f, accc[v], accm[v]) : accm[v] + accc[v]);
    }
    if constexpr (SPLIT) {
      static_assert(kSym, "the split layout is that of the symmetric form");
      double* const od = acc + ((size_t)blockIdx.x * rounds + r) * kSegDoubles;
      float* const o = reinterpret_cast<float*>(od);
      const int j = is_c ? row - kRowC : row;
      if (is_c) {
#pragma unroll
        for (int v = 0; v < 12; ++v) o[24 * v + 12 * h + j] = f[v];
      }
      if (is_z) {
#pragma unroll
        for (int v = 4; v < 12; ++v) {
          const int rw = 8 * (v / 4) + 4 * h + v % 4;
          if (rw >= kRowC) o[288 + 12 * (rw - kRowC) + j] = f[v];
        }
      }
      if (det_lane) {
#pragma unroll
        for (int v = 12; v < 15; ++v) o[432 + 24 * (v - 12) + (is_c ? j : 12 + j)] = f[v];
      }
      if (l < D) od[kSegFloats / 2 + l] = seg_eps[l];
      __syncthreads();
      return;
    } else {

    // ---- segment end
    // f[12] on the lower half is row 24 (the ones row): sum_seg x_col
    const SegLen sl = seg_len(ts, (tail ? T : ts + kSegSteps) - ts, dt, dt2);
    if (h == 0 && is_c) {
      seg_pq(seg[row - kRowC], sl.n, s, f[12]);
    }
    __syncthreads();
    {
      // flush into the FP64 Gram; on the z columns sum x is the FP64 eps
      const double P0 = is_z ? seg_eps[row] : f[12];
#pragma unroll
      for (int v = 0; v < 12; ++v) g[v] += f[v];
      if (det_lane) seg_det(gdl, sl.a, dt, dt2, P0, f[13], f[14]);
    }
    // FP64 per-segment terms on the (i, j) grid
#pragma unroll
    for (int q = 0; q < NG; ++q) {
      if (l + 64 * q < D * D) {
        const SegVec& vi = seg[gi[q]];
        const SegVec& vj = seg[gj[q]];
        bbA[q] = fma(vi.b, vj.P, fma(vi.Q, vj.b, bbA[q]));
        ebA[q] = fma(vi.E, vj.b, ebA[q]);
      }
    }
    if (l < 3 * D) {
      mb[l] += seg[mi].b * (mp == 0 ? sl.n : mp == 1 ? sl.s1 : sl.s2);
    }
    __syncthreads();
    // the next reads of b0s come two barriers into the next segment
    if (l < D) b0s[l] += s * seg_eps[l];
    }
  };
  const uint32_t full = T / kSegSteps;
  const uint32_t r1 = SPLIT && full > r0 + kSplitSegs ? r0 + kSplitSegs : full;
  for (uint32_t r = r0; r < r1; ++r) segment(r, BoolTag<false>{});
  if (r1 == full && full < rounds && (!SPLIT || full < r0 + kSplitSegs)) segment(full, BoolTag<true>{});
  if constexpr (SPLIT) return;

  // Lane indices of the output, recomputed from an opaque copy of the lane id
  // (an empty asm statement: no instruction), so that the compiler does not
  // keep the ones computed before the segment loop alive across it.
  int lx = l;
  asm volatile("" : "+v"(lx));
  const int xrow_ = lx & 31, xh = lx >> 5;
  const bool xc = xrow_ >= kRowC && xrow_ < kRowC + D, xz = xrow_ < D;

  // the Gram entries the output reads, into LDS over the row buffers (their
  // last reads came before the last segment's barriers): c lanes rows 0..23 of
  // their column, the lower half also rows 24..26; z lanes rows 24..26, and in
  // the symmetric form also rows 12..23 (the transposes of the z rows of the c
  // columns)
  if (xc) {
    double2* const gcol = reinterpret_cast<double2*>(gram + (xrow_ - kRowC) * kGramPitch + 4 * xh);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      gcol[4 * q] = make_double2(g[4 * q], g[4 * q + 1]);
      gcol[4 * q + 1] = make_double2(g[4 * q + 2], g[4 * q + 3]);
    }
  }
  if constexpr (kSym) {
    if (xz) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int r0 = 8 * q + 4 * xh;  // this lane's rows r0..r0+3 of the column
        if (r0 >= kRowC) {
          double2* const gt = reinterpret_cast<double2*>(gram + kGramT + 12 * xrow_ + (r0 - kRowC));
          gt[0] = make_double2(g[4 * q], g[4 * q + 1]);
          gt[1] = make_double2(g[4 * q + 2], g[4 * q + 3]);
        }
      }
    }
  }
  if (xh == 0 && (xc || xz)) {
    double* const gdet = xc ? gram + (xrow_ - kRowC) * kGramPitch + kRowDet : gram + kGramZ + 3 * xrow_;
    const double* const src = gd[xc ? xrow_ - kRowC : D + xrow_];
    gdet[0] = src[0];
    gdet[1] = src[1];
    gdet[2] = src[2];
  }
  __syncthreads();

  const double s2 = s * s;
  // canonical layout: [0, D^2) sum b b^T, [D^2, 2D^2) sum e b^T, then
  // sum b, sum u b, sum u^2 b, sum e, sum u e, sum u^2 e
#pragma unroll
  for (int q = 0; q < NG; ++q) {
    const int e = lx + 64 * q;
    if (e < D * D) {
      const int i = e / D, j = e % D;
      const int lo = i < j ? i : j, hi = i < j ? j : i;  // one triangle: exactly symmetric
      // symmetric form: the mean of the two transposed entries
      const double gbb = kSym ? 0.5 * (gram[hi * kGramPitch + kRowC + lo] + gram[lo * kGramPitch + kRowC + hi])
                              : gram[hi * kGramPitch + kRowC + lo];
      const double geb = kSym ? 0.5 * (gram[j * kGramPitch + i] + gram[kGramT + 12 * i + j]) : gram[j * kGramPitch + i];
      const double vbb = bbA[q] + s2 * gbb;
      const double veb = ebA[q] + s2 * geb;
      if constexpr (W == 1) {
        acc[(size_t)e * ld + walk] = vbb;
        acc[(size_t)(D * D + e) * ld + walk] = veb;
      } else {
        // packed walks: the blocks on the diagonal, in each walk's own layout
        const int w = i / DW, iw = i - w * DW, jw = j - w * DW;
        if (j / DW == w && walk + w < n_walks) {
          acc[(size_t)(iw * DW + jw) * ld + walk + w] = vbb;
          acc[(size_t)(DW * DW + iw * DW + jw) * ld + walk + w] = veb;
        }
      }
    }
  }
  if (lx < 3 * D) {
    const int xp = lx / D, xi = lx % D;
    const double vb = mb[lx] + s * gram[xi * kGramPitch + kRowDet + xp];
    const double ve = s * gram[kGramZ + 3 * xi + xp];
    const int w = xi / DW, iw = xi - w * DW;
    if (walk + w < n_walks) {
      acc[(size_t)(2 * DW * DW + xp * DW + iw) * ld + walk + w] = vb;
      acc[(size_t)(2 * DW * DW + (3 + xp) * DW + iw) * ld + walk + w] = ve;
    }
  }
}

// The moments of a split batch's walks from their segments: one workgroup per
// wave of walks, thread e < D^2 entry (i, j) of sum b b^T and sum e b^T, the next
// 3 D threads the vector moments; each adds the segments in order with the
// operations of walk_moments_mfma's flush and output.
template <int D, int W>
__global__ __launch_bounds__(192) void mfma_segments_add(uint32_t T, uint32_t n_walks, const double* __restrict__ part,
                                                         double* __restrict__ acc, size_t ld) {
  constexpr int DW = D / W;
  static_assert(D * D + 3 * D <= 192, "one thread per entry");
  const int e = threadIdx.x;
  if (e >= D * D + 3 * D) return;
  const size_t walk = (size_t)blockIdx.x * W;
  const uint32_t rounds = segment_count(T);
  const double* const p0 = part + (size_t)blockIdx.x * rounds * kSegDoubles;
  const double dt = 1.0 / (double)T, s = sqrt(dt), dt2 = dt * dt, s2 = s * s;
  auto len = [&](uint32_t r) {
    const uint32_t ts = r * kSegSteps;
    return seg_len(ts, T - ts < (uint32_t)kSegSteps ? T - ts : (uint32_t)kSegSteps, dt, dt2);
  };
  // Gram row `rw` (0..23) of c column j, and c row i (0..11) of z column j
  auto c_at = [](int rw, int j) { return 24 * (4 * (rw / 8) + rw % 4) + 12 * ((rw / 4) & 1) + j; };
  auto z_at = [](int i, int j) { return 288 + 12 * i + j; };
  if (e < D * D) {
    const int i = e / D, j = e - (e / D) * D;
    const int lo = i < j ? i : j, hi = i < j ? j : i;
    const int o0 = c_at(kRowC + lo, hi), o1 = c_at(kRowC + hi, lo), o2 = c_at(i, j), o3 = z_at(j, i);
    double g0 = 0.0, g1 = 0.0, g2 = 0.0, g3 = 0.0, bbA = 0.0, ebA = 0.0, bi = 0.0, bj = 0.0;
#pragma unroll 4
    for (uint32_t r = 0; r < rounds; ++r) {
      const double* const eps = p0 + (size_t)r * kSegDoubles + kSegFloats / 2;
      const float* const f = reinterpret_cast<const float*>(p0 + (size_t)r * kSegDoubles);
      const double ei = eps[i], ej = eps[j];
      const double n = len(r).n;
      SegVec vi, vj;
      float m;
      vi.b = seg_state(bi, s, ei, m);
      vi.E = s * ei;
      seg_pq(vi, n, s, (double)f[432 + i]);
      vj.b = seg_state(bj, s, ej, m);
      seg_pq(vj, n, s, (double)f[432 + j]);
      g0 += (double)f[o0];
      g1 += (double)f[o1];
      g2 += (double)f[o2];
      g3 += (double)f[o3];
      bbA = fma(vi.b, vj.P, fma(vi.Q, vj.b, bbA));
      ebA = fma(vi.E, vj.b, ebA);
      bi += s * ei;
      bj += s * ej;
    }
    const int w = i / DW, iw = i - w * DW, jw = j - w * DW;
    if (j / DW == w && walk + w < n_walks) {
      acc[(size_t)(iw * DW + jw) * ld + walk + w] = bbA + s2 * (0.5 * (g0 + g1));
      acc[(size_t)(DW * DW + iw * DW + jw) * ld + walk + w] = ebA + s2 * (0.5 * (g2 + g3));
    }
  } else {
    const int q = e - D * D, xp = q / D, xi = q - xp * D;
    double gc[3] = {0.0, 0.0, 0.0}, gz[3] = {0.0, 0.0, 0.0}, mb = 0.0, b0 = 0.0;
#pragma unroll 4
    for (uint32_t r = 0; r < rounds; ++r) {
      const float* const f = reinterpret_cast<const float*>(p0 + (size_t)r * kSegDoubles) + 432 + xi;
      const double eps = p0[(size_t)r * kSegDoubles + kSegFloats / 2 + xi];
      const SegLen sl = len(r);
      float m;
      const double b = seg_state(b0, s, eps, m);
      seg_det(gc, sl.a, dt, dt2, (double)f[0], (double)f[24], (double)f[48]);
      seg_det(gz, sl.a, dt, dt2, eps, (double)f[12 + 24], (double)f[12 + 48]);
      mb += b * (xp == 0 ? sl.n : xp == 1 ? sl.s1 : sl.s2);
      b0 += s * eps;
    }
    const int w = xi / DW, iw = xi - w * DW;
    if (walk + w < n_walks) {
      acc[(size_t)(2 * DW * DW + xp * DW + iw) * ld + walk + w] = mb + s * (xp == 0 ? gc[0] : xp == 1 ? gc[1] : gc[2]);
      acc[(size_t)(2 * DW * DW + (3 + xp) * DW + iw) * ld + walk + w] =
          s * (xp == 0 ? gz[0] : xp == 1 ? gz[1] : gz[2]);
    }
  }
}

static uint32_t mfma_wave_walks(int d) { return JNE_MFMA_PACK && 12 % d == 0 ? 12 / d : 1; }
size_t mfma_part_doubles(int d, int precision, uint32_t T, uint32_t n) {
  if (precision != JNE_PREC_MFMA_FP16X2) return 0;
  return segment_split_doubles((n + mfma_wave_walks(d) - 1) / mfma_wave_walks(d), T);
}

template <int D, int PREC>
static hipError_t launch_mfma_dp(const uint32_t* seeds, const double* zin, uint32_t rng_stream, uint32_t T,
                                 uint32_t n, double* acc, size_t ld, double* part, size_t part_doubles,
                                 hipStream_t st) {
  // dims dividing 12: 12 / D walks per wave as one 12-component walk
  constexpr int W = (JNE_MFMA_PACK && 12 % D == 0) ? 12 / D : 1;
  constexpr int DS = D * W;
  const unsigned grid = (n + W - 1) / W;
  if constexpr (PREC == JNE_PREC_MFMA_FP16X2) {
    const size_t need = mfma_part_doubles(D, PREC, T, n);
    if (zin == nullptr && part != nullptr && need > 0 && need <= part_doubles) {
      hipLaunchKernelGGL((walk_moments_mfma<DS, PREC, false, W, true>), dim3(grid, split_chunks(T)), dim3(64), 0, st,
                         seeds, zin, rng_stream, T, n, part, ld);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      hipLaunchKernelGGL((mfma_segments_add<DS, W>), dim3(grid), dim3(192), 0, st, T, n, part, acc, ld);
      return hipGetLastError();
    }
  }
  if (zin != nullptr)
    hipLaunchKernelGGL((walk_moments_mfma<DS, PREC, true, W>), dim3(grid), dim3(64), 0, st, seeds, zin, rng_stream, T,
                       n, acc, ld);
  else
    hipLaunchKernelGGL((walk_moments_mfma<DS, PREC, false, W>), dim3(grid), dim3(64), 0, st, seeds, zin, rng_stream,
                       T, n, acc, ld);
  return hipGetLastError();
}

template <int PREC>
static hipError_t launch_mfma_p(int d, const uint32_t* seeds, const double* zin, uint32_t rng_stream, uint32_t T,
                                uint32_t n, double* acc, size_t ld, double* part, size_t part_doubles,
                                hipStream_t st) {
  switch (d) {
#define JNE_CASE(DD) \
  case DD:           \
    return launch_mfma_dp<DD, PREC>(seeds, zin, rng_stream, T, n, acc, ld, part, part_doubles, st);
    JNE_CASE(1) JNE_CASE(2) JNE_CASE(3) JNE_CASE(4) JNE_CASE(5) JNE_CASE(6)
    JNE_CASE(7) JNE_CASE(8) JNE_CASE(9) JNE_CASE(10) JNE_CASE(11) JNE_CASE(12)
#undef JNE_CASE
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_walk_moments_mfma(int d, int precision, const uint32_t* seeds, const double* zin,
                                    uint32_t rng_stream, uint32_t T, uint32_t n, double* acc, size_t ld,
                                    double* part, size_t part_doubles, hipStream_t st) {
  switch (precision) {
    case JNE_PREC_MFMA_FP16X2: 
      return launch_mfma_p<JNE_PREC_MFMA_FP16X2>(d, seeds, zin, rng_stream, T, n, acc, ld, part, part_doubles, st);
    case JNE_PREC_MFMA_BF16X2: 
      return launch_mfma_p<JNE_PREC_MFMA_BF16X2>(d, seeds, zin, rng_stream, T, n, acc, ld, part, part_doubles, st);
    case JNE_PREC_MFMA_BF16X3: 
      return launch_mfma_p<JNE_PREC_MFMA_BF16X3>(d, seeds, zin, rng_stream, T, n, acc, ld, part, part_doubles, st);
    case JNE_PREC_MFMA_FP32: 
      return launch_mfma_p<JNE_PREC_MFMA_FP32>(d, seeds, zin, rng_stream, T, n, acc, ld, part, part_doubles, st);
    case JNE_PREC_FP32_KAHAN: 
      return launch_mfma_p<JNE_PREC_FP32_KAHAN>(d, seeds, zin, rng_stream, T, n, acc, ld, part, part_doubles, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace jne
