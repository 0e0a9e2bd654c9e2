// jne_quantile.hip -- percentiles of a device array by bucket selection.
//
// The percentile rule is the reference's get_percentile_value
// (src/simulation_analyzers.rs:4-18): rank p*(n-1) in the ascending array,
// linear interpolation between the neighbouring order statistics.  Only the
// order statistics at floor(rank) and ceil(rank) are needed, so instead of
// sorting the whole array:
//
//   1. min, max and a NaN flag per workgroup (one pass; it also clears the
//      histogram);
//   2. a histogram of kBuckets equal-width value buckets between min and max
//      (one pass).  The bucket index floor((x - min) * scale) is monotone in
//      x, so the k-th smallest value lies in the bucket where the cumulative
//      count first exceeds k;
//   3. one workgroup finds the bucket (and the rank inside it) of every needed
//      order statistic;
//   4. the values of those few buckets are gathered (one pass);
//   5. one workgroup sorts them in LDS, reads the order statistics and writes
//      the results to pinned host memory.
//
// An array of at most kMaxCand values is sorted in LDS at once.
//
// 10^6 values: 127 to 63 us a call.  Before, 1,024 workgroups met in atomics on
// one min and max (27 us, now 6 with a min and max per workgroup), 512 added
// their 8,192 counts (25 us, now 62 groups in 8), the select walked its scans
// in one thread (26 us, now 8) and a copy brought the results back.  Ending a
// pass in its last workgroup instead of a launch was slower: the fence that
// makes the others' writes visible cost 70 us.
//
// When the gathered buckets hold more than kMaxCand values (heavy ties, or a
// few extreme values stretching the bucket width), or min/max are not finite,
// the order statistics come from a radix select instead: eight passes of
// 8-bit digits over the order-preserving 64-bit keys, MSB first.  Either way
// the results are the exact order statistics, identical to sorting.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "../../include/jne.h"
#include "jne_internal.h"

namespace jne {
namespace {

constexpr int kBuckets = 8192;
constexpr int kMaxCand = 4096;
constexpr int kMaxRanks = 2 * kMaxPercentiles;

// Order-preserving map of a double to an unsigned key (NaNs sort past the
// infinities and are caught separately).
__device__ __forceinline__ uint64_t ord_key(double x) {
  const uint64_t b = (uint64_t)__double_as_longlong(x);
  return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

// Bucket selection state of one array, written by qs_hist and read by qs_gather.
struct Sel {
  uint32_t status;  // kSelect, kRadix, kNan or kEqual
  uint32_t nb;      // distinct buckets holding needed order statistics
  uint32_t m;       // values gathered
  uint32_t bucket[kMaxRanks];
  uint32_t base[kMaxRanks];     // first slot of bucket j's values
  uint32_t fill[kMaxRanks];     // gather cursors
  uint32_t pos[kMaxRanks];      // slot of rank k among the sorted gathered values
};
constexpr uint32_t kSelect = 0, kRadix = 1, kNan = 2, kEqual = 3;

// Everything a launch needs, passed by value: no host-to-device copies.
struct QsArgs {
  const double* x[kMaxArrays];
  uint64_t n;
  int np;
  uint64_t ranks[kMaxRanks];  // floor and ceil of rank i at 2i, 2i+1
  double prank[kMaxPercentiles];
};

// Workgroups of a pass over an array: up to kMaxGroups, for the histogram (whose
// LDS copy each group adds to the array's) of up to about 16,384 values each until
// kMaxGroups take more.
constexpr unsigned kMaxGroups = 256;
unsigned pass_groups(uint64_t n, uint64_t per) {
  const uint64_t g = (n + per - 1) / per;
  return g < kMaxGroups ? (unsigned)g : kMaxGroups;
}

// Per-array device scratch: the min and max keys and NaN flags of the first
// pass's workgroups, the histogram, the selection state and the gathered values.
struct QsArray {
  uint64_t lo[kMaxGroups], hi[kMaxGroups];
  uint32_t nan[kMaxGroups];
  uint32_t groups;  // of the first pass
  uint32_t hist[kBuckets];
  Sel sel;
  double cand[kMaxCand];
};
struct QsResult {
  uint32_t status, pad;
  double out[kMaxPercentiles];
};

constexpr int kThreads = 1024;

// min and max key over a workgroup (every thread gets them)
__device__ __forceinline__ void block_minmax(uint64_t& lo, uint64_t& hi, uint64_t (&smin)[16], uint64_t (&smax)[16]) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t a = __shfl_xor((unsigned long long)lo, o), b = __shfl_xor((unsigned long long)hi, o);
    lo = a < lo ? a : lo;
    hi = b > hi ? b : hi;
  }
  const int t = threadIdx.x;
  if ((t & 63) == 0) {
    smin[t >> 6] = lo;
    smax[t >> 6] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    lo = smin[w] < lo ? smin[w] : lo;
    hi = smax[w] > hi ? smax[w] : hi;
  }
}

__global__ __launch_bounds__(kThreads) void qs_minmax(QsArgs args, QsArray* arr) {
  __shared__ uint64_t smin[16], smax[16];
  const double* __restrict__ x = args.x[blockIdx.y];
  QsArray& a = arr[blockIdx.y];
  const int t = threadIdx.x;
  uint64_t lo = ~0ull, hi = 0ull;
  bool nan = false;
#pragma unroll 4
  for (uint64_t i = (uint64_t)blockIdx.x * kThreads + t; i < args.n; i += (uint64_t)gridDim.x * kThreads) {
    const double v = x[i];
    nan |= isnan(v);
    const uint64_t k = ord_key(v);
    lo = k < lo ? k : lo;
    hi = k > hi ? k : hi;
  }
  block_minmax(lo, hi, smin, smax);
  nan = __syncthreads_or(nan);
  if (t == 0) {
    a.lo[blockIdx.x] = lo;
    a.hi[blockIdx.x] = hi;
    a.nan[blockIdx.x] = nan;
  }
  for (unsigned b = blockIdx.x * kThreads + t; b < (unsigned)kBuckets; b += gridDim.x * kThreads) a.hist[b] = 0u;
  if (blockIdx.x == 0 && t == 0) a.groups = gridDim.x;
}

__device__ __forceinline__ double from_key(uint64_t k) {
  return __longlong_as_double((long long)((k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k));
}

// The bucket grid of an array from its min and max: kSelect when it is
// usable, else the reason (every thread of every workgroup decides the same).
struct Grid {
  double lo, scale;
  uint64_t min_key;
  uint32_t status;
};
__device__ __forceinline__ Grid grid_of(const QsArray& a, uint64_t (&smin)[16], uint64_t (&smax)[16]) {
  Grid g;
  const unsigned t = threadIdx.x, n = a.groups;
  uint64_t lo = t < n ? a.lo[t] : ~0ull, hi = t < n ? a.hi[t] : 0ull;
  const bool nan = __syncthreads_or(t < n && a.nan[t] != 0);
  block_minmax(lo, hi, smin, smax);
  g.min_key = lo;
  g.lo = from_key(lo);
  const double top = from_key(hi), width = top - g.lo;
  g.scale = (double)kBuckets / width;
  g.status = nan ? kNan
             : g.lo == top ? kEqual
             : isfinite(g.lo) && isfinite(top) && isfinite(width) && width > 0.0 ? kSelect : kRadix;
  return g;
}

__device__ __forceinline__ uint32_t bucket_of(double v, const Grid& g) {
  const double f = (v - g.lo) * g.scale;  // >= 0, monotone in v
  return f < (double)(kBuckets - 1) ? (uint32_t)f : (uint32_t)(kBuckets - 1);
}

// The interpolation of get_percentile_value on the order statistics s(lo), s(hi).
__device__ __forceinline__ double interp(double rank, uint64_t lo, uint64_t hi, double slo, double shi) {
  if (lo == hi) return slo;
  const double w = rank - (double)lo;
  return slo * (1.0 - w) + shi * w;
}

__global__ __launch_bounds__(kThreads) void qs_hist(QsArgs args, QsArray* arr, QsResult* res) {
  __shared__ uint32_t h[kBuckets];
  __shared__ uint64_t smin[16], smax[16];
  const double* __restrict__ x = args.x[blockIdx.y];
  QsArray& a = arr[blockIdx.y];
  const int t = threadIdx.x;
  const Grid g = grid_of(a, smin, smax);
  if (blockIdx.x == 0) {
    QsResult& r = res[blockIdx.y];
    if (t == 0) a.sel.status = r.status = g.status;
    if (g.status == kEqual && t < args.np) r.out[t] = from_key(g.min_key);  // every order statistic is the minimum
  }
  if (g.status != kSelect) return;  // the same for every workgroup
  for (int b = t; b < kBuckets; b += kThreads) h[b] = 0u;
  __syncthreads();
#pragma unroll 4
  for (uint64_t i = (uint64_t)blockIdx.x * kThreads + t; i < args.n; i += (uint64_t)gridDim.x * kThreads)
    atomicAdd(&h[bucket_of(x[i], g)], 1u);
  __syncthreads();
  for (int b = t; b < kBuckets; b += kThreads)
    if (h[b]) atomicAdd(&a.hist[b], h[b]);
}

// One workgroup per array: the buckets of the needed ranks; thread t scans
// buckets kPer t .. + kPer - 1.
__global__ __launch_bounds__(kThreads) void qs_select(QsArgs args, QsArray* arr, QsResult* res) {
  constexpr int kPer = kBuckets / kThreads;
  __shared__ uint32_t wsum[16];
  // of rank k: its bucket, the rank inside it and the bucket's count
  __shared__ uint32_t rb[kMaxRanks], rl[kMaxRanks], rc[kMaxRanks];
  QsArray& a = arr[blockIdx.y];
  Sel* const sel = &a.sel;
  const int t = threadIdx.x;
  if (sel->status != kSelect) return;
  const int nr = 2 * args.np;
  uint32_t c[kPer], sum = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    c[j] = a.hist[kPer * t + j];
    sum += c[j];
  }
  uint32_t incl = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(incl, o);
    if ((t & 63) >= o) incl += y;
  }
  if ((t & 63) == 63) wsum[t >> 6] = incl;
  __syncthreads();
  uint32_t cum = incl - sum;
  for (int w = 0; w < (t >> 6); ++w) cum += wsum[w];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    for (int k = 0; k < nr; ++k) {
      if (args.ranks[k] >= cum && args.ranks[k] < (uint64_t)cum + c[j]) {
        rb[k] = (uint32_t)(kPer * t + j);
        rl[k] = (uint32_t)args.ranks[k] - cum;
        rc[k] = c[j];
      }
    }
    cum += c[j];
  }
  __syncthreads();
  // thread k: its bucket's place among the distinct ones in increasing order,
  // and the slots of the gathered values before it
  if (t < nr) {
    uint32_t nb = 0, m = 0, at = 0, base = 0;
    bool first = true;  // no earlier rank has this bucket
    for (int j = 0; j < nr; ++j) {
      bool fj = true;
      for (int i = 0; i < j; ++i) fj &= rb[i] != rb[j];
      if (j == t) first = fj;
      if (!fj) continue;
      ++nb;
      m = m + rc[j] < m ? 0xFFFFFFFFu : m + rc[j];
      if (rb[j] < rb[t]) {
        ++at;
        base += rc[j];
      }
    }
    if (first) {
      sel->bucket[at] = rb[t];
      sel->base[at] = base;
      sel->fill[at] = 0u;
    }
    sel->pos[t] = base + rl[t];
    if (t == 0) {
      sel->nb = nb;
      sel->m = m;
      if (m > (uint32_t)kMaxCand) sel->status = res[blockIdx.y].status = kRadix;
    }
  }
}

// Sorts v[0..len) of a workgroup by key (len a power of two).
__device__ void sort_keys(uint64_t* v, uint32_t len) {
  for (uint32_t size = 2; size <= len; size <<= 1)
    for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
      for (uint32_t i = threadIdx.x; i < len / 2; i += kThreads) {
        const uint32_t lo = 2 * i - (i & (stride - 1)), hi = lo + stride;
        const uint64_t x0 = v[lo], x1 = v[hi];
        if ((x0 > x1) == ((lo & size) == 0)) {
          v[lo] = x1;
          v[hi] = x0;
        }
      }
      __syncthreads();
    }
}

__global__ __launch_bounds__(kThreads) void qs_gather(QsArgs args, QsArray* arr) {
  __shared__ uint64_t smin[16], smax[16];
  __shared__ uint32_t bk[kMaxRanks];
  const double* __restrict__ x = args.x[blockIdx.y];
  QsArray& a = arr[blockIdx.y];
  Sel* const sel = &a.sel;
  if (sel->status != kSelect) return;  // the same for every thread
  const Grid g = grid_of(a, smin, smax);
  const uint32_t nb = sel->nb;
  const int t = threadIdx.x;
  if (t < (int)nb) bk[t] = sel->bucket[t];
  __syncthreads();
#pragma unroll 4
  for (uint64_t i = (uint64_t)blockIdx.x * kThreads + t; i < args.n; i += (uint64_t)gridDim.x * kThreads) {
    const double xi = x[i];
    const uint32_t b = bucket_of(xi, g);
    for (uint32_t j = 0; j < nb; ++j)
      if (b == bk[j]) {
        const uint32_t slot = atomicAdd(&sel->fill[j], 1u);
        a.cand[sel->base[j] + slot] = xi;
      }
  }
}

// One workgroup per array: the gathered values sorted in LDS, the percentiles.
__global__ __launch_bounds__(kThreads) void qs_finish(QsArgs args, const QsArray* arr, QsResult* res) {
  __shared__ uint64_t v[kMaxCand];
  const QsArray& a = arr[blockIdx.y];
  const Sel* const sel = &a.sel;
  const int t = threadIdx.x;
  if (sel->status != kSelect) return;  // the same for every thread
  const uint32_t m = sel->m;
  uint32_t len = 1;
  while (len < m) len <<= 1;
  for (uint32_t i = t; i < len; i += kThreads) v[i] = i < m ? ord_key(a.cand[i]) : ~0ull;
  __syncthreads();
  sort_keys(v, len);
  QsResult& r = res[blockIdx.y];
  if (t < args.np)
    r.out[t] = interp(args.prank[t], args.ranks[2 * t], args.ranks[2 * t + 1], from_key(v[sel->pos[2 * t]]),
                      from_key(v[sel->pos[2 * t + 1]]));
}

// n <= kMaxCand: the whole array in one workgroup's LDS.
__global__ __launch_bounds__(kThreads) void qs_small(QsArgs args, QsResult* res) {
  __shared__ uint64_t v[kMaxCand];
  const double* __restrict__ x = args.x[blockIdx.y];
  QsResult& r = res[blockIdx.y];
  const uint32_t n = (uint32_t)args.n;
  const int t = threadIdx.x;
  uint32_t len = 1;
  while (len < n) len <<= 1;
  bool nan = false;
  for (uint32_t i = t; i < len; i += kThreads) {
    const double xi = i < n ? x[i] : 0.0;
    nan |= isnan(xi);
    v[i] = i < n ? ord_key(xi) : ~0ull;
  }
  nan = __syncthreads_or(nan);
  if (t == 0) r.status = nan ? kNan : kSelect;
  if (nan) return;
  sort_keys(v, len);
  if (t < args.np) {
    const double lo = from_key(v[0]);
    r.out[t] = lo == from_key(v[n - 1])
                   ? lo
                   : interp(args.prank[t], args.ranks[2 * t], args.ranks[2 * t + 1], from_key(v[args.ranks[2 * t]]),
                            from_key(v[args.ranks[2 * t + 1]]));
  }
}

// ---- the fallback: MSB-first radix select on the keys of ord_key.  Pass L
// histograms digit L (8 bits) of the keys whose first L digits equal the
// prefix found so far for each needed rank, one histogram per rank; the pick
// step extends each prefix by the digit whose cumulative count passes the
// rank, and the rank becomes the rank among the keys of that digit.  After
// the eighth pass each prefix is the whole key of its order statistic, exact
// whatever the ties, outliers or infinities, with no sort of the array.
constexpr int kDigits = 8;

struct Radix {
  uint64_t prefix[kMaxRanks];  // the digits found so far
  uint64_t k[kMaxRanks];       // rank among the keys with that prefix
  uint32_t hist[kMaxRanks][256];
};

__global__ void qs_radix_init(QsArgs args, Radix* rx) {
  Radix& r = rx[blockIdx.y];
  const int t = threadIdx.x;
  if (t < 2 * args.np) {
    r.prefix[t] = 0;
    r.k[t] = args.ranks[t];
  }
  for (int e = t; e < kMaxRanks * 256; e += blockDim.x) (&r.hist[0][0])[e] = 0u;
}

__global__ __launch_bounds__(256) void qs_radix_hist(QsArgs args, Radix* rx, int level) {
  __shared__ uint32_t h[kMaxRanks][256];
  __shared__ uint64_t pre[kMaxRanks];
  const double* __restrict__ x = args.x[blockIdx.y];
  Radix& r = rx[blockIdx.y];
  const int t = threadIdx.x;
  const int nr = 2 * args.np;
  for (int e = t; e < nr * 256; e += 256) (&h[0][0])[e] = 0u;
  if (t < nr) pre[t] = r.prefix[t];
  __syncthreads();
  const int shift = 56 - 8 * level;  // this pass's digit
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + t; i < args.n; i += (uint64_t)gridDim.x * 256) {
    const uint64_t key = ord_key(x[i]);
    const uint32_t d = (uint32_t)(key >> shift) & 255u;
    const uint64_t high = level == 0 ? 0ull : key >> (shift + 8);
    for (int k = 0; k < nr; ++k)
      if (high == pre[k]) atomicAdd(&h[k][d], 1u);
  }
  __syncthreads();
  for (int e = t; e < nr * 256; e += 256) {
    const uint32_t c = (&h[0][0])[e];
    if (c) atomicAdd(&(&r.hist[0][0])[e], c);
  }
}

// One thread per needed rank; the histograms are then cleared for the next pass.
__global__ void qs_radix_pick(QsArgs args, Radix* rx) {
  Radix& r = rx[blockIdx.y];
  const int t = threadIdx.x;
  if (t < 2 * args.np) {
    const uint64_t k = r.k[t];
    uint64_t cum = 0;
    uint32_t d = 0;
    for (; d < 255u; ++d) {  // the keys with this prefix number more than k
      const uint64_t c = r.hist[t][d];
      if (k < cum + c) break;
      cum += c;
    }
    r.k[t] = k - cum;
    r.prefix[t] = (r.prefix[t] << 8) | d;
  }
  __syncthreads();
  for (int e = t; e < kMaxRanks * 256; e += blockDim.x) (&r.hist[0][0])[e] = 0u;
}

__global__ void qs_radix_finish(QsArgs args, const Radix* rx, QsResult* res) {
  const Radix& r = rx[blockIdx.y];
  const int t = threadIdx.x;
  if (t < args.np)
    res[blockIdx.y].out[t] = interp(args.prank[t], args.ranks[2 * t], args.ranks[2 * t + 1], from_key(r.prefix[2 * t]),
                                    from_key(r.prefix[2 * t + 1]));
}

hipError_t grow(void** p, size_t* have, size_t need) {
  if (*have >= need) return hipSuccess;
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  *have = 0;
  const hipError_t e = hipMalloc(p, need);
  if (e == hipSuccess) *have = need;
  return e;
}

}  // namespace

QuantileScratch::~QuantileScratch() {
  if (small) (void)hipFree(small);
  if (host) (void)hipHostFree(host);
}

int quantile_select(QuantileScratch& sc, const double* const* xs, int nx, uint64_t n, const double* p, int np,
                    double* out, hipStream_t st, bool* used_fallback) {
  if (used_fallback) *used_fallback = false;
  if (nx < 1 || nx > kMaxArrays || np < 1 || np > kMaxPercentiles || n < 1 || n > 0x7FFFFFFFull)
    return JNE_ERR_INVALID_ARG;
  const size_t radix_off = ((size_t)kMaxArrays * sizeof(QsArray) + 255) & ~size_t(255);
  hipError_t e = grow(&sc.small, &sc.small_bytes, radix_off + kMaxArrays * sizeof(Radix));
  if (e != hipSuccess) return JNE_ERR_HIP;
  // the results: pinned host memory that the kernels write
  if (!sc.host && hipHostMalloc(&sc.host, kMaxArrays * sizeof(QsResult), hipHostMallocDefault) != hipSuccess) {
    sc.host = nullptr;
    return JNE_ERR_HIP;
  }
  QsArray* arr = static_cast<QsArray*>(sc.small);
  QsResult* const res = static_cast<QsResult*>(sc.host);
  Radix* radix = reinterpret_cast<Radix*>(static_cast<char*>(sc.small) + radix_off);

  // ranks of the needed order statistics (get_percentile_value's rank)
  QsArgs args = {};
  for (int a = 0; a < nx; ++a) args.x[a] = xs[a];
  args.n = n;
  args.np = np;
  for (int i = 0; i < np; ++i) {
    args.prank[i] = p[i] * (double)(n - 1);
    args.ranks[2 * i] = (uint64_t)floor(args.prank[i]);
    args.ranks[2 * i + 1] = (uint64_t)ceil(args.prank[i]);
  }
  if (n <= (uint64_t)kMaxCand) {
    hipLaunchKernelGGL(qs_small, dim3(1, nx), dim3(kThreads), 0, st, args, res);
  } else {
    hipLaunchKernelGGL(qs_minmax, dim3(pass_groups(n, 4 * kThreads), nx), dim3(kThreads), 0, st, args, arr);
    hipLaunchKernelGGL(qs_hist, dim3(pass_groups(n, 16 * kThreads), nx), dim3(kThreads), 0, st, args, arr, res);
    hipLaunchKernelGGL(qs_select, dim3(1, nx), dim3(kThreads), 0, st, args, arr, res);
    hipLaunchKernelGGL(qs_gather, dim3(pass_groups(n, 4 * kThreads), nx), dim3(kThreads), 0, st, args, arr);
    hipLaunchKernelGGL(qs_finish, dim3(1, nx), dim3(kThreads), 0, st, args, arr, res);
  }
  if ((e = hipGetLastError()) != hipSuccess || (e = hipStreamSynchronize(st)) != hipSuccess) return JNE_ERR_HIP;
  for (int a = 0; a < nx; ++a)
    if (res[a].status == kNan) return JNE_ERR_NUMERIC;
  for (int a = 0; a < nx; ++a) {
    if (res[a].status != kRadix) {
      memcpy(out + (size_t)a * np, res[a].out, np * sizeof(double));
      continue;
    }
    // the fallback: radix select of this array's order statistics
    if (used_fallback) *used_fallback = true;
    QsArgs one = args;
    one.x[0] = xs[a];
    Radix* const rx = radix + a;
    const unsigned grid = (unsigned)std::min<uint64_t>(512, (n + 255) / 256);
    hipLaunchKernelGGL(qs_radix_init, dim3(1), dim3(256), 0, st, one, rx);
    for (int level = 0; level < kDigits; ++level) {
      hipLaunchKernelGGL(qs_radix_hist, dim3(grid), dim3(256), 0, st, one, rx, level);
      hipLaunchKernelGGL(qs_radix_pick, dim3(1), dim3(256), 0, st, one, rx);
    }
    hipLaunchKernelGGL(qs_radix_finish, dim3(1), dim3(64), 0, st, one, rx, res + a);
    if ((e = hipGetLastError()) != hipSuccess || (e = hipStreamSynchronize(st)) != hipSuccess) return JNE_ERR_HIP;
    memcpy(out + (size_t)a * np, res[a].out, np * sizeof(double));
  }
  return 0;
}

}  // namespace jne
