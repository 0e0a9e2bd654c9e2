// jne_capi.hip -- the C ABI (include/jne.h): contexts, argument checks,
// chunked launches of the walk kernels, host/device copies.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/jne.h"
#include "jne_internal.h"
#include "jne_rng.h"

namespace jne {

// Groups of blockDim.x x blockDim.y = 256 threads: row y takes walk
// w0 + blockIdx.y * blockDim.y + y, its threads the walk's Philox calls
// q = blockIdx.x * blockDim.x + x, stepping by the grid width, each writing
// normals 4q..4q+3 (16-byte stores when `vec`: every walk's row of T*d floats
// starts 16-byte aligned).  blockDim.x is a multiple of 64, so a wave has one walk.
//
// Bound by the generator and then by its writes: full iterations draw two
// independent calls, and with STREAM the stores pass the caches by.  16,384
// walks of 10,000 x 12 (7.9 GB): 1.90 ms with one call at a time and a whole
// group per walk, now 1.61 ms (4.9 TB/s; a plain fill writes 6.8 TB/s);
// 100,000 walks of 100 x 5, whose 125 calls now take half a group: 53 to 43 us.
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <bool STREAM>
__global__ __launch_bounds__(256) void walk_normals_kernel(const uint32_t* __restrict__ seeds, uint32_t rng_stream,
                                                           uint32_t w0, uint32_t n, uint32_t total, uint32_t calls,
                                                           bool vec, float* __restrict__ out) {
  const uint32_t row = blockIdx.y * blockDim.y + (uint32_t)__builtin_amdgcn_readfirstlane((int)threadIdx.y);
  if (row >= n - w0) return;
  const uint32_t walk = w0 + row;
  const uint32_t seed = seeds[walk];
  float* const o = out + (size_t)walk * total;
  const uint32_t step = gridDim.x * blockDim.x;
  uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (vec) {
    const auto put = [&](uint32_t c, const float (&v)[4]) {
      f32x4* const dst = reinterpret_cast<f32x4*>(o + 4 * (size_t)c);
      const f32x4 x{v[0], v[1], v[2], v[3]};
      if constexpr (STREAM)
        __builtin_nontemporal_store(x, dst);
      else
        *dst = x;
    };
    for (; q < calls && calls - 1 - q >= step; q += 2 * step) {
      float v[2][4];
      normals4(q, seed, rng_stream, v[0]);
      normals4(q + step, seed, rng_stream, v[1]);
      put(q, v[0]);
      put(q + step, v[1]);
      if (calls - q <= 2 * step) return;  // the next q may pass 2^32
    }
    if (q < calls) {
      float v[4];
      normals4(q, seed, rng_stream, v);
      put(q, v);
    }
    return;
  }
  for (; q < calls; q += step) {
    float v[4];
    normals4(q, seed, rng_stream, v);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (4 * q + k < total) o[4 * (size_t)q + k] = v[k];
    if (calls - q <= step) break;  // q + step may pass 2^32
  }
}

hipError_t launch_walk_normals(int d, const uint32_t* seeds, uint32_t rng_stream, uint32_t T, uint32_t n,
                               float* out, hipStream_t st) {
  // the caller keeps T * d < 2^32
  const uint32_t total = T * (uint32_t)d;
  const uint32_t calls = (total + 3) / 4;
  // a walk of few calls takes one or two waves of a group, not four
  const uint32_t bx = calls <= 64 ? 64 : calls <= 128 ? 128 : 256, by = 256 / bx;
  // calls per thread: up to 8 once that leaves 2^20 threads (two rounds of the
  // GPU's), so that a wave's start is a small part of it (4 and 16: up to 1 %
  // and 3 % slower)
  const uint32_t cpt = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(8, (uint64_t)calls * n >> 20));
  const uint32_t gx = std::min<uint32_t>((uint32_t)(((uint64_t)calls + (uint64_t)bx * cpt - 1) / (bx * cpt)), 65535u);
  const bool vec = (total & 3u) == 0u && (reinterpret_cast<uintptr_t>(out) & 15u) == 0u;
  // Outputs larger than the 256 MiB last-level cache stream past it: 1.61 ms
  // against 1.64 ms for 7.9 GB.  Smaller ones stay where their reader finds them
  // (the write itself takes the same time either way).
  const bool stream = (uint64_t)total * n * sizeof(float) > (uint64_t)256 << 20;
  // a launch covers at most 65,535 rows of groups (grid y)
  for (uint32_t w0 = 0; w0 < n;) {
    const uint32_t gy = std::min<uint32_t>((n - w0 - 1) / by + 1, 65535u);
    hipLaunchKernelGGL(stream ? walk_normals_kernel<true> : walk_normals_kernel<false>, dim3(gx, gy), dim3(bx, by), 0,
                       st, seeds, rng_stream, w0, n, total, calls, vec, out);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (n - w0 <= gy * by) break;
    w0 += gy * by;
  }
  return hipSuccess;
}

}  // namespace jne

// Device scratch of jne_eigenvalues_by_seed_device_noalloc: the per-walk
// moments and the M matrices of the two-kernel eigen solve of one call, in a
// fixed array that each GPU the library runs on holds until the process ends
// (JNE_NOALLOC_SCRATCH_BYTES).  In host code `scratch` names a host-side
// stand-in, not the device address: the address of each GPU's copy is taken
// once per device with hipGetSymbolAddress (jne_create) and only that
// pointer is passed to kernels.
static __device__ __align__(256) double scratch[JNE_NOALLOC_SCRATCH_BYTES / sizeof(double)];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};  // per device: the address of its `scratch`
}  // namespace

struct jne_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  double* noalloc_scratch = nullptr;  // this device's `scratch`
  std::mutex mu;
  std::string err;
  // device scratch: per-walk moments of one chunk
  double* d_acc = nullptr;
  size_t acc_bytes = 0;
  // device scratch: M = W^T W of one chunk for the two-kernel eigen solve
  double* d_m = nullptr;
  size_t m_bytes = 0;
  // device scratch: the blocks' sums of batches split over their walks' blocks
  double* d_part = nullptr;
  size_t part_bytes = 0;
  // the scratch is shared by every call: a call on another stream than the
  // previous one first waits for the previous call's last use of it
  hipEvent_t scratch_free = nullptr;
  hipStream_t scratch_stream = nullptr;
  // device staging for the host-pointer entry points
  void* d_in = nullptr;
  size_t in_bytes = 0;
  void* d_out = nullptr;
  char* pinned = nullptr;  // seeds and eigenvalues of small host calls (kPinnedBytes, host memory)
  size_t out_bytes = 0;
  // device scratch of jne_percentiles_device
  jne::QuantileScratch qs;
  // kernel timing (jne_profile_*)
  struct TimedLaunch {
    int kernel;
    hipEvent_t start, stop;
    uint64_t walks;
  };
  bool profiling = false;
  std::vector<TimedLaunch> timed;
  std::vector<hipEvent_t> event_pool;
};

namespace {

thread_local std::string g_create_err;
constexpr size_t kChunkWalks = size_t(1) << 18;

int set_err(jne_ctx* ctx, int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  ctx->err = buf;
  return code;
}

#define JNE_HIP_CHECK(ctx, expr)                                                                   \
  do {                                                                                             \
    hipError_t e_ = (expr);                                                                        \
    if (e_ != hipSuccess) return set_err((ctx), JNE_ERR_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
  } while (0)

int ensure(jne_ctx* ctx, void** ptr, size_t* have, size_t need) {
  if (*have >= need) return JNE_OK;
  if (*ptr) {
    (void)hipFree(*ptr);
    *ptr = nullptr;
    *have = 0;
  }
  hipError_t e = hipMalloc(ptr, need);
  if (e != hipSuccess) {
    *ptr = nullptr;
    return set_err(ctx, JNE_ERR_NOMEM, "hipMalloc(%zu bytes) failed: %s", need, hipGetErrorString(e));
  }
  *have = need;
  return JNE_OK;
}

int check_args(jne_ctx* ctx, int model, int dim, uint32_t steps, int precision) {
  if (model < 0 || model > 4) return set_err(ctx, JNE_ERR_INVALID_ARG, "invalid model %d (expected 0..4)", model);
  if (dim < 1 || dim > JNE_MAX_DIM)
    return set_err(ctx, JNE_ERR_INVALID_ARG, "invalid dim %d (expected 1..%d)", dim, JNE_MAX_DIM);
  if (steps < 2 || steps > jne::kMaxSteps)
    return set_err(ctx, JNE_ERR_INVALID_ARG, "invalid steps %u (expected 2..2^30)", steps);
  switch (precision) {
    case JNE_PREC_FP64:
    case JNE_PREC_AUTO:
      return JNE_OK;
    case JNE_PREC_MFMA_FP16X2:
    case JNE_PREC_MFMA_BF16X2:
    case JNE_PREC_MFMA_BF16X3:
    case JNE_PREC_MFMA_FP32:
    case JNE_PREC_FP32_KAHAN:
      if (dim > JNE_MAX_MIXED_DIM)
        return set_err(ctx, JNE_ERR_UNSUPPORTED, "precision %d covers dims 1..%d; dim %d runs the FP64 path",
                       precision, JNE_MAX_MIXED_DIM, dim);
      return JNE_OK;
    default:
      return set_err(ctx, JNE_ERR_INVALID_ARG, "invalid precision %d", precision);
  }
}

hipEvent_t pool_event(jne_ctx* ctx) {
  if (!ctx->event_pool.empty()) {
    hipEvent_t e = ctx->event_pool.back();
    ctx->event_pool.pop_back();
    return e;
  }
  hipEvent_t e = nullptr;
  if (hipEventCreate(&e) != hipSuccess) return nullptr;
  return e;
}

void release_timed(jne_ctx* ctx) {
  for (auto& t : ctx->timed) {
    ctx->event_pool.push_back(t.start);
    ctx->event_pool.push_back(t.stop);
  }
  ctx->timed.clear();
}

// Records events around `launch` on st when profiling is enabled.
template <class F>
hipError_t timed_launch(jne_ctx* ctx, int kernel, uint64_t walks, hipStream_t st, F&& launch) {
  if (!ctx->profiling) return launch();
  hipEvent_t a = pool_event(ctx), b = pool_event(ctx);
  if (!a || !b) return hipErrorOutOfMemory;
  hipError_t e = hipEventRecord(a, st);
  if (e == hipSuccess) e = launch();
  if (e == hipSuccess) e = hipEventRecord(b, st);
  if (e != hipSuccess) {
    ctx->event_pool.push_back(a);
    ctx->event_pool.push_back(b);
    return e;
  }
  ctx->timed.push_back({kernel, a, b, walks});
  return hipSuccess;
}

// Enqueue the walk path for n walks (device pointers) on stream st.
// JNE_PREC_AUTO: the MFMA pass for dim 12 from 200 steps, dims 10-11 from 300,
// dim 9 from 500, dim 8 from 1,000 and dim 7 from 3,000; short walks carry its
// per-walk setup.  The lines were drawn where the two passes met (walks/s of the
// whole path, model 4, 262,144 walks) before the FP64 pass took blocks of steps,
// and stay, because which pass runs is part of a call's results.  Measured since,
// FP64 / MFMA in M walks/s: dim 7, T = 3,000 37.3 / 28.2, 10,000 11.9 / 8.7; dim 8,
// 1,000 83.7 / 76.5, 10,000 9.1 / 8.4; dim 9, 300 168 / 159, 500 110 / 112, 1,000 57.8
// / 63.9; dim 10, 200 200 / 179, 300 139 / 152; dim 11, 200 168 / 157, 300 118 / 135;
// dim 12, 200 172 / 150, 300 122 / 135, 10,000 5.0 / 6.3.  At dims 1-6 the FP64 pass
// keeps each walk in one lane's registers and leads by 1.2x or more (dim 6: 1.2-1.4x)
// over the MFMA pass, which packs 12 / dim walks per wave at 1, 2, 3, 4 and 6.
bool auto_uses_mfma(int dim, uint32_t steps) {
  if (dim > JNE_MAX_MIXED_DIM) return false;
  if (dim == 12) return steps >= 200;
  if (dim >= 10) return steps >= 300;
  if (dim == 9) return steps >= 500;
  if (dim == 8) return steps >= 1000;
  if (dim == 7) return steps >= 3000;
  return false;
}

int resolve_precision(int dim, uint32_t steps, int precision) {
  if (precision != JNE_PREC_AUTO) return precision;
  return auto_uses_mfma(dim, steps) ? JNE_PREC_MFMA_FP16X2 : JNE_PREC_FP64;
}

// Scratch for splitting a launch of n walks over their blocks (0: not split;
// the reduced precisions split walks given by seed only).
size_t part_doubles_for(int dim, uint32_t steps, int precision, bool by_seed, size_t n) {
  if (n == 0) return 0;
  if (dim > jne::kMaxDim) return jne::wide_part_doubles(dim, steps, (uint32_t)n);
  precision = resolve_precision(dim, steps, precision);
  if (precision != JNE_PREC_FP64) return by_seed ? jne::mfma_part_doubles(dim, precision, steps, (uint32_t)n) : 0;
  return jne::fp64_part_doubles(dim, steps, (uint32_t)n);
}

// Enqueues the walk kernels for n walks on st, in chunks of at most `chunk`
// walks over the scratch `acc` (chunk * moment_count(dim) doubles), `mbuf`
// (chunk * eigen_m_count(dim) doubles) and `part` (part_doubles; may be NULL,
// see part_doubles_for): per chunk one moment pass, then the
// eigen solve of each of the n_models models into its output (the moments of
// a walk do not depend on the model).  timed: record the launches when
// profiling is enabled.
int launch_walks(jne_ctx* ctx, const int* models, int n_models, int dim, uint32_t steps, uint32_t rng_stream,
                 const uint32_t* d_seeds, const double* d_z, size_t n, int precision, double* const* d_outs,
                 hipStream_t st, double* acc, double* mbuf, double* part, size_t part_doubles, size_t chunk,
                 bool timed) {
  precision = resolve_precision(dim, steps, precision);
  for (size_t off = 0; off < n; off += chunk) {
    const uint32_t cn = (uint32_t)std::min(chunk, n - off);
    const uint32_t* s = d_seeds ? d_seeds + off : nullptr;
    const double* z = d_z ? d_z + off * (size_t)steps * dim : nullptr;
    auto moments = [&] {
      if (dim > jne::kMaxDim)
        return jne::launch_walk_moments_wide(dim, s, z, rng_stream, steps, cn, acc, cn, part, part_doubles, st);
      if (precision == JNE_PREC_FP64)
        return jne::launch_walk_moments_fp64(dim, s, z, rng_stream, steps, cn, acc, cn, part, part_doubles, st);
      return jne::launch_walk_moments_mfma(dim, precision, s, z, rng_stream, steps, cn, acc, cn, part, part_doubles,
                                           st);
    };
    if (timed)
      JNE_HIP_CHECK(ctx, timed_launch(ctx, JNE_KERNEL_MOMENTS, cn, st, moments));
    else
      JNE_HIP_CHECK(ctx, moments());
    for (int k = 0; k < n_models; ++k) {
      const int model = models[k];
      double* const out = d_outs[k] + off * (size_t)jne::num_eigenvalues(model, dim);
      auto eigen = [&] {
        if (dim > jne::kMaxDim) return jne::launch_walk_eigen_wide(model, dim, acc, cn, steps, cn, out, st);
        return jne::launch_walk_eigen_fp64(model, dim, acc, cn, steps, cn, out, mbuf, st);
      };
      if (timed)
        JNE_HIP_CHECK(ctx, timed_launch(ctx, JNE_KERNEL_EIGEN, cn, st, eigen));
      else
        JNE_HIP_CHECK(ctx, eigen());
    }
  }
  return JNE_OK;
}

int run_walks(jne_ctx* ctx, const int* models, int n_models, int dim, uint32_t steps, uint32_t rng_stream,
              const uint32_t* d_seeds, const double* d_z, size_t n, int precision, double* const* d_outs,
              hipStream_t st) {
  const size_t mc = (size_t)jne::moment_count(dim);
  // at most 2^18 walks per launch, and at the wide dims about 1 GiB of moments
  const size_t chunk = std::min(n, std::min(kChunkWalks, std::max<size_t>(65536, (size_t(1) << 27) / mc)));
  int rc = ensure(ctx, (void**)&ctx->d_acc, &ctx->acc_bytes, chunk * mc * sizeof(double));
  if (rc) return rc;
  rc = ensure(ctx, (void**)&ctx->d_m, &ctx->m_bytes, chunk * (size_t)jne::eigen_m_count(dim) * sizeof(double));
  if (rc) return rc;
  // without room for the blocks' sums the launches are not split
  const size_t part = std::max(part_doubles_for(dim, steps, precision, d_seeds != nullptr, chunk),
                               part_doubles_for(dim, steps, precision, d_seeds != nullptr, n % chunk));
  // A captured call is not split: a smaller batch can need more room than a larger
  // one did, so a later call may replace the block sums' buffer under the graph.
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cap) != hipSuccess) (void)hipGetLastError();
  const bool captured = cap != hipStreamCaptureStatusNone;
  if (!captured && ensure(ctx, (void**)&ctx->d_part, &ctx->part_bytes, part * sizeof(double)) != JNE_OK) {
    (void)hipGetLastError();
    ctx->err.clear();
  }
  if (!ctx->scratch_free) JNE_HIP_CHECK(ctx, hipEventCreateWithFlags(&ctx->scratch_free, hipEventDisableTiming));
  if (ctx->scratch_stream && ctx->scratch_stream != st)
    JNE_HIP_CHECK(ctx, hipStreamWaitEvent(st, ctx->scratch_free, 0));
  if ((rc = launch_walks(ctx, models, n_models, dim, steps, rng_stream, d_seeds, d_z, n, precision, d_outs, st,
                         ctx->d_acc, ctx->d_m, captured ? nullptr : ctx->d_part,
                         captured ? 0 : ctx->part_bytes / sizeof(double), chunk, true)))
    return rc;
  JNE_HIP_CHECK(ctx, hipEventRecord(ctx->scratch_free, st));
  ctx->scratch_stream = st;
  return JNE_OK;
}

// The stream a device entry point enqueues on: JNE_STREAM_CONTEXT is the
// context's own stream, anything else (NULL included: HIP's null stream) is
// the caller's.
hipStream_t stream_of(jne_ctx* ctx, void* hip_stream) {
  return hip_stream == JNE_STREAM_CONTEXT ? ctx->stream : (hipStream_t)hip_stream;
}

// Host calls of few walks: their seeds and eigenvalues are in the context's
// pinned host memory, which the kernels read and write over the bus; each of
// the two copies of pageable memory costs as much as a small kernel.
// One walk of 1,000 x 5: 66 to 51 us; 5,000 walks 148 to 132, 20,000 walks
// (0.9 MB) 307 to 291: 15 us per call at every size tried.  Above 1 MiB the
// call is bound by the walks, and a context would hold more host memory.
constexpr size_t kPinnedBytes = size_t(1) << 20;

// The pinned memory when `need` bytes fit it, else null (also when the host has
// none to pin: the call copies then).
char* pinned_for(jne_ctx* ctx, size_t need) {
  if (need > kPinnedBytes) return nullptr;
  if (!ctx->pinned && hipHostMalloc((void**)&ctx->pinned, kPinnedBytes, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    ctx->pinned = nullptr;
  }
  return ctx->pinned;
}

// n rows of nf eigenvalues from the context's device buffer, or from `pinned`
// when the kernels wrote them there; a NaN row (S11 not positive definite) makes
// the call return JNE_ERR_NUMERIC, naming the first such walk (0-based row).
int finish_host_out(jne_ctx* ctx, const double* pinned, double* out, size_t n, size_t nf) {
  const size_t count = n * nf;
  if (!pinned)
    JNE_HIP_CHECK(ctx, hipMemcpyAsync(out, ctx->d_out, count * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  JNE_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  if (pinned) memcpy(out, pinned, count * sizeof(double));
  for (size_t i = 0; i < count; ++i)
    if (isnan(out[i]))
      return set_err(ctx, JNE_ERR_NUMERIC, "walk %zu: S11 is not positive definite", i / nf);
  return JNE_OK;
}

}  // namespace

extern "C" {

int jne_create(int device, jne_ctx** out) {
  if (!out) {
    g_create_err = "jne_create: out is NULL";
    return JNE_ERR_INVALID_ARG;
  }
  *out = nullptr;
  int count = 0;
  hipError_t e = hipGetDeviceCount(&count);
  if (e != hipSuccess || count <= 0) {
    g_create_err = std::string("jne_create: no HIP device: ") + hipGetErrorString(e);
    return JNE_ERR_HIP;
  }
  if (device < 0 || device >= count) {
    g_create_err = "jne_create: device index out of range";
    return JNE_ERR_INVALID_ARG;
  }
  if (device >= kMaxDevices) {
    g_create_err = "jne_create: device index above 63";
    return JNE_ERR_INVALID_ARG;
  }
  jne_ctx* ctx = new jne_ctx();
  ctx->device = device;
  if ((e = hipSetDevice(device)) != hipSuccess || (e = hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking)) != hipSuccess) {
    g_create_err = std::string("jne_create: ") + hipGetErrorString(e);
    delete ctx;
    return JNE_ERR_HIP;
  }
  {
    // the address of this device's copy of the no-alloc scratch, once per
    // device (with the device current)
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
      void* p = nullptr;
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess || !p) {
        g_create_err = std::string("jne_create: hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
        (void)hipStreamDestroy(ctx->stream);
        delete ctx;
        return JNE_ERR_HIP;
      }
      g_scratch_ptr[device] = static_cast<double*>(p);
    }
    ctx->noalloc_scratch = g_scratch_ptr[device];
  }
  *out = ctx;
  return JNE_OK;
}

void jne_destroy(jne_ctx* ctx) {
  if (!ctx) return;
  (void)hipSetDevice(ctx->device);
  if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
  release_timed(ctx);
  for (hipEvent_t e : ctx->event_pool) (void)hipEventDestroy(e);
  if (ctx->d_acc) (void)hipFree(ctx->d_acc);
  if (ctx->d_m) (void)hipFree(ctx->d_m);
  if (ctx->d_part) (void)hipFree(ctx->d_part);
  if (ctx->scratch_free) (void)hipEventDestroy(ctx->scratch_free);
  if (ctx->d_in) (void)hipFree(ctx->d_in);
  if (ctx->d_out) (void)hipFree(ctx->d_out);
  if (ctx->pinned) (void)hipHostFree(ctx->pinned);
  if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
  delete ctx;
}

const char* jne_last_error(const jne_ctx* ctx) { return ctx ? ctx->err.c_str() : g_create_err.c_str(); }

int jne_num_eigenvalues(int model, int dim) {
  if (model < 0 || model > 4 || dim < 1 || dim > 255) return JNE_ERR_INVALID_ARG;
  return jne::num_eigenvalues(model, dim);
}

int jne_eigenvalues_by_seed(jne_ctx* ctx, int model, int dim, uint32_t steps, uint32_t rng_stream,
                            const uint32_t* seeds, size_t n, int precision, double* out) {
  if (!ctx) return JNE_ERR_INVALID_ARG;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->err.clear();
  int rc = check_args(ctx, model, dim, steps, precision);
  if (rc) return rc;
  if (n == 0) return JNE_OK;
  if (!seeds || !out) return set_err(ctx, JNE_ERR_INVALID_ARG, "seeds/out must not be NULL");
  JNE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  const size_t nf = (size_t)jne::num_eigenvalues(model, dim);
  const size_t out_bytes = n * nf * sizeof(double), seed_bytes = n * sizeof(uint32_t);
  char* const pin = pinned_for(ctx, out_bytes + seed_bytes);
  const uint32_t* s;
  double* outs[1];
  if (pin) {
    memcpy(pin + out_bytes, seeds, seed_bytes);
    s = reinterpret_cast<const uint32_t*>(pin + out_bytes);
    outs[0] = reinterpret_cast<double*>(pin);
  } else {
    if ((rc = ensure(ctx, &ctx->d_in, &ctx->in_bytes, seed_bytes))) return rc;
    if ((rc = ensure(ctx, &ctx->d_out, &ctx->out_bytes, out_bytes))) return rc;
    JNE_HIP_CHECK(ctx, hipMemcpyAsync(ctx->d_in, seeds, seed_bytes, hipMemcpyHostToDevice, ctx->stream));
    s = (const uint32_t*)ctx->d_in;
    outs[0] = (double*)ctx->d_out;
  }
  if ((rc = run_walks(ctx, &model, 1, dim, steps, rng_stream, s, nullptr, n, precision, outs, ctx->stream))) {
    if (pin) (void)hipStreamSynchronize(ctx->stream);  // nothing reads or writes the pinned memory after the call
    return rc;
  }
  return finish_host_out(ctx, pin ? outs[0] : nullptr, out, n, nf);
}

int jne_eigenvalues_by_seed_device(jne_ctx* ctx, int model, int dim, uint32_t steps, uint32_t rng_stream,
                                   const uint32_t* d_seeds, size_t n, int precision, double* d_out,
                                   void* hip_stream) {
  if (!ctx) return JNE_ERR_INVALID_ARG;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->err.clear();
  int rc = check_args(ctx, model, dim, steps, precision);
  if (rc) return rc;
  if (n == 0) return JNE_OK;
  if (!d_seeds || !d_out) return set_err(ctx, JNE_ERR_INVALID_ARG, "d_seeds/d_out must not be NULL");
  JNE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  hipStream_t st = stream_of(ctx, hip_stream);
  double* const outs[1] = {d_out};
  return run_walks(ctx, &model, 1, dim, steps, rng_stream, d_seeds, nullptr, n, precision, outs, st);
}

int jne_eigenvalues_by_seed_models_device(jne_ctx* ctx, const int* models, int n_models, int dim, uint32_t steps,
                                          uint32_t rng_stream, const uint32_t* d_seeds, size_t n, int precision,
                                          double* const* d_outs, void* hip_stream) {
  if (!ctx) return JNE_ERR_INVALID_ARG;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->err.clear();
  if (!models || !d_outs || n_models < 1 || n_models > 5)
    return set_err(ctx, JNE_ERR_INVALID_ARG, "models/d_outs must not be NULL and n_models must be in 1..5");
  for (int k = 0; k < n_models; ++k) {
    int rc = check_args(ctx, models[k], dim, steps, precision);
    if (rc) return rc;
    if (n > 0 && !d_outs[k]) return set_err(ctx, JNE_ERR_INVALID_ARG, "d_outs[%d] must not be NULL", k);
  }
  if (n == 0) return JNE_OK;
  if (!d_seeds) return set_err(ctx, JNE_ERR_INVALID_ARG, "d_seeds must not be NULL");
  JNE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  return run_walks(ctx, models, n_models, dim, steps, rng_stream, d_seeds, nullptr, n, precision, d_outs,
                   stream_of(ctx, hip_stream));
}

int jne_eigenvalues_by_seed_device_noalloc(jne_ctx* ctx, int model, int dim, uint32_t steps, uint32_t rng_stream,
                                           const uint32_t* d_seeds, size_t n, int precision, double* d_out,
                                           void* hip_stream) {
  if (!ctx) return JNE_ERR_INVALID_ARG;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->err.clear();
  int rc = check_args(ctx, model, dim, steps, precision);
  if (rc) return rc;
  if (n == 0) return JNE_OK;
  if (!d_seeds || !d_out) return set_err(ctx, JNE_ERR_INVALID_ARG, "d_seeds/d_out must not be NULL");
  const size_t mc = (size_t)jne::moment_count(dim);
  const size_t per_walk = mc + (size_t)jne::eigen_m_count(dim);
  const size_t cap_doubles = JNE_NOALLOC_SCRATCH_BYTES / sizeof(double);
  const size_t cap = cap_doubles / per_walk;
  if (n > cap)
    return set_err(ctx, JNE_ERR_INVALID_ARG,
                   "jne_eigenvalues_by_seed_device_noalloc: %zu walks exceed the scratch of %zu walks at dim %d "
                   "(%zu bytes per walk in %d MiB)",
                   n, cap, dim, per_walk * sizeof(double), (int)(JNE_NOALLOC_SCRATCH_BYTES >> 20));
  if (!ctx->noalloc_scratch) return set_err(ctx, JNE_ERR_HIP, "the no-alloc scratch has no device address");
  JNE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  double* const acc = ctx->noalloc_scratch;
  double* const outs[1] = {d_out};
  // what n leaves of the scratch takes the blocks' sums when it is enough
  return launch_walks(ctx, &model, 1, dim, steps, rng_stream, d_seeds, nullptr, n, precision, outs,
                      stream_of(ctx, hip_stream), acc, acc + mc * n, acc + per_walk * n, (cap_doubles - per_walk * n), n,
                      false);
}

int jne_eigenvalues_from_normals(jne_ctx* ctx, int model, int dim, uint32_t steps, const double* z, size_t n,
                                 int precision, double* out) {
  if (!ctx) return JNE_ERR_INVALID_ARG;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->err.clear();
  int rc = check_args(ctx, model, dim, steps, precision);
  if (rc) return rc;
  if (n == 0) return JNE_OK;
  if (!z || !out) return set_err(ctx, JNE_ERR_INVALID_ARG, "z/out must not be NULL");
  JNE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  const size_t nf = (size_t)jne::num_eigenvalues(model, dim);
  const size_t zcount = n * (size_t)steps * dim;
  if ((rc = ensure(ctx, &ctx->d_in, &ctx->in_bytes, zcount * sizeof(double)))) return rc;
  if ((rc = ensure(ctx, &ctx->d_out, &ctx->out_bytes, n * nf * sizeof(double)))) return rc;
  JNE_HIP_CHECK(ctx, hipMemcpyAsync(ctx->d_in, z, zcount * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
  double* const outs[1] = {(double*)ctx->d_out};
  if ((rc = run_walks(ctx, &model, 1, dim, steps, 0, nullptr, (const double*)ctx->d_in, n, precision, outs,
                      ctx->stream)))
    return rc;
  return finish_host_out(ctx, nullptr, out, n, nf);
}

namespace {
int check_normals_args(jne_ctx* ctx, int dim, uint32_t steps, size_t n) {
  if (dim < 1 || dim > 255) return set_err(ctx, JNE_ERR_INVALID_ARG, "invalid dim %d", dim);
  if (steps < 1 || steps > (1u << 30)) return set_err(ctx, JNE_ERR_INVALID_ARG, "invalid steps %u", steps);
  if ((uint64_t)steps * dim > 0xFFFFFFFCull)
    return set_err(ctx, JNE_ERR_INVALID_ARG, "jne_walk_normals: steps * dim must stay below 2^32");
  if (n > 0xFFFFFFFFull) return set_err(ctx, JNE_ERR_INVALID_ARG, "jne_walk_normals: at most 2^32-1 walks");
  return JNE_OK;
}
}  // namespace

int jne_walk_normals(jne_ctx* ctx, int dim, uint32_t steps, uint32_t rng_stream, const uint32_t* seeds, size_t n,
                     float* out) {
  if (!ctx) return JNE_ERR_INVALID_ARG;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->err.clear();
  int rc = check_normals_args(ctx, dim, steps, n);
  if (rc) return rc;
  if (n == 0) return JNE_OK;
  if (!seeds || !out) return set_err(ctx, JNE_ERR_INVALID_ARG, "seeds/out must not be NULL");
  JNE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  const size_t total = n * (size_t)steps * dim;
  if ((rc = ensure(ctx, &ctx->d_in, &ctx->in_bytes, n * sizeof(uint32_t)))) return rc;
  if ((rc = ensure(ctx, &ctx->d_out, &ctx->out_bytes, total * sizeof(float)))) return rc;
  JNE_HIP_CHECK(ctx, hipMemcpyAsync(ctx->d_in, seeds, n * sizeof(uint32_t), hipMemcpyHostToDevice, ctx->stream));
  JNE_HIP_CHECK(ctx, timed_launch(ctx, JNE_KERNEL_NORMALS, n, ctx->stream, [&] {
                  return jne::launch_walk_normals(dim, (const uint32_t*)ctx->d_in, rng_stream, steps, (uint32_t)n,
                                                  (float*)ctx->d_out, ctx->stream);
                }));
  JNE_HIP_CHECK(ctx, hipMemcpyAsync(out, ctx->d_out, total * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
  JNE_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  return JNE_OK;
}

int jne_walk_normals_device(jne_ctx* ctx, int dim, uint32_t steps, uint32_t rng_stream, const uint32_t* d_seeds,
                            size_t n, float* d_out, void* hip_stream) {
  if (!ctx) return JNE_ERR_INVALID_ARG;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->err.clear();
  int rc = check_normals_args(ctx, dim, steps, n);
  if (rc) return rc;
  if (n == 0) return JNE_OK;
  if (!d_seeds || !d_out) return set_err(ctx, JNE_ERR_INVALID_ARG, "d_seeds/d_out must not be NULL");
  JNE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  hipStream_t st = stream_of(ctx, hip_stream);
  JNE_HIP_CHECK(ctx, timed_launch(ctx, JNE_KERNEL_NORMALS, n, st, [&] {
                  return jne::launch_walk_normals(dim, d_seeds, rng_stream, steps, (uint32_t)n, d_out, st);
                }));
  return JNE_OK;
}

int jne_percentiles_device(jne_ctx* ctx, const double* d_values, uint64_t n, const double* p, size_t np,
                           double* out, void* hip_stream) {
  if (!ctx) return JNE_ERR_INVALID_ARG;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->err.clear();
  if (!p || !out || np < 1 || np > (size_t)jne::kMaxPercentiles)
    return set_err(ctx, JNE_ERR_INVALID_ARG, "p/out must not be NULL and np must be 1..%d", jne::kMaxPercentiles);
  for (size_t i = 0; i < np; ++i)
    if (!(p[i] >= 0.0 && p[i] <= 1.0)) return set_err(ctx, JNE_ERR_INVALID_ARG, "p[%zu] is not in [0, 1]", i);
  if (n > 0x7FFFFFFFull) return set_err(ctx, JNE_ERR_INVALID_ARG, "n must be below 2^31");
  if (n == 0) {  // as jne_percentiles: no order statistics
    for (size_t i = 0; i < np; ++i) out[i] = NAN;
    return JNE_OK;
  }
  if (!d_values) return set_err(ctx, JNE_ERR_INVALID_ARG, "d_values must not be NULL");
  JNE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  hipStream_t st = stream_of(ctx, hip_stream);
  const int rc = jne::quantile_select(ctx->qs, &d_values, 1, n, p, (int)np, out, st, nullptr);
  if (rc == JNE_ERR_NUMERIC) return set_err(ctx, rc, "a value is NaN");
  if (rc) return set_err(ctx, rc, "percentile selection failed");
  return JNE_OK;
}

int jne_synchronize(jne_ctx* ctx) {
  if (!ctx) return JNE_ERR_INVALID_ARG;
  std::lock_guard<std::mutex> lock(ctx->mu);
  JNE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  JNE_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  return JNE_OK;
}

int jne_profile_enable(jne_ctx* ctx, int enable) {
  if (!ctx) return JNE_ERR_INVALID_ARG;
  std::lock_guard<std::mutex> lock(ctx->mu);
  JNE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  for (auto& t : ctx->timed) {
    (void)hipEventSynchronize(t.stop);
  }
  release_timed(ctx);
  ctx->profiling = enable != 0;
  return JNE_OK;
}

int jne_profile_read(jne_ctx* ctx, int kernel, double* total_ms, uint64_t* launches, uint64_t* walks) {
  if (!ctx || !total_ms || !launches || !walks) return JNE_ERR_INVALID_ARG;
  std::lock_guard<std::mutex> lock(ctx->mu);
  JNE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  double ms = 0.0;
  uint64_t nl = 0, nw = 0;
  for (auto& t : ctx->timed) {
    if (t.kernel != kernel) continue;
    JNE_HIP_CHECK(ctx, hipEventSynchronize(t.stop));
    float e = 0.0f;
    JNE_HIP_CHECK(ctx, hipEventElapsedTime(&e, t.start, t.stop));
    ms += e;
    ++nl;
    nw += t.walks;
  }
  *total_ms = ms;
  *launches = nl;
  *walks = nw;
  return JNE_OK;
}

}  // extern "C"
