// jne_rng_check.hip -- the square root of the normal transform (sqrt_cr of
// jne_rng.h) at every radius word.
//
// sqrt_cr rests on v_rsq_f32's own results: its error bound does not prove the
// last bit, so it is compared, for all 2^32 words wa, with what a correctly rounded
// root of y = -2 ln(u1(wa)) is: the float r with (r - ulp/2)^2 < y < (r + ulp/2)^2.
// r and its neighbours have 24 bits, so the midpoints and their squares are exact
// in double (25 and 50 bits), and no midpoint is itself a root: y has 24 bits and an
// odd 25-bit number's square more.  y = -0 (u1 = 1) has the root -0.
//
// Prints one JSON line: the words compared, how many roots differ, the least word
// that does.  Exits 1 on any difference.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "jne_rng.h"

namespace {

constexpr unsigned kBlock = 256, kBlocks = 4096;
constexpr unsigned kPerThread = (1ull << 32) / kBlock / kBlocks;

struct Result {
  unsigned long long words, differ;
  unsigned least;
};

__global__ __launch_bounds__(kBlock) void check_kernel(Result* res) {
  const uint32_t first = (blockIdx.x * kBlock + threadIdx.x) * kPerThread;
  unsigned differ = 0, least = 0xFFFFFFFFu;
  for (uint32_t i = 0; i < kPerThread; ++i) {
    const uint32_t wa = first + i;
    const float u1 = __builtin_fmaf((float)wa, 0x1p-32f, 0x1p-33f);  // as normal_pair forms it
    const float y = -jne::two_ln(u1);
    const float r = jne::sqrt_cr(y);
    const uint32_t rb = __float_as_uint(r);
    bool good;
    if (y == 0.0f) {
      good = rb == __float_as_uint(y);
    } else {
      const double lo = 0.5 * ((double)__uint_as_float(rb - 1u) + (double)r);
      const double hi = 0.5 * ((double)r + (double)__uint_as_float(rb + 1u));
      good = r > 0.0f && lo * lo < (double)y && (double)y < hi * hi;
    }
    if (!good) {
      ++differ;
      least = wa < least ? wa : least;
    }
  }
  atomicAdd(&res->words, (unsigned long long)kPerThread);
  if (differ) {
    atomicAdd(&res->differ, (unsigned long long)differ);
    atomicMin(&res->least, least);
  }
}

int fail(const char* what, hipError_t e) {
  std::fprintf(stderr, "jne_rng_check: %s: %s\n", what, hipGetErrorString(e));
  return 2;
}

}  // namespace

int main() {
  Result h = {0, 0, 0xFFFFFFFFu}, *d = nullptr;
  hipError_t e = hipMalloc(&d, sizeof h);
  if (e != hipSuccess) return fail("hipMalloc", e);
  if ((e = hipMemcpy(d, &h, sizeof h, hipMemcpyHostToDevice)) != hipSuccess) return fail("hipMemcpy", e);
  hipLaunchKernelGGL(check_kernel, dim3(kBlocks), dim3(kBlock), 0, nullptr, d);
  if ((e = hipGetLastError()) != hipSuccess) return fail("launch", e);
  if ((e = hipMemcpy(&h, d, sizeof h, hipMemcpyDeviceToHost)) != hipSuccess) return fail("hipMemcpy", e);
  if ((e = hipFree(d)) != hipSuccess) return fail("hipFree", e);
  std::printf("{\"words\": %llu, \"differ\": %llu, \"least_word\": %u}\n", h.words, h.differ, h.least);
  return h.differ || h.words != 1ull << 32 ? 1 : 0;
}
