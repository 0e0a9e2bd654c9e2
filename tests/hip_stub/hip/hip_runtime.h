// A stand-in for HIP's header under which jne_rng.h builds for the host: the
// qualifiers it uses and its device builtins as the plain operations they are
// (test_device_stream_forms.py).
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>

#define __device__
#define __forceinline__ inline

static inline uint32_t __float_as_uint(float x) {
  uint32_t u;
  std::memcpy(&u, &x, 4);
  return u;
}
static inline float __uint_as_float(uint32_t u) {
  float x;
  std::memcpy(&x, &u, 4);
  return x;
}
// v_bitop3_b32: bit 4a + 2b + c of the truth table
static inline uint32_t host_bitop3(uint32_t a, uint32_t b, uint32_t c, uint32_t table) {
  uint32_t r = 0;
  for (uint32_t k = 0; k < 8; ++k)
    if (table >> k & 1u) r |= (k & 4u ? a : ~a) & (k & 2u ? b : ~b) & (k & 1u ? c : ~c);
  return r;
}
#define __builtin_amdgcn_bitop3_b32(a, b, c, table) host_bitop3(a, b, c, table)
// the reciprocal root, rounded (the instruction is within 1 ulp of it)
#define __builtin_amdgcn_rsqf(x) ((float)(1.0 / std::sqrt((double)(x))))
