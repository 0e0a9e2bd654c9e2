// stream_forms.cpp -- the normal transform of jne_rng.h, as the device code
// includes it, built for the host (test_device_stream_forms.py).
#include "jne_rng.h"

extern "C" {
float device_minus_two_ln(float u) { return -jne::two_ln(u); }
void device_normal_pair(uint32_t wa, uint32_t wb, float out[2]) { jne::normal_pair(wa, wb, out[0], out[1]); }
void device_philox(const uint32_t c[4], const uint32_t k[2], uint32_t out[4]) {
  const jne::u32x4 w = jne::philox4x32_10(c[0], c[1], c[2], c[3], k[0], k[1]);
  out[0] = w.x, out[1] = w.y, out[2] = w.z, out[3] = w.w;
}
}
