/* stream_forms_oracle.c -- compares the forms of stream_forms.cpp with the
 * oracle's (oracle/jne_oracle.c, included for its static functions), bit for bit:
 *   radius: every float u1 in [2^-33, 1] (all u1 the stream can produce);
 *   turn:   every quadrant, the angle word's low 30 bits over the 2^21 values at
 *           each end of the range and a stride-1021 sample of the rest, for three
 *           radius words (u1 = 1, whose radius is -0, among them);
 *   Philox: 100,000 counters and keys.
 * Prints one line of counts and exits 1 on any difference. */
#include <stdio.h>

#include "jne_oracle.c"

float device_minus_two_ln(float u);
void device_normal_pair(uint32_t wa, uint32_t wb, float out[2]);
void device_philox(const uint32_t c[4], const uint32_t k[2], uint32_t out[4]);

int main(void) {
    long radius_bad = 0, radius_n = 0, turn_bad = 0, turn_n = 0, philox_bad = 0, philox_n = 0;
    for (uint32_t ub = f2u(0x1p-33f); ub <= f2u(1.0f); ++ub, ++radius_n)
        radius_bad += f2u(device_minus_two_ln(u2f(ub))) != f2u(-2.0f * ln_poly(u2f(ub)));
    const uint32_t was[3] = {0xFFFFFFFFu, 0u, 0x9E3779B9u};
    for (uint32_t low = 0; low < (1u << 30); low += (low < (1u << 21) || low >= (1u << 30) - (1u << 21)) ? 1u : 1021u)
        for (uint32_t q = 0; q < 4; ++q)
            for (int k = 0; k < 3; ++k, ++turn_n) {
                float o[2], d[2];
                jo_normal_pair(was[k], (q << 30) | low, o);
                device_normal_pair(was[k], (q << 30) | low, d);
                turn_bad += f2u(o[0]) != f2u(d[0]) || f2u(o[1]) != f2u(d[1]);
            }
    uint32_t s = 1u;
    for (; philox_n < 100000; ++philox_n) {
        uint32_t c[4], k[2], d[4], o[4];
        for (int i = 0; i < 4; ++i) c[i] = s = s * 1664525u + 1013904223u;
        for (int i = 0; i < 2; ++i) k[i] = s = s * 1664525u + 1013904223u;
        device_philox(c, k, d);
        jo_philox4x32_10(c, k, o);
        for (int i = 0; i < 4; ++i) philox_bad += d[i] != o[i];
    }
    printf("radius %ld/%ld differ, turn %ld/%ld differ, philox %ld/%ld differ\n", radius_bad, radius_n, turn_bad, turn_n,
           philox_bad, philox_n);
    return (radius_bad || turn_bad || philox_bad) ? 1 : 0;
}
