// The Snake of the codec decoder's kernels (snake.h), compiled for the host: tests/test_snake_cpu.py calls it.
#include "snake.h"

extern "C" {

// sin^2 of n arguments as a kernel would take them, one at a time (wide: through the 64-bit reduction)
void sin2_values(const float *u, int n, int wide, float *out) {
    for (int i = 0; i < n; ++i) out[i] = wide ? navi_amd::sin2_wide(u[i]) : navi_amd::sin2(u[i]);
}

// the 16 values of one channel that a lane of a conv's epilogue holds
void snake16(const float *v, float za, float zb, float *out) {
    float a[16], o[16];
    for (int i = 0; i < 16; ++i) a[i] = v[i];
    navi_amd::snake_n(a, za, zb, o);
    for (int i = 0; i < 16; ++i) out[i] = o[i];
}

float sin2_max() { return navi_amd::SIN2_MAX; }

}
