// The codec decoder's Snake activation, v + b sin^2(a v), in plain f32 code for host and device.
//
// sin^2 needs no sinf: it is even and has period pi, and sin^2(r + pi / 2) = 1 - sin^2(r). So u is reduced
// to r = u - n pi / 2, |r| <= pi / 4 (pi / 2 as two floats; n pi / 2's first product and its difference
// from u are exact), and with z = r^2 sin^2 is s = z + z^2 P(z), or 1 - s where n is odd. P is a cubic fitted
// to (sin^2(sqrt z) - z) / z^2 on z <= (pi / 4)^2 (least squares on Chebyshev nodes, reweighted towards the
// smallest maximum of z^2 P's error: 2.8e-9 with the coefficients rounded to f32).
//
// Root mean square error 1.9e-8 for arguments of any size up to SIN2_MAX, where a correctly rounded sinf,
// squared, has 2.7e-8, and one polynomial over the whole period (|r| <= pi / 2) 3.4e-8: above pi / 4 the
// rounding of r, z and z^2 weighs more than the result's own. 14 instructions; sinf(u)^2 takes about three times
// as many and a branch to its reduction for large arguments at every use, and the epilogues' sines took longer
// than their MFMAs (a 240-frame block 5.50 ms, with the whole-period polynomial 4.84; other steps since: that one
// 4.64, this one 4.66).
#pragma once

#include <hip/hip_runtime.h>

namespace navi_amd {

constexpr float SIN2_MAX = 1048576.f;

// sin^2 of r, or of r + pi / 2 (odd), |r| <= pi / 4
__host__ __device__ __forceinline__ float sin2_reduced(float r, bool odd) {
    const float z = r * r;
    float p = fmaf(1.3411097461357713e-4f, z, -3.1704693101346493e-3f);
    p = fmaf(p, z, 4.444342106580734e-2f);
    p = fmaf(p, z, -3.3333325386047363e-1f);
    const float s = fmaf(z * z, p, z);
    return odd ? 1.f - s : s;
}

// |u| <= SIN2_MAX. The sum with 1.5 2^23 is rounded to a whole number, whose last bit it shows.
__host__ __device__ __forceinline__ float sin2(float u) {
    const float t = fmaf(u, 0.636619772f, 12582912.f), n = t - 12582912.f;
    uint32_t bits;
    __builtin_memcpy(&bits, &t, 4);
    return sin2_reduced(fmaf(-n, -4.37113883e-8f, fmaf(-n, 1.57079637f, u)), (bits & 1u) != 0);
}

// Any u, in 64 bits: larger arguments, which no activation inside the f16 range gives with a sane alpha. A
// pass leaves less than 2^-51 of an argument whose multiple of pi has more than 53 bits (2.8e16 on): three
// bring every finite float into range. The phase holds up to about 2^80; infinities give NaN.
__host__ __device__ __forceinline__ float sin2_wide(float u) {
    double r = static_cast<double>(u);
#pragma unroll 1
    for (int pass = 0; pass < 3; ++pass) {
        const double m = rint(r * 0.3183098861837907);
        r = fma(-m, 1.2246467991473532e-16, fma(-m, 3.141592653589793, r));
    }
    r = fabs(r);
    const bool odd = r > 0.7853981633974483;
    return sin2_reduced(static_cast<float>(odd ? 1.5707963267948966 - r : r), odd);
}

// out = v + zb sin^2(za v) for N values of one channel: one branch for all of them, their chains interleaved.
template <int N>
__host__ __device__ __forceinline__ void snake_n(const float (&v)[N], float za, float zb, float (&out)[N]) {
    float big = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) big = fmaxf(big, fabsf(v[i] * za));
    if (__builtin_expect(big > SIN2_MAX, 0)) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float u = v[i] * za;
            out[i] = fmaf(fabsf(u) > SIN2_MAX ? sin2_wide(u) : sin2(u), zb, v[i]);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) out[i] = fmaf(sin2(v[i] * za), zb, v[i]);
}
__host__ __device__ __forceinline__ float snake(float v, float za, float zb) {
    const float a[1] = {v};
    float o[1];
    snake_n(a, za, zb, o);
    return o[0];
}

} // namespace navi_amd
