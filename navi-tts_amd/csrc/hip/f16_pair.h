// The split of an f32 activation into two f16 halves, which the matrix units multiply one after the other.
#pragma once

#include "dev_common.h"

namespace navi_amd {

// The f16 pair of an f32 value: h + o is v to 22 bits. The barrier makes v a rounded f32 value: where v is a
// product or an fma, the compiler may otherwise round h once, from the exact one (v_fma_mixlo_f16), in one of
// its two uses and twice (v_cvt_pk_f16_f32) in the other, which differ where v is halfway between two f16
// values: the pair is then off by a whole f16 unit, 5.4e-6 of the value in root mean square (4 million products of
// N(0, 1) values and weights about 1) instead of 5.2e-8.
__device__ __forceinline__ void f16_pair(float v, _Float16 &h, _Float16 &o) {
    asm("" : "+v"(v));
    h = static_cast<_Float16>(v);
    o = static_cast<_Float16>(v - static_cast<float>(h));
}

} // namespace navi_amd
