// An f32 pair as bf16 parts for the bf16 matrix products.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace airkv {

// (x, y) as three bf16 pairs, x in the low half: the hardware's rounding to
// nearest of the values, then of what is left.  Each remainder (exact) is one
// v_dot2_f32_bf16, x - h: 7 instructions a pair against 11 with the halves
// widened and subtracted.
__device__ __forceinline__ void split3(float x, float y, uint32_t &h, uint32_t &m, uint32_t &l) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    // (-1, 0) and (0, -1) in scalar registers: as an inline constant the
    // hardware does not read the pair the compiler means
    uint32_t c0 = 0x0000BF80u, c1 = 0xBF800000u;
    asm("" : "+s"(c0), "+s"(c1));
    const bf16x2 first = __builtin_bit_cast(bf16x2, c0), second = __builtin_bit_cast(bf16x2, c1);
    const bf16x2 hv = __builtin_convertvector((f32x2{x, y}), bf16x2);
    x = __builtin_amdgcn_fdot2_f32_bf16(hv, first, x, false);
    y = __builtin_amdgcn_fdot2_f32_bf16(hv, second, y, false);
    const bf16x2 mv = __builtin_convertvector((f32x2{x, y}), bf16x2);
    x = __builtin_amdgcn_fdot2_f32_bf16(mv, first, x, false);
    y = __builtin_amdgcn_fdot2_f32_bf16(mv, second, y, false);
    h = __builtin_bit_cast(uint32_t, hv);
    m = __builtin_bit_cast(uint32_t, mv);
    l = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x, y}), bf16x2));
}

}  // namespace airkv
