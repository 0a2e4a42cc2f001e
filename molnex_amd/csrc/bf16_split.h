// Exact three-way bf16 split of fp32 values for fp32-accurate products on the
// bf16 matrix cores: v = v0 + v1 + v2 to 2^-25 |v| with v0 = bf16(v),
// v1 = bf16(v - v0), v2 = bf16(v - v0 - v1), each rounded to nearest.
//
// Two values at a time: one packed conversion gives both bf16 halves, whose fp32
// values are then one shift and one mask of the packed word, 5.5 vector
// instructions per value.  (Converted one by one, the compiler repeats the
// conversion for the packed operand: 7.5.)
#pragma once

#include "common.h"

namespace mnx {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t bf16_pack2(float a, float b) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 h2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, h2));
}

// The three planes of values (a, b), packed (a in the low half).
__device__ __forceinline__ void bf16_split2(float a, float b, uint32_t& p0, uint32_t& p1, uint32_t& p2) {
    p0 = bf16_pack2(a, b);
    a -= __uint_as_float(p0 << 16);
    b -= __uint_as_float(p0 & 0xffff0000u);
    p1 = bf16_pack2(a, b);
    a -= __uint_as_float(p1 << 16);
    b -= __uint_as_float(p1 & 0xffff0000u);
    p2 = bf16_pack2(a, b);
}

// The three planes of eight values, one MFMA operand each.
__device__ __forceinline__ void bf16_split8(const float (&v)[8], bf16x8_t& b0, bf16x8_t& b1, bf16x8_t& b2) {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    u4 q0, q1, q2;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t p0, p1, p2;
        bf16_split2(v[2 * j], v[2 * j + 1], p0, p1, p2);
        q0[j] = p0;
        q1[j] = p1;
        q2[j] = p2;
    }
    b0 = __builtin_bit_cast(bf16x8_t, q0);
    b1 = __builtin_bit_cast(bf16x8_t, q1);
    b2 = __builtin_bit_cast(bf16x8_t, q2);
}

}  // namespace mnx
