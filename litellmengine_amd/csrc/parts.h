// A float32 number as the sum of three bfloat16 numbers.
#pragma once
#include "common.h"

// Two numbers as their three bfloat16 parts, packed: x1 = x rounded, x2 = what is left rounded, x3 = the rest (3 x 8 significand bits and
// two signs hold 24, down to 2^-133, where bfloat16 ends: of numbers below 2^-109 the last bits are lost).
__device__ __forceinline__ void split2(float a, float b, uint32_t& p1, uint32_t& p2, uint32_t& p3) {
    typedef bf16_t pair __attribute__((ext_vector_type(2)));
    typedef float fpair __attribute__((ext_vector_type(2)));
    auto pack = [](float x, float y) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(fpair{x, y}, pair)); };
    p1 = pack(a, b);
    a -= __builtin_bit_cast(float, p1 << 16);
    b -= __builtin_bit_cast(float, p1 & 0xffff0000u);
    p2 = pack(a, b);
    a -= __builtin_bit_cast(float, p2 << 16);
    b -= __builtin_bit_cast(float, p2 & 0xffff0000u);
    p3 = pack(a, b);
}
