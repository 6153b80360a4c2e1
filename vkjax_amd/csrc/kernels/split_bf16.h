// What the kernels that compute fp32 products on the bf16 matrix cores share (how a number is taken apart: conv_split.h).
#pragma once
#include "common.h"

typedef __bf16   bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16   bf16x2 __attribute__((ext_vector_type(2)));
typedef float    f32x2  __attribute__((ext_vector_type(2)));

// the two numbers' nearest bf16, the first in the low half
__device__ __forceinline__ uint32_t to_bf16x2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
}
// Consecutive workgroup ids go to the 8 XCDs in turn: renumbers [0, n) so that every XCD works through a contiguous range.
__device__ __forceinline__ int xcd_range(int id, int n) {
    const int per = n / 8;
    return per > 0 && id < per * 8 ? (id & 7) * per + (id >> 3) : id;
}
