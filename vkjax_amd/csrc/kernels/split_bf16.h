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
// What is left of a number when the low (high) half of `parts` has been taken off: one instruction instead of a shift or mask and a
// subtraction, with the same bits for every number up to the largest bf16 (2^24 pairs over all exponents compared). Beyond it the half is
// infinite and leaves a NaN beside it too, in a row of the product that is not finite anyway. (The vector instructions of a split hardly
// overlap with the matrix instructions: ResNet-50 at batch 64 3.87 -> 3.78 ms, its training step 13.82 -> 13.31 ms.)
// (The low half's factors are kept from the compiler, which takes {-1, 0} for its inline constant -1.0, whose -1 is the high half.)
__device__ __forceinline__ float minus_low(uint32_t parts, float v) {
    uint32_t factors = 0x0000BF80u;
    asm("" : "+s"(factors));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, parts), __builtin_bit_cast(bf16x2, factors), v, false);
}
__device__ __forceinline__ float minus_high(uint32_t parts, float v) {
    uint32_t factors = 0xBF800000u;
    asm("" : "+s"(factors));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, parts), __builtin_bit_cast(bf16x2, factors), v, false);
}
// Consecutive workgroup ids go to the 8 XCDs in turn: renumbers [0, n) so that every XCD works through a contiguous range.
__device__ __forceinline__ int xcd_range(int id, int n) {
    const int per = n / 8;
    return per > 0 && id < per * 8 ? (id & 7) * per + (id >> 3) : id;
}
// max(high, |a|, |b|); NaN if one of them is
__device__ __forceinline__ float higher_of(float high, float a, float b) {
    asm("v_maximum3_f32 %0, %0, |%1|, |%2|" : "+v"(high) : "v"(a), "v"(b));
    return high;
}
// threadIdx.x of a one-dimensional block, from the wave's number
__device__ __forceinline__ int tid_again(int wave) {
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
    return wave * 64 + lane;
}
