// Shared device helpers for the vkJAX gfx950 kernels (wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

typedef float    f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float    f32x16 __attribute__((ext_vector_type(16)));

#define VKJ_WAVE 64

__device__ __forceinline__ uint32_t f2u(float x) { return __float_as_uint(x); }
__device__ __forceinline__ float    u2f(uint32_t x) { return __uint_as_float(x); }

// The value of lane ^ S, in vector instructions: __shfl_xor goes through LDS, a round trip of some 100 cycles, of which a butterfly makes six in a row.
// (Needs the lanes it reads to be active, like __shfl_xor.)
template <int S>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
    static_assert(S == 1 || S == 2 || S == 4 || S == 8 || S == 16 || S == 32, "a step of a butterfly");
    if constexpr (S == 1) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);           // quads: 1 0 3 2
    else if constexpr (S == 2) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true);      // quads: 2 3 0 1
    else if constexpr (S == 4) {                                        // quads 0 and 2 of a row of 16 lanes take the next quad, 1 and 3 the one before
        const int up = __builtin_amdgcn_update_dpp((int)v, (int)v, 0x104, 0xF, 0x5, false);
        return (uint32_t)__builtin_amdgcn_update_dpp(up, (int)v, 0x114, 0xF, 0xA, false);
    }
    else if constexpr (S == 8) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xF, 0xF, true);     // a row turned by 8
    else {                                                              // [0]: the even rows (the lower half) twice, [1]: the odd ones (the upper half) twice
        const bool second = (__lane_id() & (uint32_t)S) != 0u;
        if constexpr (S == 16) { const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false); return second ? r[0] : r[1]; }
        else                   { const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false); return second ? r[0] : r[1]; }
    }
}
template <int S> __device__ __forceinline__ float lane_xor(float v) { return u2f(lane_xor<S>(f2u(v))); }
template <int S> __device__ __forceinline__ uint64_t lane_xor(uint64_t v) {
    return (uint64_t)lane_xor<S>((uint32_t)(v >> 32)) << 32 | lane_xor<S>((uint32_t)v);
}
// step(std::integral_constant<int, S>) for S = 32, 16 .. 1
template <class F>
__device__ __forceinline__ void wave_butterfly(F step) {
    step(std::integral_constant<int, 32>{}); step(std::integral_constant<int, 16>{}); step(std::integral_constant<int, 8>{});
    step(std::integral_constant<int, 4>{});  step(std::integral_constant<int, 2>{});  step(std::integral_constant<int, 1>{});
}
// Butterfly across groups of `lanes` lanes (a power of two, the same in the whole wave), the widest step first.
template <class T, class F>
__device__ __forceinline__ T lanes_allreduce(T v, uint32_t lanes, F f) {
    if (lanes > 32u) v = f(v, lane_xor<32>(v));
    if (lanes > 16u) v = f(v, lane_xor<16>(v));
    if (lanes > 8u)  v = f(v, lane_xor<8>(v));
    if (lanes > 4u)  v = f(v, lane_xor<4>(v));
    if (lanes > 2u)  v = f(v, lane_xor<2>(v));
    if (lanes > 1u)  v = f(v, lane_xor<1>(v));
    return v;
}

// Buffer-descriptor access: loads beyond `bytes` return 0 and stores there are dropped, so a lane
// that must not touch memory is given an offset of 0x80000000.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
// voff: per-lane byte offset, soff: wave-uniform byte offset; the range check covers their sum
__device__ __forceinline__ f32x4 buffer_load_x4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff = 0) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ __forceinline__ float buffer_load_x1(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff = 0) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ void buffer_store_x1(float v, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff = 0) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, voff, soff, 0);
}
// the same for data that is touched once (nontemporal: not kept in the caches at the expense of what is reused)
__device__ __forceinline__ float buffer_load_x1_nt(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff = 0) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 2));
}
// Bit 31 of the first word of a kernel's parameters (an element count below 2^31 in every kernel that looks at it):
// the result is stored with the nontemporal hint. The host sets it for large results that no later launch of the
// program reads (they leave for the host, or stay where they are): such an array only pushes out of the caches what
// could be reused, and the stores of a launch that reads and writes run faster past the L2 (relu on 64 M elements
// 92 -> 76 us). Results that the next launch reads are left to the caches (256 MB behind the L2s: a training step
// whose backward kernels streamed their results was 0.15 ms slower). Only for results below 4 GiB (a buffer
// addresses 32 bits); the host checks.
#define STREAM_RESULT_BIT 0x80000000u
__device__ __forceinline__ bool streams_result(uint32_t first_word) { return (first_word & STREAM_RESULT_BIT) != 0u; }
__device__ __forceinline__ uint32_t without_stream_bit(uint32_t first_word) { return first_word & ~STREAM_RESULT_BIT; }
// base[element .. element + 4) = v; `stream`: past the caches. (Through a buffer: written as two stores through one
// pointer, one of them nontemporal, the compiler merges them into one plain store.)
__device__ __forceinline__ void store_x4(uint32_t* base, uint64_t element, u32x4 v, bool stream, uint32_t result_bytes) {
    if (stream) __builtin_amdgcn_raw_buffer_store_b128(v, make_rsrc(base, result_bytes), (uint32_t)element * 4u, 0, 2);
    else *reinterpret_cast<u32x4*>(base + element) = v;
}
__device__ __forceinline__ int magic_div(int n, uint32_t magic, uint32_t shift) {
    return magic ? (int)(__umulhi((uint32_t)n, magic) >> shift) : n;
}

// Requests every 64 bytes of a kernel's first BYTES of arguments at once. Left to itself the compiler fetches an argument where it is first used, and each
// line of 64 bytes that no fetch has touched before is a round trip to memory of its own, some 0.7 us one after the other in front of a launch's first load.
// (For kernels that do not read their arguments in one go by themselves. Replays with and without: a convolutional network's training step 227.2, 225.8 us,
// ResNet-50 on six images of 160 x 160 607, 603, on 64 images 3.90, 3.86 ms.)
template <size_t BYTES>
__device__ __forceinline__ void request_arguments() {
    const uint32_t* const words = reinterpret_cast<const uint32_t*>(__builtin_amdgcn_kernarg_segment_ptr());
    uint32_t all = words[(BYTES - 4) / 4];
#pragma unroll
    for (size_t at = 0; at + 4 < BYTES; at += 64) all |= words[at / 4];
    asm volatile("" :: "s"(all));
}

// Consecutive workgroup ids are handed to the 8 XCDs in turn, and every XCD has an L2 of its own.
// This renumbers the workgroups of a 1-D grid so that each XCD works through a contiguous range:
// kernels whose neighbouring workgroups read overlapping data (windows, halos) then find the
// overlap in their own L2 instead of fetching it once per XCD. A bijection on [0, gridDim.x).
__device__ __forceinline__ uint32_t xcd_contiguous_block() {
    const uint32_t b = blockIdx.x, per = gridDim.x / 8u;
    return (per > 0u && b < per * 8u) ? (b & 7u) * per + (b >> 3) : b;
}
