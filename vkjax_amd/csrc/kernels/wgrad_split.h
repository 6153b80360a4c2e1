// Kernel gradients on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16) at fp32's accuracy: the contraction of wgrad_gemm.hip, whose
// parameter block these kernels share, with both operands taken apart into three bf16 numbers (conv_split.h says how and how exactly).
#pragma once
#include "split_bf16.h"

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Block = 2 x 2 waves (twice as many where PAIR, below), each with TM x TN tiles of 32 x 32; k tile: 32 pixels. The matrix cores want eight consecutive pixels of one
// column per lane where memory has consecutive columns of one pixel, so a thread loads eight pixels of four columns (16 bytes each)
// and finds every column's eight numbers in its own registers: taken apart they are 16 bytes of LDS per column and part,
// [part][octet of pixels][column]. Columns lie by their number modulo 4 first (what 32 threads of a wave write at once is contiguous),
// xor-ed so that the four groups of eight which a wave reads for a tile of 32 columns lie in banks of their own.
// A tile's row r stands for column 4 (r % 8) + r / 8 of its 32, in both operands: the stores of a wave stay whole lines.
//
// Pixels: a wave's lanes compute where the (up to 32) pixels of its next items lie, once per k tile, and hand that round through LDS:
// a byte offset and the pixel's (y, x) as two 16-bit numbers, to which a column's tap is added and compared with the image's size.
// Rows of a matrix, and convolutions of 1 x 1 with a stride of 1, have no such table: a pixel's offset is its number.
//
// What it gives (MI355X, ResNet-50 at batch 64; through wgrad_gemm.hip's v_mfma_f32_32x32x2_f32 in brackets): 3x3x256x256 on 12544 pixels
// 81 us (147), 3x3x128x128 on 50176 81 (147), 1x1x512x128 on 50176 42 (65), 3x3x64x64 on 200704 108 (140), 1x1x64x256 on 200704 51 (69; the
// two operands alone are 46 us of HBM reads), the stem's 7x7x3x64 on 802816 180 (243; its words are loaded one by one). Error against
// 64-bit sums 0.3 to 0.65 times that of the fp32 products (3136 to 50176 pixels).
// Sums: the twelve products of a k tile are chained from zero and added to the accumulators by fp32 operations, G's sign changed in
// every other k tile (the matrix cores cut sums off, see conv_split.h).
// Scale: both operands are multiplied by 2^24 before they are taken apart and the sums by 2^-48, so the smallest numbers have all their bits
// (a bf16 part of a number below 2^-102 would not). It costs 1 to 2 % of the kernel. (Looking behind the loop for sums that such numbers could
// matter to, and through their columns, costs as much for the columns' largest numbers and far more where it finds some: sums of nothing but
// zeros are everywhere behind a ReLU, ResNet-50's training step took 17.7 ms instead of 12.6.)
constexpr float WGRAD_SCALE = 0x1p24f;
//
// PAIR: a block is two such groups of four waves, each with LDS of its own and half of the slice's k tiles; they take turns, the one
// takes its tile apart while the other one multiplies, and add their sums up in LDS in the end: half as many partial results are written, and
// read by the sum behind, as by two blocks per CU that each have a slice. ResNet-50's training step at batch 64: 12.59 -> 12.40 ms, the
// launch that adds the partial results 288 -> 185 us.
template <int TM, int TN, bool VEC_A, bool VEC_B, bool PAIR>
__device__ __forceinline__ void wgrad_split_body(u32x4* __restrict__ lds, u32x2* __restrict__ table, float* __restrict__ out,
                                                 const float* __restrict__ x, const float* __restrict__ g, const WgradParams& P, const WgradSplitParams& Q) {
    constexpr int BM = 64 * TM, BN = 64 * TN, BK = 32;
    const int tid = threadIdx.x, lane = tid & 63, wave_of_block = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = wave_of_block & 3, group = PAIR ? wave_of_block >> 2 : 0;
    float* const exchange = reinterpret_cast<float*>(lds);
    lds += group * 12 * (BM + BN);
    table += group * 4 * 32;
    u32x4 *const As = lds, *const Bs = lds + 12 * BM;             // [3 parts][4 octets][columns]
    const int wm = wave >> 1, wn = wave & 1, l32 = lane & 31, half = lane >> 5;
    // the blocks of one slice read the same pixels: neighbours on one XCD
    const int work = xcd_range((int)blockIdx.x, (int)gridDim.x), tiles = Q.tiles_m * Q.tiles_n;
    const int slice = work / tiles, tile = work - slice * tiles, tile_m = tile / Q.tiles_n, tile_n = tile - tile_m * Q.tiles_n;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    int kbeg = slice * P.pix_per_split, kend = min(P.pixels, kbeg + P.pix_per_split), nk = kbeg < kend ? (kend - kbeg + BK - 1) / BK : 0, turns = nk;
    if constexpr (PAIR) {                                         // the first group has the odd k tile
        turns = (nk + 1) / 2;
        if (group == 0) { kend = min(kend, kbeg + turns * BK); nk = turns; }
        else            { kbeg += turns * BK; nk -= turns; }
    }
    const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(x, P.x_bytes), g_rsrc = make_rsrc(g, P.g_bytes);
    const bool flat = Q.flat != 0;

    // ---- what this thread loads: eight pixels (an octet of the k tile) of four columns, of X in the first waves, of G in the next
    const bool is_a = wave < BM / 64, is_b = !is_a && wave < (BM + BN) / 64;
    const int cols4 = (is_a ? BM : BN) / 4, item = (is_a ? wave : wave - BM / 64) * 64 + lane;
    const int cg = item & (cols4 - 1), oct = item / cols4;
    const int wave_px = oct - ((lane / cols4)), pixels_per_wave = 64 / cols4 * 8;   // first octet of the wave, and its pixels
    constexpr int NA = VEC_A ? 1 : 4;
    uint32_t a_off[NA];
    u16x2 a_yx[NA];
    uint32_t b_off[4];
    const int first = (is_a ? m0 : n0) + 4 * cg;
    if (is_a) {
#pragma unroll
        for (int q = 0; q < NA; ++q) {
            const int m   = first + q;
            const int tap = magic_div(m, P.c_magic, P.c_shift);
            const int ky  = magic_div(tap, P.kw_magic, P.kw_shift);
            const int ci = m - tap * P.C, dy = ky * P.DH - P.PH, dx = (tap - ky * P.KW) * P.DW - P.PW;
            if (flat) a_off[q] = m < P.M ? (uint32_t)((kbeg + oct * 8) * P.C + m) * 4u : WG_OOB;
            else      a_off[q] = (uint32_t)((dy * P.W + dx) * P.C + ci) * 4u;
            a_yx[q] = m < P.M ? u16x2{(uint16_t)dx, (uint16_t)dy} : u16x2{0x7000, 0x7000};
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) b_off[q] = first + q < P.N ? (uint32_t)((kbeg + oct * 8) * P.N + first + q) * 4u : WG_OOB;
    const u16x2 last_yx = {(uint16_t)(P.W - 1), (uint16_t)(P.H - 1)};
    float raw[8][4];
    auto load_tile = [&](int kt) {
        if (is_b) {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const uint32_t soff = (uint32_t)((kt * BK + q) * P.N) * 4u;
                if constexpr (VEC_B) {
                    const f32x4 v = buffer_load_x4(g_rsrc, b_off[0], soff);
#pragma unroll
                    for (int e = 0; e < 4; ++e) raw[q][e] = v[e];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) raw[q][e] = buffer_load_x1(g_rsrc, b_off[e], soff);
                }
            }
        } else if (is_a && flat) {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const uint32_t soff = (uint32_t)((kt * BK + q) * P.C) * 4u;
                if constexpr (VEC_A) {
                    const f32x4 v = buffer_load_x4(x_rsrc, a_off[0], soff);
#pragma unroll
                    for (int e = 0; e < 4; ++e) raw[q][e] = v[e];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) raw[q][e] = buffer_load_x1(x_rsrc, a_off[e], soff);
                }
            }
        } else if (is_a) {
            if (lane < pixels_per_wave) {
                const int p   = kbeg + kt * BK + wave_px * 8 + lane;
                const int img = magic_div(p, P.howo_magic, P.howo_shift), r = p - img * (P.Ho * P.Wo);
                const int ho  = magic_div(r, P.wo_magic, P.wo_shift), y0 = ho * P.SH, x0 = (r - ho * P.Wo) * P.SW;
                table[wave * 32 + lane] = u32x2{(uint32_t)(((img * P.H + y0) * P.W + x0) * P.C) * 4u,
                                                p < kend ? (uint32_t)y0 << 16 | (uint32_t)x0 : 0x70007000u};
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const u32x2* const from = table + wave * 32 + (oct - wave_px) * 8;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const uint32_t px_off = from[q].x, px_yx = from[q].y;
#pragma unroll
                for (int e = 0; e < NA; ++e) {
                    const u16x2 at = __builtin_bit_cast(u16x2, px_yx) + a_yx[e];
                    const bool ok  = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(at, last_yx)) == __builtin_bit_cast(uint32_t, at);
                    const uint32_t off = ok ? px_off + a_off[e] : WG_OOB;
                    if constexpr (VEC_A) {
                        const f32x4 v = buffer_load_x4(x_rsrc, off);
#pragma unroll
                        for (int c = 0; c < 4; ++c) raw[q][c] = v[c];
                    } else {
                        raw[q][e] = buffer_load_x1(x_rsrc, off);
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    };
    u32x4* const to = (is_a ? As : Bs) + oct * (is_a ? BM : BN);
    const int part_step = 4 * (is_a ? BM : BN);
    auto park_tile = [&](bool odd) {
        if (!is_a && !is_b) return;
        const float scale = odd && is_b ? -WGRAD_SCALE : WGRAD_SCALE;
#pragma unroll
        for (int q = 0; q < 8; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) raw[q][e] *= scale;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            u32x4* const slot = to + e * cols4 + (cg ^ ((e * 8) & (cols4 - 1)));
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                u32x4 part;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t v = to_bf16x2(raw[2 * q][e], raw[2 * q + 1][e]);
                    if (t < 2 && TM * TN == 1) {
                        raw[2 * q][e] = minus_low(v, raw[2 * q][e]); raw[2 * q + 1][e] = minus_high(v, raw[2 * q + 1][e]);
                    } else if (t < 2) {                          // larger tiles are slower with it: 3x3x128x128 on 50176 pixels 96 us against 87
                        raw[2 * q][e] -= u2f(v << 16); raw[2 * q + 1][e] -= u2f(v & 0xFFFF0000u);
                    }
                    part[q] = v;
                }
                slot[t * part_step] = part;
            }
        }
    };
    // where lane l of a wave reads tile `block` of 32 columns (k16 step 0, part 0)
    auto read_slot = [&](int block, int columns) {
        const int e = l32 >> 3, c = block * 8 + (l32 & 7), n4 = columns / 4;
        return half * columns + e * n4 + (c ^ ((e * 8) & (n4 - 1)));
    };
    const u32x4 *a_from[TM], *b_from[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) a_from[i] = As + read_slot(wm * TM + i, BM);
#pragma unroll
    for (int j = 0; j < TN; ++j) b_from[j] = Bs + read_slot(wn * TN + j, BN);

    f32x16 acc[TM][TN] = {};
    constexpr int PA[6] = {2, 1, 1, 0, 0, 0}, PB[6] = {0, 0, 1, 1, 2, 0};
    if (nk > 0) load_tile(0);
    if (PAIR && group == 1) __syncthreads();
    for (int kt = 0; kt < turns; ++kt) {
        if (!PAIR || kt < nk) park_tile(kt & 1);
        __syncthreads();
        if (PAIR && kt >= nk) { __syncthreads(); continue; }
        if (kt + 1 < nk) load_tile(kt + 1);
        const float sign = kt & 1 ? -1.f / (WGRAD_SCALE * WGRAD_SCALE) : 1.f / (WGRAD_SCALE * WGRAD_SCALE);
        bf16x8 af[TM][2][3];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int t = 0; t < 3; ++t) af[i][ks][t] = __builtin_bit_cast(bf16x8, a_from[i][(t * 4 + 2 * ks) * BM]);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            bf16x8 bf[2][3];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int t = 0; t < 3; ++t) bf[ks][t] = __builtin_bit_cast(bf16x8, b_from[j][(t * 4 + 2 * ks) * BN]);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                f32x16 sum = {};
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                    for (int t = 0; t < 6; ++t) sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i][ks][PA[t]], bf[ks][PB[t]], sum, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = __builtin_fmaf(sum[v], sign, acc[i][j][v]);
            }
        }
        __syncthreads();
    }
    if (PAIR && group == 0) __syncthreads();

    // Sums that are not finite (an operand that is infinite, not a number, or beyond 2^104; a sum beyond 2^80): again, with fp32 products. The
    // finite ones beside them stay as they are.
    float high = 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; v += 2) high = higher_of(high, acc[i][j][v], acc[i][j][v + 1]);
    if (__builtin_amdgcn_ballot_w64(!(high < __builtin_inff()))) {
        // Steps of eight pixels per half of the wave, the next step's words requested before this one's products. 12544 pixels, 2304 x 256 with NaN
        // only: 465 us (95 without; 868 with the words requested one after the other), through the fp32 kernels 160.
        constexpr int U = 8;
        int dy[TM], dx[TM];
        uint32_t x_at[TM];
        bool in_m[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int m   = m0 + (wm * TM + i) * 32 + 4 * (l32 & 7) + (l32 >> 3);
            const int tap = magic_div(m, P.c_magic, P.c_shift), ky = magic_div(tap, P.kw_magic, P.kw_shift);
            dy[i] = ky * P.DH - P.PH; dx[i] = (tap - ky * P.KW) * P.DW - P.PW;
            x_at[i] = (uint32_t)((dy[i] * P.W + dx[i]) * P.C + m - tap * P.C) * 4u;
            in_m[i] = m < P.M;
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            bool any = false;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int v = 0; v < 16; ++v) any |= !__builtin_isfinite(acc[i][j][v]);
            if (!__builtin_amdgcn_ballot_w64(any)) continue;
            const int n = n0 + (wn * TN + j) * 32 + 4 * (l32 & 7) + (l32 >> 3);
            f32x16 again[TM] = {}, total[TM] = {};                // (summed by 64 pixels)
            float x_next[TM][U], g_next[U];
            auto request = [&](int p0) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int p   = p0 + 2 * u + half;
                    const int img = magic_div(p, P.howo_magic, P.howo_shift), r = p - img * (P.Ho * P.Wo);
                    const int ho  = magic_div(r, P.wo_magic, P.wo_shift), y0 = ho * P.SH, x0 = (r - ho * P.Wo) * P.SW;
                    const uint32_t px = (uint32_t)(((img * P.H + y0) * P.W + x0) * P.C) * 4u;
#pragma unroll
                    for (int i = 0; i < TM; ++i) {
                        const bool ok = p < kend && in_m[i] && (uint32_t)(y0 + dy[i]) < (uint32_t)P.H && (uint32_t)(x0 + dx[i]) < (uint32_t)P.W;
                        x_next[i][u] = buffer_load_x1(x_rsrc, ok ? px + x_at[i] : WG_OOB);
                    }
                    g_next[u] = buffer_load_x1(g_rsrc, p < kend && n < P.N ? (uint32_t)(p * P.N + n) * 4u : WG_OOB);
                }
            };
            request(kbeg);
#pragma nounroll
            for (int p0 = kbeg; p0 < kend; p0 += 2 * U) {
                float xv[TM][U], gv[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
#pragma unroll
                    for (int i = 0; i < TM; ++i) xv[i][u] = x_next[i][u];
                    gv[u] = g_next[u];
                }
                request(p0 + 2 * U);
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int i = 0; i < TM; ++i) again[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[i][u], gv[u], again[i], 0, 0, 0);
                if ((p0 - kbeg) % 64 == 48 || p0 + 2 * U >= kend) {
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int v = 0; v < 16; ++v) { total[i][v] += again[i][v]; again[i][v] = 0.f; }
                }
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = __builtin_isfinite(acc[i][j][v]) ? acc[i][j][v] : total[i][v];
        }
    }
    float* const result = out + (size_t)slice * P.M * P.N;
    auto store_row_of_tiles = [&](auto i_) {
        constexpr int i = decltype(i_)::value;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int col = n0 + (wn * TN + j) * 32 + 4 * (l32 & 7) + (l32 >> 3);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = m0 + (wm * TM + i) * 32 + 4 * (4 * half + v % 4) + v / 4;
                if (row < P.M && col < P.N) result[(size_t)row * P.N + col] = acc[i][j][v];
            }
        }
    };
    if constexpr (PAIR) {
        // group i finishes row i of its waves' tiles, with the other group's sums of it
        static_assert(TM == 2, "a row of tiles for each group");
        auto hand_over = [&](auto i_) {
            constexpr int i = decltype(i_)::value;
            float* const to = exchange + i * (4 * TN * 16 * 64) + wave * (TN * 16 * 64) + lane;
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) to[(j * 16 + v) * 64] = acc[i][j][v];
        };
        auto finish = [&](auto i_) {
            constexpr int i = decltype(i_)::value;
            const float* const from = exchange + i * (4 * TN * 16 * 64) + wave * (TN * 16 * 64) + lane;
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] += from[(j * 16 + v) * 64];
            store_row_of_tiles(i_);
        };
        if (group == 0) hand_over(std::integral_constant<int, 1>{}); else hand_over(std::integral_constant<int, 0>{});
        __syncthreads();
        if (group == 0) finish(std::integral_constant<int, 0>{}); else finish(std::integral_constant<int, 1>{});
    } else {
        store_row_of_tiles(std::integral_constant<int, 0>{});
        if constexpr (TM == 2) store_row_of_tiles(std::integral_constant<int, 1>{});
    }
}

#define WGRAD_SPLIT_KERNEL(name, TM, TN, VA, VB, WPE, PAIR)                                                                         \
    extern "C" __global__ __launch_bounds__(PAIR ? 512 : 256) __attribute__((amdgpu_waves_per_eu(WPE))) void name(                         \
        float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ g, WgradParams P, WgradSplitParams Q) { \
        __shared__ __attribute__((aligned(16))) u32x4 lds[(PAIR ? 2 : 1) * 12 * 64 * (TM + TN)];                                               \
        __shared__ __attribute__((aligned(16))) u32x2 table[(PAIR ? 2 : 1) * 4 * 32];                                                          \
        request_arguments<3 * sizeof(void*) + sizeof(WgradParams) + sizeof(WgradSplitParams)>();                                    \
        wgrad_split_body<TM, TN, VA, VB, PAIR>(lds, table, out, x, g, P, Q);                                                        \
    }
WGRAD_SPLIT_KERNEL(wgrad_split_128x128_aa, 2, 2, true, true, 2, true)
WGRAD_SPLIT_KERNEL(wgrad_split_128x64_aa, 2, 1, true, true, 3, false)
WGRAD_SPLIT_KERNEL(wgrad_split_64x128_aa, 1, 2, true, true, 3, false)
WGRAD_SPLIT_KERNEL(wgrad_split_64x64_aa, 1, 1, true, true, 4, false)
WGRAD_SPLIT_KERNEL(wgrad_split_64x64_sa, 1, 1, false, true, 4, false)
