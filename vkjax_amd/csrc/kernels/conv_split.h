// fp32 implicit GEMM on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16). Included by conv_gemm.hip, whose parameter block,
// epilogue and addressing these kernels share.
//
// An fp32 number is the sum of three bf16 numbers: hi = its nearest bf16, mid = the nearest bf16 of what is left, lo = the
// rest, which has at most 8 significant bits by then (24 = 8 + 8 + 8). A product of two such numbers is taken as the six
// products hi.hi, hi.mid, mid.hi, hi.lo, mid.mid, lo.hi, each exact in fp32 and added in fp32 accumulators; the three that are
// left out are below 2^-24 of the product together, the rounding of an fp32 accumulation. The matrix cores run bf16 sixteen
// times as fast as fp32, so six products instead of one are still 2.6 times as fast at peak.
//   - a number below 2^-102 has parts that a bf16 holds with fewer bits, or not at all: both operands are multiplied by 2^24 before they are
//     taken apart, and the sums by 2^-48, so the smallest numbers have all their bits (which costs 1 to 2 % of the kernel);
//   - operands that are infinite, NaN or beyond 2^104 (then beyond the largest bf16) leave sums that are not finite, because a part that is
//     infinite meets parts that are zero, and so do sums beyond 2^80: a wave whose results are not all finite computes those that are not again
//     with v_mfma_f32_32x32x2_f32 and fp32 operands, so that such results are what fp32 products give.
// Measured against 64-bit sums (4096 x K x 128, normal data): an error of 0.76, 0.56 and 0.30 times that of
// v_mfma_f32_32x32x2_f32 at K = 64, 576 and 2304 (which rounds after every second product, this after every sixteenth). Sums of which less than
// a fifth of the terms are not zero are further off than those: 1.3 times at 16 of 512, 1.4 times at one (which is cut off, not rounded).
// The kernels that serve products the fp32 kernels would be nearly as fast at (_short, _fine) are not: see CONV_FINE_PA.
#pragma once
#include "split_bf16.h"

// ---- the kernel operand, taken apart and laid out for the matrix cores ----------------------------------------------
// A program's weights serve every row of a product: a launch of this kernel takes them apart once, instead of every tile of
// rows doing it again, and lays them out in the order in which the lanes of a wave want them, so that the product's waves
// load them straight into registers (16 bytes per lane, 1 KB per wave and load), past the LDS:
//     [block of 32 columns][k16 step][part hi, mid, lo][lane] x 8 bf16
// Lane l of a k16 step holds column l % 32 and octet o = 2 (step % 2) + l / 32 of its k tile of 32: k = 4o .. 4o+3 and
// 16+4o .. 16+4o+3 (the order in which four lanes that share a row of the other operand load 64 contiguous bytes each time).
// The kernel operand may lie in any order (strides, negative ones too), which makes the transposed and reversed kernels of a
// backward pass no work of their own.
// For the kernels that hold a patch of the input in LDS (PATCH below) a step is 16 input features under one tap of a 3 x 3 window, the nine taps
// one after the other: [block of 32 columns][16 features][tap][part][lane], lane l: features 4o .. 4o+3 and 8+4o .. of them for o = l / 32.
struct ConvPackParams {
    int32_t N, K, Cin, KW;               // k = (ky * KW + kx) * Cin + c; K below 0: -K, in the order for a patch
    int32_t ws_r, ws_s, ws_c, ws_n;      // element strides of ky, kx, c, n
};
struct ConvPackEntry {
    uint32_t first_block, pad;
    u32x4*       out;
    const float* w;
    ConvPackParams P;
};
static_assert(sizeof(ConvPackEntry) == 56, "the host lays the table out with 56-byte entries");

// A number that the scale takes beyond the largest bf16 is stored as it is: a NaN of its own kind in front, which has the column's sums computed
// again with fp32 products, and its two halves behind it.
constexpr float CONV_SPLIT_SCALE = 0x1p24f;
constexpr uint32_t CONV_PACK_RAW = 0x7FC1u;

constexpr uint32_t CONV_SPLIT_MASKED = 1u << 25;      // ConvParams::flags; the host has it under the same name

__device__ __forceinline__ void conv_pack_body(u32x4* __restrict__ out, const float* __restrict__ w, const ConvPackParams& P, int block) {
    const bool patch = P.K < 0;
    const int K = patch ? -P.K : P.K;
    const int id = block * 256 + (int)threadIdx.x, lane = id & 63, step = id >> 6, ksteps = patch ? K / 16 : (K + 63) / 64 * 4;
    const int nb = step / ksteps, s = step - nb * ksteps, o = 2 * (s & 1) + (lane >> 5), n = nb * 32 + (lane & 31);
    if (nb * 32 >= P.N) return;
    const int sixteen = s / 9, tap = s - 9 * sixteen;
    const bool negative = patch ? s / 3 & 1 : s & 4;        // every other group of steps: see the product's sums
    float x[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int c_patch = 16 * sixteen + 8 * h + 4 * (lane >> 5), k0 = (s >> 1) * 32 + h * 16 + 4 * o, rs = patch ? tap : k0 / P.Cin;
        int c = patch ? c_patch : k0 - rs * P.Cin, ky = rs / P.KW, kx = rs - ky * P.KW;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            // (the last vector of a patch, where features are left for a part of one only, ends with the last feature: it begins with ones that were there before)
            if (patch) c = c_patch + 4 > P.Cin && c_patch < P.Cin ? P.Cin - 4 + q : c_patch + q;
            const float v = ((patch ? c >= c_patch && c < P.Cin : k0 + q < K) && n < P.N) ? w[(int64_t)ky * P.ws_r + (int64_t)kx * P.ws_s + (int64_t)c * P.ws_c + (int64_t)n * P.ws_n] : 0.f;
            x[4 * h + q] = negative ? -v : v;
            if (++c == P.Cin && !patch) { c = 0; if (++kx == P.KW) { kx = 0; ++ky; } }
        }
    }
    u32x4 part[3];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float rest[2] = {x[2 * q] * CONV_SPLIT_SCALE, x[2 * q + 1] * CONV_SPLIT_SCALE};
        uint32_t v[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            v[t] = to_bf16x2(rest[0], rest[1]);
            rest[0] -= u2f(v[t] << 16);
            rest[1] -= u2f(v[t] & 0xFFFF0000u);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t shift = 16 * h, bits = f2u(x[2 * q + h]), keep = h ? 0xFFFFu : 0xFFFF0000u;
            if ((v[0] >> shift & 0x7F80u) != 0x7F80u) continue;
            const bool raw = __builtin_isfinite(x[2 * q + h]);
            const uint32_t front = raw ? CONV_PACK_RAW : bits << 1 > 0xFF000000u ? 0x7FC0u : bits >> 16;
            v[0] = (v[0] & keep) | front << shift;
            v[1] = (v[1] & keep) | (raw ? bits >> 16 : 0u) << shift;
            v[2] = (v[2] & keep) | (raw ? bits & 0xFFFFu : 0u) << shift;
        }
#pragma unroll
        for (int t = 0; t < 3; ++t) part[t][q] = v[t];
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) out[(size_t)step * 192 + t * 64 + lane] = part[t];
}
extern "C" __global__ __launch_bounds__(256) void conv_split_pack(u32x4* __restrict__ out, const float* __restrict__ w, ConvPackParams P) {
    conv_pack_body(out, w, P, blockIdx.x);
}
// The weights of several layers in one launch: workgroup b belongs to the last entry of the table whose first_block is <= b.
extern "C" __global__ __launch_bounds__(256) void conv_split_pack_layers(const ConvPackEntry* __restrict__ table, uint32_t entries) {
    uint32_t lo = 0, hi = entries;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (table[mid].first_block <= blockIdx.x) lo = mid; else hi = mid;
    }
    const ConvPackEntry& e = table[__builtin_amdgcn_readfirstlane(lo)];
    conv_pack_body(e.out, e.w, e.P, (int)(blockIdx.x - e.first_block));
}

__device__ __forceinline__ uint32_t conv_split_step_desc(const ConvParams& P, int e) {
    return ((e < 3 ? P.epi_desc[0] : P.epi_desc[1]) >> (10 * (e < 3 ? e : e - 3))) & 1023u;
}
// The epilogue's scalars and per-column vectors, to LDS
template <int BN>
__device__ __forceinline__ void conv_split_epilogue_operands(float* __restrict__ Es, const ConvEpiPtrs& epi, const ConvDerivedPtrs& Dp, const ConvParams& P,
                                                             const ConvDerived& Dk, int tid, int n0) {
    if (tid < BN) {
        float e_reg[CONV_MAX_EPI], d_in[CONV_MAX_DERIVED + 1];
#pragma unroll
        for (int e = 0; e < CONV_MAX_EPI; ++e) {
            const uint32_t kind = conv_split_step_desc(P, e) >> 8;
            const uint32_t present = epi.p[e] != nullptr ? 1u : 0u;
            e_reg[e] = buffer_load_x1(make_rsrc(epi.p[e], kind == 1 ? 4u * present : kind == 2 ? (uint32_t)P.N * 4u * present : 0u),
                                      kind == 2 ? (uint32_t)(n0 + tid) * 4u : 0u);
        }
        if (Dk.nsteps) {
#pragma unroll
            for (int k = 0; k <= CONV_MAX_DERIVED; ++k) {
                const bool vec = (Dk.vector_mask >> k) & 1u;
                d_in[k] = buffer_load_x1(make_rsrc(Dp.p[k], Dp.p[k] == nullptr ? 0u : vec ? (uint32_t)P.N * 4u : 4u),
                                         vec ? (uint32_t)(n0 + tid) * 4u : 0u);
            }
            const float v = conv_derived_value(d_in, Dk);
#pragma unroll
            for (int e = 0; e < CONV_MAX_EPI; ++e)
                if (e == (int)Dk.step) e_reg[e] = v;
        }
#pragma unroll
        for (int e = 0; e < CONV_MAX_EPI; ++e)
            if (e < (int)((P.flags >> 8) & 15u)) Es[e * BN + tid] = e_reg[e];
    }
}

#define FENCE() __builtin_amdgcn_sched_barrier(0)
// The next part of two neighbouring numbers of an item's eight, and what is left of them: their nearest bf16
__device__ __forceinline__ uint32_t conv_split_word(f32x4 (&x)[2], int t, int q) {
    f32x4& v = x[q >> 1];
    const int e = 2 * (q & 1);
    if (t == 0) { v[e] *= CONV_SPLIT_SCALE; v[e + 1] *= CONV_SPLIT_SCALE; }
    const uint32_t w2 = to_bf16x2(v[e], v[e + 1]);
    if (t < 2) { v[e] = minus_low(w2, v[e]); v[e + 1] = minus_high(w2, v[e + 1]); }
    return w2;
}
// (A part, B part) of the six products of a k16 step, in their order
__device__ constexpr int CONV_SPLIT_PA[6] = {2, 1, 1, 0, 0, 0}, CONV_SPLIT_PB[6] = {0, 0, 1, 1, 2, 0};
// Where sums of few terms have to be as close to 64 bits as fp32 products give them: the seven products beside the largest, the smallest first. The largest,
// of the two parts of 8 bits that come first, is summed for itself: such products are 16 bits long, so few bits are cut off where they are added,
// and the others are a 256th of them. (Without the first two a sum of one term is 1.03 times as far off as its fp32 product.)
__device__ constexpr int CONV_FINE_PA[7] = {2, 1, 2, 1, 1, 0, 0}, CONV_FINE_PB[7] = {1, 2, 0, 0, 1, 1, 2};

// ---- the product ------------------------------------------------------------------------------------------------------
// Block = WGM x WGN waves, each with TM x TN tiles of 32 x 32; k tile 32, i.e. two k16 steps, taken in pairs. A tile of the
// rows' operand is loaded as fp32 (two items per thread, each a row's octet in two 16-byte vectors), taken apart in registers and
// put into one of two LDS buffers, [part][octet][row] x 8 bf16 (rows permuted by the octet: neither the writes nor the reads
// of eight lanes in a row meet in a bank); the packed kernel operand goes straight into registers. Between the MFMAs of a k16
// step: the next step's A parts are read from LDS as soon as this step has used a part for its last column, one item of the
// next k tile (the next but one behind the barrier) is taken apart, written to LDS and requested for the k tile after it, and
// the columns' parts are requested for the next k tile. Everything a wave waits for has been requested some 40 MFMAs of
// 32 cycles before. One barrier per k tile, in its second step. The order of instructions is written down (FENCE): left
// alone, the compiler gathers loads and splitting in front of or behind the MFMAs (a 128 x 128 x 4608 tile alone on a CU:
// 273 us with one stage after the other, 193 without a branch in the loop, 147 with the order written down).
//
// What bounds it: power. On 8192 x 2048 x 8192 the matrix cores are busy 73 to 79 % of the time at 1.64 to 1.71 GHz, 200 to 221
// TFLOP/s of fp32 products (133 through v_mfma_f32_32x32x2_f32, which cannot exceed 157); a loop of these MFMAs and nothing
// else runs at 1.8 to 1.9 GHz. So what moves less data is faster: 128 x 64 tiles reach 0.88 of the 128 x 128 tiles' rate. The
// layers of a network are shorter: start, stores and the last round of blocks count (12544 x 2304 x 256: 147 to 163 TFLOP/s, by the card).
//
// Sharing out: the first P.split_tiles_m tiles of the grid are computed by one block each, the contraction of every tile behind
// them by P.m_blocks blocks (slices of P.m_each or one more pairs of k tiles). A slice's sums go to `partial`, and whichever block arrives
// last at the tile's counter adds all slices in their order and applies the epilogue: no block waits for another. The
// counters are left at zero for the next launch.

// ---- the sums of a tile, from a patch of the input in LDS ----------------------------------------------------------------
// 3 x 3 windows at a stride of 1 over an input with a border of one: the rows of a tile are consecutive positions m of the images laid end to
// end, and under tap (r, s) position m sees position m + (r - 1) W + s - 1. So the 128 + 2 W + 2 positions m0 - W - 1 .. of 16 input features
// are loaded, taken apart and put into LDS once and serve nine k16 steps, where the kernel above loads and takes apart 128 positions in each
// of them. A tap that lies outside the image for some rows (their neighbour belongs to another row or image there) has those lanes read zeros
// that stand behind the patch.
//   LDS: [2 buffers][3 parts][2 octets][264 positions] x 8 bf16; octet o: features 4o .. 4o+3 and 8+4o .. of the 16; positions 256 .. 258 are zeros;
//     264: neither the writes nor the reads of lanes that go together meet in a bank.
// While one buffer serves its nine steps, the next 16 features' two items per thread are taken apart into the other one, in the first
// eight steps, and requested again for the 16 features behind them. One barrier per nine steps, in the last. The products of three steps, not
// four, are summed from zero before they are added to the accumulators: errors against 64-bit sums of 1.06e-7 and 1.28e-7 of the 2-norm for 64 and 512
// features where every tap is loaded anew 1.24e-7 and 1.37e-7.
// What bounds it: power, as below; what it saves is vector instructions, LDS writes and loads, which take their share of it. Products alone, before and after:
// 64 x 56 x 56 x 64 x 64 91.5 -> 78.0 us, 28 x 28 x 128 x 128 88.1 -> 74.2, 14 x 14 x 256 x 256 87.5 -> 73.5, 7 x 7 x 512 x 512 88.3 -> 79.0 (187 to 201 TFLOP/s);
// 32 x 56 x 56 x 64 x 64 52.5 -> 44.9, 50 x 24 x 24 x 128 x 64 38.3 -> 25.6. ResNet-50 at batch 64 3.94 -> 3.83 ms, its training step 13.10 -> 12.82.
// (The body of the loop has no branch: skipping the second item where a patch is short cost more in spilled registers than it saved.)
// FINE: the eight products and two sums of CONV_FINE_PA, each sum with accumulators of its own, which meet behind the last slice. For products that the
// fp32 kernels would compute: errors of 0.3 to 0.96 times theirs however few terms are not zero, 1.00 for sums of one term (with six products in one sum 1.2 to
// 1.3 times where less than a tenth of the terms are not zero). A third more products and twice the accumulators, two blocks per CU: 64 x 56 x 56 x 64 x 32 68
// -> 86 us (fp32 114), 33 x 7 x 7 x 512 x 512 55 -> 67 (101), 1 x 7 x 7 x 480 x 480 27 -> 32 (93).
constexpr int CONV_PATCH_ROWS = 264, CONV_PATCH_ZEROS = 256;

template <int WGM, int WGN, int TM, int TN, bool FINE, bool RAGGED>
__device__ __forceinline__ void conv_patch_sums(u32x4* __restrict__ As, float* __restrict__ Es, float (&acc)[TM][TN][16],
                                                float (&acc_large)[FINE ? TM : 1][FINE ? TN : 1][16], const uint32_t (&b_soff)[TN],
                                                const float* __restrict__ x, __amdgpu_buffer_rsrc_t w_rsrc, const ConvEpiPtrs& epi, const ConvDerivedPtrs& Dp,
                                                const ConvParams& P, const ConvDerived& Dk, int wave, int m0, int n0, int kbeg, int kend) {
    constexpr int BN = 32 * WGN * TN, NT = 64 * WGM * WGN, ROWS = CONV_PATCH_ROWS;
    static_assert(WGM * TM == 4 && NT == 256, "tiles of 128 rows, two items per thread");
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5, wm = wave / WGN;
    const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(x, P.x_bytes);
    // ---- items: (position of the patch, octet)
    const int p_octet = tid & 1, p_row = tid >> 1;                      // item p: position p_row + 128 p
    uint32_t p_voff[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int at = m0 - P.W - 1 + p_row + 128 * p;
        p_voff[p] = at >= 0 && at < P.M && p_row + 128 * p < 130 + 2 * P.W ? (uint32_t)(at * P.xs_w + 4 * p_octet) * 4u : CONV_OOB;
    }
    const int p_slot = p_octet * ROWS + p_row;
    constexpr int RAWS = TN == 1 ? 2 : 1;                               // items in registers: there is no room for two beside 128 columns
    f32x4 raw[RAWS][2];
    // RAGGED: the vectors of the last eight features that are not all there; those of one octet behind the last feature are not, and those that reach beyond it begin earlier
    const int last_eight = RAGGED ? (P.Cin - 1) >> 3 : 0, into = RAGGED ? P.Cin - 8 * last_eight - 4 * p_octet : 4;
    const uint32_t p_last = into <= 0 ? CONV_OOB : (uint32_t)(8 * last_eight + min(into - 4, 0)) * 4u;      // (all in the lane's offset, which must not be negative)
    auto load_eight = [&](int eight, int p) {
        if constexpr (!RAGGED) return buffer_load_x4(x_rsrc, p_voff[p], (uint32_t)eight * 32u);
        const uint32_t v = p_voff[p] + (eight == last_eight ? p_last : 0u);
        return buffer_load_x4(x_rsrc, p_voff[p] == CONV_OOB ? CONV_OOB : v, eight > last_eight ? CONV_OOB : eight == last_eight ? 0u : (uint32_t)eight * 32u);
    };
    auto load_item = [&](f32x4 (&to)[2], int sixteen, int p) {
        to[0] = load_eight(2 * sixteen, p);
        to[1] = load_eight(2 * sixteen + 1, p);
    };
    u32x4 part;
    auto park = [&](u32x4* to, int p, int t) { to[t * 2 * ROWS + p_slot + 128 * p] = part; };
    // ---- the rows of this wave's tiles, and which of their neighbours lie outside the image
    const int a_zero = (half * ROWS + CONV_PATCH_ZEROS) * 16, row_bytes = P.W * 16;
    int a_slot[TM];
    uint64_t above[TM], below[TM], before[TM], behind[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int row = (wm * TM + i) * 32 + l32, m = m0 + row;
        const int b = magic_div(m, P.howo_magic, P.howo_shift), r2 = m - b * P.Ho * P.Wo;
        const int ho = magic_div(r2, P.wo_magic, P.wo_shift), wo = r2 - ho * P.Wo;
        a_slot[i] = (half * ROWS + row) * 16;
        above[i]  = __builtin_amdgcn_ballot_w64(ho == 0);
        below[i]  = __builtin_amdgcn_ballot_w64(ho == P.H - 1);
        before[i] = __builtin_amdgcn_ballot_w64(wo == 0);
        behind[i] = __builtin_amdgcn_ballot_w64(wo == P.W - 1);
    }
    u32x4 bf[2][TN][3], af[TM][3];
    // where tile i's rows lie under tap (r, s), and their part t from there (s is in the read's own offset)
    int a_at[TM];
    auto find_a = [&](int r, int s, int i) {
        const uint64_t outside = (r == 0 ? above[i] : r == 2 ? below[i] : 0u) | (s == 0 ? before[i] : s == 2 ? behind[i] : 0u);
        a_at[i] = a_slot[i] + r * row_bytes;
        if (r != 1 || s != 1) asm volatile("v_cndmask_b32_e64 %0, %0, %1, %2" : "+v"(a_at[i]) : "v"(a_zero), "s"(outside));
    };
    auto read_a = [&](const u32x4* from, int s, int t, int i) {
        af[i][t] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(from + t * 2 * ROWS + s) + a_at[i]);
    };
    const uint32_t b_lane = (uint32_t)lane * 16u;
    auto load_b = [&](int step, int parity, int t, int j) {
        bf[parity][j][t] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, b_lane, b_soff[j] + (uint32_t)step * 3072u + t * 1024u, 0);
    };
    f32x16 sum[TM * TN] = {}, large[FINE ? TM * TN : 1] = {};
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                acc[i][j][v] = 0.f;
                if constexpr (FINE) acc_large[i][j][v] = 0.f;
            }
    // products of a step, and behind which of them the parts 2, 1 and 0 of A have met their last
    constexpr int NP = FINE ? 8 : 6, LAST[3] = {NP - 1, FINE ? 5 : 4, FINE ? 3 : 2};
    constexpr int CH = TM * TN, NS = NP * CH, BARRIER = NP * (TN - 1) + LAST[2];
    constexpr auto pa = [](int t) { return FINE ? t < 7 ? CONV_FINE_PA[t] : 0 : CONV_SPLIT_PA[t]; };
    constexpr auto pb = [](int t) { return FINE ? t < 7 ? CONV_FINE_PB[t] : 0 : CONV_SPLIT_PB[t]; };
    // which of the two items' twelve pieces follows a product of the nine steps, -1: none. One item in registers: the second is requested when
    // the first has been taken apart, and has a step and a half to arrive.
    constexpr auto item_piece = [](int place) {
        for (int e = 0; e < 12; ++e) {
            const int at = RAWS == 2 ? (e + 1) * 8 * NS / 12 - 1 : (e < 6 ? 3 * NS / 2 : 11 * NS / 2) + (e % 6 + 1) * 5 * NS / 12 - 1;
            if (place == at) return e;
        }
        return -1;
    };
    float sign = 1.f / (CONV_SPLIT_SCALE * CONV_SPLIT_SCALE);            // (six groups of three steps per turn of the loop)
    auto nine_steps = [&](auto buffer_, int sixteen) {
        constexpr int buffer = decltype(buffer_)::value;
        u32x4 *const mine = As + buffer * 6 * ROWS, *const other = As + (buffer ^ 1) * 6 * ROWS;
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            const int parity = (tap + buffer) & 1, next = tap == 8 ? 0 : tap + 1;
            FENCE();
#pragma unroll
            for (int n = 0; n < NS; ++n) {
                const int c = n / NP, t = n % NP, i = c / TN, j = c % TN;
                if (tap == 8 && n == BARRIER) { __syncthreads(); FENCE(); }
                f32x16& to = FINE && t == NP - 1 ? large[FINE ? c : 0] : sum[c];
                to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, af[i][pa(t)]), __builtin_bit_cast(bf16x8, bf[parity][j][pb(t)]),
                                                             tap % 3 == 0 && (t == 0 || (FINE && t == NP - 1)) ? f32x16{} : to, 0, 0, 0);
                // the chain before has seen its last product
                if (tap % 3 == (c > 0 ? 2 : 0) && t >= NP - 4) {
                    const int pc = (c + CH - 1) % CH, v0 = 4 * (t - NP + 4);
#pragma unroll
                    for (int v = v0; v < v0 + 4; ++v) {
                        acc[pc / TN][pc % TN][v] = __builtin_fmaf(sum[pc][v], sign, acc[pc / TN][pc % TN][v]);
                        if constexpr (FINE) acc_large[pc / TN][pc % TN][v] = __builtin_fmaf(large[pc][v], sign, acc_large[pc / TN][pc % TN][v]);
                    }
                }
                // parts of A that have met their last column are replaced by the next step's
                if (j == TN - 1 && t == LAST[2]) find_a(next / 3, next % 3, i);
#pragma unroll
                for (int q = 2; q >= 0; --q)
                    if (j == TN - 1 && t == LAST[q]) read_a(tap == 8 ? other : mine, next % 3, q, i);
                // an item of the next 16 features: its three parts, in halves, then the request of a later one
                const int place = tap * NS + n, e = item_piece(place), h = e % 6, item = e / 6;
                if (e >= 0) {
                    f32x4 (&numbers)[2] = raw[item % RAWS];
                    part[2 * (h & 1)] = conv_split_word(numbers, h / 2, 2 * (h & 1));
                    part[2 * (h & 1) + 1] = conv_split_word(numbers, h / 2, 2 * (h & 1) + 1);
                    if (h & 1) park(other, item, h / 2);
                    if (h == 5) load_item(numbers, sixteen + (RAWS == 2 || item == 1 ? 2 : 1), RAWS == 2 ? item : item ^ 1);
                }
                // the columns' parts of the next step but one
#pragma unroll
                for (int q = 0; q < TN; ++q)
                    if (q < TN - 1 ? n == (CH - TN + q + 1) * NP + 1 : n == NS - 1) {
#pragma unroll
                        for (int t2 = 0; t2 < 3; ++t2) load_b(9 * sixteen + tap + 2, parity, t2, q);
                    }
                FENCE();
            }
            if (tap % 3 == 0 && (tap > 0 || sixteen > kbeg)) sign = -sign;
        }
    };

    f32x4 first[2][2];
    load_item(first[0], kbeg, 0);
    load_item(first[1], kbeg, 1);
    FENCE();
#pragma unroll
    for (int p = 0; p < RAWS; ++p) load_item(raw[p], kbeg + 1, p);
    FENCE();
#pragma unroll
    for (int parity = 0; parity < 2; ++parity)
#pragma unroll
        for (int q = 0; q < TN; ++q)
#pragma unroll
            for (int t = 0; t < 3; ++t) { load_b(9 * kbeg + parity, parity, t, q); FENCE(); }
    conv_split_epilogue_operands<BN>(Es, epi, Dp, P, Dk, tid, n0);
    if (tid < 36) As[(tid / 3) * ROWS + CONV_PATCH_ZEROS + tid % 3] = u32x4{0u, 0u, 0u, 0u};      // (no item lies there)
#pragma unroll
    for (int f = 0; f < 2; ++f) {
#pragma unroll
        for (int t = 0; t < 3; ++t) {
#pragma unroll
            for (int q = 0; q < 4; ++q) part[q] = conv_split_word(first[f], t, q);
            park(As, f, t);
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        find_a(0, 0, i);
#pragma unroll
        for (int t = 0; t < 3; ++t) read_a(As, 0, t, i);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);                                  // (as in the kernel below)
    for (int sixteen = kbeg; sixteen < kend; sixteen += 2) {             // (no branch inside: registers would spill)
        nine_steps(std::integral_constant<int, 0>{}, sixteen);
        nine_steps(std::integral_constant<int, 1>{}, sixteen + 1);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        acc[TM - 1][TN - 1][v] = __builtin_fmaf(sum[CH - 1][v], sign, acc[TM - 1][TN - 1][v]);
        if constexpr (FINE) acc_large[TM - 1][TN - 1][v] = __builtin_fmaf(large[CH - 1][v], sign, acc_large[TM - 1][TN - 1][v]);
    }
    __syncthreads();
}

// STEPS: an epilogue other than the straight-line one, step by step (ReLU6, a scalar or a vector in another place, a residual that is subtracted).
// FINE: products and sums of CONV_FINE_PA; a slice leaves both its sums.
// RAGGED (with a patch): any number of features from four on. The kernel operand is laid out for a multiple of 32 of them, with zeros behind the last. A
// vector of the input that would reach beyond a position's last feature ends there instead and begins with features of the vector in front, which meet zeros:
// nothing of another position is read, so sums are what they are whatever their neighbours hold.
template <int WGM, int WGN, int TM, int TN, bool STEPS, bool PATCH, bool FINE, bool RAGGED = false>
__device__ __forceinline__ void conv_split_body(u32x4* __restrict__ pool, float* __restrict__ Es, int* __restrict__ Rs,
                                                float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w,
                                                float* __restrict__ partial, uint32_t* __restrict__ arrivals, const ConvEpiPtrs& epi, const ConvDerivedPtrs& Dp,
                                                const ConvParams& P, const ConvDerived& Dk) {
    constexpr int BM = 32 * WGM * TM, BN = 32 * WGN * TN, NT = 64 * WGM * WGN, BK = 32;
    u32x4* const As = pool;                         // [2 buffers][3 parts][4 octets][BM rows]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave / WGN, wn = wave % WGN;
    const bool c_contig = P.flags & 1u, flat_rows = P.flags & 2u, masked = P.flags & 4u;
    const int nepi = (P.flags >> 8) & 15u, epi_first_full = (int)((P.flags >> 16) & 15u) - 1;
    auto step_desc = [&](int e) -> uint32_t { return conv_split_step_desc(P, e); };

    // k16 steps; what a slice is made of: k tiles, in pairs, or (PATCH) groups of nine steps, in pairs too
    const int ktiles = (P.K + 2 * BK - 1) / (2 * BK) * 2, ksteps = PATCH ? P.K / 16 : 2 * ktiles, slices = P.m_blocks, whole = P.split_tiles_m;
    int work = (int)blockIdx.x, tile, slice = 0, kbeg = 0, kend = PATCH ? ksteps / 9 : ktiles;
    if (work < whole) {
        tile = xcd_range(work, whole);
    } else {
        const int rest = P.tiles_m * P.tiles_n - whole;
        work  = xcd_range(work - whole, rest * slices);
        slice = work / rest;
        tile  = whole + work - slice * rest;
        kbeg  = 2 * (slice * P.m_each + min(slice, P.m_extra));
        kend  = kbeg + 2 * (P.m_each + (slice < P.m_extra ? 1 : 0));
    }
    const bool sliced = (int)blockIdx.x >= whole;
    const int tile_m = tile / P.tiles_n, tile_n = tile - tile_m * P.tiles_n;
    const int m0 = tile_m * BM, n0 = tile_n * BN, HoWo = P.Ho * P.Wo;

    const uint32_t x_bias = (uint32_t)(P.PH * P.xs_h + P.PW * P.xs_w) * 4u;
    const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(reinterpret_cast<const char*>(x) - x_bias, P.x_bytes + x_bias),
                                 w_rsrc = make_rsrc(w, P.w_bytes), o_rsrc = make_rsrc(out, P.out_bytes);

    const uint32_t rowb = (uint32_t)P.N * 4u;
    float acc[TM][TN][16], acc_large[FINE ? TM : 1][FINE ? TN : 1][16];
    uint32_t b_soff[TN];                             // the packed columns of this wave
    // (blocks of columns beyond the last one lie outside the descriptor and read as zeros)
#pragma unroll
    for (int j = 0; j < TN; ++j) b_soff[j] = (uint32_t)(n0 / 32 + wn * TN + j) * (uint32_t)ksteps * 3072u;
    if constexpr (PATCH) {
        conv_patch_sums<WGM, WGN, TM, TN, FINE, RAGGED>(pool, Es, acc, acc_large, b_soff, x, w_rsrc, epi, Dp, P, Dk, wave, m0, n0, kbeg, kend);
    } else {
    static_assert(!FINE, "only with a patch");
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
    // ---- load assignment: A item = (row, octet of k); octet o holds k = 4o..4o+3 and 16+4o..16+4o+3 of the k tile
    constexpr int A_NI = BM * 4 / NT, A_RSTEP = NT / 4;
    const int a_o = tid & 3, a_r0 = tid >> 2;
    uint32_t a_voff[A_NI], a_inv[A_NI];
#pragma unroll
    for (int p = 0; p < A_NI; ++p) {
        const int m = m0 + a_r0 + p * A_RSTEP;
        a_inv[p] = 0u;
        if (flat_rows) {
            a_voff[p] = m < P.M ? (uint32_t)(m * P.xs_h + a_o * 4) * 4u : CONV_OOB;
            continue;
        }
        const int b = magic_div(m, P.howo_magic, P.howo_shift);
        const int r2 = m - b * HoWo;
        const int ho = magic_div(r2, P.wo_magic, P.wo_shift);
        const int wo = r2 - ho * P.Wo;
        a_voff[p] = m < P.M ? (uint32_t)(b * P.xs_b + ho * P.SH * P.xs_h + wo * P.SW * P.xs_w + a_o * 4) * 4u : CONV_OOB;
        if (masked) {
            const int hi0 = ho * P.SH - P.PH, wi0 = wo * P.SW - P.PW;
            uint32_t wbad = 0u;
            for (int s = 0; s < P.KW; ++s) wbad |= ((uint32_t)(wi0 + s * P.DW) >= (uint32_t)P.W ? 1u : 0u) << s;
            const uint32_t wall = (2u << (P.KW - 1)) - 1u;
            for (int r = 0; r < P.KH; ++r)
                a_inv[p] |= ((uint32_t)(hi0 + r * P.DH) >= (uint32_t)P.H ? wall : wbad) << (r * P.KW);
        }
    }
    const uint32_t b_lane = (uint32_t)lane * 16u;
    int t_r = 0, t_s = 0, t_c = kbeg * BK;          // kernel tap and first feature of the next k tile to load
    if (kbeg > 0 && P.KH * P.KW > 1) {
        const int rs = t_c / P.Cin;
        t_c -= rs * P.Cin; t_r = rs / P.KW; t_s = rs - t_r * P.KW;
    }
    static_assert(A_NI == 2 && TM == 2, "two items per thread, two rows of tiles per wave: the schedule below");
    f32x4 raw[2][2];
    // requests item p of k tile kt (beyond the contraction: zeros)
    auto load_item = [&](f32x4 (&to)[2], int kt, int p) {
        const uint32_t soff = (uint32_t)(t_r * P.DH * P.xs_h + t_s * P.DW * P.xs_w + t_c) * 4u, sh = 31u - (uint32_t)(t_r * P.KW + t_s);
        const uint32_t bad0 = kt * BK + a_o * 4 >= P.K ? CONV_OOB : 0u, bad1 = kt * BK + 16 + a_o * 4 >= P.K ? CONV_OOB : 0u;
        const uint32_t v = a_voff[p] | ((a_inv[p] << sh) & CONV_OOB);
        to[0] = buffer_load_x4(x_rsrc, v | bad0, soff);
        to[1] = buffer_load_x4(x_rsrc, v | bad1, soff + 64u);
    };
    auto advance = [&]() {
        t_c += BK;
        const bool wrap_c = t_c >= P.Cin; t_c = wrap_c ? 0 : t_c; t_s += wrap_c ? 1 : 0;
        const bool wrap_s = t_s == P.KW; t_s = wrap_s ? 0 : t_s; t_r += wrap_s ? 1 : 0;
    };
    f32x16 sum[TM * TN] = {};                        // the products of a pair of k tiles
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    u32x4 bf[2][TN][3], af[TM][3];
    auto load_b = [&](int kt, int ks, int t, int j) {
        bf[ks][j][t] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, b_lane, b_soff[j] + (uint32_t)(2 * kt + ks) * 3072u + t * 1024u, 0);
    };
    int a_slot[TM];                                  // k16 step 0; the other one: two octets on
#pragma unroll
    for (int i = 0; i < TM; ++i) a_slot[i] = half * BM + (((wm * TM + i) * 32 + l32) ^ (half * 2));
    auto read_a = [&](const u32x4* from, int ks, int t, int i) { af[i][t] = from[(t * 4 + 2 * ks) * BM + (a_slot[i] ^ (ks * 4))]; };
    const int p_slot = a_o * BM + (a_r0 ^ (a_o * 2));
    u32x4 part;
    auto park = [&](u32x4* to, int p, int t) { to[t * 4 * BM + (p_slot ^ (p * A_RSTEP))] = part; };

    // The matrix cores cut off what lies below the last bit of a sum, towards minus infinity. So the products of a pair of k
    // tiles are summed from zero (TM x TN chains of four times six products each) and added to the accumulators by fp32
    // operations, rounded to nearest, while the next chain runs; and the packed operand has its sign changed in every
    // other pair, whose sums are subtracted, so that what is cut off goes up as often as down. (All products into one
    // accumulator: an error 1.7 to 2.7 times that of fp32 products at K = 576, of mean -3e-8 of the results' rms; chains of
    // one sign: that mean, the same in every layer, left ResNet-50's logits 1.3e-6 from 64-bit ones where fp32 products are
    // 4.1e-7 off and these 3.5e-7.)
    // The small products of a k step come first, (A part, B part): a sum that begins there is cut off once at its full size and not four
    // times. (Of 512 terms 512, 16 and 1 that are not zero: errors of 1.22e-7, 7.6e-8 and 3.5e-8 of the results' 2-norm, with the largest
    // product first 1.36e-7, 8.9e-8 and 5.3e-8, through fp32 products 2.1e-7, 5.9e-8 and 2.5e-8; no slower.)
    constexpr int CH = TM * TN, NS = 6 * CH;
    float sign = kbeg & 2 ? -1.f / (CONV_SPLIT_SCALE * CONV_SPLIT_SCALE) : 1.f / (CONV_SPLIT_SCALE * CONV_SPLIT_SCALE);
    auto k16_step = [&](auto step_, int kt) {
        constexpr int step = decltype(step_)::value, ks = step & 1, item = 1 - ks;   // step of the pair of k tiles, the second of its k tile
        u32x4 *const mine = As + (step >> 1) * 12 * BM, *const other = As + ((step >> 1) ^ 1) * 12 * BM;
        constexpr int BARRIER = 6 * TN - 4;                                     // second step only: in front of the first part of the next tile
        constexpr int SPLIT = ks == 0 ? 0 : BARRIER, EACH = (NS - SPLIT) / 6;   // an item's three parts, in halves, then its reload
        u32x4* const to = ks == 0 ? other : mine;                               // k tile kt + 1, or kt + 2
        FENCE();
#pragma unroll
        for (int n = 0; n < NS; ++n) {
            const int c = n / 6, t = n % 6, i = c / TN, j = c % TN;
            if (ks == 1 && n == BARRIER) { __syncthreads(); FENCE(); }
            sum[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, af[i][CONV_SPLIT_PA[t]]), __builtin_bit_cast(bf16x8, bf[ks][j][CONV_SPLIT_PB[t]]),
                                                             step == 0 && t == 0 ? f32x16{} : sum[c], 0, 0, 0);
            // the chain before has seen its last product
            if (step == (c > 0 ? 3 : 0) && t >= 2) {
                const int pc = (c + CH - 1) % CH;
#pragma unroll
                for (int v = 4 * t - 8; v < 4 * t - 4; ++v) acc[pc / TN][pc % TN][v] = __builtin_fmaf(sum[pc][v], sign, acc[pc / TN][pc % TN][v]);
            }
            // parts of A that have met their last column are replaced by the next step's
            if (j == TN - 1 && (t == 2 || t == 4 || t == 5)) read_a(ks == 1 ? other : mine, 1 - ks, t == 2 ? 2 : t == 4 ? 1 : 0, i);
            // an item of a later k tile
            if (n >= SPLIT && (n - SPLIT) % EACH == EACH - 1 && (n - SPLIT) / EACH < 6) {
                const int h = (n - SPLIT) / EACH, pt = h / 2;
                part[2 * (h & 1)] = conv_split_word(raw[item], pt, 2 * (h & 1));
                part[2 * (h & 1) + 1] = conv_split_word(raw[item], pt, 2 * (h & 1) + 1);
                if (h & 1) park(to, item, pt);
                if (h == 5) load_item(raw[item], kt + (ks == 0 ? 2 : 3), item);
            }
            // the columns' parts of the next k tile
#pragma unroll
            for (int q = 0; q < TN; ++q)
                if (q < TN - 1 ? n == (CH - TN + q + 1) * 6 + 1 : n == NS - 1) { load_b(kt + 1, ks, 0, q); load_b(kt + 1, ks, 1, q); load_b(kt + 1, ks, 2, q); }
            FENCE();
        }
        if constexpr (ks == 0) advance();
        if constexpr (step == 0) { if (kt > kbeg) sign = -sign; }
    };

    // The loads of the first k tiles, the last of them in the order in which the loop below issues those of later ones.
    f32x4 first[3][2];
    load_item(first[0], kbeg, 0);
    load_item(first[1], kbeg, 1);
    advance();
    load_item(first[2], kbeg + 1, 0);
    FENCE();
    load_item(raw[1], kbeg + 1, 1);
    advance();
    FENCE();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int q = 0; q < TN; ++q) {
            if (ks == 1 && q == TN - 1) { load_item(raw[0], kbeg + 2, 0); FENCE(); }
#pragma unroll
            for (int t = 0; t < 3; ++t) { load_b(kbeg, ks, t, q); FENCE(); }
        }
    conv_split_epilogue_operands<BN>(Es, epi, Dp, P, Dk, tid, n0);

    {
#pragma unroll
        for (int f = 0; f < 3; ++f) {
#pragma unroll
            for (int t = 0; t < 3; ++t) {
#pragma unroll
                for (int q = 0; q < 4; ++q) part[q] = conv_split_word(first[f], t, q);
                park(As + f / 2 * 12 * BM, f & 1, t);
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int t = 0; t < 3; ++t) read_a(As, 0, t, i);
        // Everything requested so far has arrived when the loop begins: the compiler then counts in the loop which of its own loads it waits
        // for. (Left alone it may wait for all of them once per pair of k tiles, where the paths into the loop differ in their order: 12544 x
        // 2304 x 256, one block per CU, 95.5 us instead of 92.)
        __builtin_amdgcn_s_waitcnt(0x0F70);
        for (int kt = kbeg; kt < kend; kt += 2) {
            k16_step(std::integral_constant<int, 0>{}, kt);
            k16_step(std::integral_constant<int, 1>{}, kt);
            k16_step(std::integral_constant<int, 2>{}, kt + 1);
            k16_step(std::integral_constant<int, 3>{}, kt + 1);
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[TM - 1][TN - 1][v] = __builtin_fmaf(sum[CH - 1][v], sign, acc[TM - 1][TN - 1][v]);
        __syncthreads();
    }
    }

    // (behind the loop the lane's number is asked for again: kept over the loop, it and what depends on it would cost registers there)
    const int tid = tid_again(wave), lane = tid & 63, l32 = lane & 31, half = lane >> 5;
    const uint32_t b_lane = (uint32_t)lane * 16u;
    if (sliced) {
        // store this slice's sums; the block that arrives last adds all of them, in the order of the slices
        const int mine = tile - whole;
        constexpr int SUMS = FINE ? 2 : 1;
        const uint32_t tile_bytes = BM * BN * 4 * SUMS;
        const __amdgpu_buffer_rsrc_t p_rsrc = make_rsrc(reinterpret_cast<char*>(partial) + (size_t)mine * slices * tile_bytes, (uint32_t)slices * tile_bytes);
        auto each = [&](auto&& fn) {                              // fn(four of this lane's sums, their place in a slice)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; v += 4) {
                        fn(&acc[i][j][v], (uint32_t)((i * TN + j) * 4 + v / 4) * (NT * 16u));
                        if constexpr (FINE) fn(&acc_large[i][j][v], (uint32_t)((TM * TN + i * TN + j) * 4 + v / 4) * (NT * 16u));
                    }
        };
        each([&](float* four, uint32_t place) {
            buffer_store_x4_agent(f32x4{four[0], four[1], four[2], four[3]}, p_rsrc, (uint32_t)tid * 16u, (uint32_t)slice * tile_bytes + place);
        });
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the stores above have reached memory
        __syncthreads();
        if (tid == 0) {
            const uint32_t n = __hip_atomic_fetch_add(arrivals + mine, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (n + 1u == (uint32_t)slices) __hip_atomic_store(arrivals + mine, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            Rs[0] = (int)n;
        }
        __syncthreads();
        if (Rs[0] + 1 != slices) return;
        each([&](float* four, uint32_t) {
#pragma unroll
            for (int u = 0; u < 4; ++u) four[u] = 0.f;
        });
#pragma nounroll
        for (int s = 0; s < slices; ++s)
            each([&](float* four, uint32_t place) {
                const f32x4 q = buffer_load_x4_agent(p_rsrc, (uint32_t)tid * 16u, (uint32_t)s * tile_bytes + place);
#pragma unroll
                for (int u = 0; u < 4; ++u) four[u] += q[u];
            });
    }
    if constexpr (FINE) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] += acc_large[i][j][v];
    }

    // Sums that are not finite are computed again with fp32 products. The others beside them stay as they are, so a row's results do not
    // depend on what the rows in its tile hold.
    float high = 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; v += 2) high = higher_of(high, acc[i][j][v], acc[i][j][v + 1]);
    if (__builtin_amdgcn_ballot_w64(!(high < __builtin_inff()))) {
        // In the order of the packed operand: lane l of a k16 step takes row l % 32, column l % 32 and the octet of its half of the wave,
        // so both operands come in 16-byte loads, the next step's while this one's 8 TN products run. 12544 x 2304 x 256 with NaN only: 454 us
        // (102 without; 1560 with single words requested one after the other), 3x3x128x128 on 50176 rows 356 (91; 1350), through the fp32
        // kernels 131 and 132.
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            bool any = false;
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) any |= !__builtin_isfinite(acc[i][j][v]);
            if (!__builtin_amdgcn_ballot_w64(any)) continue;
            const int m = m0 + (wm * TM + i) * 32 + l32;
            const int b = flat_rows ? 0 : magic_div(m, P.howo_magic, P.howo_shift), r2 = m - b * HoWo;
            const int ho = flat_rows ? 0 : magic_div(r2, P.wo_magic, P.wo_shift), wo = r2 - ho * P.Wo;
            const int hi0 = ho * P.SH - P.PH, wi0 = wo * P.SW - P.PW;
            const uint32_t row = (uint32_t)(flat_rows ? m * P.xs_h : b * P.xs_b + ho * P.SH * P.xs_h + wo * P.SW * P.xs_w) * 4u;
            int r = 0, s = 0, c = 0;
            f32x4 a_next[2];
            int c_next = 0;                                      // (RAGGED) the first feature of the vectors in a_next
            u32x4 b_next[TN][3];
            auto request = [&](int step) {
                const int hi = hi0 + r * P.DH, wi = wi0 + s * P.DW, o = PATCH ? half : 2 * (step & 1) + half, k = PATCH ? 16 * step : (step >> 1) * BK + 4 * o;
                c_next = RAGGED ? c + 4 * half : 0;
                const bool ok = m < P.M && (flat_rows || ((uint32_t)hi < (uint32_t)P.H && (uint32_t)wi < (uint32_t)P.W));
                const uint32_t at = row + (uint32_t)(r * P.DH * P.xs_h + s * P.DW * P.xs_w + c + 4 * o) * 4u;
                const int over0 = RAGGED ? max(0, c_next + 4 - P.Cin) : 0, over1 = RAGGED ? max(0, c_next + 12 - P.Cin) : 0;      // (4 or more: nothing is left)
                a_next[0] = buffer_load_x4(x_rsrc, ok && k < P.K && over0 < 4 ? at - (uint32_t)over0 * 4u : CONV_OOB);
                a_next[1] = buffer_load_x4(x_rsrc, ok && k + (PATCH ? 8 : 16) < P.K && over1 < 4 ? at + (PATCH ? 32u : 64u) - (uint32_t)over1 * 4u : CONV_OOB);
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        b_next[j][q] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, b_lane, b_soff[j] + (uint32_t)step * 3072u + (uint32_t)q * 1024u, 0);
                if constexpr (PATCH) {
                    if (++s == 3) { s = 0; if (++r == 3) { r = 0; c += 16; } }
                } else if (step & 1) {
                    c += BK;
                    if (c >= P.Cin) { c = 0; if (++s == P.KW) { s = 0; ++r; } }
                }
            };
            f32x16 again[TN] = {}, total[TN] = {};          // (summed by as many k, as rounded as in the loop above)
            request(0);
#pragma nounroll
            for (int step = 0; step < ksteps; ++step) {
                float av[8], bv[TN][8];
                const float sign_k = (PATCH ? step / 3 & 1 : step & 4) ? -1.f : 1.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    av[e] = !RAGGED || (e & 3) >= c_next + 8 * (e >> 2) + 4 - P.Cin ? a_next[e >> 2][e & 3] : 0.f;      // (not the features that were there before)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        uint32_t part_e[3];
#pragma unroll
                        for (int q = 0; q < 3; ++q) part_e[q] = e & 1 ? b_next[j][q][e >> 1] & 0xFFFF0000u : b_next[j][q][e >> 1] << 16;
                        const float value = ((u2f(part_e[2]) + u2f(part_e[1])) + u2f(part_e[0])) * (1.f / CONV_SPLIT_SCALE);
                        bv[j][e] = (part_e[0] == CONV_PACK_RAW << 16 ? u2f(part_e[1] | part_e[2] >> 16) : value) * sign_k;
                    }
                }
                request(step + 1);                          // (behind the last step: zeros, or the next columns' first, unused)
#pragma unroll
                for (int e = 0; e < 8; ++e)
#pragma unroll
                    for (int j = 0; j < TN; ++j) again[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[e], bv[j][e], again[j], 0, 0, 0);
                if (PATCH ? step % 3 == 2 : (step & 3) == 3) {
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int v = 0; v < 16; ++v) { total[j][v] += again[j][v]; again[j][v] = 0.f; }
                }
            }
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = __builtin_isfinite(acc[i][j][v]) ? acc[i][j][v] : total[j][v];
        }
    }

    if (!c_contig) {
        __syncthreads();
        for (int r = tid; r < BM; r += NT) {
            const int m = m0 + r;
            const int b = m / HoWo, r2 = m - b * HoWo, ho = r2 / P.Wo, wo = r2 - ho * P.Wo;
            Rs[r] = m < P.M ? b * P.os_b + ho * P.os_h + wo * P.os_w : -1;
        }
        __syncthreads();
    }
    auto sub_tile = [&](int i, int j, auto&& fn) {
        const int n  = n0 + (wn * TN + j) * 32 + l32;
        const int r0 = (wm * TM + i) * 32 + 4 * half;
        if (c_contig) {
            const uint32_t base = n < P.N ? (uint32_t)((m0 + r0) * P.N + n) * 4u : CONV_OOB;
#pragma unroll
            for (int v = 0; v < 16; ++v) fn(v, base, (uint32_t)(8 * (v / 4) + (v % 4)) * rowb);
        } else {
            const int* ro = Rs + r0;
            const int  cn = n < P.N ? n * P.os_n : -(1 << 30);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int r = ro[8 * (v / 4) + (v % 4)];
                fn(v, (r >= 0 && cn >= 0) ? (uint32_t)(r + cn) * 4u : CONV_OOB, 0u);
            }
        }
    };
    if constexpr (STEPS) {
        // (the pointer table is read from the argument block: indexing the by-value argument with a run-time value would make the compiler copy
        // it to scratch memory)
        const float* const* table = reinterpret_cast<const float* const*>(reinterpret_cast<const char*>(__builtin_amdgcn_kernarg_segment_ptr()) + 40);
#pragma nounroll
        for (int e = 0; e < nepi; ++e) {
            const uint32_t kind = step_desc(e) >> 8, code = step_desc(e) & 255u;
            const __amdgpu_buffer_rsrc_t e_rsrc = make_rsrc(table[e], kind == 3 ? P.out_bytes : 0u);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if (kind == 3) {
                        float ov[16];
                        sub_tile(i, j, [&](int v, uint32_t vo, uint32_t so) { ov[v] = buffer_load_x1_nt(e_rsrc, vo, so); });
                        conv_epilogue_step(code, acc[i][j], [&](int v) { return ov[v]; });
                    } else {
                        const float o = Es[e * BN + (wn * TN + j) * 32 + l32];
                        conv_epilogue_step(code, acc[i][j], [&](int) { return o; });
                    }
                }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) sub_tile(i, j, [&](int v, uint32_t vo, uint32_t so) { buffer_store_x1(acc[i][j][v], o_rsrc, vo, so); });
        return;
    }
    const float* full_ptr = epi.p[0];
#pragma unroll
    for (int t = 1; t < CONV_MAX_EPI; ++t) full_ptr = epi_first_full == t ? epi.p[t] : full_ptr;
    const __amdgpu_buffer_rsrc_t f_rsrc = make_rsrc(full_ptr, P.out_bytes);
    const uint32_t slots = (P.flags >> 20) & 31u;
    const int tap = (int)((P.flags >> 12) & 15u) - 1;
    // The epilogue of a backward pass: + full tensor (operand 0), kept where an activation (operand 1) lies above a limit (3) and
    // replaced by a constant (4) elsewhere, stored as a second result, * vector (2). The launches it replaces moved four to six times
    // the result; ResNet-50's training step at batch 64: 13.31 -> 12.11 ms.
    const bool masked_form = P.flags & CONV_SPLIT_MASKED;
    const __amdgpu_buffer_rsrc_t m_rsrc = make_rsrc(epi.p[1], masked_form ? P.out_bytes : 0u);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            float y[16], ov[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) y[v] = acc[i][j][v];
            const int col = (wn * TN + j) * 32 + l32;
            if (slots & 8u) sub_tile(i, j, [&](int v, uint32_t vo, uint32_t so) { ov[v] = buffer_load_x1_nt(f_rsrc, vo, so); });
            auto tap_store = [&]() {
                const __amdgpu_buffer_rsrc_t t_rsrc = make_rsrc(epi.p[CONV_MAX_EPI - 1], P.out_bytes);
                sub_tile(i, j, [&](int v, uint32_t vo, uint32_t so) { buffer_store_x1(y[v], t_rsrc, vo, so); });
            };
            if (masked_form) {
                float av[16];
                sub_tile(i, j, [&](int v, uint32_t vo, uint32_t so) { av[v] = buffer_load_x1_nt(m_rsrc, vo, so); });
                const float limit = Es[3 * BN + col], otherwise = Es[4 * BN + col], o = Es[2 * BN + col];
                if (slots & 8u) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) y[v] = y[v] + ov[v];
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) y[v] = av[v] > limit ? y[v] : otherwise;
                if (tap >= 0) tap_store();
                if (slots & 2u) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) y[v] = y[v] * o;
                }
                sub_tile(i, j, [&](int v, uint32_t vo, uint32_t so) { buffer_store_x1(y[v], o_rsrc, vo, so); });
                continue;
            }
            conv_straight_steps<16>(y, ov, slots, tap, Es, BN, col, tap_store);
            sub_tile(i, j, [&](int v, uint32_t vo, uint32_t so) { buffer_store_x1(y[v], o_rsrc, vo, so); });
        }
}

#define CONV_SPLIT_KERNEL(name, WGM, WGN, TM, TN, WPE, STEPS, PATCH, FINE, ...)                                              \
    extern "C" __global__ __launch_bounds__(64 * WGM * WGN) __attribute__((amdgpu_waves_per_eu(WPE))) void name(             \
        float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w,                                   \
        float* __restrict__ partial, uint32_t* __restrict__ arrivals, ConvEpiPtrs epi, ConvDerivedPtrs dp, ConvParams P, ConvDerived D) { \
        __shared__ __attribute__((aligned(16))) u32x4 pool[PATCH ? 12 * CONV_PATCH_ROWS : 24 * 32 * WGM * TM];               \
        __shared__ float Es[CONV_MAX_EPI * 32 * WGN * TN];                                                                   \
        __shared__ int Rs[32 * WGM * TM];                                                                                    \
        request_arguments<5 * sizeof(void*) + sizeof(ConvEpiPtrs) + sizeof(ConvDerivedPtrs) + sizeof(ConvParams) + sizeof(ConvDerived)>(); \
        conv_split_body<WGM, WGN, TM, TN, STEPS, PATCH, FINE, ##__VA_ARGS__>(pool, Es, Rs, out, x, w, partial, arrivals, epi, dp, P, D);    \
    }
// _steps: 50176 x 128 x 512 with a ReLU6 68 us, with a scalar 62, with `relu(y) + r` 82 (each as launches of its own behind the product: 83, 82, 94;
// in the fp32 kernels 73, 71, 73); 50176 x 256 x 512 97, 89, 108 (127, 120, 130). (Words of a full tensor requested for two tiles at a time
// instead of one: 80 instead of 82, not kept; for four: registers spill.)
// (2 x 2 waves of 64 x 64: 255 registers, two blocks per CU; 1 x 4 waves of 128 x 32, which load every column once, were 1 % slower)
CONV_SPLIT_KERNEL(conv_gemm_split_128x128, 2, 2, 2, 2, 2, false, false, false)
CONV_SPLIT_KERNEL(conv_gemm_split_128x128_patch, 2, 2, 2, 2, 2, false, true, false)
CONV_SPLIT_KERNEL(conv_gemm_split_128x128_steps, 2, 2, 2, 2, 2, true, false, false)
CONV_SPLIT_KERNEL(conv_gemm_split_128x128_patch_steps, 2, 2, 2, 2, 2, true, true, false)
// for at most 64 columns, or where the smaller tile divides the rows better among the CUs: three blocks per CU
CONV_SPLIT_KERNEL(conv_gemm_split_128x64, 2, 2, 2, 1, 3, false, false, false)
CONV_SPLIT_KERNEL(conv_gemm_split_128x64_patch, 2, 2, 2, 1, 3, false, true, false)
CONV_SPLIT_KERNEL(conv_gemm_split_128x64_steps, 2, 2, 2, 1, 3, true, false, false)
CONV_SPLIT_KERNEL(conv_gemm_split_128x64_patch_steps, 2, 2, 2, 1, 3, true, true, false)
// (242 registers: two blocks per CU)
CONV_SPLIT_KERNEL(conv_gemm_split_128x64_patch_fine, 2, 2, 2, 1, 2, false, true, true)
CONV_SPLIT_KERNEL(conv_gemm_split_128x64_patch_fine_steps, 2, 2, 2, 1, 2, true, true, true)
// (11 x 31 x 31 x 397 x 397 589 -> 209 us, 4 x 37 x 37 x 191 x 191 186 -> 44, 9 x 62 x 62 x 152 x 152 169 -> 115, 1 x 11 x 11 x 105 x 105 57 -> 18; before: the fp32 kernels)
CONV_SPLIT_KERNEL(conv_gemm_split_128x64_ragged, 2, 2, 2, 1, 2, false, true, true, true)
CONV_SPLIT_KERNEL(conv_gemm_split_128x64_ragged_steps, 2, 2, 2, 1, 2, true, true, true, true)

// ---- short contractions -------------------------------------------------------------------------------------------------
// Dense rows [M, K] with K <= 64: a product whose time is that of its result, and of the arrays its epilogue reads. A block holds the packed
// kernel operand of 256 columns in LDS (96 KB) for good; its 12 waves take 32 rows each, by themselves, keep their parts in registers and walk
// the columns. No barrier behind the first, nothing loaded twice, and while some waves of a SIMD wait for memory others multiply.
// Eight products of parts, not six (all but lo.lo, which is 2^-36 of the whole), and those of the two largest parts in a sum of their own: they are 16
// bits long, so few of them are cut off where they are added, and the other seven are a 256th of them. The two sums meet in one addition that is
// rounded. Errors against 64-bit sums, as a multiple of those of v_mfma_f32_32x32x2_f32, 64 terms of which 1, 2, 4, 16 and 64 are not zero: 1.00,
// 0.83, 0.66, 0.45, 0.34 (all of six products in one sum: 1.37, 1.56, 1.65, 1.36, 0.76, and 1.04 for activations of which half are zero; six in
// two sums: 1.03, 0.85, 0.68, 0.45, 0.35).
// What bounds it: HBM, at 0.7 to 0.85 of a copy's rate. 200704 x 64 x 256 alone (replays, packing included) 77 -> 60 us, with a residual 103 -> 83 (67 us
// of memory time; the fp32 tiles and those above load the rows once per 64 or 128 columns, and start and end a block for two k tiles), and with the
// backward pass of a ReLU, which the fp32 tiles leave to a launch of its own, 179 -> 82. (Six products in one sum: 52, 80 and 79; six in two sums: 53, 81, 80.
// Holding the next tile's rows in registers too, with 8 waves of 256 registers, was slower by 4 us with a residual.)
constexpr int CONV_SHORT_ROWS = 32, CONV_SHORT_COLS = 256, CONV_SHORT_WAVES = 12;

template <bool STEPS>
__device__ __forceinline__ void conv_short_body(u32x4* __restrict__ Bs, float* __restrict__ Es, float* __restrict__ out, const float* __restrict__ x,
                                                const float* __restrict__ w, const ConvEpiPtrs& epi, const ConvDerivedPtrs& Dp, const ConvParams& P,
                                                const ConvDerived& Dk) {
    constexpr int COLS = CONV_SHORT_COLS, KSTEPS = 4, WAVES = CONV_SHORT_WAVES, NT = 64 * WAVES;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // blocks that share rows stand behind the same L2
    const int work = xcd_range((int)blockIdx.x, (int)gridDim.x), walkers = (int)gridDim.x / P.tiles_n;
    const int walker = work / P.tiles_n, n0 = (work - walker * P.tiles_n) * P.m_each * 32;         // (m_each blocks of 32 columns per block, 8 at most)
    const int blocks_here = min(P.m_each, (P.N - n0 + 31) / 32);
    const uint32_t out_bytes = min(P.out_bytes, (uint32_t)P.M * (uint32_t)P.N * 4u), rowb = (uint32_t)P.N * 4u;
    const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(x, P.x_bytes), w_rsrc = make_rsrc(w, P.w_bytes), o_rsrc = make_rsrc(out, out_bytes);
    const int nepi = (P.flags >> 8) & 15u, epi_first_full = (int)((P.flags >> 16) & 15u) - 1;
    const uint32_t slots = (P.flags >> 20) & 31u;
    const int tap = (int)((P.flags >> 12) & 15u) - 1;
    const bool masked_form = P.flags & CONV_SPLIT_MASKED;
    const float* full_ptr = epi.p[0];
#pragma unroll
    for (int t = 1; t < CONV_MAX_EPI; ++t) full_ptr = epi_first_full == t ? epi.p[t] : full_ptr;
    const __amdgpu_buffer_rsrc_t f_rsrc = make_rsrc(full_ptr, slots & 8u ? out_bytes : 0u),
                                 m_rsrc = make_rsrc(epi.p[1], masked_form ? out_bytes : 0u),
                                 t_rsrc = make_rsrc(epi.p[CONV_MAX_EPI - 1], tap >= 0 ? out_bytes : 0u);

    auto request_rows = [&](f32x4 (&raw)[KSTEPS][2], int tile) {                     // (rows and features that do not exist: zeros)
        const int m = tile * CONV_SHORT_ROWS + l32;
        const uint32_t row = m < P.M ? (uint32_t)(m * P.xs_h) * 4u : CONV_OOB;
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int k = (s >> 1) * 32 + 16 * h + 4 * (2 * (s & 1) + half);
                raw[s][h] = buffer_load_x4(x_rsrc, k < P.K ? row + (uint32_t)k * 4u : CONV_OOB);
            }
    };
    const int tiles = (P.M + CONV_SHORT_ROWS - 1) / CONV_SHORT_ROWS;
    for (int i = tid; i < blocks_here * KSTEPS * 192; i += NT)
        Bs[i] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (uint32_t)i * 16u, (uint32_t)(n0 / 32 * KSTEPS) * 3072u, 0);
    conv_split_epilogue_operands<COLS>(Es, epi, Dp, P, Dk, tid, n0);
    __syncthreads();

    for (int tile = wave * walkers + walker; tile < tiles; tile += WAVES * walkers) {
        f32x4 raw[KSTEPS][2];
        request_rows(raw, tile);
        u32x4 af[KSTEPS][3];
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
            for (int t = 0; t < 3; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q) af[s][t][q] = conv_split_word(raw[s], t, q);
        const int m0 = tile * CONV_SHORT_ROWS;
#pragma nounroll
        for (int cb = 0; cb < blocks_here; ++cb) {
            const int col = cb * 32 + l32, n = n0 + col;
            const uint32_t base = n < P.N ? (uint32_t)((m0 + 4 * half) * P.N + n) * 4u : CONV_OOB;
            auto at = [&](int v) { return (uint32_t)(8 * (v / 4) + (v % 4)) * rowb; };
            float y[16], ov[16], av[16];
            if constexpr (!STEPS) {
                if (slots & 8u) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) ov[v] = buffer_load_x1_nt(f_rsrc, base, at(v));
                }
                if (masked_form) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) av[v] = buffer_load_x1_nt(m_rsrc, base, at(v));
                }
            }
            const u32x4* b_at = Bs + cb * KSTEPS * 192 + lane;
            f32x16 sum = {}, large = {};
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) {
                u32x4 bf[3];
#pragma unroll
                for (int t = 0; t < 3; ++t) bf[t] = b_at[s * 192 + t * 64];
                if (s & 1) FENCE();                         // (all of the columns' parts at once: registers would spill)
#pragma unroll
                for (int t = 0; t < 7; ++t)
                    sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, af[s][CONV_FINE_PA[t]]), __builtin_bit_cast(bf16x8, bf[CONV_FINE_PB[t]]), sum, 0, 0, 0);
                large = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, af[s][0]), __builtin_bit_cast(bf16x8, bf[0]), large, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) y[v] = (sum[v] + large[v]) * (1.f / (CONV_SPLIT_SCALE * CONV_SPLIT_SCALE));
            // sums that are not finite: again with fp32 products, as above
            float high = 0.f;
#pragma unroll
            for (int v = 0; v < 16; v += 2) high = higher_of(high, y[v], y[v + 1]);
            if (__builtin_amdgcn_ballot_w64(!(high < __builtin_inff()))) {
                f32x16 again = {};
                const int m = m0 + l32;
                const uint32_t row = m < P.M ? (uint32_t)(m * P.xs_h) * 4u : CONV_OOB;
#pragma nounroll
                for (int s = 0; s < KSTEPS; ++s) {
                    const int k = (s >> 1) * 32 + 4 * (2 * (s & 1) + half);
                    f32x4 a[2] = {buffer_load_x4(x_rsrc, k < P.K ? row + (uint32_t)k * 4u : CONV_OOB),
                                  buffer_load_x4(x_rsrc, k + 16 < P.K ? row + (uint32_t)(k + 16) * 4u : CONV_OOB)};
                    u32x4 b[3];
#pragma unroll
                    for (int t = 0; t < 3; ++t) b[t] = b_at[s * 192 + t * 64];
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        uint32_t part_e[3];
#pragma unroll
                        for (int t = 0; t < 3; ++t) part_e[t] = e & 1 ? b[t][e >> 1] & 0xFFFF0000u : b[t][e >> 1] << 16;
                        const float value = ((u2f(part_e[2]) + u2f(part_e[1])) + u2f(part_e[0])) * (1.f / CONV_SPLIT_SCALE);
                        const float bv = part_e[0] == CONV_PACK_RAW << 16 ? u2f(part_e[1] | part_e[2] >> 16) : value;
                        again = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e >> 2][e & 3], bv, again, 0, 0, 0);
                    }
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) y[v] = __builtin_isfinite(y[v]) ? y[v] : again[v];
            }
            auto store = [&](__amdgpu_buffer_rsrc_t to) {
#pragma unroll
                for (int v = 0; v < 16; ++v) buffer_store_x1(y[v], to, base, at(v));
            };
            if constexpr (STEPS) {
                // (the pointer table is read from the argument block, as above)
                const float* const* table = reinterpret_cast<const float* const*>(reinterpret_cast<const char*>(__builtin_amdgcn_kernarg_segment_ptr()) + 40);
#pragma nounroll
                for (int e = 0; e < nepi; ++e) {
                    const uint32_t desc = conv_split_step_desc(P, e);
                    if (desc >> 8 == 3) {
                        const __amdgpu_buffer_rsrc_t e_rsrc = make_rsrc(table[e], out_bytes);
#pragma unroll
                        for (int v = 0; v < 16; ++v) ov[v] = buffer_load_x1_nt(e_rsrc, base, at(v));
                        conv_epilogue_step(desc & 255u, y, [&](int v) { return ov[v]; });
                    } else {
                        const float o = Es[e * COLS + col];
                        conv_epilogue_step(desc & 255u, y, [&](int) { return o; });
                    }
                }
                store(o_rsrc);
                continue;
            }
            if (masked_form) {
                const float limit = Es[3 * COLS + col], otherwise = Es[4 * COLS + col], o = Es[2 * COLS + col];
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    if (slots & 8u) y[v] = y[v] + ov[v];
                    y[v] = av[v] > limit ? y[v] : otherwise;
                }
                if (tap >= 0) store(t_rsrc);
                if (slots & 2u) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) y[v] = y[v] * o;
                }
                store(o_rsrc);
                continue;
            }
            conv_straight_steps<16>(y, ov, slots, tap, Es, COLS, col, [&]() { store(t_rsrc); });
            store(o_rsrc);
        }
    }
}

#define CONV_SHORT_KERNEL(name, STEPS)                                                                                       \
    extern "C" __global__ __launch_bounds__(64 * CONV_SHORT_WAVES) __attribute__((amdgpu_waves_per_eu(CONV_SHORT_WAVES / 4, CONV_SHORT_WAVES / 4))) void name( \
        float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w,                                   \
        float* __restrict__ partial, uint32_t* __restrict__ arrivals, ConvEpiPtrs epi, ConvDerivedPtrs dp, ConvParams P, ConvDerived D) { \
        __shared__ __attribute__((aligned(16))) u32x4 Bs[CONV_SHORT_COLS / 32 * 4 * 192];                                    \
        __shared__ float Es[CONV_MAX_EPI * CONV_SHORT_COLS];                                                                 \
        request_arguments<5 * sizeof(void*) + sizeof(ConvEpiPtrs) + sizeof(ConvDerivedPtrs) + sizeof(ConvParams) + sizeof(ConvDerived)>(); \
        conv_short_body<STEPS>(Bs, Es, out, x, w, epi, dp, P, D);                                                            \
    }
CONV_SHORT_KERNEL(conv_gemm_split_short, false)
CONV_SHORT_KERNEL(conv_gemm_split_short_steps, true)
