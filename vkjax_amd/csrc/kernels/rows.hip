// Row programs: a run of element-wise steps and row reductions over the same [outer, R] array in one launch, one row to a
// wave (several where they are short). The loss of a classifier and its gradient are such a run: maximum of a row, exp,
// sum, log, products, two more sums - eleven launches of 3 to 5 us each on a thousand rows of ten.
//
// The host (fusion.fuse_row_programs) writes the run down as a program for this kernel: what it reads from memory is
// loaded first, everything at once, into slots of LDS; every instruction then works on an accumulator (R values, spread
// over the lanes as reduce_rows spreads them) and on slots, and results that something outside the run reads are stored.
// A slot belongs to the thread that wrote it, so no barrier is needed. Element-wise steps are those of ew_apply.h and
// sums and maxima are taken in the order of reduce_rows, so every value has the bits that the separate launches give.
//
// What bounds it: for arrays of a few thousand values the latency of one round of loads and some twenty-five dependent
// instructions, each a branch and the code of its step (replays of a loss and its gradient on 1000 rows of 10: 38 -> 15.5
// us, 15 launches -> 4; the words of an instruction requested when it begins, not one ahead, 16.2; one launch less and the arguments
// read in one go 10.5 -> 9.9). Steps on one value per row are worked out once, not in every word of a lane (64 x 1000 22.3 -> 18.6, 65536 x 1000 450 -> 378). Large arrays: the
// element-wise steps, which read and write LDS where the launches it replaces went through memory (65536 x 1000: 838 ->
// 462 us). Training steps: MLP on 1000 samples 171 -> 145 us, conv net on 50 images 353 -> 329.
#include "ew_apply.h"

enum RowsOp : uint32_t { ROWS_LOAD = 0, ROWS_APPLY = 1, ROWS_SUM = 2, ROWS_MAX = 3, ROWS_PUT = 4, ROWS_OUT = 5 };

struct RowsParams {
    uint32_t outer, R, lanes_log2, n_in, n_code;      // lanes_log2: bits 0-7; the block's threads in bits 8-31
    uint32_t in_bytes[8];                 // readable bytes behind each input pointer
    uint32_t in_base[8];                  // element of row 0, column 0
    int32_t  in_row[8], in_col[8];        // element strides
    uint32_t in_slot[8];                  // bits 0-15: first word of the slot; bit 16: one word (the same for a whole row); bit 17: 16-byte loads
    // two words per instruction: bits 0-3 RowsOp, 4-15 opcode of ew_opcodes.h, 16 the operand is the LEFT argument, 17 one word per row,
    // 18 there is an operand, 19 accumulator and operand are one value per row, 20-31 first word of the slot (or number of the output); then the step's immediate
    uint32_t code[96];
};
struct RowsIn  { const uint32_t* p[8]; };
struct RowsOut { uint32_t* p[6]; };
constexpr int ROWS_MAX_IN = 8;

template <int VEC, int NV>
__device__ __forceinline__ void rows_body(const RowsOut& out, const RowsIn& in, const RowsParams& Pk) {
    constexpr int W = VEC * NV;
    extern __shared__ uint32_t slots[];
    // The argument block is read in one go, and a word of every 64 bytes of the program with it: left to itself the compiler fetches words where they are
    // used, one round trip to memory after the other.
    const uint32_t* const code = reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(__builtin_amdgcn_kernarg_segment_ptr())
                                                                   + sizeof(RowsOut) + sizeof(RowsIn) + offsetof(RowsParams, code));
    struct { uint32_t outer, R, lanes_log2, n_in, n_code, in_bytes[8], in_base[8]; int32_t in_row[8], in_col[8]; uint32_t in_slot[8]; } P;
    P.outer = Pk.outer; P.R = Pk.R; P.lanes_log2 = Pk.lanes_log2; P.n_in = Pk.n_in; P.n_code = Pk.n_code;
    uint32_t next = code[0], next_imm = code[1];
    asm volatile("" : "+s"(P.outer), "+s"(P.R), "+s"(P.lanes_log2), "+s"(P.n_in), "+s"(P.n_code), "+s"(next), "+s"(next_imm)
                 : "s"(code[16]), "s"(code[32]), "s"(code[48]), "s"(code[64]), "s"(code[80]), "s"(in.p[0]), "s"(in.p[1]), "s"(in.p[2]), "s"(in.p[3]));
#pragma unroll
    for (int k = 0; k < ROWS_MAX_IN; ++k) {
        P.in_bytes[k] = Pk.in_bytes[k]; P.in_base[k] = Pk.in_base[k]; P.in_row[k] = Pk.in_row[k]; P.in_col[k] = Pk.in_col[k]; P.in_slot[k] = Pk.in_slot[k];
        asm volatile("" : "+s"(P.in_bytes[k]), "+s"(P.in_base[k]), "+s"(P.in_row[k]), "+s"(P.in_col[k]), "+s"(P.in_slot[k]));
    }
    const uint32_t nt = P.lanes_log2 >> 8, lane = threadIdx.x & 63u;
    const uint32_t log2_lanes = NV == 1 ? P.lanes_log2 & 255u : 6u, lanes = 1u << log2_lanes, rows = 64u >> log2_lanes;
    const uint32_t first = (blockIdx.x * (nt >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * rows;
    if (first >= P.outer) return;                                     // whole wave leaves together
    const uint32_t l = lane & (lanes - 1u), row = first + (lane >> log2_lanes);
    const bool row_ok = row < P.outer;
    uint32_t col[NV];                                                 // first column of a lane's vector i
    bool ok[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) { col[i] = (l + i * lanes) * VEC; ok[i] = row_ok && col[i] < P.R; }
    uint32_t* const mine = slots + threadIdx.x;

    // ---- everything the program reads, requested together (absent inputs: descriptors of no bytes)
    uint32_t got[ROWS_MAX_IN][W];
#pragma unroll
    for (int k = 0; k < ROWS_MAX_IN; ++k) {
        const __amdgpu_buffer_rsrc_t r = make_rsrc(in.p[k], k < (int)P.n_in ? P.in_bytes[k] : 0u);
        const uint32_t base = P.in_base[k] + row * (uint32_t)P.in_row[k], how = P.in_slot[k] >> 16;
        if (how & 1u) {
            got[k][0] = __builtin_amdgcn_raw_buffer_load_b32(r, row_ok ? base * 4u : 0x80000000u, 0, 0);
            continue;
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            if (VEC == 4 && (how & 2u)) {
                const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(r, ok[i] ? (base + col[i]) * 4u : 0x80000000u, 0, 0);
#pragma unroll
                for (int j = 0; j < VEC; ++j) got[k][i * VEC + j] = t[j];
            } else {
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                    got[k][i * VEC + j] = __builtin_amdgcn_raw_buffer_load_b32(r, ok[i] ? (base + (col[i] + j) * (uint32_t)P.in_col[k]) * 4u : 0x80000000u, 0, 0);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < ROWS_MAX_IN; ++k) {
        if (k >= (int)P.n_in) continue;
        const uint32_t at = P.in_slot[k] & 0xFFFFu;
        mine[at * nt] = got[k][0];
        if (P.in_slot[k] & 0x10000u) continue;
#pragma unroll
        for (int e = 1; e < W; ++e) mine[(at + e) * nt] = got[k][e];
    }

    // ---- the program. (Its words are read from the argument block itself: indexing the by-value argument with a run-time value would make
    // the compiler copy it to scratch memory.)
    uint32_t* const* outs = reinterpret_cast<uint32_t* const*>(reinterpret_cast<const char*>(__builtin_amdgcn_kernarg_segment_ptr()));
    uint32_t acc[W];
#pragma unroll
    for (int e = 0; e < W; ++e) acc[e] = 0u;
    const uint32_t n_code = P.n_code;
#pragma nounroll
    for (uint32_t pc = 0; pc < n_code; ++pc) {
        const uint32_t word = next, imm = next_imm, kind = word & 15u, slot = word >> 20;
        const uint32_t after = min(2u * pc + 2u, 94u);                // (requested an instruction ahead)
        next = code[after]; next_imm = code[after + 1];
        const bool single = word & (1u << 17);
        if (kind <= ROWS_APPLY) {
            uint32_t v[W];
            if (kind == ROWS_LOAD || (word & (1u << 18))) {
                v[0] = mine[slot * nt];
#pragma unroll
                for (int e = 1; e < W; ++e) v[e] = v[0];
                if (!single) {
#pragma unroll
                    for (int e = 1; e < W; ++e) v[e] = mine[(slot + e) * nt];
                }
            } else {
#pragma unroll
                for (int e = 0; e < W; ++e) v[e] = acc[e];
            }
            if (kind == ROWS_LOAD) {
#pragma unroll
                for (int e = 0; e < W; ++e) acc[e] = v[e];
            } else if (W > 1 && (word & (1u << 19))) {                // the same in every word: worked out once
                uint32_t one[1] = {acc[0]};
                const uint32_t operand[1] = {v[0]};
                ew_apply_vec<1>(word >> 4 & 0xFFFu, one, operand, word & (1u << 16), imm);
#pragma unroll
                for (int e = 0; e < W; ++e) acc[e] = one[0];
            } else {
                ew_apply_vec<W>(word >> 4 & 0xFFFu, acc, v, word & (1u << 16), imm);
            }
        } else if (kind == ROWS_SUM) {
            float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < NV; ++i)
#pragma unroll
                for (int j = 0; j < VEC; ++j) s[VEC == 4 ? j : i & 3] += ok[i] ? u2f(acc[i * VEC + j]) : 0.f;
            float total = (s[0] + s[1]) + (s[2] + s[3]);
            total = lanes_allreduce(total, lanes, [](float a, float b) { return a + b; });
#pragma unroll
            for (int e = 0; e < W; ++e) acc[e] = f2u(total);
        } else if (kind == ROWS_MAX) {
            auto higher = [](float a, float b) { return (a > b || a != a) ? a : b; };      // a NaN wins; of two zeros the later one
            float s[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
            for (int i = 0; i < NV; ++i)
#pragma unroll
                for (int j = 0; j < VEC; ++j) s[VEC == 4 ? j : i & 3] = higher(s[VEC == 4 ? j : i & 3], ok[i] ? u2f(acc[i * VEC + j]) : -INFINITY);
            float top = higher(higher(s[0], s[1]), higher(s[2], s[3]));
            top = lanes_allreduce(top, lanes, higher);
            top = __shfl(top, lane & ~(lanes - 1u), 64);              // (the first lane's, as reduce_rows stores it)
#pragma unroll
            for (int e = 0; e < W; ++e) acc[e] = f2u(top);
        } else if (kind == ROWS_PUT) {
            mine[slot * nt] = acc[0];
            if (!single) {
#pragma unroll
                for (int e = 1; e < W; ++e) mine[(slot + e) * nt] = acc[e];
            }
        } else {
            uint32_t* const to = outs[slot];
            if (single) {
                if (row_ok && l == 0) to[row] = acc[0];
                continue;
            }
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                if (!ok[i]) continue;
                uint32_t* const at = to + (size_t)row * P.R + col[i];
                if constexpr (VEC == 4) *reinterpret_cast<u32x4*>(at) = u32x4{acc[4 * i], acc[4 * i + 1], acc[4 * i + 2], acc[4 * i + 3]};
                else at[0] = acc[i];
            }
        }
    }
}

#define ROWS_KERNEL(name, VEC, NV)                                                                                          \
    extern "C" __global__ __launch_bounds__(256) void name(RowsOut out, RowsIn in, RowsParams P) { rows_body<VEC, NV>(out, in, P); }
// _v4: R % 4 == 0, in the order of the 16-byte reduce_rows kernel. _n<NV>: vectors per lane, rows of up to 64 * VEC * NV values
ROWS_KERNEL(rows_v4_n1, 4, 1)
ROWS_KERNEL(rows_v4_n4, 4, 4)
ROWS_KERNEL(rows_v1_n1, 1, 1)
ROWS_KERNEL(rows_v1_n4, 1, 4)
ROWS_KERNEL(rows_v1_n16, 1, 16)
