// Four waves share one 32 x 32 tile of a product on the fp32 matrix cores (v_mfma_f32_32x32x2_f32): for products with so few tiles that one wave per
// tile would leave most matrix cores idle (a wave can drive only one). Every wave takes a quarter of each k step: it loads, parks in LDS and consumes
// its own slice, so the k loop has no barrier; the four sums meet in LDS behind it, and every wave finishes a quarter of the tile.
//
// A block of these kernels is usually alone on its CU, and its time is what it waits for: the path to its first loads, their way from memory, and in
// every k step the way through LDS. So
//   - divisions by what is known when the launch is recorded are multiplications by constants from the host, and whether a tap lies inside the input is
//     worked out for the tap a load is for instead of for all of them beforehand;
//   - the operands of the epilogue are requested behind the first tiles, and used behind the loop;
//   - a wave reads the fragments of the coming k step, stores that step's tiles before it and requests a later step's between the matrix instructions of
//     the one it computes: each slot below is one matrix instruction (64 cycles) and what fits beside it.
// A k step of 128 takes 0.5 us where a block is alone on its CU (0.43 at the rate of the matrix cores) and everything else 3.5 us. Before, one k step after the
// other, epilogue operands in front of the loop and long divisions at the start: 0.8 and 4.4 us. In ResNet-50 on one image, where the kernel operands come
// from behind the L2s: 49 x 4608 x 512 in four slices 12.4 -> 9.3 us, 49 x 512 x 2048 7.1 -> 5.5, 3136 x 576 x 64 (steps of 64) 10.2 -> 8.2; the whole replay
// 483 -> 429 us, on six images of 160 x 160 690 -> 609, its training step on four of 128 x 128 2.54 -> 2.35 ms, a conv block 2 x 28 x 28 x 256 30.4 -> 25.6 us.
// With the loads of two more k steps on their way instead of one only three blocks fit a CU (164 registers, 126): 1960 x 2048 x 512 (992 tiles) 44.0
// instead of 37.5 us, 900 x 256 x 512 6.4 instead of 5.9; 1960 x 2048 x 128 11.4 instead of 11.5.
#pragma once

// How the kernel operand is loaded: element by element; 16-byte vectors along the columns; 16-byte vectors along the contraction, contiguous there (a
// transposed matrix: one tap only), which is then handled like the A operand. 40 x 1000 x 2048 21.3 us element by element, 7.2 in vectors; 300 x 2000 x 500 38.1, 11.0.
enum { QUAD_B_WORDS = 0, QUAD_B_COLUMNS = 1, QUAD_B_ROWS = 2 };

// LDS of one wave: its slices of the A tile ([32][BKW + 4]) and the B tile ([BKW][36], or like A's)
template <int BK> constexpr int conv_quad_wave_floats() { return 32 * (BK / 4 + 4) + BK / 4 * 36; }
// ... of a block: those, the per-column epilogue operands, and a word (floats)
template <int BK> constexpr int conv_quad_floats() { return 4 * conv_quad_wave_floats<BK>() + CONV_MAX_EPI * 32 + 4; }

// BK: k step of the block. SHARED: several blocks share a tile, each summing a slice
// of the contraction; a slice leaves its sums in `partial`, and the block that arrives last at the tile's counter adds them.
// STRIDED: the result's rows lie apart (a class of the outputs of a convolution over a dilated input): ConvParams' ws_* are its strides, and there is no epilogue.
// Requirements (the host checks them): 16-byte loads of A, K = KH * KW * Cin with one tap or Cin a multiple of BK / 4, a row-major result (or STRIDED) and an
// epilogue that conv_straight_steps takes. ConvParams' os_* and LH, LW hold divisors here (see there).
template <int BK, int B_LOADS, bool SHARED, bool STRIDED = false>
__device__ __forceinline__ void conv_quad_body(float* __restrict__ pool, const ConvRegion region, float* __restrict__ out, const float* __restrict__ x,
                                               const float* __restrict__ w, const ConvEpiPtrs& epi, const ConvDerivedPtrs& Dp, const ConvParams& Pk,
                                               const ConvDerived& Dk, float* __restrict__ partial = nullptr, uint32_t* __restrict__ arrivals = nullptr) {
    constexpr int BKW = BK / 4, LDA = BKW + 4, LDB = 36;               // a wave's slice of a k step; row pitches in LDS (no bank conflicts)
    constexpr int G = BKW / 8, SLOTS = 4 * G;                          // groups of four matrix instructions: a lane holds four k, its half's, of each
    constexpr int A_VPR = BKW / 4, A_RSTEP = 64 / A_VPR, A_NV = 32 / A_RSTEP, B_NV = BKW / 8, NV = A_NV + B_NV;
    static_assert(B_LOADS != QUAD_B_ROWS || A_NV == B_NV, "the B tile has the A tile's layout");
    constexpr uint32_t TILE = 32 * 32 * 4;

    // every argument that the way to the loads needs, in one batch
    struct {
        int32_t M, N, K, Ho, Wo, H, W, Cin, KH, KW, SH, SW, PH, PW, DH, DW, xs_b, xs_h, xs_w, per, slices;
        uint32_t flags, x_bytes, w_bytes, out_bytes, howo_magic, howo_shift, wo_magic, wo_shift, inner_magic, inner_shift, all_magic, all_shift, cin_magic, cin_shift;
    } P;
#define QUAD_PIN(f, from) P.f = Pk.from; asm volatile("" : "+s"(P.f));
    asm volatile("" : "+s"(out), "+s"(x), "+s"(w));
    QUAD_PIN(M, M) QUAD_PIN(N, N) QUAD_PIN(K, K) QUAD_PIN(Ho, Ho) QUAD_PIN(Wo, Wo) QUAD_PIN(H, H) QUAD_PIN(W, W) QUAD_PIN(Cin, Cin)
    QUAD_PIN(KH, KH) QUAD_PIN(KW, KW) QUAD_PIN(SH, SH) QUAD_PIN(SW, SW) QUAD_PIN(PH, PH) QUAD_PIN(PW, PW) QUAD_PIN(DH, DH) QUAD_PIN(DW, DW)
    QUAD_PIN(xs_b, xs_b) QUAD_PIN(xs_h, xs_h) QUAD_PIN(xs_w, xs_w) QUAD_PIN(flags, flags) QUAD_PIN(x_bytes, x_bytes) QUAD_PIN(w_bytes, w_bytes)
    QUAD_PIN(out_bytes, out_bytes) QUAD_PIN(howo_magic, howo_magic) QUAD_PIN(howo_shift, howo_shift) QUAD_PIN(wo_magic, wo_magic) QUAD_PIN(wo_shift, wo_shift)
    QUAD_PIN(inner_magic, os_b) QUAD_PIN(inner_shift, os_h) QUAD_PIN(all_magic, os_w) QUAD_PIN(all_shift, os_n) QUAD_PIN(cin_magic, LH) QUAD_PIN(cin_shift, LW)
    QUAD_PIN(per, k_split_steps) QUAD_PIN(slices, m_each)
#undef QUAD_PIN
    const bool flat_rows = P.flags & 2u, masked = P.flags & 4u, taps = B_LOADS != QUAD_B_ROWS && P.KH * P.KW != 1;
    const int tid = threadIdx.x, lane = tid & 63, kw = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, half = lane >> 5;
    float* const As = pool + kw * conv_quad_wave_floats<BK>();          // [32][LDA], this wave's
    float* const Bs = As + 32 * LDA;                                    // [BKW][LDB]
    float* const Es = pool + 4 * conv_quad_wave_floats<BK>();           // [CONV_MAX_EPI][32]
    int*   const Rs = reinterpret_cast<int*>(Es + CONV_MAX_EPI * 32);

    // ---------------- which tile, which part of its contraction ----------------
    // Consecutive block ids go to different XCDs (8 of them, each with its own L2): every XCD is handed a contiguous range of tiles, row by row
    // or column by column, or (flags bits 29-31: 1 + log2 xn, xn up to 8) a rectangle of 8 / xn x xn of them.
    int work = (int)blockIdx.x - region.first_block;
    const int all = region.tiles_m * region.tiles_n;
    int kbase = 0, ktiles = max(1, (P.K + BK - 1) / BK), slice = 0;        // K = 0 runs as one k step whose loads are all out of range
    if (P.per > 0) {
        slice = magic_div(work, P.all_magic, P.all_shift);
        work -= slice * all;
        kbase = slice * P.per;
        ktiles = min(P.per, ktiles - kbase);
        if constexpr (!SHARED) out += (size_t)slice * (size_t)P.M * (size_t)P.N;
    }
    const uint32_t xcd_code = P.flags >> 29;
    int tile_m, tile_n;
    if (xcd_code > 0 && xcd_code < CONV_XCD_COLUMNWISE) {
        const int xn = 1 << (xcd_code - 1), sub_n = region.tiles_n / xn, sub_m = region.tiles_m >> (4 - xcd_code);       // (both divisible)
        const int xcd = work & 7, l = work >> 3, lm = l / sub_n;
        tile_m = (xcd >> (xcd_code - 1)) * sub_m + lm;
        tile_n = (xcd & (xn - 1)) * sub_n + (l - lm * sub_n);
    } else {
        const int each = all / 8;
        if (each > 0 && work < each * 8) work = (work & 7) * each + (work >> 3);
        const int q = magic_div(work, P.inner_magic, P.inner_shift);
        if (xcd_code == CONV_XCD_COLUMNWISE) { tile_n = q; tile_m = work - q * region.tiles_m; }
        else                                 { tile_m = q; tile_n = work - q * region.tiles_n; }
    }
    const int m0 = region.m_base + tile_m * 32, n0 = tile_n * 32;

    // ---------------- what a lane loads ----------------
    // A: 16-byte vectors along k, addressed from (PH, PW) positions before the input's start, so that the offset of a row's top-left tap is never
    // negative (a negative offset is out of range for the descriptor even when a later addition brings it back). Out of range: reads zeros.
    const uint32_t x_bias = (uint32_t)(P.PH * P.xs_h + P.PW * P.xs_w) * 4u;
    const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(reinterpret_cast<const char*>(x) - x_bias, P.x_bytes + x_bias),
                                 w_rsrc = make_rsrc(w, P.w_bytes), o_rsrc = make_rsrc(out, P.out_bytes);
    const int a_row = lane / A_VPR, a_k = 4 * (lane % A_VPR);           // (k within the wave's slice)
    const int b_k = lane / 8, b_n = n0 + 4 * (lane % 8);
    uint32_t a_voff[A_NV], a_at[A_NV];                                  // of tap 0; of the tap that is loaded, out of range where that lies outside
    int a_h[A_NV], a_w[A_NV];
#pragma unroll
    for (int p = 0; p < A_NV; ++p) {
        const int m = m0 + a_row + p * A_RSTEP;
        a_h[p] = a_w[p] = 0;
        if (flat_rows) {
            a_voff[p] = (uint32_t)(m * P.xs_h + a_k) * 4u;
        } else {
            const int b = magic_div(m, P.howo_magic, P.howo_shift), r2 = m - b * (P.Ho * P.Wo);
            const int ho = magic_div(r2, P.wo_magic, P.wo_shift), wo = r2 - ho * P.Wo;
            a_voff[p] = (uint32_t)(b * P.xs_b + ho * P.SH * P.xs_h + wo * P.SW * P.xs_w + a_k) * 4u;
            a_h[p] = ho * P.SH - P.PH;
            a_w[p] = wo * P.SW - P.PW;
        }
        if (m >= P.M) a_voff[p] = CONV_OOB;
        a_at[p] = a_voff[p];
    }
    // the position of the step that is loaded next: its first k (this wave's), tap and feature
    int k = kbase * BK + kw * BKW, t_r = 0, t_s = 0, t_c = k;
    if (taps) {
        const int rs = magic_div(k, P.cin_magic, P.cin_shift);
        t_c = k - rs * P.Cin;
        t_s = rs;
        while (t_s >= P.KW) { t_s -= P.KW; ++t_r; }
    }
    auto at_tap = [&]() {                                               // a new tap: which rows read nothing there
        if (!masked) return;
#pragma unroll
        for (int p = 0; p < A_NV; ++p) {
            const bool in = (uint32_t)(a_h[p] + t_r * P.DH) < (uint32_t)P.H && (uint32_t)(a_w[p] + t_s * P.DW) < (uint32_t)P.W;
            a_at[p] = in ? a_voff[p] : CONV_OOB;
        }
    };
    at_tap();
    // what a step's loads have in common: worked out once, then the loads are issued one by one
    uint32_t a_soff = 0u, b_soff = 0u, b_at[B_NV];                      // (b_at: of vectors along the contraction)
    if constexpr (B_LOADS == QUAD_B_ROWS) {
#pragma unroll
        for (int p = 0; p < B_NV; ++p) {
            const int n = n0 + a_row + p * A_RSTEP;
            b_at[p] = n < P.N ? (uint32_t)(n * Pk.ws_n + a_k) * 4u : CONV_OOB;
        }
    }
    int b_first = 0;
    const int k_end = min(P.K, (kbase + ktiles) * BK);
    auto begin_loads = [&]() {
        if (k + BKW > k_end) {                                          // the contraction (the slice) ends here: later loads of this wave read nothing
#pragma unroll
            for (int p = 0; p < A_NV; ++p) {
                a_at[p] = k + a_k >= k_end ? CONV_OOB : a_at[p];
                if constexpr (B_LOADS == QUAD_B_ROWS) b_at[p] = k + a_k >= k_end ? CONV_OOB : b_at[p];
            }
        }
        a_soff = (uint32_t)(t_r * P.DH * P.xs_h + t_s * P.DW * P.xs_w + t_c) * 4u;
        if constexpr (B_LOADS == QUAD_B_COLUMNS) b_soff = k < k_end ? (uint32_t)k * (uint32_t)P.N * 4u : CONV_OOB - 4u;
        else if constexpr (B_LOADS == QUAD_B_ROWS) b_soff = (uint32_t)k * 4u;
        else b_first = t_r * Pk.ws_r + t_s * Pk.ws_s + t_c * Pk.ws_c;
    };
    const uint32_t b_voff = b_n < P.N ? (uint32_t)(b_k * P.N + b_n) * 4u : CONV_OOB;       // vectors along the columns; rows k >= K lie beyond the descriptor
    const float* const b_words = w + (B_LOADS != QUAD_B_WORDS ? 0 : (n0 + l32) * Pk.ws_n + half * (BKW / 2) * Pk.ws_c);
    struct Stage { f32x4 a[A_NV]; f32x4 b[B_NV]; };                      // what is on its way for one k step (B element by element: BKW / 2 numbers of a column)
    auto load_one = [&](Stage& st, int v) {
        if (v < A_NV) { st.a[v < A_NV ? v : 0] = buffer_load_x4(x_rsrc, a_at[v < A_NV ? v : 0], a_soff); return; }
        const int p = v - A_NV;
        if constexpr (B_LOADS == QUAD_B_COLUMNS) st.b[p] = buffer_load_x4(w_rsrc, b_voff, b_soff + (uint32_t)(p * 8) * (uint32_t)P.N * 4u);
        else if constexpr (B_LOADS == QUAD_B_ROWS) st.b[p] = buffer_load_x4(w_rsrc, b_at[p], b_soff);
        else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = 4 * p + q;
                st.b[p][q] = n0 + l32 < P.N && k + half * (BKW / 2) + j < k_end ? b_words[b_first + j * Pk.ws_c] : 0.f;
            }
        }
    };
    auto end_loads = [&]() {
        k += BK;
        t_c += BK;
        if (taps && t_c >= P.Cin && k < k_end) {
            while (t_c >= P.Cin) { t_c -= P.Cin; if (++t_s == P.KW) { t_s = 0; ++t_r; } }
            at_tap();
        }
    };
    auto load_all = [&](Stage& st) {
        begin_loads();
#pragma unroll
        for (int v = 0; v < NV; ++v) load_one(st, v);
        end_loads();
    };
    // A contraction that ends within a vector (only with a single tap): what lies behind it is the next row's, and zeros on the other side would not leave
    // a value alone that is not finite.
    auto clear_tail = [&](Stage& st, int step) {
        const int first = step * BK + kw * BKW;
        if ((P.K & 3) != 0 && first + BKW > P.K) {
#pragma unroll
            for (int p = 0; p < A_NV; ++p)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    st.a[p][q] = first + a_k + q < P.K ? st.a[p][q] : 0.f;
                    if constexpr (B_LOADS == QUAD_B_ROWS) st.b[p][q] = first + a_k + q < P.K ? st.b[p][q] : 0.f;
                }
        }
    };
    auto store_one = [&](const Stage& st, int v) {
        if (v < A_NV) { *reinterpret_cast<f32x4*>(&As[(a_row + (v < A_NV ? v : 0) * A_RSTEP) * LDA + a_k]) = st.a[v < A_NV ? v : 0]; return; }
        const int p = v - A_NV;
        if constexpr (B_LOADS == QUAD_B_ROWS) *reinterpret_cast<f32x4*>(&Bs[(a_row + p * A_RSTEP) * LDA + a_k]) = st.b[p];
        else if constexpr (B_LOADS == QUAD_B_COLUMNS) *reinterpret_cast<f32x4*>(&Bs[(b_k + p * 8) * LDB + 4 * (lane % 8)]) = st.b[p];
        else {
#pragma unroll
            for (int q = 0; q < 4; ++q) Bs[(half * (BKW / 2) + 4 * p + q) * LDB + l32] = st.b[p][q];
        }
    };
    f32x4 fa[G], fb[G];                                                 // fragments of the k step that is computed
    uint32_t a_frag = (uint32_t)(l32 * LDA + half * (BKW / 2)), b_frag = (uint32_t)(32 * LDA + (B_LOADS == QUAD_B_ROWS ? l32 * LDA + half * (BKW / 2) : half * (BKW / 2) * LDB + l32));
    asm volatile("" : "+v"(a_frag), "+v"(b_frag));                      // (one register each, not one per group)
    auto read_group = [&](int g) {                                      // lanes 0-31 take the first half of the wave's slice, lanes 32-63 the second
        fa[g] = *reinterpret_cast<const f32x4*>(&As[a_frag + g * 4]);
        if constexpr (B_LOADS == QUAD_B_ROWS) fb[g] = *reinterpret_cast<const f32x4*>(&As[b_frag + g * 4]);
        else {
#pragma unroll
            for (int q = 0; q < 4; ++q) fb[g][q] = As[b_frag + (g * 4 + q) * LDB];
        }
    };
    // LDS accesses of a wave execute in order; the compiler has to keep them in order, too
    auto in_order = [&]() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };

    // a wave's quarter of the tile: rows 8 kw + 4 half .. + 3 of its column
    auto quarter_tile = [&](auto&& fn) {
        const int n = n0 + l32;
        const uint32_t base = n < P.N ? (uint32_t)((m0 + 4 * half) * P.N + n) * 4u : CONV_OOB, rowb = (uint32_t)P.N * 4u;
#pragma unroll
        for (int v = 0; v < 4; ++v) fn(v, base, (uint32_t)(8 * kw + v) * rowb);
    };

    Stage next;
    load_all(next);
    // Epilogue operands: thread t fetches column t of every step. Every step issues one load, whatever its kind, so that none waits for the one before: an
    // absent operand, one that is derived behind the loop, or a full tensor has a descriptor of size 0, which reads nothing and returns 0.
    float e_reg[CONV_MAX_EPI], d_in[CONV_MAX_DERIVED + 1], quarter[4] = {0.f, 0.f, 0.f, 0.f};
    const int nepi = (P.flags >> 8) & 15u, first_full = (int)((P.flags >> 16) & 15u) - 1;
    if (nepi) {
        uint32_t e_bytes[CONV_MAX_EPI], e_scale[CONV_MAX_EPI];          // (the same in every lane: worked out before the lanes part)
#pragma unroll
        for (int e = 0; e < CONV_MAX_EPI; ++e) {
            const uint32_t kind = ((Pk.epi_desc[e / 3] >> (10 * (e % 3))) & 1023u) >> 8;       // 0 beyond the last step
            const uint32_t present = epi.p[e] != nullptr ? 1u : 0u;
            e_bytes[e] = (uint32_t)__builtin_amdgcn_readfirstlane((int)(kind == 1 ? 4u * present : kind == 2 ? (uint32_t)P.N * 4u * present : 0u));
            e_scale[e] = kind == 2 ? 4u : 0u;
        }
        if (tid < 32) {
#pragma unroll
            for (int e = 0; e < CONV_MAX_EPI; ++e) e_reg[e] = buffer_load_x1(make_rsrc(epi.p[e], e_bytes[e]), (uint32_t)(n0 + tid) * e_scale[e]);
            if (Dk.nsteps) {
#pragma unroll
                for (int q = 0; q <= CONV_MAX_DERIVED; ++q) {
                    const bool vec = (Dk.vector_mask >> q) & 1u;
                    d_in[q] = buffer_load_x1(make_rsrc(Dp.p[q], Dp.p[q] == nullptr ? 0u : vec ? (uint32_t)P.N * 4u : 4u), vec ? (uint32_t)(n0 + tid) * 4u : 0u);
                }
            }
        }
        if (P.flags & (8u << 20)) {
            const float* full_ptr = epi.p[0];
#pragma unroll
            for (int t = 1; t < CONV_MAX_EPI; ++t) full_ptr = first_full == t ? epi.p[t] : full_ptr;
            const __amdgpu_buffer_rsrc_t f_rsrc = make_rsrc(full_ptr, P.out_bytes);
            quarter_tile([&](int v, uint32_t vo, uint32_t so) { quarter[v] = buffer_load_x1_nt(f_rsrc, vo, so); });
        }
    }

    f32x16 acc = f32x16{};
    clear_tail(next, kbase);
#pragma unroll
    for (int v = 0; v < NV; ++v) store_one(next, v);
    in_order();
    load_all(next);
#pragma unroll
    for (int g = 0; g < G; ++g) read_group(g);
    // One k step: the matrix instructions of the fragments at hand; between them the tiles of the next step go to LDS, the loads of the one behind it are
    // issued into the registers that frees (beyond the end they read nothing), and the next step's fragments are read, each group behind the last
    // instruction that uses the one before.
#pragma nounroll
    for (int at = 1; at < ktiles; ++at) {
        clear_tail(next, kbase + at);
        in_order();
        begin_loads();
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) {
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[s / 4][s % 4], fb[s / 4][s % 4], acc, 0, 0, 0);
            if (s < NV) {
                store_one(next, s);
                load_one(next, s);
                if (s == NV - 1) in_order();
            }
#pragma unroll
            for (int g = 0; g < G; ++g)
                if (s == (NV + g > 4 * g + 3 ? NV + g : 4 * g + 3)) read_group(g);
            __builtin_amdgcn_sched_barrier(0);
        }
        end_loads();
    }
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[s / 4][s % 4], fb[s / 4][s % 4], acc, 0, 0, 0);

    // ---------------- the four sums, the epilogue ----------------
    if (nepi && tid < 32) {
        if (Dk.nsteps) {
            const float v = conv_derived_value(d_in, Dk);
#pragma unroll
            for (int e = 0; e < CONV_MAX_EPI; ++e)
                if (e == (int)Dk.step) e_reg[e] = v;
        }
#pragma unroll
        for (int e = 0; e < CONV_MAX_EPI; ++e)
            if (e < nepi) Es[e * 32 + tid] = e_reg[e];
    }
    static_assert(16 * 64 <= conv_quad_wave_floats<BK>(), "a wave's sums replace its tiles");
    in_order();
    f32x4* const red = reinterpret_cast<f32x4*>(As);
#pragma unroll
    for (int q = 0; q < 4; ++q) red[q * 64 + lane] = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    __syncthreads();
    auto quarter_of = [&](int s) { return reinterpret_cast<const f32x4*>(pool + s * conv_quad_wave_floats<BK>())[kw * 64 + lane]; };
    f32x4 sum = quarter_of(0);
#pragma unroll
    for (int s = 1; s < 4; ++s) sum += quarter_of(s);
    if constexpr (SHARED) {
        // A slice leaves its sums in memory; the block that arrives last at the tile's counter, which it sets back, adds all of them in
        // their order. No block waits for another.
        const int tile = tile_m * region.tiles_n + tile_n;
        const __amdgpu_buffer_rsrc_t p_rsrc = make_rsrc(reinterpret_cast<const char*>(partial) + (size_t)tile * (size_t)P.slices * TILE, (uint32_t)P.slices * TILE);
        buffer_store_x4_agent(sum, p_rsrc, (uint32_t)tid * 16u, (uint32_t)slice * TILE);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");               // the sums have reached memory
        __syncthreads();
        if (tid == 0) {
            const uint32_t n = __hip_atomic_fetch_add(arrivals + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (n + 1u == (uint32_t)P.slices) __hip_atomic_store(arrivals + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            Rs[0] = (int)n;
        }
        __syncthreads();
        if (Rs[0] + 1 != P.slices) return;
        f32x4 q[CONV_MAX_SHARES];                                       // requested together; beyond the last slice the loads read zeros, which are not added
#pragma unroll
        for (int s = 0; s < CONV_MAX_SHARES; ++s) q[s] = buffer_load_x4_agent(p_rsrc, (uint32_t)tid * 16u, (uint32_t)s * TILE);
        sum = q[0];
#pragma unroll
        for (int s = 1; s < CONV_MAX_SHARES; ++s)
            if (s < P.slices) sum += q[s];
    }
    if constexpr (STRIDED) {
        static_assert(B_LOADS == QUAD_B_COLUMNS, "the strides' places are free there");
        const int n = n0 + l32;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int m = m0 + 8 * kw + 4 * half + v, b = magic_div(m, P.howo_magic, P.howo_shift), r2 = m - b * (P.Ho * P.Wo);
            const int ho = magic_div(r2, P.wo_magic, P.wo_shift), wo = r2 - ho * P.Wo;
            const uint32_t at = (uint32_t)(b * Pk.ws_r + ho * Pk.ws_s + wo * Pk.ws_c + n * Pk.ws_n) * 4u;
            buffer_store_x1(sum[v], o_rsrc, m < P.M && n < P.N ? at : CONV_OOB);
        }
        return;
    }
    float y[4] = {sum[0], sum[1], sum[2], sum[3]};
    conv_straight_steps<4>(y, quarter, (P.flags >> 20) & 31u, (int)((P.flags >> 12) & 15u) - 1, Es, 32, l32, [&]() {
        quarter_tile([&](int v, uint32_t vo, uint32_t so) { buffer_store_x1(y[v], make_rsrc(epi.p[CONV_MAX_EPI - 1], P.out_bytes), vo, so); });
    });
    quarter_tile([&](int v, uint32_t vo, uint32_t so) { buffer_store_x1(y[v], o_rsrc, vo, so); });
}
