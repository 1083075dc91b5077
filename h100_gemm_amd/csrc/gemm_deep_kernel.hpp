// gemm_deep_kernel.hpp -- gfx950 tiled GEMM kernel on a deep ring of whole cache lines:
//
//   C[M,N] = A[M,K] . B[N,K]^T     any M and N; K % 8 == 0, K >= 128, A and B on 16-byte boundaries
//
// For outputs of up to a few tiles per CU.  With one workgroup on a CU nothing hides its loads
// but the loads themselves, and the two stages of the 16x16x32 kernel leave a load one K step to land:
// less than the way to memory.  Here the ring has as many 64-deep slabs as fit the LDS (128x128: five
// of 32 KB), and a slab has NS - 1 steps.
//   * 2 x 2 waves over the tile, one barrier per K step, in its middle: the slab the second half reads
//     from has landed, and every wave holds all it needs of the slab before, whose stage takes the
//     request NS slabs ahead.  Fragment reads are dealt out over the first three quarters of a half
//     step's MFMAs, loads over the second half's.  (Waves that take 32-deep halves of every slab instead of quarters of
//     the tile read a quarter less LDS, and lost 5-9 %: the loads bind, not the LDS.)
//   * LINES, K % 64 != 0: rows start inside a 128-byte line, and loading 64 elements of every row a step
//     touches two lines a row and halves what a CU takes in from its L2 (59 -> 30 bytes a clock, measured
//     with loads alone).  The ring therefore holds whole lines of every row, each loaded once: K step t
//     of a row lies in its lines t and t + 1, the row's phase (chunks between the start of its line and its
//     first element) says where.  Rows r and r + 16 have the same phase, as 16 rows of K % 8 == 0 elements are
//     whole lines, and a lane reads fragments of rows 16 apart only: the phase costs one LDS address
//     per lane and half step, no work in the loop.  A slab must have landed a step earlier, so
//     the ring hides one step less.  Chunks outside their row (in front of it in line 0, past K in the last ones) are
//     never read from memory: their lanes load from past the descriptor's end and get the zeros that fill up K.
// Bound by what a CU takes in: 128x128 on 64 CUs 0.275 us a step, its loads alone 0.2515, its MFMAs alone 0.217; on all
// 256 the L2s' fills bind (2048x2048: 0.40 / 0.334 / 0.242).
// Against the kernels these calls took before, us with operands from memory / in the caches: 1472x3264x1216 22.0 / 17.6 -> 16.3 /
// 14.0, 1536x1536x1536 11.8 / 11.9 -> 11.0 / 10.0, 896x1408x1536 10.0 / 9.6 -> 8.7 / 7.9, 640x256x256 3.3 / 3.1 ->
// 2.9 / 2.8; with K % 64 != 0: 976x2808x2712 41.7 / 31.8 -> 24.1 / 22.5, 3008x968x2224 31.2 / 27.1 -> 23.6 / 18.8.
// The reference has no counterpart: its kernels use one tile size (matmul_utils.cuh:362).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

#include "deep_lines.hpp"
#include "gemm_kernel.hpp"
#include "gemm_mfma16_kernel.hpp"   // mfma_16x16x32, f32x4_t
#include "splitk_common.hpp"        // TraceRec

namespace mi {

// f(integral_constant<int, FIRST>) ... f(integral_constant<int, FIRST + N - 1>), in order
template <int FIRST, class F, int... Is>
__device__ __forceinline__ void deep_for_each(F&& f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, FIRST + Is>{}), ...);
}
template <int N, int FIRST = 0, class F>
__device__ __forceinline__ void deep_for(F&& f) {
    deep_for_each<FIRST>(f, std::make_integer_sequence<int, N>{});
}

template <int BM_, int BN_, int NS_, int GROUP_, int DT_, bool LINES_, int OCC_ = 1>
struct DeepConfig {
    static constexpr int BM = BM_, BN = BN_, WM = 2, WN = 2, NS = NS_, GROUP = GROUP_, DT = DT_;
    static constexpr bool LINES = LINES_;
    static constexpr int NW = 4, NT = NW * 64;
    static constexpr int OCC = OCC_;                                  // workgroups per CU the registers are sized for
    static constexpr int TM = BM / WM, TN = BN / WN;
    static constexpr int MI = TM / 16, NI = TN / 16;
    static constexpr int LA = BM / (8 * NW), LB = BN / (8 * NW);      // load instructions per wave and slab
    static constexpr int L = LA + LB;
    static constexpr int A_STAGE = BM * 128, STAGE = (BM + BN) * 128;
    static constexpr int LDS_BYTES = NS * STAGE;
    static constexpr int NMMA = MI * NI, NFR = MI + NI;
    static constexpr int AHEAD = LINES ? 2 : 1;                       // slabs past the current one a step reads from
    static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "tile rows divide over the waves");
    static_assert(TM % 16 == 0 && TN % 16 == 0, "wave tile must be a multiple of 16x16");
    static_assert(NS >= AHEAD + 1 && (NS - AHEAD) * L <= 63, "vmcnt is a 6-bit counter");
    static_assert(LDS_BYTES * OCC <= 160 * 1024, "LDS budget of one CU");
    static_assert(BM * BN * 2 <= LDS_BYTES, "the epilogue stages the C tile in the ring");
};

// SPLITK: the workgroup multiplies one piece of K of its tile (blockIdx.y) and leaves fp32 sums in the workspace.
// TRACE: the per-workgroup timing record (TraceRec) for launches that pass a trace buffer.
template <class Cfg, bool TRACE = false, bool SPLITK = false>
__global__ void __launch_bounds__(Cfg::NT) __attribute__((amdgpu_waves_per_eu(Cfg::OCC, Cfg::OCC)))
gemm_deep_kernel(const GemmArgs p) {
    constexpr int BM = Cfg::BM, BN = Cfg::BN, WN = Cfg::WN, NS = Cfg::NS, DT = Cfg::DT;
    constexpr int MI = Cfg::MI, NI = Cfg::NI, LA = Cfg::LA, LB = Cfg::LB, L = Cfg::L;
    constexpr int A_STAGE = Cfg::A_STAGE, STAGE = Cfg::STAGE;
    constexpr int NMMA = Cfg::NMMA, NFR = Cfg::NFR, TM = Cfg::TM, TN = Cfg::TN;
    constexpr bool LINES = Cfg::LINES;
    constexpr int AHEAD = Cfg::AHEAD;

    __shared__ __attribute__((aligned(128))) unsigned char lds[Cfg::LDS_BYTES];
    TraceRec<TRACE> tr;
    tr.begin();

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    int tm, tn;
    tile_of_block<Cfg::GROUP>(blockIdx.x, gridDim.x, p.tiles_m, p.tiles_n, tm, tn);
    const int row0 = tm * BM, col0 = tn * BN;
    // split-K: the K range [k0, k0 + K) of the tile; k_per_split is a multiple of 64
    const int k0 = SPLITK ? (int)blockIdx.y * p.k_per_split : 0;
    const int M = p.M, N = p.N;
    const int K = SPLITK ? ((p.K - k0) < p.k_per_split ? (p.K - k0) : p.k_per_split) : p.K;
    const int KT = (K + 63) / 64;                            // K steps
    const int slabs = deep_slabs(LINES, K);

    const int rowsA = (M - row0) < BM ? (M - row0) : BM;
    const int rowsB = (N - col0) < BN ? (N - col0) : BN;
    const unsigned char* Ab = (const unsigned char*)p.A + ((size_t)row0 * p.lda + k0) * 2;
    const unsigned char* Bb = (const unsigned char*)p.B + ((size_t)col0 * p.ldb + k0) * 2;
    // LINES: descriptors start on the 128-byte line that holds the first row's first element
    const uint32_t misA = LINES ? (uint32_t)(uintptr_t)Ab & 127u : 0u, misB = LINES ? (uint32_t)(uintptr_t)Bb & 127u : 0u;
    // descriptors end at the last element (of this K range) of the last valid row
    const uint32_t bytesA = deep_bytes(misA, rowsA, p.lda, K);
    const uint32_t bytesB = deep_bytes(misB, rowsB, p.ldb, K);
    const __amdgpu_buffer_rsrc_t rsrcA = __builtin_amdgcn_make_buffer_rsrc((void*)(Ab - misA), 0, (int)bytesA, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcB = __builtin_amdgcn_make_buffer_rsrc((void*)(Bb - misB), 0, (int)bytesB, 0x00020000);

    // load instruction d of A (of B) of this wave fills rows (wave * LA + d) * 8 .. + 7
    const int lr = lane >> 3, lc = lane & 7;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
    constexpr int GA = LA % 4 == 0 ? 4 : LA % 3 == 0 ? 3 : LA % 2 == 0 ? 2 : 1;
    constexpr int GB = LB % 4 == 0 ? 4 : LB % 3 == 0 ? 3 : LB % 2 == 0 ? 2 : 1;
    uint32_t voffs[L];
#pragma unroll
    for (int d = 0; d < L; ++d) {
        const bool a = d < LA;
        const int e = a ? d : d - LA;
        const int row = (wave * (a ? LA : LB) + e) * 8 + lr;
        voffs[d] = deep_chunk_offset(LINES, a ? misA : misB, row, a ? rowsA : rowsB, a ? p.lda : p.ldb, lc ^ deep_swizzle(row)) -
                   (uint32_t)((e % (a ? GA : GB)) * 1024);
    }
    // LINES: chunk and phase repeat every 16 rows, so there are two of each operand, for even and odd e
    int left[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int row = (wave * (a ? LA : LB) + e) * 8 + lr;
            left[a][e] = deep_chunks_left(a ? misA : misB, row, a ? p.lda : p.ldb, K, lc ^ deep_swizzle(row));
        }
    auto dma = [](__amdgpu_buffer_rsrc_t rsrc, uint32_t voff, uint32_t soff, uint32_t dst) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :: "s"(dst), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
    };
    // same M0 as the load before, LDS (and global) address IMM bytes further
    auto dma_next = [](__amdgpu_buffer_rsrc_t rsrc, uint32_t voff, uint32_t soff, auto imm_c) __attribute__((always_inline)) {
        asm volatile("buffer_load_dwordx4 %0, %1, %2 offen offset:%3 lds"
                     :: "v"(voff), "s"(rsrc), "s"(soff), "n"(decltype(imm_c)::value) : "memory");
    };
    // load d of slab t into stage s.  Plain: the slab lies inside every row, and the K offset is the load's scalar one.
    // Otherwise (EDGE) it goes into the lanes' offsets, and chunks outside their row, and slabs past the last one, come
    // from nowhere (FRONT: slab 0, where some lie in front of their row).
    auto load_one = [&](int t, auto s_c, auto d_c, auto edge_c, auto front_c) __attribute__((always_inline)) {
        constexpr int s = decltype(s_c)::value, d = decltype(d_c)::value;
        constexpr bool edge = decltype(edge_c)::value, a = d < LA;
        constexpr int e = a ? d : d - LA, G = a ? GA : GB;
        uint32_t kb = (uint32_t)t * 128u;
        uint32_t vo = voffs[d];
        const __amdgpu_buffer_rsrc_t rs = a ? rsrcA : rsrcB;
        if constexpr (edge) {
            const bool ok = LINES ? deep_chunk_inside(left[a][e & 1], t, K, decltype(front_c)::value) : t < slabs;
            vo = ok ? vo + kb : kDeepNowhere;
            kb = 0;
        }
        const uint32_t dst = lds_base + (uint32_t)(s * STAGE + (a ? 0 : A_STAGE) + ((int)wave * (a ? LA : LB) + (e / G) * G) * 1024);
        if constexpr (e % G == 0) dma(rs, vo, kb, dst);
        else dma_next(rs, vo, kb, std::integral_constant<int, (e % G) * 1024>{});
    };

    // fragment reads: lane holds row (lane & 15) of a 16-row block, chunk 4*ks + (lane >> 4) of the K step;
    // LINES: chunk phase + 4*ks + (lane >> 4) of the two slabs t and t + 1
    const int l16 = lane & 15, q = lane >> 4;
    int rdA[2], rdB[2];
    bool upA[2], upB[2];
#pragma unroll
    for (int ph = 0; ph < 2; ++ph) {
        const int ga = (LINES ? deep_phase(misA, l16, p.lda) : 0) + 4 * ph + q;
        const int gb = (LINES ? deep_phase(misB, l16, p.ldb) : 0) + 4 * ph + q;
        upA[ph] = ga >= 8;
        upB[ph] = gb >= 8;
        rdA[ph] = (wm * TM + l16) * 128 + (((ga & 7) ^ deep_swizzle(l16)) << 4);
        rdB[ph] = A_STAGE + (wn * TN + l16) * 128 + (((gb & 7) ^ deep_swizzle(l16)) << 4);
    }

    u32x4_t fa[2][MI], fb[2][NI];
    f32x4_t acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto mma_one = [&](int ph, int idx) __attribute__((always_inline)) {
        const int i = idx / NI, j = (i & 1) ? NI - 1 - idx % NI : idx % NI;
        acc[i][j] = mfma_16x16x32<DT>(fb[ph][j], fa[ph][i], acc[i][j]);
    };
    // fragment r of half ph of the K step whose (first) slab is in stage s, in the order the MFMAs need them
    auto read_one = [&](auto s_c, int ph, int r) __attribute__((always_inline)) {
        constexpr int s = decltype(s_c)::value, n = (s + 1) % NS;
        if (r == 0 || r > NI) {
            const int i = r == 0 ? 0 : r - NI;
            const int base = LINES && upA[ph] ? n * STAGE : s * STAGE;
            fa[ph][i] = *(const u32x4_t*)(lds + base + rdA[ph] + i * 2048);
        } else {
            const int base = LINES && upB[ph] ? n * STAGE : s * STAGE;
            fb[ph][r - 1] = *(const u32x4_t*)(lds + base + rdB[ph] + (r - 1) * 2048);
        }
    };

    // One K step, t = s mod NS: slice 0 multiplies while slice 1's fragments are read; then, behind the barrier,
    // slice 1 multiplies while slice 0 of the next step is read and slab t + NS is requested.
    auto step = [&](int t, auto s_c, auto edge_c) __attribute__((always_inline)) {
        constexpr int s = decltype(s_c)::value;
        using S = std::integral_constant<int, s>;
        using SN = std::integral_constant<int, (s + 1) % NS>;
        deep_for<2>([&](auto ph_c) __attribute__((always_inline)) {
            constexpr int ph = decltype(ph_c)::value;
            constexpr bool last = ph == 1;
            if constexpr (last) {
                tr.wait_begin();
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((NS - 1 - AHEAD) * L) : "memory");
                tr.wait_end();
            }
            deep_for<NMMA>([&](auto idx_c) __attribute__((always_inline)) {
                constexpr int idx = decltype(idx_c)::value;
                mma_one(ph, idx);
                // (read r behind MFMA r * NMMA * 3 / (4 * NFR): over the first three quarters; load d behind d * NMMA / L: over
                // all.  Which of them this MFMA has is computed, not asked of each: every lambda is a function until it is
                // inlined, and ten times as many took the compiler four minutes a tile)
                constexpr int r0 = (idx * 4 * NFR + NMMA * 3 - 1) / (NMMA * 3), r1 = ((idx + 1) * 4 * NFR + NMMA * 3 - 1) / (NMMA * 3);
                constexpr int r_end = r1 < NFR ? r1 : NFR;
#pragma unroll
                for (int r = r0; r < r_end; ++r) {
                    if constexpr (last) read_one(SN{}, 0, r);
                    else read_one(S{}, 1, r);
                }
                if constexpr (last) {
                    constexpr int d0 = (idx * L + NMMA - 1) / NMMA, d1 = ((idx + 1) * L + NMMA - 1) / NMMA;
                    deep_for<d1 - d0, d0>([&](auto d_c) __attribute__((always_inline)) {
                        load_one(t + NS, S{}, d_c, edge_c, std::false_type{});
                    });
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
    };
    using T = std::true_type;
    using F = std::false_type;

    // ---- prologue: slabs 0 .. NS-1 ----
    deep_for<NS>([&](auto s_c) __attribute__((always_inline)) {
        deep_for<L>([&](auto d_c) __attribute__((always_inline)) {
            load_one(decltype(s_c)::value, s_c, d_c, T{}, std::integral_constant<bool, decltype(s_c)::value == 0>{});
        });
    });
    // the accumulators in AGPRs, zeroed while the first slabs are on their way
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) asm volatile("" : "+a"(acc[i][j]));
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((NS - AHEAD) * L) : "memory");
#pragma unroll
    for (int r = 0; r < NFR; ++r) read_one(std::integral_constant<int, 0>{}, 0, r);

    // ---- NS steps a trip (the stage a compile-time index); the last trips may request chunks past the rows' ends ----
    const int whole = deep_whole_slabs(LINES, K);            // slabs < whole lie inside every row
    int t = 0;
    for (; t + 2 * NS - 1 < whole; t += NS)
        deep_for<NS>([&](auto s_c) __attribute__((always_inline)) { step(t + decltype(s_c)::value, s_c, F{}); });
    for (; t < KT; t += NS)
        deep_for<NS>([&](auto s_c) __attribute__((always_inline)) {
            if (t + decltype(s_c)::value < KT) step(t + decltype(s_c)::value, s_c, T{});
        });
    // requests past the last slab are still heading for the ring: drain before C takes its place
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    tr.loop_end();

    // ---- epilogue ----
    // acc[i][j][e] of lane l is C[m][n], m = i*16 + (l & 15), n = j*16 + 4*(l >> 4) + e of the wave's TM x TN
    const int cn0 = col0 + wn * TN;
    if constexpr (SPLITK) {
        float* P = p.ws + ((size_t)blockIdx.y * M + row0) * N;
        const __amdgpu_buffer_rsrc_t rsrcP =
            __builtin_amdgcn_make_buffer_rsrc((void*)P, 0, (int)((uint32_t)(rowsA * N) * 4u), 0x00020000);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int m_loc = wm * TM + i * 16 + l16;
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const int n = cn0 + j * 16 + 4 * q;
                if (n < N)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[i][j]), rsrcP,
                                                           (uint32_t)(m_loc * N + n) * 4u, 0, 0);
            }
        }
    } else {
        unsigned char* Cb = (unsigned char*)p.C + (size_t)row0 * p.ldc * 2;
        const __amdgpu_buffer_rsrc_t rsrcC =
            __builtin_amdgcn_make_buffer_rsrc((void*)Cb, 0, (int)((uint32_t)(rowsA * p.ldc) * 2u), 0x00020000);
        constexpr int CPR = TN / 8;                          // 16-byte chunks per row of the wave tile
        constexpr bool POW2 = (CPR & (CPR - 1)) == 0;
        static_assert(CPR % 2 == 0, "C staging layout");
        // (the swizzle stays inside a row: CPR is a power of two, or a multiple of 4 or 2)
        auto cswz = [](int row) __attribute__((always_inline)) {
            return POW2 ? (row & (CPR - 1)) : CPR % 4 == 0 ? ((row >> 2) & 3) : ((row >> 2) & 1);
        };
        unsigned char* stg = lds + wave * (TM * TN * 2);
        constexpr int CH_ROWS = (TM % 32 == 0 && (32 * CPR) % 64 == 0) ? 32 : TM;
        auto epilogue = [&](auto scaled_c, auto whole_c) __attribute__((always_inline)) {
            constexpr bool SCALED = decltype(scaled_c)::value, WHOLE = decltype(whole_c)::value;
            const float alpha = p.alpha, beta = p.beta;
#pragma unroll
            for (int c = 0; c < TM / CH_ROWS; ++c) {
#pragma unroll
                for (int i = c * (CH_ROWS / 16); i < (c + 1) * (CH_ROWS / 16); ++i) {
                    const int row = i * 16 + l16;
#pragma unroll
                    for (int j = 0; j < NI; ++j) {
                        const int chunk = (j * 2 + (q >> 1)) ^ cswz(row);
                        u32x2_t w;
                        w[0] = cvt_store2<DT>(scale_acc<SCALED>(acc[i][j][0], alpha, beta), scale_acc<SCALED>(acc[i][j][1], alpha, beta));
                        w[1] = cvt_store2<DT>(scale_acc<SCALED>(acc[i][j][2], alpha, beta), scale_acc<SCALED>(acc[i][j][3], alpha, beta));
                        *(u32x2_t*)(stg + row * (TN * 2) + chunk * 16 + (q & 1) * 8) = w;
                    }
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                for (int r = 0; r < (CH_ROWS * CPR + 63) / 64; ++r) {
                    const int idx = c * (CH_ROWS * CPR) + r * 64 + lane;
                    if (CH_ROWS * CPR % 64 != 0 && idx >= (c + 1) * (CH_ROWS * CPR)) continue;
                    const int row = idx / CPR, rc = idx % CPR;
                    const u32x4_t v = *(const u32x4_t*)(stg + row * (TN * 2) + ((rc ^ cswz(row)) << 4));
                    const int m_loc = wm * TM + row;
                    const int n = cn0 + rc * 8;
                    const uint32_t off = ((uint32_t)m_loc * (uint32_t)p.ldc + (uint32_t)n) * 2u;
                    if constexpr (WHOLE) {
                        if (n < N) __builtin_amdgcn_raw_buffer_store_b128(v, rsrcC, off, 0, 2);      // non-temporal
                    } else if (m_loc < rowsA) {
                        if (n + 7 < N) {
                            __builtin_amdgcn_raw_buffer_store_b128(v, rsrcC, off, 0, 0);
                        } else {
#pragma unroll
                            for (int e = 0; e < 8; ++e)
                                if (n + e < N)
                                    __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(v[e >> 1] >> ((e & 1) * 16)), rsrcC, off + 2 * e, 0, 0);
                        }
                    }
                }
            }
        };
        // WHOLE leaves rows past M to the range check, so a tile's rows have to lie within 32-bit offsets (of 2^24 columns row
        // 128 is 2^32 bytes away and would come round into C below the descriptor's end)
        const bool whole_lines = ((p.ldc & 63) | (int)((uintptr_t)p.C & 127u)) == 0 && (uint64_t)p.ldc * (BM * 2) <= 0x80000000u;
        const bool scaled = p.alpha != 1.0f || p.beta != 0.0f;
        if (whole_lines) {
            if (scaled) epilogue(T{}, T{}); else epilogue(F{}, T{});
        } else {
            if (scaled) epilogue(T{}, F{}); else epilogue(F{}, F{});
        }
    }
    tr.finish(p.DB, KT);
}

template <class Cfg>
hipError_t launch_deep_kernel(const GemmArgs& args, hipStream_t stream) {
    const dim3 grid(args.tiles_m * args.tiles_n, args.splits);
    if (args.splits > 1)
        return args.DB ? launch_kernel(gemm_deep_kernel<Cfg, true, true>, grid, dim3(Cfg::NT), stream, args)
                       : launch_kernel(gemm_deep_kernel<Cfg, false, true>, grid, dim3(Cfg::NT), stream, args);
    return args.DB ? launch_kernel(gemm_deep_kernel<Cfg, true, false>, grid, dim3(Cfg::NT), stream, args)
                   : launch_kernel(gemm_deep_kernel<Cfg, false, false>, grid, dim3(Cfg::NT), stream, args);
}

}  // namespace mi
