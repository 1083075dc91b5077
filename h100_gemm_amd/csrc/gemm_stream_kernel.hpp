// gemm_stream_kernel.hpp -- gfx950 GEMM kernel for the thinnest decode shapes (M <= 64):
//
//   C[M,N] = A[M,K] . B[N,K]^T     one pass over B, one kernel, no workspace
//
// B (the weights) is read exactly once from HBM and that read is the whole cost, so the
// kernel is a set of independent streams, one per wave:
//   * a workgroup owns BN = 8, 16, 24 or 32 rows of B (columns of C) over all of K.  A CU takes in
//     ~26 GB/s whatever it keeps in flight, so BN is the narrowest that keeps N / BN workgroups
//     within one round of the CUs (stream_time_us in the kernel table): 1 x 4096 x 4096 with 32
//     columns on 128 workgroups 9.2 us (3.6 TB/s), with 16 on 256 7.1 (4.7); 1 x 2048 x 4096 with 8
//     5.4, 16 x 6144 x 4096 with 24 10.2 (32: 11.3).  Narrower still reads more of A, which every
//     workgroup walks whole: 16 x 8192 x 8192 with 32 21.9 us, with 16 24.0, with 8 30.2;
//   * its four waves split K between them, 64-deep slab by slab (wave w takes slabs
//     w, w+4, ...), so the workgroup as a whole walks 512 contiguous bytes of every row;
//   * each wave has a private ring of NS stages in LDS, filled by direct-to-LDS buffer
//     loads (B rows and the matching k range of A, 128-byte rows, XOR-swizzled) and
//     drained by its own MFMAs (32x32x16 with 24 or 32 columns, 16x16x32 with fewer); a wave
//     waits only on its own `vmcnt`, there is no barrier in the loop, and NS-1 slabs per wave
//     are always in flight (narrow stages are small: rings of five where 32 columns have three);
//   * workgroup b starts its walk over K at slab 37*b mod K/64 and wraps around: with every
//     workgroup at the same k at the same time, all requests in flight would share their
//     low address bits (rows are K*2 bytes apart) and crowd a few HBM channels; staggered
//     starts measured 6.7 TB/s against 4.7 TB/s for the same bytes;
//   * the four partial fp32 tiles are added in wave order through LDS (a fixed order:
//     results are reproducible), rounded once and stored.
// A is re-read by every workgroup; it is at most 64 x K and stays in L2.
// Rows of A past M and rows of B past N are never fetched (the buffer descriptors end at
// the last valid row; out-of-range lanes load nothing that reaches a stored element).
// The reference has no counterpart: its kernels assert M % 128 == 0 (matmul_utils.cuh:362).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_kernel.hpp"
#include "gemm_mfma16_kernel.hpp"   // mfma_16x16x32
#include "splitk_common.hpp"

namespace mi {

template <int BM_, int NS_, int DT_, int BN_ = 32>
struct StreamConfig {
    static constexpr int BM = BM_, BN = BN_, NS = NS_, DT = DT_;
    static constexpr int NT = 256, NW = 4;
    static constexpr int ROWS = BM + BN;                     // rows of one stage: A then B
    static constexpr int STAGE = ROWS * 128;
    static constexpr int L = ROWS / 8;                       // load instructions per slab
    static constexpr int RING = NS * STAGE;                  // one wave's ring
    static constexpr int LDS_BYTES = NW * RING;
    static constexpr bool WIDE = BN > 16;                   // 32x32x16 MFMAs, else 16x16x32
    static constexpr int R = WIDE ? 32 : 16;                 // rows and columns of an MFMA block
    static constexpr int KS = WIDE ? 4 : 2;                  // MFMAs deep a slab is
    static constexpr int MI = (BM + R - 1) / R;              // MFMA blocks of A
    static_assert(BN == 32 || BN == 24 || BN == 16 || BN == 8, "columns of a workgroup: one MFMA block or part of one");
    static_assert(BM == 16 || BM % 32 == 0, "A block is half of or whole MFMA operands");
    static_assert(NS >= 2 && (NS - 1) * L <= 63, "vmcnt is a 6-bit counter");
    static_assert(RING >= MI * R * R * 4, "a ring holds the wave's fp32 partial tile");
    static_assert(LDS_BYTES <= 160 * 1024, "LDS budget of one CU");
};

// TRACE: the per-workgroup timing record (TraceRec; thread 0 is in wave 0, so the waits and the
// K units are that wave's) for launches that pass a trace buffer.
template <class Cfg, bool TRACE = false>
__global__ void __launch_bounds__(256) gemm_stream_kernel(const DecodeArgs p) {
    constexpr int BM = Cfg::BM, NS = Cfg::NS, DT = Cfg::DT;
    constexpr int L = Cfg::L, STAGE = Cfg::STAGE, RING = Cfg::RING, MI = Cfg::MI;
    constexpr int BN = Cfg::BN, R = Cfg::R, KS = Cfg::KS;
    constexpr bool WIDE = Cfg::WIDE;

    __shared__ __attribute__((aligned(128))) unsigned char lds[Cfg::LDS_BYTES];
    TraceRec<TRACE> tr;
    tr.begin();

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col0 = blockIdx.x * BN;
    const int M = p.M, N = p.N, K = p.K;
    const int KT = K / 64;                                   // slabs (K % 64 == 0 is a launch precondition)
    const int cnt = (KT - wave + 3) / 4;                     // slabs of this wave: wave, wave+4, ...

    const int rowsA = M < BM ? M : BM;
    const int rowsB = (N - col0) < BN ? (N - col0) : BN;
    const unsigned char* Ab = (const unsigned char*)p.A;
    const unsigned char* Bb = (const unsigned char*)p.B + (size_t)col0 * p.ldb * 2;
    const uint32_t bytesA = (uint32_t)((rowsA - 1) * p.lda + K) * 2u;
    const uint32_t bytesB = (uint32_t)((rowsB - 1) * p.ldb + K) * 2u;
    const __amdgpu_buffer_rsrc_t rsrcA = __builtin_amdgcn_make_buffer_rsrc((void*)Ab, 0, (int)bytesA, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcB = __builtin_amdgcn_make_buffer_rsrc((void*)Bb, 0, (int)bytesB, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcNone = __builtin_amdgcn_make_buffer_rsrc((void*)Ab, 0, 0, 0x00020000);

    // One load instruction fills 8 consecutive 128-byte rows of a stage: lane l lands on
    // chunk position l & 7 of row l >> 3 and fetches logical chunk (l & 7) ^ swz(row).
    const int lr = lane >> 3, lc = lane & 7;
    auto swz = [](int row) __attribute__((always_inline)) { return (row >> 1) & 7; };
    const uint32_t ring_base =
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds + (uint32_t)wave * RING;
    auto dma = [&](const __amdgpu_buffer_rsrc_t& rsrc, uint32_t voff, uint32_t dst) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                     :: "s"(dst), "v"(voff), "s"(rsrc) : "memory");
    };
    // B is read once: non-temporal, so that it does not push A (re-read by every workgroup) out of the L2s
    auto dma_nt = [&](const __amdgpu_buffer_rsrc_t& rsrc, uint32_t voff, uint32_t dst) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds"
                     :: "s"(dst), "v"(voff), "s"(rsrc) : "memory");
    };
    // this lane's byte offsets inside A and B for instruction q of a slab (k offset added later)
    uint32_t voff[L];
#pragma unroll
    for (int q = 0; q < L; ++q) {
        const int row = q * 8 + lr;                          // stage row: A rows first, then B rows
        const int chunk = lc ^ swz(row);
        voff[q] = q * 8 < BM ? (uint32_t)(row * p.lda + chunk * 8) * 2u
                             : (uint32_t)((row - BM) * p.ldb + chunk * 8) * 2u;
    }
    // slab i of this wave is slab (wave + 4*i + rot) mod KT of the matrix; `gs` follows the
    // slab about to be requested
    int gs = (int)(((unsigned)wave + blockIdx.x * 37u) % (unsigned)KT);
    auto dma_slab = [&](int i, int s) __attribute__((always_inline)) {
        const bool live = i < cnt;
        const uint32_t kb = (uint32_t)gs * 128u;
        gs += 4;
        while (gs >= KT) gs -= KT;
#pragma unroll
        for (int q = 0; q < L; ++q) {
            if (q * 8 < BM) dma(live ? rsrcA : rsrcNone, voff[q] + kb, ring_base + (uint32_t)(s * STAGE + q * 1024));
            else dma_nt(live ? rsrcB : rsrcNone, voff[q] + kb, ring_base + (uint32_t)(s * STAGE + q * 1024));
        }
    };

    // fragment reads: lane holds row (lane % R), k chunk ks * 64 / R + lane / R.  With BN = 32 and
    // BM = 16 the upper half of the A operand reads B rows, with BN = 8 the upper half of the B
    // operand repeats the lower: values that only reach elements of the accumulator that are
    // never stored.
    const int lrow = lane % R, lh = lane / R;
    const int lb = lrow < BN ? lrow : lrow - BN;                // (BN = 24, 8: the block's upper columns repeat the lower)
    int rd_a[KS], rd_b[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        rd_a[ks] = lrow * 128 + (((ks * (64 / R) + lh) ^ swz(lrow)) << 4);
        rd_b[ks] = lb * 128 + (((ks * (64 / R) + lh) ^ swz(lb)) << 4);
    }

    std::conditional_t<WIDE, f32x16_t, f32x4_t> acc[MI];
#pragma unroll
    for (int a = 0; a < MI; ++a)
#pragma unroll
        for (int e = 0; e < R * R / 64; ++e) acc[a][e] = 0.0f;

#pragma unroll
    for (int i = 0; i < NS - 1; ++i) dma_slab(i, i);

    const unsigned char* ring = lds + wave * RING;
    int s = 0;
    for (int i = 0; i < cnt; ++i) {
        // slab i of this wave has landed; its predecessor's fragments are in registers
        tr.wait_begin();
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((NS - 2) * L) : "memory");
        tr.wait_end();
        dma_slab(i + NS - 1, s == 0 ? NS - 1 : s - 1);
        const unsigned char* st = ring + s * STAGE;
        u32x4_t fa[MI][KS], fb[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
            for (int a = 0; a < MI; ++a) fa[a][ks] = *(const u32x4_t*)(st + a * R * 128 + rd_a[ks]);
            fb[ks] = *(const u32x4_t*)(st + BM * 128 + rd_b[ks]);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int a = 0; a < MI; ++a) {
                if constexpr (WIDE) acc[a] = mfma_32x32x16<DT>(fb[ks], fa[a][ks], acc[a]);
                else acc[a] = mfma_16x16x32<DT>(fb[ks], fa[a][ks], acc[a]);
            }
        s = s + 1 == NS ? 0 : s + 1;
    }
    // requests past K are still heading for the ring: drain before it is reused
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    tr.loop_end();

    // ---- add the four partial tiles in wave order, round, store ----
    // lane holds P[m][n .. n+3], m = R*a + lane % R, n = (256/R)*g + 4*(lane / R): the partial tile is
    // MI*R rows of BN columns
    float* part = (float*)(lds + wave * RING);
#pragma unroll
    for (int a = 0; a < MI; ++a)
#pragma unroll
        for (int g = 0; g < R * R / 256; ++g) {
            const float4 v = {acc[a][g * 4 + 0], acc[a][g * 4 + 1], acc[a][g * 4 + 2], acc[a][g * 4 + 3]};
            const int n = g * (256 / R) + lh * 4;
            if (BN >= R || n < BN) *(float4*)(part + (a * R + lrow) * BN + n) = v;
        }
    __syncthreads();
    constexpr int RP = 256 / (BN / 4);                       // rows of C a pass of the 256 threads covers
#pragma unroll
    for (int a = 0; a < (MI * R + RP - 1) / RP; ++a) {
        const int m = a * RP + tid / (BN / 4), n = tid % (BN / 4) * 4;
        if (tid >= RP * (BN / 4) || m >= MI * R) break;
        float4 sum = *(const float4*)((const float*)lds + m * BN + n);
#pragma unroll
        for (int w = 1; w < 4; ++w) {
            const float4 v = *(const float4*)((const float*)(lds + w * RING) + m * BN + n);
            sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
        }
        if (p.alpha != 1.0f || p.beta != 0.0f) {
            sum.x = mul_add_unfused(sum.x, p.alpha, p.beta);
            sum.y = mul_add_unfused(sum.y, p.alpha, p.beta);
            sum.z = mul_add_unfused(sum.z, p.alpha, p.beta);
            sum.w = mul_add_unfused(sum.w, p.alpha, p.beta);
        }
        if (m < M && col0 + n < N) {                         // N % 4 == 0 is a launch precondition
            u32x2_t w2;
            w2[0] = cvt_store2<DT>(sum.x, sum.y);
            w2[1] = cvt_store2<DT>(sum.z, sum.w);
            *(u32x2_t*)((unsigned char*)p.C + ((size_t)m * p.ldc + col0 + n) * 2) = w2;
        }
    }
    tr.finish(p.DB, cnt);
}

template <class Cfg>
hipError_t launch_stream_kernel(const DecodeArgs& a, hipStream_t stream) {
    return a.DB ? launch_kernel(gemm_stream_kernel<Cfg, true>, dim3((a.N + Cfg::BN - 1) / Cfg::BN), dim3(256), stream, a)
                : launch_kernel(gemm_stream_kernel<Cfg, false>, dim3((a.N + Cfg::BN - 1) / Cfg::BN), dim3(256), stream, a);
}

}  // namespace mi
