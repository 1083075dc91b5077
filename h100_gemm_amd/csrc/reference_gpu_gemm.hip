// reference_gpu_gemm.hip -- the order-preserving GPU GEMM the harness checks the GEMM kernels
// against.  It takes the place of reference_gpu_gemm / reference_gpu_gemm_kernel
// (reference.h:49-90), which the reference's own harness uses as golden
// (matmul_h100.cu.jinja:1043-1047), and keeps that kernel's contract: one fp32
// accumulator per C element fed in ascending k, nothing added for k >= K, stores are
// predicated on m < M and n < N, and C = (CType)(acc * alpha + beta) with beta a plain
// scalar.  acc * alpha and + beta are two separately rounded operations, as in the host
// version of the same formula (reference.h:40).
//
// The fp32 matrix instructions of depth ONE (v_mfma_f32_32x32x1 / 16x16x1 / 4x4x1) keep that
// order: each adds a single product to every accumulator, rounded to nearest even like an fma
// (and the product of two bf16 or fp16 values is exact in fp32, so that is the same number as a
// rounded product added), at twice the rate of the vector units' fma.  The bound is those
// instructions' rate, 64 flops per SIMD and cycle whatever their shape (157 TFLOP/s at 2.4 GHz).
//   * A wave owns 64 rows (m) x TN columns (n) of C: lane l holds row l of A and column l % TN of B,
//     and the instruction broadcasts one block of B's columns to all blocks of A's rows.  Both
//     operands are unpacked to fp32 in registers, eight k's at a time.
//   * The four waves of a workgroup share a ring of LDS stages of 64 k's, filled by direct-to-LDS
//     loads.  (Every lane loading its own row from memory, without LDS, ran 4096^3 in 1060 us but
//     costs 64 line accesses per load: 150 us at 1024 x 1024 x 4096, 380 at 3000 x 2000 x 1001.)
//   * TN is chosen so that every SIMD of the chip has a tile: the K products of an element are a
//     serial chain, 2 * TN cycles per k.
// 4096^3: 2.77 ms (49.6 TFLOP/s, vector fma) -> 1.12 ms (123); 512^3: 81 -> 8.7 us; 256 x 256 x 4096:
// 724 -> 51.  At 4096^3 the matrix units are busy 88 % of the time at 2.07 GHz, the rest is the unpacking.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/mi_gemm.h"
#include "gemm_kernel.hpp"

namespace {

using mi::u32x4_t;
typedef __attribute__((ext_vector_type(32))) float f32x32_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
struct __attribute__((packed, aligned(2))) Chunk16 { u32x4_t v; };      // 16 bytes at any 2-byte boundary

template <int DT>
__device__ __forceinline__ float elem(uint32_t word, int half) {
    if constexpr (DT == MI_DTYPE_BF16) {
        return __builtin_bit_cast(float, half ? word & 0xffff0000u : word << 16);
    } else {
        return (float)__builtin_bit_cast(_Float16, (uint16_t)(half ? word >> 16 : word));
    }
}

// R x R matrix instruction of depth one: 64 / R blocks of R rows of A against block ABID of B's
// columns.  Accumulator register 4*g + e of block b holds, in lane l, row m = b*R + l % R and
// column n = ABID*R + 8*g + 4*(l / 32) + e (R = 32), 4*(l / 16) + e (16), e (4).
template <int R> struct Mma;
template <> struct Mma<32> {
    typedef f32x32_t Acc;
    template <int ABID> static __device__ __forceinline__ Acc run(float b, float a, Acc c) {
        return __builtin_amdgcn_mfma_f32_32x32x1f32(b, a, c, 1, ABID, 0);
    }
};
template <> struct Mma<16> {
    typedef f32x16_t Acc;
    template <int ABID> static __device__ __forceinline__ Acc run(float b, float a, Acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x1f32(b, a, c, 2, ABID, 0);
    }
};
template <> struct Mma<4> {
    typedef f32x4_t Acc;
    template <int ABID> static __device__ __forceinline__ Acc run(float b, float a, Acc c) {
        return __builtin_amdgcn_mfma_f32_4x4x1f32(b, a, c, 4, ABID, 0);
    }
};

template <int DT, int TN_>
struct GoldenConfig {
    static constexpr int TN = TN_;
    static constexpr int R = TN >= 32 ? 32 : TN >= 16 ? 16 : 4;             // block size of the matrix instruction
    static constexpr int NB = TN / R;                        // blocks of columns
    static constexpr int WM = TN >= 32 ? 2 : 1, WN = 4 / WM; // wave grid of a workgroup
    static constexpr int BM = 64 * WM, BN = TN * WN;
    static constexpr int ROWS = BM + BN;                     // rows of a stage: A's, then B's
    static constexpr int STAGE = ROWS * 128;
    static constexpr int NS = TN == 64 ? 2 : 3;              // stages of the ring
    static constexpr int LW = (ROWS / 8 + 3) / 4;            // load instructions per wave and unit
    static_assert(ROWS % 8 == 0 && (NS - 1) * LW <= 63 && NS * STAGE <= 80 * 1024, "two workgroups per CU");
};

template <int DT, int TN>
__global__ void __launch_bounds__(256)
golden_gemm_kernel(int M, int N, int K, const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                   uint16_t* __restrict__ C, float alpha, float beta) {
    using Cfg = GoldenConfig<DT, TN>;
    using Acc = typename Mma<Cfg::R>::Acc;
    constexpr int R = Cfg::R, NB = Cfg::NB, NS = Cfg::NS, LW = Cfg::LW, STAGE = Cfg::STAGE, BM = Cfg::BM;
    __shared__ __attribute__((aligned(128))) unsigned char lds[NS * STAGE];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
    int tm, tn;
    mi::tile_of_block<8>(blockIdx.x, gridDim.x, (M + BM - 1) / BM, (N + Cfg::BN - 1) / Cfg::BN, tm, tn);
    const int row0 = tm * BM, col0 = tn * Cfg::BN;
    const int m0 = row0 + wm * 64, n0 = col0 + wn * TN;

    Acc acc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int e = 0; e < R; ++e) acc[j][e] = 0.0f;

    // one k of the tile: the lane's element of its row of A and of its column of B
    auto mul = [&](float a, float b) __attribute__((always_inline)) {
        acc[0] = Mma<R>::template run<0>(b, a, acc[0]);
        if constexpr (NB > 1) acc[1] = Mma<R>::template run<1>(b, a, acc[1]);
    };

    // ---- whole 64-deep units of K through a ring of LDS stages ----
    // A unit is ROWS rows of 128 bytes, the 16-byte chunks of a row at chunk ^ ((row >> 1) & 7).
    // One load instruction fills 8 rows: lane l lands on position l & 7 of row l >> 3.  Rows past
    // M or N repeat the last one (their sums are not stored), so every load is inside the matrix.
    const int units = K / 64;
    auto swz = [](int row) __attribute__((always_inline)) { return (row >> 1) & 7; };
    if (units > 0) {
        const __amdgpu_buffer_rsrc_t rsrcA = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(A + (size_t)row0 * K), 0, (int)((uint32_t)((M - row0 < BM ? M - row0 : BM) * K) * 2u), 0x00020000);
        const __amdgpu_buffer_rsrc_t rsrcB = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(B + (size_t)col0 * K), 0, (int)((uint32_t)((N - col0 < Cfg::BN ? N - col0 : Cfg::BN) * K) * 2u), 0x00020000);
        const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
        uint32_t voff[LW], dst[LW];
        bool of_a[LW];
#pragma unroll
        for (int i = 0; i < LW; ++i) {
            // (where the instructions do not divide by four, the last ones are loaded twice)
            const int inst = wave * LW + i < Cfg::ROWS / 8 ? wave * LW + i : Cfg::ROWS / 8 - 1;
            const int r = inst * 8 + (lane >> 3);
            of_a[i] = inst * 8 < BM;
            const int last = of_a[i] ? M - row0 - 1 : N - col0 - 1;
            const int src = of_a[i] ? r : r - BM;
            voff[i] = (uint32_t)((src < last ? src : last) * K + ((lane & 7) ^ swz(r)) * 8) * 2u;
            dst[i] = lds_base + (uint32_t)inst * 1024u;
        }
        auto request = [&](int u, int stage) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < LW; ++i) {
                const uint32_t soff = (uint32_t)u * 128u;
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                             :: "s"(dst[i] + (uint32_t)(stage * STAGE)), "v"(voff[i]), "s"(of_a[i] ? rsrcA : rsrcB), "s"(soff)
                             : "memory");
            }
        };
        const int ra = wm * 64 + lane, rb = BM + wn * TN + lane % TN;
        // Chunk g (8 k's) is multiplied out of the floats fl[g & 1] while chunk g + 2 is read from LDS;
        // chunk g + 1 is unpacked in one go behind it.  The fp32 matrix instructions and the vector
        // ALU do not overlap, not even across waves, and every change from one to the other costs a
        // drained pipeline: unpacking two values between one k and the next took 34 cycles per k on
        // top of the matrix instructions, 16 values every 8 k's 22.  The order is pinned.
        u32x4_t raw_a[2], raw_b[2];
        float fl_a[2][8], fl_b[2][8];
        uint32_t rd_a[8], rd_b[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            rd_a[c] = (uint32_t)(ra * 128 + ((c ^ swz(ra)) << 4));
            rd_b[c] = (uint32_t)(rb * 128 + ((c ^ swz(rb)) << 4));
        }
        auto read = [&](int stage, int c) __attribute__((always_inline)) {
            raw_a[c & 1] = *(const u32x4_t*)(lds + stage * STAGE + rd_a[c]);
            raw_b[c & 1] = *(const u32x4_t*)(lds + stage * STAGE + rd_b[c]);
        };
        auto unpack = [&](int c) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                fl_a[c & 1][i] = elem<DT>(raw_a[c & 1][i >> 1], i & 1);
                fl_b[c & 1][i] = elem<DT>(raw_b[c & 1][i >> 1], i & 1);
            }
        };
        auto unit = [&](int u, int s) __attribute__((always_inline)) {
            const int next = s + 1 == NS ? 0 : s + 1;
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                if (c == 6 && u + 1 < units) {
                    // this wave holds its last chunk of the unit and its loads of the next one have
                    // landed; after the barrier that is so for every wave, and the stage is free
                    if (u + NS <= units) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((NS - 2) * LW) : "memory");
                    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    if (u + NS < units) request(u + NS, s);
                }
                if (c < 6) read(s, c + 2);
                else read(next, c - 6);                      // (behind the last unit: stale rows, never multiplied)
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 8; ++i) mul(fl_a[c & 1][i], fl_b[c & 1][i]);
                __builtin_amdgcn_sched_barrier(0);
                unpack(c + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
#pragma unroll
        for (int i = 0; i < NS; ++i)
            if (i < units) request(i, i);
        if (units >= NS) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((NS - 1) * LW) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        read(0, 0);
        read(0, 1);
        unpack(0);
        for (int u = 0; u < units; u += NS) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
                if (u + s < units) unit(u + s, s);
        }
    }
    // ---- what is left of the row: whole 16-byte pieces, then single elements, nothing past its end ----
    const int k0 = units * 64, left = K - k0;
    if (left > 0) {
        const uint16_t* pa = A + (size_t)(m0 + lane < M ? m0 + lane : M - 1) * K + k0;
        const uint16_t* pb = B + (size_t)(n0 + lane % TN < N ? n0 + lane % TN : N - 1) * K + k0;
        u32x4_t a[8], b[8];
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            if (left >= 8 * p + 8) {
                a[p] = ((const Chunk16*)(pa + 8 * p))->v;
                b[p] = ((const Chunk16*)(pb + 8 * p))->v;
            } else if (left > 8 * p) {
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const int k = 8 * p + 2 * w;
                    uint32_t va = 0, vb = 0;
                    if (k < left) va = pa[k], vb = pb[k];
                    if (k + 1 < left) va |= (uint32_t)pa[k + 1] << 16, vb |= (uint32_t)pb[k + 1] << 16;
                    a[p][w] = va;
                    b[p][w] = vb;
                }
            } else {
                a[p] = b[p] = u32x4_t{0u, 0u, 0u, 0u};
            }
        }
#pragma unroll
        for (int i = 0; i < 63; ++i)
            if (i < left) mul(elem<DT>(a[i >> 3][(i >> 1) & 3], i & 1), elem<DT>(b[i >> 3][(i >> 1) & 3], i & 1));
    }

    // ---- store: a lane holds groups of four consecutive n of one row ----
    const bool vec = (N & 3) == 0 && ((uintptr_t)C & 7u) == 0;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int g = 0; g < R / 4; ++g) {
            constexpr int GB = R * R / 256 > 0 ? R * R / 256 : 1;      // groups per block of rows: 4, 1, 1
            const int m = m0 + (g / GB) * R + lane % R;
            const int n = n0 + j * R + (g % GB) * 8 + (R == 4 ? 0 : 4 * ((lane / R) % (R / 4)));
            // (4x4: block lane / 4 of the one instruction, so the row is the lane)
            const int mm = R == 4 ? m0 + lane : m;
            if (mm >= M || n >= N) continue;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = mi::mul_add_unfused(acc[j][4 * g + e], alpha, beta);
            uint16_t* dst = C + (size_t)mm * N + n;
            const mi::u32x2_t w = {mi::cvt_store2<DT>(v[0], v[1]), mi::cvt_store2<DT>(v[2], v[3])};
            if (vec) {
                *(mi::u32x2_t*)dst = w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) dst[e] = (uint16_t)(w[e >> 1] >> ((e & 1) * 16));
            }
        }
}

template <int DT, int TN>
hipError_t launch_golden(int M, int N, int K, const void* A, const void* B, void* C, float alpha, float beta,
                         hipStream_t stream) {
    using Cfg = GoldenConfig<DT, TN>;
    const long long tiles = (long long)((M + Cfg::BM - 1) / Cfg::BM) * ((N + Cfg::BN - 1) / Cfg::BN);
    // (the status of this launch, not an error some earlier call of the process left behind)
    return mi::launch_kernel(golden_gemm_kernel<DT, TN>, dim3((unsigned)tiles), dim3(256), stream, M, N, K,
                             (const uint16_t*)A, (const uint16_t*)B, (uint16_t*)C, alpha, beta);
}

// Columns of a wave's tile.  Every workgroup puts one wave on each SIMD of a CU, so a launch takes
// K * max(serial chain of one tile, workgroups of the busiest CU * issue time of one tile), and narrow
// tiles trade matrix-unit efficiency (fewer matrix instructions per value unpacked) for a
// shorter chain and more CUs at work.  Nanoseconds per k, measured: `chain` on 256 x 256 x 4096
// (one wave per SIMD), `issue` on 2048^3 and 4096^3 (all SIMDs busy).  4096^3 in us, TN = 64 / 32 / 16 /
// 8 / 4: 1121 / 1194 / 1305 / 1555 / 2196; 1024^3: 67 / 39 / 24.9 / 28.1 / 38.4; 512^3: 35.6 / 21.0 / 13.2 /
// 9.8 / 8.7; 1500^3: 106 / 109 / 91.0 / 91.5 / 117.
int columns_per_wave(int M, int N, int cus) {
    static const struct { int tn, bm, bn; double chain, issue; } kinds[] = {
        {64, 128, 128, 62.1, 68.4}, {32, 128, 64, 34.7, 36.0}, {16, 64, 64, 20.7, 19.3}, {8, 64, 32, 14.2, 11.5}, {4, 64, 16, 12.4, 8.1}};
    int best = 0;
    double best_t = 0.0;
    for (const auto& k : kinds) {
        const long long wgs = (long long)((M + k.bm - 1) / k.bm) * ((N + k.bn - 1) / k.bn);
        const double issue = (double)((wgs + cus - 1) / cus) * k.issue;
        const double t = issue > k.chain ? issue : k.chain;
        if (best == 0 || t < best_t) {
            best = k.tn;
            best_t = t;
        }
    }
    return best;
}

template <int DT>
hipError_t launch_dtype(int M, int N, int K, const void* A, const void* B, void* C, float alpha, float beta,
                        int cus, hipStream_t stream) {
    switch (columns_per_wave(M, N, cus)) {
        case 64: return launch_golden<DT, 64>(M, N, K, A, B, C, alpha, beta, stream);
        case 32: return launch_golden<DT, 32>(M, N, K, A, B, C, alpha, beta, stream);
        case 16: return launch_golden<DT, 16>(M, N, K, A, B, C, alpha, beta, stream);
        case 8: return launch_golden<DT, 8>(M, N, K, A, B, C, alpha, beta, stream);
        default: return launch_golden<DT, 4>(M, N, K, A, B, C, alpha, beta, stream);
    }
}

}  // namespace

namespace mi {
hipError_t launch_reference_gpu_gemm(int dtype, int M, int N, int K, const void* A, const void* B,
                                     void* C, float alpha, float beta, int cus, hipStream_t stream) {
    return dtype == MI_DTYPE_BF16 ? launch_dtype<MI_DTYPE_BF16>(M, N, K, A, B, C, alpha, beta, cus, stream)
                                  : launch_dtype<MI_DTYPE_FP16>(M, N, K, A, B, C, alpha, beta, cus, stream);
}
}  // namespace mi
