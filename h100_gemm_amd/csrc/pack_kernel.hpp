// pack_kernel.hpp -- copies A and B into a workspace whose rows start on 128-byte lines.
//
// A row pitch that is no multiple of 128 bytes (K % 64 != 0) makes every 128-byte piece that the
// tiled kernels load straddle two cache lines, and each line is fetched by two consecutive K
// steps; the K loop then runs at 0.69-0.83 of its rate on whole lines.  The copy reads each
// operand once and writes it once; past a certain size that is less than what it saves (the rule
// is choose_packing in mi_gemm.hip).  Rows are padded with zeros to a whole number of 64-deep slabs:
// zero products at the end of every sum, so C is bit for bit the same.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_kernel.hpp"

namespace mi {

struct PackArgs {
    const uint16_t* src[2];  // the operands to copy (one of them: rows_first covers all)
    uint16_t* out;           // rows of the first, then of the second, each of 8 * chunks elements
    uint32_t rows_first;
    uint32_t total;          // 16-byte chunks of the copy: rows * chunks
    uint32_t chunks;         // ... of a row
    int K;
};
constexpr int kPackChunks = 4;           // 16-byte chunks per thread, their loads in flight together

// Bound by memory: each byte of A and B read once (streamed past the caches), written once.
__global__ void __launch_bounds__(256) pack_operands_kernel(const PackArgs p) {
    struct __attribute__((packed, aligned(2))) Chunk { u32x4_t v; };       // 16 bytes at any 2-byte boundary
    u32x4_t v[kPackChunks];
    const uint32_t first = blockIdx.x * (256u * kPackChunks) + threadIdx.x;
#pragma unroll
    for (int i = 0; i < kPackChunks; ++i) {
        const uint32_t idx = first + 256u * i;
        v[i] = u32x4_t{0u, 0u, 0u, 0u};
        if (idx >= p.total) continue;
        const uint32_t row = idx / p.chunks;
        const int k = (int)(idx - row * p.chunks) * 8;
        const uint16_t* src = (row < p.rows_first ? p.src[0] + (size_t)row * p.K : p.src[1] + (size_t)(row - p.rows_first) * p.K) + k;
        if (k + 8 <= p.K) {
            v[i] = ((const Chunk*)src)->v;
        } else {
            // the end of the row: element by element, nothing past it
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (k + e < p.K) v[i][e >> 1] |= (uint32_t)src[e] << (16 * (e & 1));
        }
    }
#pragma unroll
    for (int i = 0; i < kPackChunks; ++i) {
        const uint32_t idx = first + 256u * i;
        if (idx < p.total) ((u32x4_t*)p.out)[idx] = v[i];
    }
}

}  // namespace mi
