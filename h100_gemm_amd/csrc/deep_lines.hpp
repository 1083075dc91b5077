// deep_lines.hpp -- where the loads of the deep-ring kernel (gemm_deep_kernel.hpp) go: plain arithmetic, for the kernel
// and for a host program that walks over it.
//
// A tile of an operand is `rows` rows of `ld` elements, K of them multiplied (K % 8 == 0), in 16-byte chunks.  Plain: slab t of a
// row is its 8 chunks from 8 * t on.  Lines: slab t is the row's t-th 128-byte line, counted from the line that
// holds its first element; `mis` bytes lie between the start of the first row's line, where the descriptor starts,
// and that row.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define MI_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define MI_HOST_DEVICE inline
#endif

namespace mi {

// past the end of every descriptor (an operand's 256 rows end below it): no access, zeros
constexpr uint32_t kDeepNowhere = 0x80000000u;

// where chunk c of a row is kept among the row's eight in LDS: at c ^ deep_swizzle(row)
MI_HOST_DEVICE int deep_swizzle(int row) { return (row >> 1) & 7; }

// chunks between the start of the row's 128-byte line and its first element (rows r and r + 16 have the same:
// 16 rows of whole chunks are whole lines)
MI_HOST_DEVICE int deep_phase(uint32_t mis, int row, int ld) { return (int)(((mis + (uint32_t)(row * ld) * 2u) >> 4) & 7u); }

// bytes of a descriptor: up to the last element of the last row
MI_HOST_DEVICE uint32_t deep_bytes(uint32_t mis, int rows, int ld, int K) { return mis + (uint32_t)((rows - 1) * ld + K) * 2u; }

// byte of chunk c (0 .. 7) of slab 0 of a row.  A row past the operand's last has none: rounded down to its line, the first
// one's start can lie below the descriptor's end, and whether the K offset a load adds in its scalar operand takes part in the
// range check is not something to rely on.
MI_HOST_DEVICE uint32_t deep_chunk_offset(bool lines, uint32_t mis, int row, int rows, int ld, int c) {
    if (lines && row >= rows) return kDeepNowhere;
    const uint32_t start = (uint32_t)(row * ld) * 2u + mis;
    return (lines ? start & ~127u : start) + (uint32_t)c * 16u;
}

// lines: chunks from chunk c of slab 0 to the row's end; more than K / 8: the chunk lies in front of the row
MI_HOST_DEVICE int deep_chunks_left(uint32_t mis, int row, int ld, int K, int c) { return K / 8 + deep_phase(mis, row, ld) - c; }

// lines: whether that chunk of slab t lies inside its row (`front`: t may be 0)
MI_HOST_DEVICE bool deep_chunk_inside(int left, int t, int K, bool front) { return left > 8 * t && !(front && left > K / 8); }

// slabs the walk over K requests, and the first of them that may reach past a row's end
MI_HOST_DEVICE int deep_slabs(bool lines, int K) { return (K + 63) / 64 + (lines ? 1 : 0); }
MI_HOST_DEVICE int deep_whole_slabs(bool lines, int K) { return lines ? K / 64 : (K + 63) / 64; }

}  // namespace mi
