// The loads of the deep-ring kernel, walked on the CPU with the kernel's own arithmetic (deep_lines.hpp): every
// chunk of every row is loaded once, and no load touches memory outside its row, whether or not the range
// check of a buffer load counts the scalar offset.
#include <stdint.h>
#include <stdio.h>

#include <vector>

#include "../../h100_gemm_amd/csrc/deep_lines.hpp"

namespace {

int faults = 0;

// `rows` of a tile of `tile` rows; K elements of rows of `ld` are multiplied, the first at byte `mis` of its line
void walk(bool lines, int tile, int rows, int ld, int K, uint32_t mis, int NS) {
    if (!lines) mis = 0;
    const int KT = (K + 63) / 64, slabs = mi::deep_slabs(lines, K), whole = mi::deep_whole_slabs(lines, K);
    const uint32_t bytes = mi::deep_bytes(mis, rows, ld, K);
    std::vector<int> loaded((size_t)rows * (K / 8));
    const char* what = nullptr;
    auto load = [&](int t, bool edge, bool front) {
        for (int row = 0; row < tile; ++row)
            for (int c = 0; c < 8; ++c) {
                uint32_t lane = mi::deep_chunk_offset(lines, mis, row, rows, ld, c), scalar = (uint32_t)t * 128u;
                if (edge) {
                    const bool ok = lines ? mi::deep_chunk_inside(mi::deep_chunks_left(mis, row, ld, K, c), t, K, front) : t < slabs;
                    lane = ok ? lane + scalar : mi::kDeepNowhere;
                    scalar = 0;
                }
                const bool by_sum = (uint64_t)lane + scalar + 16 <= bytes, by_lane = (uint64_t)lane + 16 <= bytes;
                const int64_t at = (int64_t)lane + scalar - mis - (int64_t)row * ld * 2;     // byte of the row
                const bool inside = row < rows && at >= 0 && at + 16 <= (int64_t)K * 2;
                if (by_sum != by_lane) what = "whether a load is made depends on the scalar offset";
                if ((by_sum || by_lane) && !inside) what = "a load outside its row";
                if (inside && by_sum) ++loaded[(size_t)row * (K / 8) + (size_t)(at / 16)];
            }
    };
    for (int s = 0; s < NS; ++s) load(s, true, s == 0);
    int t = 0;
    for (; t + 2 * NS - 1 < whole; t += NS)
        for (int s = 0; s < NS; ++s) load(t + s + NS, false, false);
    for (; t < KT; t += NS)
        for (int s = 0; s < NS; ++s)
            if (t + s < KT) load(t + s + NS, true, false);
    for (int n : loaded)
        if (n != 1) what = "a chunk not loaded, or more than once";
    if (what && faults++ < 20)
        fprintf(stderr, "%s, %d of %d rows of %d, K = %d, %u bytes into a line, %d stages: %s\n", lines ? "lines" : "plain", rows, tile, ld, K,
                mis, NS, what);
}

}  // namespace

int main() {
    for (int NS : {3, 4, 5, 6, 8})
        for (int rows : {1, 2, 7, 8, 31, 32}) {
            for (int k = 2; k < 4 * NS + 2; ++k) walk(false, 32, rows, 64 * k, 64 * k, 0, NS);
            for (int K = 128; K < 64 * (3 * NS + 2); K += K < 256 ? 8 : 72)
                for (uint32_t mis = 0; mis < 128; mis += 16) walk(true, 32, rows, K, K, mis, NS);
            // a piece of a longer K
            for (int K : {8, 120, 512, 640})
                for (uint32_t mis = 0; mis < 128; mis += 16) walk(true, 32, rows, 2568, K, mis, NS);
            for (int K : {128, 512, 640}) walk(false, 32, rows, 2560, K, 0, NS);
        }
    return faults != 0;
}
