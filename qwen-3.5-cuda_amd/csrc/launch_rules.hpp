// Launch shapes and the index arithmetic that kernels derive from them, where the two have to agree. Plain C++ (no
// HIP), so that a test walks them on the host over the sizes the entry points accept.
#pragma once

#include <cstddef>
#include <cstdint>

namespace qk {

// Grid of the chunked GDN recurrence's prep (csrc/gdn_chunk.hip): x = chunk; y = the workgroup's first value head h0,
// of which it takes h0, h0 + step, ... < value_heads. Value head h reads key head h % key_heads, and step is a multiple
// of key_heads or covers every head, so a workgroup's heads share one key head; the workgroups with y < key_heads write
// that head's K and Q out. y < heads <= value_heads: no workgroup starts past the last value head, also where
// value_heads is no multiple of key_heads.
// A value head's share is a third of a workgroup's serial chain: while one workgroup per (chunk, value head) has a CU
// to itself, every value head has its own (both launches, 64 tokens 20.0 -> 16.2 us, 128 24.1 -> 20.7, 400 38.9 -> 36.3;
// two to a CU gains nothing, 777 tokens 52.1 -> 52.9).
constexpr int kSpreadGroups = 256;
struct PrepGrid {
    int heads, step;
};
constexpr PrepGrid prep_grid(int chunks, int key_heads, int value_heads) {
    if (static_cast<int64_t>(chunks) * value_heads <= kSpreadGroups) return {value_heads, value_heads};
    return {key_heads < value_heads ? key_heads : value_heads, key_heads};
}

// Whether a lane's byte offset into a K-quant matrix's rows (csrc/gemm.hip), row * blocks of a row * block bytes and the
// block's own, stays below 2^32: Q4_K offsets may start at the matrix's first row (the 128 x 256 tiles), Q6_K ones at
// the first of a workgroup's rows, of which no tile has more than kGemmTileRows.
constexpr int kGemmTileRows = 256;
constexpr bool gemm_offsets_fit(bool from_first_row, int block_bytes, int M, int K) {
    const uint64_t rows = from_first_row || M < kGemmTileRows ? M : kGemmTileRows;
    return rows * static_cast<uint64_t>(K / 256) * static_cast<uint64_t>(block_bytes) < (uint64_t{1} << 32);
}

// Whether n floats at a and m floats at b share a byte. Calls that stand in for a sequence of launches, in which an
// output may replace an input that the sequence has finished with, run as that sequence where the two overlap.
inline bool floats_overlap(const float* a, size_t n, const float* b, size_t m) {
    const auto x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x < y + 4 * m && y < x + 4 * n;
}

}  // namespace qk
