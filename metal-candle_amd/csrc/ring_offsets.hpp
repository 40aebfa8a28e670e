// Offsets of buffer loads that a kernel computes once and then advances
// through soffset. Plain C++: tests/test_ring_offsets_cpu.py checks them
// against the operand's extent.
#pragma once

#include <cstdint>

namespace mc {

// A byte offset past every buffer resource (common.hpp).
constexpr uint32_t kOOB = 0x80000000u;

// The fp32 ring GEMM's loads of a B stored [k][N]: byte offset, from the first
// element of the step's first k row, of the 16-byte chunk that lane `lane` of
// wave `wave` requests with load j (k rows 8 wave + 4 j + lane / 16; chunk c of
// row k goes to LDS slot c ^ 8 ((k / 4) % 2)). `cols` = N - n0, a multiple of
// 4: chunks past them are given up here, because the step's advance is in
// soffset, which the range check of the load need not include: in the last k
// row such a chunk lies behind the operand.
constexpr uint32_t nn_chunk_offset(int wave, int lane, int j, uint32_t ldb, int64_t cols) {
    const uint32_t row = (uint32_t)(8 * wave + 4 * j + (lane >> 4));
    const uint32_t col = 4u * (uint32_t)((lane & 15) ^ (8 * j));
    return (int64_t)col < cols ? (row * ldb + col) * 4u : kOOB;
}

}  // namespace mc
