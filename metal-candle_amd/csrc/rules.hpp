// Rules that choose between two kernels for one call by its sizes. Plain C++:
// tests/test_dispatch_rules_cpu.py holds each against times measured on both
// sides of its line.
#pragma once

#include <cstdint>

namespace mc {

// Float32 row projection of few tokens and ranks: a workgroup per token
// (rowproj_f32_rows) instead of one per 16 tokens, which leaves most CUs
// without a row to read. Projection and its product, us, per token / per 16:
// r 4: K 768, T 32 7.7 / 9.0, T 512 8.5 / 9.5, T 1024 10.1 / 9.6; K 8960, T 32
// 14.8 / 28.6, T 512 23.6 / 29.3, T 1024 39.8 / 31.3; r 1: K 3584, T 1024
// 11.0 / 17.1, T 4096 23.8 / 20.6.
constexpr bool rowproj_f32_by_token(int64_t T, int r) { return r <= 4 && T * r <= 2048; }

}  // namespace mc
