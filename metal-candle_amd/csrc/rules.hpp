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

// Tile of the float32 column reduction: 16 rt ranks by 16 ct columns per
// workgroup; `cols` of all its outputs together. A workgroup walks all of T, so
// small outputs take the smallest tile to fill the CUs, and wide ones the
// largest that still does, since every group of ranks reads X again. Measured
// for one output, us, rt x ct:
//   cols 768,  r 64,  T 512:  1x1 4.9, 1x4 7.1, 4x4 18.3; T 4096: 16.6 / 29.1 / 92.0
//   cols 2304, r 16,  T 2048: 1x1 10.9, 1x4 16.9
//   cols 4608, r 16,  T 2048: 1x1 25.8, 1x4 20.6; T 32: 3.2 / 4.5
//   cols 1536, r 64,  T 2048: 1x1 15.7, 1x4 17.4 (384 of the small tiles)
//   cols 2304, r 64,  T 2048: 1x1 22.9, 1x4 17.8 (576)
//   cols 4608, r 64,  T 2048: 1x4 33.0, 2x4 35.9
//   cols 8960, r 128, T 2048: 1x4 98.1, 2x4 82.5, 4x4 104
//   cols 8960, r 64,  T 4096: 1x4 110, 2x4 107, 4x4 103
struct ColF32Tile {
    int rt, ct;
};
constexpr ColF32Tile colreduce_f32_tile(int64_t T, int64_t cols, int r) {
    const int64_t small = (cols + 15) / 16 * ((r + 15) / 16);  // workgroups of the smallest tile
    if (T <= 32 || (cols <= 3072 && small <= 448)) return ColF32Tile{1, 1};
    if (r <= 16 || cols <= 6144) return ColF32Tile{1, 4};
    return ColF32Tile{r > 32 && r <= 64 && T >= 4096 ? 4 : 2, 4};
}

}  // namespace mc
