// Rules that choose between two kernels for one call by its sizes. Plain C++:
// tests/test_dispatch_rules_cpu.py holds each against times measured on both
// sides of its line.
#pragma once

#include <cstdint>

namespace mc {

// Cross-entropy rows on 1024 threads instead of 256, where so few rows leave
// CUs short of loads in flight and a row has work for all the threads. Forward and backward,
// us, 1024 / 256 threads:
//   rows 64    fp32 8001 14.0 / 15.9, 50257 21.7 / 40.5; bf16 8192 12.9 / 11.7, 32000 18.6 / 23.0
//   rows 256   fp32 8192 15.3 / 15.7, 32000 25.8 / 30.3; bf16 16384 16.0 / 16.6, 151936 50.5 / 78.0
//   rows 384   fp32 8192 19.0 / 16.3, 32000 36.8 / 40.2; bf16 16384 19.7 / 17.9, 50257 34.8 / 36.3
//   rows 512   fp32 16384 27.6 / 24.7, 50257 63.3 / 64.9; bf16 32000 29.4 / 27.7, 151936 95.3 / 116
//   rows 1000  fp32 8192 30.5 / 23.9, 151936 333 / 333; bf16 8192 26.4 / 19.1, 50257 66.3 / 62.8
constexpr bool xent_wide_rows(int64_t rows, int64_t vocab, int elem_size) {
    const int64_t vectors = vocab * elem_size / 16;
    return rows <= 256 ? vectors >= 1536 : rows <= 512 && vectors >= 6144;
}

// Gradients of the logits stored past the caches, once they are 64 MB, a quarter
// of the last-level cache. Below, the product that reads the gradients finds
// them in the cache, and forward and backward alone lose nothing by it; above,
// ordinary stores push out logits that the backward has yet to read, and more
// of the next step's. Time of streamed over ordinary stores: forward and
// backward in a loop over three inputs; on logits not seen before; followed by a
// LoRA backward; between the product that made the logits and the one that
// reads the gradients (torch.matmul, 896 features).
//   20 MB   0.96-1.01  0.97-1.01  1.00-1.31  1.00-1.01
//   50 MB   0.98-1.01  0.98-1.03  1.01-1.28  1.00-1.02
//   85 MB   0.83-0.96  0.95-0.99  0.99-1.24  1.00 (70 MB, bf16 1.03)
//   120 MB  0.77-0.86  0.82-0.95  0.97-1.18  1.00-1.01
//   300 MB             0.84-0.90  0.92-1.01  0.98
// 2036 bf16 rows of 151936 (619 MB), not seen before: 333 / 384 us, 621 / 629 with
// a LoRA backward, 1685 / 1704 between products. From 900 MB on the two differ by
// less than 6% either way.
constexpr bool xent_stream_gradients(int64_t rows, int64_t vocab, int elem_size) {
    return rows * vocab * elem_size > (int64_t)64 << 20;
}

// Softmax rows that are not whole 16-byte vectors: the covering vectors of the
// one-wave kernels, or for short rows a lane per element (the scalar kernels),
// where the vectors keep only a few lanes busy and pay for the shared edges.
// us, elements / vectors, 56 heads of S x S, or 112 causal ones:
//   fp32 forward   S 65 3.0 / 3.1 (3.8 / 4.1), S 99 3.7 / 3.5 (5.4 / 5.1), S 201 8.4 / 5.3
//   fp32 backward  S 99 3.5 / 4.0 (5.0 / 5.7), S 161 6.5 / 5.5 (7.7 / 7.7), S 201 8.0 / 6.9
//   bf16 forward   S 99 3.5 / 4.2 (5.0 / 6.0), S 161 6.0 / 5.4 (8.5 / 8.9), S 201 8.0 / 6.2
//   bf16 backward  S 99 3.0 / 4.4 (4.5 / 6.2), S 201 7.0 / 6.2 (9.1 / 9.8), S 257 8.8 / 7.3
// Enough whole rows to be bound by memory, forward, backward: 65536 rows of 77,
// fp32 20.7 / 15.0, 21.3 / 19.0, bf16 20.4 / 21.1, 15.7 / 19.1; of 129, bf16
// 26.6 / 21.2, 27.3 / 20.9; of 33, fp32 14.6 / 15.0, 11.1 / 17.8.
constexpr bool softmax_ragged_vectors(int64_t rows, int64_t dim, bool causal, int elem_size, bool backward) {
    if (rows >= 32768 && !causal) return dim >= (elem_size == 4 ? 64 : 112);
    return dim >= (elem_size == 4 ? (backward ? 160 : 96) : (backward ? 224 : 176));
}

// Float32 attention of short sequences: the row kernels (attn_*_generic, a wave
// per row) in the place of the 32 x 32 tiles, whose work and four-wave
// combination do not shrink with S. The row backward walks the query heads of a
// K/V head (rep of them) one after the other. Ratio of tiles to rows, forward:
// D 32 S 3 1.18-1.27, S 5 0.92-0.99; D 64 S 6 1.06-1.19, S 8 0.89-0.98; D 128 S 8
// 1.07-1.19, S 10 0.94-1.05. Backward: D 32 rep 1 S 5 1.02-1.10, S 8 0.82-0.90;
// D 64 rep 1 S 10 1.07-1.19, S 16 0.81-0.88, rep 6 S 4 0.98-1.10, S 5 0.84-0.92;
// D 96 rep 1 S 12 1.27-1.42, D 128 rep 6 S 5 1.02-1.17, rep 7 S 6 0.77-0.94.
constexpr bool attention_f32_rows_fwd(int64_t S, int D) { return S <= (D <= 32 ? 4 : D <= 64 ? 7 : 9); }
constexpr bool attention_f32_rows_bwd(int64_t S, int D, int rep) {
    return S * (rep + 2) <= (D <= 32 ? 18 : D <= 64 ? 33 : 45);
}

// The tiles' launches, 256 threads per 32 rows of a head, stay within 2^32 - 1
// work-items (the row kernels take 64 per row, fewer where S is 1 to 3).
constexpr bool attention_f32_tiles_fit(int64_t S, int64_t batch_heads) {
    return (S + 31) / 32 * batch_heads <= (((int64_t)1 << 32) - 1) / 256;
}

// Few-token LoRA forward (lora_small.hip) for one projection, else the tiled
// path. A projection of a group takes the path that it would take alone, so
// that the group's results are those of single calls. Up to 16 tokens it was
// never the slower of the two by more than 10%; past that its workgroups are 32
// rows of W, and it is ahead while a round of the CUs holds them all (N 8192).
// Forward, us, few-token / tiled (before the tiles for small grids):
//   T 16: 1536 -> 8960, r 8 18.7 / 17.0 (27.6), 3584 -> 18944, r 64 54.2 / 57.4 (66.5)
//   T 17: 1536 -> 1536, r 8 12.6 / 16.9 (27.8), 3584 -> 18944, r 64 65.3 / 57.3 (66.3)
//   T 32: 896 -> 896, r 8 10.1 / 11.6 (19.1), 1536 -> 8960, r 8 21.6 / 17.3 (28.1),
//         18944 -> 3584, r 64 91.8 / 136 (202), 1536 -> 18944, r 64 48.2 / 40.2 (41.6),
//         3584 -> 3584, r 64 30.7 / 39.9 (51.7), 3584 -> 18944, r 64 71.7 / 60.7 (67.1)
// Groups, T 32: 1536 -> 8960, 8960, r 64 48.0 / 39.7 (41.0); 3584 -> 18944, 18944
// gains nothing from the line: r 64 102.6 / 103.5 (104.6), r 16 81.6 / 87.4 (106).
constexpr int kSmallTokens = 32, kSmallRanks = 64;
constexpr bool lora_few_tokens(int64_t T, int64_t N, int r) {
    return r <= kSmallRanks && (T <= 16 || (T <= kSmallTokens && N <= 8192));
}

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
