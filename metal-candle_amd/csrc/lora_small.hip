// LoRA linear forward of a few tokens (decode steps), bf16, gfx950.
//
// y = x.W^T + b + s Hd.B, Hd = (x.A) (.) mask / (1-p)
// (src/training/lora.rs:320-339 over src/models/transformer.rs:189-192), for
// at most kSmallTokens (32) tokens and kSmallRanks (64) ranks, every projection
// of a group in each launch:
//
//   small_hidden  H = x.A in fp32 on v_mfma_f32_16x16x4_f32, 1024 columns of x
//                 per workgroup, partial sums [split][T][r];
//   small_linear  16 (32) rows of W per workgroup against all tokens, the waves
//                 taking every nw-th step of 64 columns, W straight from memory
//                 into the operands of v_mfma_f32_16x16x32_bf16; the rank-r
//                 term is added in fp32 from the partial sums of H.
//
// Bound by the read of W and, for small ones, by launches: the tiled path runs
// an operand preparation, a row projection (one launch up to 32 ranks and 4095
// columns) and a GEMM, whose few workgroups each walk all of K. The device's
// time, inputs not in the caches, tiled path / this, K -> N (the rule between
// the two is lora_few_tokens):
//   T  8,  1536 -> 1536,  r 8    16.6 /  9.4 us
//   T  8,  3584 -> 18944, r 64   56.4 / 50.1 us (W alone: 22 us at 6.2 TB/s)
//   T  8, 18944 -> 3584,  r 64    134 / 51.8 us
//   T 16,  3584 -> 3584,  r 8    31.6 / 14.1 us
//   T 32,  3584 -> 3584,  r 64   39.9 / 30.7 us
//   T 32, 18944 -> 3584,  r 64    136 / 91.8 us
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "lora_kernels.hpp"
#include "profile.hpp"
#include "rules.hpp"

namespace mc {
namespace {

struct SmallJob {
    int64_t N;
    const uint16_t* W;     // [N][K] or null
    const uint16_t* bias;  // [N] or null
    const float* A;        // [K][r]
    const float* B;        // [r][N]
    const uint8_t* mask;   // [T][r] or null
    uint16_t* y;           // [T][N]
    float* h_save;         // [r][T] or null
};
struct SmallArgs {
    SmallJob job[kMaxProj];
    int64_t tile0[kMaxProj + 1];  // first row tile of each projection
    int count, T, r, splits;
    int64_t K;
    const uint16_t* x;
    float* part;  // [count][splits][T][r]
    float scale, keep;
};

// Grid (splits, 16-token tiles, projections). Lane l supplies token (rank)
// l % 16 and, for MFMA q of a 16-column group, column 4 (l / 16) + q; a wave
// takes every nw-th block of 32 columns of the split.
constexpr int kHiddenCols = 1024;
template <int RT> constexpr int kHiddenWaves = RT <= 2 ? 16 : 8;
template <int RT>
__global__ __launch_bounds__(64 * kHiddenWaves<RT>) void small_hidden(SmallArgs a) {
    constexpr int NW = kHiddenWaves<RT>, NI = kHiddenCols / (32 * NW);  // blocks per wave
    const int lane = lane_id(), wave = wave_id(), l16 = lane & 15, g = lane >> 4;
    const int t0 = 16 * (int)blockIdx.y, r = a.r;
    const int64_t K = a.K;
    const float* A = a.job[blockIdx.z].A;
    const uint16_t* xr = a.x + (int64_t)std::min(t0 + l16, a.T - 1) * K;  // rows past T are dropped below
    const int64_t cbase = (int64_t)blockIdx.x * kHiddenCols + 32 * wave;
    // Every load first (of clamped addresses; the value selects come with the
    // products): left to itself the compiler moves each next to its use, one
    // memory latency after the other.
    u32x2 xv[NI][2];
    float p[NI][RT][2][4];
    auto col = [&](int it, int i) { return cbase + 32 * NW * it + 16 * i + 4 * g; };
#pragma unroll
    for (int it = 0; it < NI; ++it)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int64_t c = std::min(col(it, i), K - 4);  // K % 8 == 0: four columns are in or out together
            xv[it][i] = *reinterpret_cast<const u32x2*>(xr + c);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const float* pr = A + c * r + std::min(16 * rt + l16, r - 1);
#pragma unroll
                for (int q = 0; q < 4; ++q) p[it][rt][i][q] = pr[q * r];
            }
        }
    __builtin_amdgcn_sched_barrier(0);
    f32x4 tot[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) tot[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int it = 0; it < NI; ++it)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const bool in = col(it, i) < K;
            float xf[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t w = xv[it][i][q >> 1];
                xf[q] = in ? (q & 1 ? bf16_hi(w) : bf16_lo(w)) : 0.f;
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                f32x4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    part = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        xf[q], in && 16 * rt + l16 < r ? p[it][rt][i][q] : 0.f, part, 0, 0, 0);
                tot[rt] += part;
            }
        }
    __shared__ float red[NW][RT][16][17];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][rt][4 * g + i][l16] = tot[rt][i];
    __syncthreads();
    float* out = a.part + ((int64_t)blockIdx.z * a.splits + blockIdx.x) * a.T * r;
    for (int o = (int)threadIdx.x; o < 256 * RT; o += 64 * NW) {
        const int jl = o & 15, tl = (o >> 4) & 15, rt = o >> 8, t = t0 + tl, j = 16 * rt + jl;
        if (t < a.T && j < r) out[t * r + j] = sum_tree(NW, [&](int w) { return red[w][rt][tl][jl]; });
    }
}

// The partial sums of H added up (in split order), where every workgroup of
// small_linear adding them for itself would read more than its part of W.
__global__ __launch_bounds__(256) void small_hidden_sum(const float* __restrict__ part, float* __restrict__ out, int n,
                                                        int splits) {
    const int i = (int)(blockIdx.x * 256 + threadIdx.x);
    if (i >= n) return;
    const float* p = part + (int64_t)blockIdx.y * splits * n + i;
    out[(int64_t)blockIdx.y * n + i] = sum_tree(splits, [&](int s) { return p[(int64_t)s * n]; });
}

// TT 16-token tiles, RW 16-row tiles of W per workgroup, NW waves, U steps of W
// requested ahead. RW and U change no sum: a wave takes every NW-th step in
// order and the waves are added in order.
template <int TT, int RW, int NW, int U>
__global__ __launch_bounds__(64 * NW) void small_linear(SmallArgs a) {
    constexpr int ROWS = 16 * RW, LD = ROWS + 4;
    const int lane = lane_id(), wave = wave_id(), l16 = lane & 15, g = lane >> 4, tid = (int)threadIdx.x;
    int pj = 0;
    while (pj + 1 < a.count && (int64_t)blockIdx.x >= a.tile0[pj + 1]) ++pj;  // workgroup-uniform
    const SmallJob& J = a.job[pj];
    const int64_t tile = (int64_t)blockIdx.x - a.tile0[pj], n0 = tile * ROWS, N = J.N, K = a.K;
    const int T = a.T, r = a.r;
    const int64_t rows = std::min<int64_t>(N - n0, ROWS);
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(J.W + n0 * K, J.W ? rows * K * 2 : 0);
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x, J.W ? (int64_t)T * K * 2 : 0);
    const uint32_t lrow = (uint32_t)l16 * (uint32_t)K + 8u * (uint32_t)g;  // MFMA operand: row l % 16, k chunk l / 16
    // the 16-row tiles of v, U steps from column c0 (columns past K, rows past the resource: zeros)
    auto fetch = [&](__amdgpu_buffer_rsrc_t rs, int64_t c0, auto& v) {
        constexpr int R16 = sizeof(v[0]) / sizeof(v[0][0]);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < R16; ++k)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int64_t c = c0 + 64 * NW * u + 32 * i;
                    v[u][k][i] = buf_load16(
                        rs, c + 8 * g < K ? (lrow + (uint32_t)c + 16u * (uint32_t)k * (uint32_t)K) * 2u : kOOB);
                }
    };
    f32x4 acc[RW][TT];
#pragma unroll
    for (int k = 0; k < RW; ++k)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[k][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    i32x4 w[U][RW][2], wn[U][RW][2], xv[U][TT][2], xn[U][TT][2];
    const int64_t kend = J.W ? K : 0;
    int64_t c0 = 64 * (int64_t)wave;
    if (c0 < kend) {  // on their way while the rank-r operands are staged
        fetch(rw, c0, w);
        fetch(rx, c0, xv);
    }

    // s Hd [tokens][ranks] and B^T [ranks][ROWS], ranks in steps of 4 (zeros past r)
    constexpr int HLD = kSmallRanks + 1;
    __shared__ float hs[16 * TT][HLD];
    __shared__ float bl[kSmallRanks][ROWS];
    __shared__ __attribute__((aligned(16))) float red[NW][16][LD];
    const int r4 = (r + 3) / 4 * 4;
    for (int i = tid; i < 16 * TT * r4; i += 64 * NW) {
        const int t = i / r4, j = i - t * r4;
        float v = 0.f;
        if (t < T && j < r) {
            const float* p = a.part + (int64_t)pj * a.splits * T * r + t * r + j;
            v = sum_tree(a.splits, [&](int s) { return p[(int64_t)s * T * r]; });
            if (J.mask) v = J.mask[t * r + j] ? v * a.keep : 0.f;
            if (J.h_save && tile == 0) J.h_save[(int64_t)j * T + t] = v;
        }
        hs[t][j] = v * a.scale;
    }
    for (int i = tid; i < r4 * ROWS; i += 64 * NW) {
        const int j = i / ROWS, n = i % ROWS;
        bl[j][n] = j < r && n0 + n < N ? J.B[(int64_t)j * N + n0 + n] : 0.f;
    }
    for (; c0 < kend; c0 += 64 * NW * U) {
        if (c0 + 64 * NW * U < kend) {
            fetch(rw, c0 + 64 * NW * U, wn);
            fetch(rx, c0 + 64 * NW * U, xn);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int k = 0; k < RW; ++k)
#pragma unroll
                    for (int t = 0; t < TT; ++t)
                        acc[k][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[u][k][i]),
                                                                            __builtin_bit_cast(bf16x8, xv[u][t][i]),
                                                                            acc[k][t], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int k = 0; k < RW; ++k) w[u][k][i] = wn[u][k][i];
#pragma unroll
                for (int t = 0; t < TT; ++t) xv[u][t][i] = xn[u][t][i];
            }
    }
    // the rank-r term in fp32, four ranks per MFMA, the steps spread over the waves
    __syncthreads();
    for (int j0 = 4 * wave; j0 < r4; j0 += 4 * NW)
#pragma unroll
        for (int k = 0; k < RW; ++k)
#pragma unroll
            for (int t = 0; t < TT; ++t)
                acc[k][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(bl[j0 + g][16 * k + l16], hs[16 * t + l16][j0 + g],
                                                                 acc[k][t], 0, 0, 0);
    // accumulator i of lane l: row 4 (l / 16) + i of W, token l % 16
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        if (16 * t >= T) break;  // workgroup-uniform
        if (t > 0) __syncthreads();
#pragma unroll
        for (int k = 0; k < RW; ++k) *reinterpret_cast<f32x4*>(&red[wave][l16][16 * k + 4 * g]) = acc[k][t];
        __syncthreads();
        const int tokens = std::min(T - 16 * t, 16);
        for (int o = tid; o < tokens * ROWS; o += 64 * NW) {
            const int n = o % ROWS, tl = o / ROWS, tok = 16 * t + tl;
            if (n0 + n >= N) continue;
            float v = sum_tree(NW, [&](int q) { return red[q][tl][n]; });
            if (J.bias) v += bf16_to_f32(J.bias[n0 + n]);
            J.y[(int64_t)tok * N + n0 + n] = f32_to_bf16(v);
        }
    }
}

}  // namespace

int lora_small_splits(int64_t K) { return (int)((K + kHiddenCols - 1) / kHiddenCols); }

size_t lora_small_ws(int64_t T, int64_t K, int r, int count) {
    return (size_t)count * (lora_small_splits(K) + 1) * T * r * 4;  // the partial sums of H, then H
}

hipError_t launch_lora_small_fwd(const mc_lora_desc& d, const void* x, const LoraProj* proj, int count, void* const* y,
                                 float* const* h_save, void* ws, hipStream_t st) {
    SmallArgs a{};
    a.count = count;
    a.T = (int)d.tokens;
    a.r = d.rank;
    a.K = d.in_features;
    a.x = static_cast<const uint16_t*>(x);
    a.part = static_cast<float*>(ws);
    a.splits = lora_small_splits(a.K);
    a.scale = d.scale;
    a.keep = d.dropout_p > 0.f ? 1.0f / (1.0f - d.dropout_p) : 1.0f;
    // Rows of W per workgroup: enough workgroups for the CUs first, then more
    // rows for each read of x and of the rank-r operands.
    int64_t sumN = 0;
    for (int g = 0; g < count; ++g) sumN += proj[g].N;
    const bool wide = sumN >= 16384;
    const int rows = (a.T <= 16 ? 16 : 32) * (wide ? 2 : 1);
    for (int g = 0; g < count; ++g) {
        a.job[g] = SmallJob{proj[g].N, static_cast<const uint16_t*>(proj[g].W),
                            static_cast<const uint16_t*>(proj[g].bias), proj[g].A, proj[g].B, proj[g].mask,
                            static_cast<uint16_t*>(y[g]), h_save ? h_save[g] : nullptr};
        a.tile0[g + 1] = a.tile0[g] + (proj[g].N + rows - 1) / rows;
    }
    double flops = 0, bytes = 2.0 * a.T * (a.K + sumN);  // of the products; x and y
    for (int g = 0; g < count; ++g) {
        const double k = proj[g].W ? (double)a.K : 0.0;
        flops += 2.0 * a.T * proj[g].N * (k > 0 ? k : a.r);
        bytes += proj[g].N * (2.0 * k + 4.0 * a.r);
    }
    {
        // h: [splits] partial sums of each projection, then one sum where they are many
        auto sc = prof::Scope(prof::kLowRank, st, 2.0 * a.T * a.K * a.r * count,
                              2.0 * a.T * a.K + 4.0 * a.r * (a.K + a.T) * count);
        const dim3 gh((unsigned)a.splits, (unsigned)((a.T + 15) / 16), (unsigned)count);
        if (a.r <= 16) small_hidden<1><<<gh, 64 * kHiddenWaves<1>, 0, st>>>(a);
        else if (a.r <= 32) small_hidden<2><<<gh, 64 * kHiddenWaves<2>, 0, st>>>(a);
        else small_hidden<4><<<gh, 64 * kHiddenWaves<4>, 0, st>>>(a);
        const int n = a.T * a.r;
        if (a.splits > 1 && n * a.splits > 8192) {  // 32 KB of partial sums per workgroup of small_linear
            float* sum = a.part + (size_t)count * a.splits * n;
            small_hidden_sum<<<dim3((unsigned)((n + 255) / 256), (unsigned)count), 256, 0, st>>>(a.part, sum, n,
                                                                                                 a.splits);
            a.part = sum;
            a.splits = 1;
        }
    }
    auto sc = prof::Scope(prof::kGemm, st, flops, bytes);
    const dim3 grid((unsigned)a.tile0[count]);
    if (a.T <= 16) {
        if (wide) small_linear<1, 2, 16, 1><<<grid, 1024, 0, st>>>(a);
        else small_linear<1, 1, 16, 2><<<grid, 1024, 0, st>>>(a);
    } else {
        if (wide) small_linear<2, 4, 8, 1><<<grid, 512, 0, st>>>(a);
        else small_linear<2, 2, 8, 2><<<grid, 512, 0, st>>>(a);
    }
    return hipGetLastError();
}

}  // namespace mc
