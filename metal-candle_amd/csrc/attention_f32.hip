// Float32 attention core on the fp32 matrix cores, gfx950.
//
// The same composite as attention.hip (src/models/transformer.rs:258-319) for
// float32 tensors with a head dim that is a multiple of 4, at most 128. Every
// product is v_mfma_f32_32x32x2_f32 (fp32 operands and sums), the softmax
// arithmetic fp32, so the precision is that of the row-per-wave kernels these
// replaced (attn_*_generic<float>, now for the other head dims and for sequences
// of a few tokens, attention_f32_rows_fwd / _bwd).
//
// What bounds it: the fp32 MFMA rate (157 TFLOP/s; a 32 x 32 block of scores
// costs D / 2 MFMAs of 64 cycles per product), far below what LDS and L2 can
// feed at 32 queries (keys) per wave. So the tiles are small and the split is
// made for parallelism: a workgroup owns 32 queries (dK/dV: 32 keys) of one
// head and its 4 waves take every 4th block of 32 keys (queries), each with a
// private LDS tile and no barrier in the loop; the waves' partial sums are
// added in wave order at the end. A call of a few hundred tokens thus still
// has a wave for every SIMD.
//
// Layouts. Accumulator register q of lane l (half h = l / 32) is row
// 8 (q / 4) + 4 h + q % 4, column l % 32. The scores are formed so that this
// is also the operand order of the next product: with S^T = K.Q^T a lane holds
// 16 keys of one query, and step q of O^T += V^T.P^T multiplies key rows
// 8 (q / 4) + q % 4 and that + 4, so p goes from accumulator to operand
// without moving. The other operand of that step is a row of V (of K, Q, dO in
// the backward): output row i stands for dims DT i .. DT i + DT - 1 over the
// DT = D / 32 tiles, so lane i reads DT consecutive floats and 32 lanes a
// whole row.
//
// B 4, H 12, Hkv 2, S 509, D 64, causal (rocprofv3, cold caches; row-per-wave
// kernels -> these): forward 1050 -> 35 us, dQ with Delta 626 -> 46 us, dK/dV
// 2011 -> 58 us and 5 us for the sum over the groups. The products alone would
// take 11, 16 and 21 us at the MFMA rate.
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "rules.hpp"

namespace mc {
namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_inff();

struct F32AttnArgs {
    const float *q, *k, *v, *mask, *o, *dout;
    float *out, *lse;  // forward outputs (lse may be null; the backward's input)
    float *delta;      // backward: rowsum(dO (.) O) [B, H, S]
    float *dq, *dk, *dv;
    int64_t S;
    int B, H, Hkv, D, nblk, causal;
    int groups;  // dK/dV: groups of H / Hkv / groups query heads, one partial each
    float scale;
};

// Orders a wave's LDS accesses for the compiler (the hardware keeps them in
// order): the tiles below are private to a wave.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float half_swap(float v) { return __shfl_xor(v, 32, kWave); }

// Row of accumulator register q.
__device__ __forceinline__ int acc_row(int q, int h) { return 8 * (q >> 2) + 4 * h + (q & 3); }

// A 32-row tile [32][DP] of fp32, DP = D rounded up to 32, 64 or 128. Rows in
// LDS are DP + 4 floats apart: 16 consecutive rows of one 16-byte column, and
// one row's consecutive columns, each fall on distinct banks.
template <int DP> struct Tile32 {
    static constexpr int LD = DP + 4, CPR = DP / 4, LOADS = DP / 8, DT = DP / 32;
    static constexpr int FLOATS = 32 * LD;
    typedef float vec __attribute__((ext_vector_type(DT)));

    // Resource over rows row0 .. of an operand whose rows are ld floats apart
    // (`rows` of them in all); rows past the end load as zeros.
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const float* base, int64_t row0, int64_t rows,
                                                                  int64_t ld, int D) {
        const int64_t left = rows - row0;
        return make_rsrc(base + row0 * ld, left > 0 ? ((left - 1) * ld + D) * 4 : 0);
    }
    // Whole row segments: lane l loads 16-byte chunk l % CPR of rows
    // l / CPR + i (64 / CPR); chunks past D load as zeros.
    static __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, uint32_t ld, int D, f32x4 (&t)[LOADS]) {
        const int lane = lane_id(), c = lane % CPR;
        uint32_t off = 4 * c < D ? ((uint32_t)(lane / CPR) * ld + 4u * c) * 4u : kOOB;
        asm volatile("" : "+v"(off));  // keeps the LOADS offsets out of registers across the caller's loop
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            t[i] = __builtin_bit_cast(f32x4, buf_load16(r, off + (uint32_t)i * (64u / CPR) * ld * 4u));
    }
    static __device__ __forceinline__ void store(float* lds, const f32x4 (&t)[LOADS]) {
        const int lane = lane_id(), c = lane % CPR;
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            *reinterpret_cast<f32x4*>(&lds[(lane / CPR + i * (64 / CPR)) * LD + 4 * c]) = t[i];
    }
    // Operand of a product over the head dim: lane's row l % 32, dims
    // 8 j + 4 h .. + 3 for step group j.
    static __device__ __forceinline__ f32x4 along_d(const float* lds, int j) {
        const int lane = lane_id();
        return *reinterpret_cast<const f32x4*>(&lds[(lane & 31) * LD + 8 * j + 4 * (lane >> 5)]);
    }
    // The same straight from memory (an operand held for the whole kernel).
    static __device__ __forceinline__ void load_along_d(__amdgpu_buffer_rsrc_t r, uint32_t ld, int D,
                                                        f32x4 (&t)[DP / 8]) {
        const int lane = lane_id();
#pragma unroll
        for (int j = 0; j < DP / 8; ++j) {
            const int d = 8 * j + 4 * (lane >> 5);
            t[j] = __builtin_bit_cast(f32x4, buf_load16(r, d < D ? ((uint32_t)(lane & 31) * ld + d) * 4u : kOOB));
        }
    }
    // Operand of step q of a product over the rows: row acc_row(q, h), the
    // DT dims of output row l % 32.
    static __device__ __forceinline__ vec along_rows(const float* lds, int q) {
        const int lane = lane_id();
        return *reinterpret_cast<const vec*>(&lds[acc_row(q, lane >> 5) * LD + DT * (lane & 31)]);
    }
    // acc^T (DT tiles, rows = dims, lane = row l % 32) -> lds rows
    static __device__ __forceinline__ void store_acc(float* lds, const f32x16 (&acc)[DT]) {
        const int lane = lane_id();
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float v[4 * DT];
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int t = 0; t < DT; ++t) v[e * DT + t] = acc[t][4 * g + e];
            float* dst = &lds[(lane & 31) * LD + DT * (8 * g + 4 * (lane >> 5))];
#pragma unroll
            for (int e = 0; e < DT; ++e)
                *reinterpret_cast<f32x4*>(dst + 4 * e) = f32x4{v[4 * e], v[4 * e + 1], v[4 * e + 2], v[4 * e + 3]};
        }
    }
};

__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int q = 0; q < 16; ++q) z[q] = 0.f;
    return z;
}

// A.B over the head dim: A rows from an LDS tile, B from b(j) (held in
// registers, or read from a second tile). Each step's operand is read one step
// (256 cycles of MFMA) ahead; the scheduling barriers keep the compiler from
// hoisting more of them than the registers hold. Every 8 dims are summed on
// their own, added in pairs and the pairs to the total, so the rounding of a
// score is that of short chains (one chain over the whole head dim was up to
// 1.4 times further from the 64-bit result than the row kernels at short
// sequences).
template <int DP, typename Bf>
__device__ __forceinline__ f32x16 mma_d(const float* lds, Bf&& b) {
    constexpr int NJ = DP / 8;
    f32x16 acc, even;
    f32x4 x = Tile32<DP>::along_d(lds, 0), y = b(0);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        f32x4 nx = x, ny = y;
        if (j + 1 < NJ) {
            nx = Tile32<DP>::along_d(lds, j + 1);
            ny = b(j + 1);
        }
        f32x16 part = zero16();
#pragma unroll
        for (int p = 0; p < 4; ++p) part = __builtin_amdgcn_mfma_f32_32x32x2f32(x[p], y[p], part, 0, 0, 0);
        if (j % 2 == 0) {
            even = part;
        } else {
            acc = j == 1 ? even + part : acc + (even + part);
            asm volatile("" : "+v"(acc));  // adds it here, not after the last chain
        }
        x = nx;
        y = ny;
        __builtin_amdgcn_sched_barrier(0);
    }
    return acc;
}

// acc^T += X^T.P over the 32 rows of an LDS tile X, P from an accumulator
// (operands read four steps ahead).
template <int DP>
__device__ __forceinline__ void mma_rows(const float* lds, const f32x16& p, f32x16 (&acc)[DP / 32]) {
    typename Tile32<DP>::vec x[2][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[0][e] = Tile32<DP>::along_rows(lds, e);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        if (g < 3)
#pragma unroll
            for (int e = 0; e < 4; ++e) x[(g + 1) & 1][e] = Tile32<DP>::along_rows(lds, 4 * (g + 1) + e);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int t = 0; t < DP / 32; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[g & 1][e][t], p[4 * g + e], acc[t], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// A causal diagonal block multiplies zero scores with rows that a query (key)
// must not see, and 0 * inf is not 0. Blocks with a non-finite row there (a
// padded tail of uninitialised memory, say) take this detour, so that such a
// row reaches exactly the results that it reached one row at a time: the
// non-finite elements are added element by element where the row is visible,
// then zeroed in the tile for the matrix product. KEYS: rows are keys and
// visible to queries at or past them; otherwise queries, for keys up to them.
__device__ __forceinline__ bool nonfinite(float v) { return !(__builtin_fabsf(v) <= 3.402823466e38f); }
template <int DP, bool KEYS>
__device__ __forceinline__ void add_nonfinite(float* tile, const f32x16& p, f32x16 (&acc)[DP / 32]) {
    constexpr int DT = DP / 32, LD = Tile32<DP>::LD;
    const int lane = lane_id(), col = lane & 31, h = lane >> 5;
#pragma unroll 1
    for (int r = 0; r < 32; ++r) {  // row r is register 4 (r / 8) + r % 4 of lane half (r / 4) % 2
        const float pr = __shfl(p[4 * (r >> 3) + (r & 3)], col + 32 * ((r >> 2) & 1), kWave);
        const bool visible = KEYS ? r <= col : r >= col;
#pragma unroll
        for (int g = 0; g < 16; ++g)
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                const float v = tile[r * LD + DT * acc_row(g, h) + t];
                acc[t][g] += visible && nonfinite(v) ? pr * v : 0.f;
            }
    }
    wave_lds_fence();
#pragma unroll 1
    for (int i = lane; i < Tile32<DP>::FLOATS; i += 64)
        if (nonfinite(tile[i])) tile[i] = 0.f;
    wave_lds_fence();
}
template <int N>
__device__ __forceinline__ bool any_nonfinite(const f32x4 (&t)[N]) {
    bool bad = false;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) bad |= nonfinite(t[i][e]);
    return __any(bad);
}

// Last row of the key block at k0 that this lane's query (q0 + l % 32) reads.
__device__ __forceinline__ int last_key(const F32AttnArgs& a, int64_t q0, int64_t k0) {
    const int end = (int)(a.S - 1 - k0 < 31 ? a.S - 1 - k0 : 31);
    const int own = (int)(q0 - k0 < 64 ? q0 - k0 : 64) + (lane_id() & 31);
    return a.causal && own < end ? own : end;
}

// Head of workgroup j of a round of nbh: with the round a multiple of 8 long
// each XCD (workgroup id mod 8) takes a contiguous run of heads, so the heads
// that share a K/V head share an L2.
__device__ __forceinline__ int head_of(int j, int nbh) { return (nbh & 7) ? j : (j & 7) * (nbh >> 3) + (j >> 3); }

// Two waves per SIMD where the registers allow it (D <= 64); D = 128 holds
// twice the operands and accumulators and runs one.
template <int DP> constexpr int kWgPerCu = DP <= 64 ? 2 : 1;

// ---------------------------------------------------------------- forward
// A zero mask gives the result of no mask bit for bit: both keep the running
// max over scale * product.
template <int DP, bool MASK>
__global__ __launch_bounds__(256, kWgPerCu<DP>) void attn_f32_fwd(F32AttnArgs a) {
    typedef Tile32<DP> TL;
    constexpr int DT = TL::DT;
    __shared__ __attribute__((aligned(16))) float tiles[4][TL::FLOATS];
    __shared__ float stat[4][2][32];
    const int lane = lane_id(), wave = wave_id(), col = lane & 31, h = lane >> 5;
    const int nbh = a.B * a.H;
    const int qb = a.nblk - 1 - (int)(blockIdx.x / nbh);  // heaviest (causal) query blocks first
    const int bh = head_of((int)(blockIdx.x % nbh), nbh);
    const int b = bh / a.H, hq = bh % a.H;
    const int64_t S = a.S, D = a.D;
    const int64_t bhk = (int64_t)b * a.Hkv + hq / (a.H / a.Hkv);
    const int64_t q0 = (int64_t)qb * 32, qi = q0 + col;
    const float *kh = a.k + bhk * S * D, *vh = a.v + bhk * S * D;
    float* kt = tiles[wave];

    f32x4 qf[DP / 8];
    TL::load_along_d(TL::rsrc(a.q + (int64_t)bh * S * D, q0, S, D, a.D), a.D, a.D, qf);
    const int nkb = a.causal ? qb + 1 : a.nblk;
    float m = kNegInf, l = 0.f;
    f32x16 acc[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[t] = zero16();

    f32x4 kr[TL::LOADS];
    if (wave < nkb) TL::load(TL::rsrc(kh, (int64_t)wave * 32, S, D, a.D), a.D, a.D, kr);
    for (int kb = wave; kb < nkb; kb += 4) {
        const int64_t k0 = (int64_t)kb * 32;
        TL::store(kt, kr);
        // V rows of this block, one step's operand per register group
        typename TL::vec vr[16];
        {
            const __amdgpu_buffer_rsrc_t rv = TL::rsrc(vh, k0, S, D, a.D);
            const uint32_t d0 = (uint32_t)(DT * col);
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int off = (int)(d0 < (uint32_t)a.D ? ((uint32_t)acc_row(q, h) * (uint32_t)a.D + d0) * 4u : kOOB);
                if constexpr (DT == 4)
                    vr[q] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rv, off, 0, 0));
                else if constexpr (DT == 2)
                    vr[q] = __builtin_bit_cast(typename TL::vec, __builtin_amdgcn_raw_buffer_load_b64(rv, off, 0, 0));
                else
                    vr[q][0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rv, off, 0, 0));
            }
        }
        wave_lds_fence();
        f32x16 s = mma_d<DP>(kt, [&](int j) { return qf[j]; });  // S^T: lane = query, registers = keys
        wave_lds_fence();
        if (kb + 4 < nkb) TL::load(TL::rsrc(kh, k0 + 128, S, D, a.D), a.D, a.D, kr);
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            s[q] *= a.scale;
            if constexpr (MASK)
                if (qi < S && k0 + acc_row(q, h) < S) s[q] += a.mask[qi * S + k0 + acc_row(q, h)];
        }
        if (k0 + 32 > S || (a.causal && kb == qb)) {  // past the end, or the diagonal block
            const int last = last_key(a, q0, k0) - 4 * h;
#pragma unroll
            for (int q = 0; q < 16; ++q)
                if (acc_row(q, 0) > last) s[q] = kNegInf;
        }
        float mb = s[0];
#pragma unroll
        for (int q = 1; q < 16; ++q) mb = fmaxf(mb, s[q]);
        mb = fmaxf(mb, half_swap(mb));
        const float mn = fmaxf(m, mb);
        const float mu = mn == kNegInf ? 0.f : mn;  // no key seen yet: p = 0
        if (__any(mn != m)) {
            const float alpha = exp2_hw((m - mu) * kLog2e);
            l *= alpha;
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
                for (int q = 0; q < 16; ++q) acc[t][q] *= alpha;
            m = mn;
        }
        float lb = 0.f;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            s[q] = exp2_hw((s[q] - mu) * kLog2e);
            lb += s[q];
        }
        l += lb;
        if (a.causal && kb == qb) {
            bool bad = false;
#pragma unroll
            for (int q = 0; q < 16; ++q)
#pragma unroll
                for (int t = 0; t < DT; ++t) bad |= nonfinite(vr[q][t]);
            if (__any(bad)) {
#pragma unroll
                for (int q = 0; q < 16; ++q)
                    *reinterpret_cast<typename TL::vec*>(&kt[acc_row(q, h) * TL::LD + DT * col]) = vr[q];
                wave_lds_fence();
                add_nonfinite<DP, true>(kt, s, acc);
#pragma unroll
                for (int q = 0; q < 16; ++q) vr[q] = TL::along_rows(kt, q);
                wave_lds_fence();
            }
        }
#pragma unroll
        for (int q = 0; q < 16; ++q)
#pragma unroll
            for (int t = 0; t < DT; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[q][t], s[q], acc[t], 0, 0, 0);
    }
    l += half_swap(l);
    if (h == 0) {
        stat[wave][0][col] = m;
        stat[wave][1][col] = l;
    }
    wave_lds_fence();
    TL::store_acc(kt, acc);
    __syncthreads();
    // o = sum_w O_w 2^(m_w - M) / sum_w l_w 2^(m_w - M), waves in order
#pragma unroll
    for (int i = 0; i < DT; ++i) {
        const int ch = (int)threadIdx.x + 256 * i, row = ch / TL::CPR, d = 4 * (ch % TL::CPR);
        float M = stat[0][0][row];
#pragma unroll
        for (int w = 1; w < 4; ++w) M = fmaxf(M, stat[w][0][row]);
        const float mu = M == kNegInf ? 0.f : M;
        float L = 0.f;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float e = exp2_hw((stat[w][0][row] - mu) * kLog2e);
            L += stat[w][1][row] * e;
            const f32x4 x = *reinterpret_cast<const f32x4*>(&tiles[w][row * TL::LD + d]);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] += x[j] * e;
        }
        const int64_t qr = q0 + row;
        if (qr >= S) continue;
        const float inv = 1.f / L;
        if (d < a.D)
            *reinterpret_cast<f32x4*>(&a.out[(((int64_t)b * S + qr) * a.H + hq) * D + d]) =
                f32x4{v[0] * inv, v[1] * inv, v[2] * inv, v[3] * inv};
        if (d == 0 && a.lse) a.lse[(int64_t)bh * S + qr] = M + logf(L);
    }
}

// ------------------------------------------------------------- dQ (and Delta)
// Shaped like the forward: S^T = K.Q^T, dP^T = V.dO^T, dQ^T += K^T.dS^T with K
// read both ways from its LDS tile. It runs before dK/dV and also writes
// Delta_i = sum_d dO_id O_id of its 32 queries for it.
template <int DP, bool MASK>
__global__ __launch_bounds__(256, kWgPerCu<DP>) void attn_f32_bwd_dq(F32AttnArgs a) {
    typedef Tile32<DP> TL;
    constexpr int DT = TL::DT;
    __shared__ __attribute__((aligned(16))) float tiles[4][2][TL::FLOATS];
    __shared__ float sdelta[32];
    const int lane = lane_id(), wave = wave_id(), col = lane & 31, h = lane >> 5;
    const int nbh = a.B * a.H;
    const int qb = a.nblk - 1 - (int)(blockIdx.x / nbh);
    const int bh = head_of((int)(blockIdx.x % nbh), nbh);
    const int b = bh / a.H, hq = bh % a.H;
    const int64_t S = a.S, D = a.D, HD = (int64_t)a.H * D;
    const int64_t bhk = (int64_t)b * a.Hkv + hq / (a.H / a.Hkv);
    const int64_t q0 = (int64_t)qb * 32, qi = q0 + col;
    const float *kh = a.k + bhk * S * D, *vh = a.v + bhk * S * D;
    const int64_t obase = (int64_t)b * S * HD + (int64_t)hq * D;
    float *kt = tiles[wave][0], *vt = tiles[wave][1];

    {  // Delta: 8 threads per query, in a fixed order
        const int row = (int)threadIdx.x >> 3, part = (int)threadIdx.x & 7;
        float s = 0.f;
        if (q0 + row < S) {
            const int64_t base = obase + (q0 + row) * HD;
            for (int d = 4 * part; d < a.D; d += 32) {
                const f32x4 x = *reinterpret_cast<const f32x4*>(a.o + base + d);
                const f32x4 y = *reinterpret_cast<const f32x4*>(a.dout + base + d);
                s += (x[0] * y[0] + x[1] * y[1]) + (x[2] * y[2] + x[3] * y[3]);
            }
        }
        s += __shfl_xor(s, 1, kWave);
        s += __shfl_xor(s, 2, kWave);
        s += __shfl_xor(s, 4, kWave);
        if (part == 0) {
            sdelta[row] = s;
            if (q0 + row < S) a.delta[(int64_t)bh * S + q0 + row] = s;
        }
    }
    f32x4 qf[DP / 8], gf[DP / 8];
    TL::load_along_d(TL::rsrc(a.q + (int64_t)bh * S * D, q0, S, D, a.D), a.D, a.D, qf);
    TL::load_along_d(TL::rsrc(a.dout + obase, q0, S, HD, a.D), (uint32_t)HD, a.D, gf);
    const float li = qi < S ? a.lse[(int64_t)bh * S + qi] : 0.f;
    __syncthreads();
    const float di = sdelta[col];
    const int nkb = a.causal ? qb + 1 : a.nblk;
    f32x16 acc[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[t] = zero16();

    f32x4 kr[TL::LOADS], vr[TL::LOADS];
    if (wave < nkb) {
        TL::load(TL::rsrc(kh, (int64_t)wave * 32, S, D, a.D), a.D, a.D, kr);
        TL::load(TL::rsrc(vh, (int64_t)wave * 32, S, D, a.D), a.D, a.D, vr);
    }
    for (int kb = wave; kb < nkb; kb += 4) {
        const int64_t k0 = (int64_t)kb * 32;
        TL::store(kt, kr);
        TL::store(vt, vr);
        const bool bad = a.causal && kb == qb && any_nonfinite(kr);
        wave_lds_fence();
        if (kb + 4 < nkb) {
            TL::load(TL::rsrc(kh, k0 + 128, S, D, a.D), a.D, a.D, kr);
            TL::load(TL::rsrc(vh, k0 + 128, S, D, a.D), a.D, a.D, vr);
        }
        f32x16 s = mma_d<DP>(kt, [&](int j) { return qf[j]; });
        const f32x16 dp = mma_d<DP>(vt, [&](int j) { return gf[j]; });
        // last key of this lane's query inside the block, from row 4 h
        const int last = (k0 + 32 > S || (a.causal && kb == qb) ? last_key(a, q0, k0) : 31) - 4 * h;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            float x = s[q] * a.scale;
            if constexpr (MASK)
                if (qi < S && k0 + acc_row(q, h) < S) x += a.mask[qi * S + k0 + acc_row(q, h)];
            const float ds = exp2_hw((x - li) * kLog2e) * (dp[q] - di);
            s[q] = acc_row(q, 0) > last ? 0.f : ds;
        }
        if (bad) add_nonfinite<DP, true>(kt, s, acc);
        mma_rows<DP>(kt, s, acc);
        wave_lds_fence();
    }
    TL::store_acc(kt, acc);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < DT; ++i) {
        const int ch = (int)threadIdx.x + 256 * i, row = ch / TL::CPR, d = 4 * (ch % TL::CPR);
        f32x4 v = *reinterpret_cast<const f32x4*>(&tiles[0][0][row * TL::LD + d]);
#pragma unroll
        for (int w = 1; w < 4; ++w) v += *reinterpret_cast<const f32x4*>(&tiles[w][0][row * TL::LD + d]);
        if (q0 + row < S && d < a.D)
            *reinterpret_cast<f32x4*>(&a.dq[((int64_t)bh * S + q0 + row) * D + d]) = v * a.scale;
    }
}

// -------------------------------------------------------------------- dK, dV
// One workgroup per (b, K/V head, group of query heads, 32 keys): the waves
// take every 4th (head, query block) of the group. K stays in registers and V
// in an LDS tile that the waves share (at D = 64 this form spills 16 VGPRs, 24
// with a mask, and both in registers spilled more);
// Q and dO rows go through the wave's LDS tiles and are read both ways:
// S = Q.K^T, dP = dO.V^T (lane = key, registers = queries), dV^T += dO^T.P,
// dK^T += Q^T.dS.
template <int DP, bool MASK>
__global__ __launch_bounds__(256, kWgPerCu<DP>) void attn_f32_bwd_dkdv(F32AttnArgs a) {
    typedef Tile32<DP> TL;
    constexpr int DT = TL::DT;
    __shared__ __attribute__((aligned(16))) float tiles[4][2][TL::FLOATS];
    __shared__ __attribute__((aligned(16))) float vtile[TL::FLOATS];  // the workgroup's V rows
    __shared__ __attribute__((aligned(16))) float stat[4][2][32];     // lse, Delta of the wave's queries
    const int lane = lane_id(), wave = wave_id(), col = lane & 31, h = lane >> 5;
    const int ngrp = a.B * a.Hkv * a.groups;
    const int kb = (int)(blockIdx.x / ngrp);  // heaviest (causal) key blocks first
    const int grp = head_of((int)(blockIdx.x % ngrp), ngrp);
    const int b = grp / (a.Hkv * a.groups), hk = grp / a.groups % a.Hkv, g = grp % a.groups;
    const int rep = a.H / a.Hkv, per = rep / a.groups;  // query heads per K/V head, per group
    const int64_t S = a.S, D = a.D, HD = (int64_t)a.H * D;
    const int64_t k0 = (int64_t)kb * 32, bhk = (int64_t)b * a.Hkv + hk;
    float *qt = tiles[wave][0], *gt = tiles[wave][1];

    f32x4 kf[DP / 8];
    TL::load_along_d(TL::rsrc(a.k + bhk * S * D, k0, S, D, a.D), a.D, a.D, kf);
    if (wave == 0) {
        f32x4 t[TL::LOADS];
        TL::load(TL::rsrc(a.v + bhk * S * D, k0, S, D, a.D), a.D, a.D, t);
        TL::store(vtile, t);
    }
    __syncthreads();
    const int first = a.causal ? kb : 0, nqb = a.nblk - first, total = nqb * per;
    f32x16 ak[DT], av[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) ak[t] = av[t] = zero16();

    f32x4 qr[TL::LOADS], gr[TL::LOADS];
    float st = 0.f;
    // the next block's rows are requested in two steps, each once the registers
    // of a finished product are free, with the remaining products to land
    auto fetch_q = [&](int it) {
        const int hq = hk * rep + g * per + it / nqb;
        const int64_t bh = (int64_t)b * a.H + hq, q0 = (int64_t)(first + it % nqb) * 32;
        TL::load(TL::rsrc(a.q + bh * S * D, q0, S, D, a.D), a.D, a.D, qr);
        st = q0 + col < S ? (h ? a.delta : a.lse)[bh * S + q0 + col] : 0.f;
    };
    auto fetch_g = [&](int it) {
        const int hq = hk * rep + g * per + it / nqb;
        const int64_t q0 = (int64_t)(first + it % nqb) * 32;
        TL::load(TL::rsrc(a.dout + (int64_t)b * S * HD + (int64_t)hq * D, q0, S, HD, a.D), (uint32_t)HD, a.D, gr);
    };
    if (wave < total) {
        fetch_q(wave);
        fetch_g(wave);
    }
    for (int it = wave; it < total; it += 4) {
        const int qb = first + it % nqb;
        const int64_t q0 = (int64_t)qb * 32;
        TL::store(qt, qr);
        TL::store(gt, gr);
        stat[wave][h][col] = st;
        const bool bad = a.causal && qb == kb && (any_nonfinite(qr) || any_nonfinite(gr));
        wave_lds_fence();
        f32x16 s = mma_d<DP>(qt, [&](int j) { return kf[j]; });
        f32x16 dp = mma_d<DP>(gt, [&](int j) { return TL::along_d(vtile, j); });
        if (it + 4 < total) fetch_q(it + 4);
        // queries [lo, hi] of the block read this lane's key, from row 4 h
        const int lo = (a.causal && qb == kb ? col : 0) - 4 * h;
        const int hi = (q0 + 32 > S ? (int)(S - 1 - q0) : 31) - 4 * h;
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
            const f32x4 li = *reinterpret_cast<const f32x4*>(&stat[wave][0][8 * g4 + 4 * h]);
            const f32x4 di = *reinterpret_cast<const f32x4*>(&stat[wave][1][8 * g4 + 4 * h]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int q = 4 * g4 + e;
                float x = s[q] * a.scale;
                if constexpr (MASK) {
                    const int64_t qi = q0 + acc_row(q, h), key = k0 + col;
                    if (qi < S && key < S) x += a.mask[qi * S + key];
                }
                const bool off = acc_row(q, 0) < lo || acc_row(q, 0) > hi;
                const float p = exp2_hw(off ? kNegInf : (x - li[e]) * kLog2e);
                const float ds = p * (dp[q] - di[e]);
                s[q] = p;
                dp[q] = off ? 0.f : ds;
            }
            __builtin_amdgcn_sched_barrier(0);  // lse and Delta of one row group at a time
        }
        if (bad) {
            add_nonfinite<DP, false>(gt, s, av);
            add_nonfinite<DP, false>(qt, dp, ak);
        }
        mma_rows<DP>(gt, s, av);
        if (it + 4 < total) fetch_g(it + 4);
        mma_rows<DP>(qt, dp, ak);
        wave_lds_fence();
    }
    TL::store_acc(qt, ak);
    TL::store_acc(gt, av);
    __syncthreads();
    const int64_t part = (bhk * a.groups + g) * S;  // groups == 1: the outputs themselves
#pragma unroll
    for (int i = 0; i < 2 * DT; ++i) {
        const int which = i / DT, ch = (int)threadIdx.x + 256 * (i % DT), row = ch / TL::CPR, d = 4 * (ch % TL::CPR);
        f32x4 v = *reinterpret_cast<const f32x4*>(&tiles[0][which][row * TL::LD + d]);
#pragma unroll
        for (int w = 1; w < 4; ++w) v += *reinterpret_cast<const f32x4*>(&tiles[w][which][row * TL::LD + d]);
        if (which == 0) v *= a.scale;
        if (k0 + row < S && d < a.D)
            *reinterpret_cast<f32x4*>(&(which ? a.dv : a.dk)[(part + k0 + row) * D + d]) = v;
    }
}

// dk, dv = the groups' partials summed in group order; n4 16-byte vectors
// each, per_head4 of them per K/V head.
__global__ __launch_bounds__(256) void attn_f32_bwd_sum(const f32x4* __restrict__ pk, const f32x4* __restrict__ pv,
                                                        f32x4* __restrict__ dk, f32x4* __restrict__ dv, int groups,
                                                        int64_t per_head4, int64_t n4) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= 2 * n4) return;
    const bool second = i >= n4;
    const int64_t j = second ? i - n4 : i;
    const f32x4* src = (second ? pv : pk) + j / per_head4 * per_head4 * groups + j % per_head4;
    f32x4 v = src[0];
    for (int g = 1; g < groups; ++g) v += src[g * per_head4];
    (second ? dv : dk)[j] = v;
}

F32AttnArgs base_args(const mc_attn_desc& d, const void* q, const void* k, const void* v, const float* mask) {
    F32AttnArgs a{};
    a.q = static_cast<const float*>(q);
    a.k = static_cast<const float*>(k);
    a.v = static_cast<const float*>(v);
    a.mask = mask;
    a.S = d.seq;
    a.B = (int)d.batch; a.H = d.heads; a.Hkv = d.kv_heads; a.D = d.head_dim;
    a.nblk = (int)((d.seq + 31) / 32);
    a.causal = d.causal ? 1 : 0;
    a.scale = d.scale;
    a.groups = 1;
    return a;
}

}  // namespace

namespace {
bool tiles_take(const mc_attn_desc& d) {
    return d.dtype == MC_F32 && d.head_dim % 4 == 0 && d.head_dim <= 128 &&
           attention_f32_tiles_fit(d.seq, d.batch * d.heads);
}
}  // namespace
bool attention_f32_mfma_fwd(const mc_attn_desc& d) {
    return tiles_take(d) && !attention_f32_rows_fwd(d.seq, d.head_dim);
}
bool attention_f32_mfma_bwd(const mc_attn_desc& d) {
    return tiles_take(d) && !attention_f32_rows_bwd(d.seq, d.head_dim, d.heads / d.kv_heads);
}

int attention_f32_groups(const mc_attn_desc& d) {
    const int rep = d.heads / d.kv_heads;
    const int64_t per_group = (d.seq + 31) / 32 * d.batch * d.kv_heads;
    for (int groups = 1; groups < rep; ++groups)
        if (rep % groups == 0 && per_group * groups >= 1024) return groups;
    return rep;
}

hipError_t launch_attention_f32_fwd(const mc_attn_desc& d, const void* q, const void* k, const void* v,
                                    const float* mask, void* o, float* lse, hipStream_t stream) {
    F32AttnArgs a = base_args(d, q, k, v, mask);
    a.out = static_cast<float*>(o);
    a.lse = lse;
    const dim3 grid((unsigned)((int64_t)a.nblk * a.B * a.H));
    auto go = [&](auto dp) {
        constexpr int DP = decltype(dp)::value;
        if (mask) attn_f32_fwd<DP, true><<<grid, 256, 0, stream>>>(a);
        else attn_f32_fwd<DP, false><<<grid, 256, 0, stream>>>(a);
    };
    if (d.head_dim <= 32) go(std::integral_constant<int, 32>{});
    else if (d.head_dim <= 64) go(std::integral_constant<int, 64>{});
    else go(std::integral_constant<int, 128>{});
    return hipGetLastError();
}

hipError_t launch_attention_f32_bwd(const mc_attn_desc& d, const void* q, const void* k, const void* v,
                                    const float* mask, const void* o, const float* lse, const void* dout, void* dq,
                                    void* dk, void* dv, float* delta, float* dk_part, float* dv_part,
                                    hipStream_t stream) {
    F32AttnArgs a = base_args(d, q, k, v, mask);
    a.o = static_cast<const float*>(o);
    a.dout = static_cast<const float*>(dout);
    a.lse = const_cast<float*>(lse);
    a.delta = delta;
    a.groups = attention_f32_groups(d);
    a.dq = static_cast<float*>(dq);
    a.dk = a.groups > 1 ? dk_part : static_cast<float*>(dk);
    a.dv = a.groups > 1 ? dv_part : static_cast<float*>(dv);
    const dim3 gq((unsigned)((int64_t)a.nblk * a.B * a.H));
    const dim3 gk((unsigned)((int64_t)a.nblk * a.B * a.Hkv * a.groups));
    auto go = [&](auto dp) {
        constexpr int DP = decltype(dp)::value;
        if (mask) {
            attn_f32_bwd_dq<DP, true><<<gq, 256, 0, stream>>>(a);
            attn_f32_bwd_dkdv<DP, true><<<gk, 256, 0, stream>>>(a);
        } else {
            attn_f32_bwd_dq<DP, false><<<gq, 256, 0, stream>>>(a);
            attn_f32_bwd_dkdv<DP, false><<<gk, 256, 0, stream>>>(a);
        }
    };
    if (d.head_dim <= 32) go(std::integral_constant<int, 32>{});
    else if (d.head_dim <= 64) go(std::integral_constant<int, 64>{});
    else go(std::integral_constant<int, 128>{});
    if (a.groups > 1) {
        const int64_t per4 = d.seq * d.head_dim / 4, n4 = per4 * d.batch * d.kv_heads;
        attn_f32_bwd_sum<<<dim3((unsigned)((2 * n4 + 255) / 256)), 256, 0, stream>>>(
            reinterpret_cast<const f32x4*>(dk_part), reinterpret_cast<const f32x4*>(dv_part),
            static_cast<f32x4*>(dk), static_cast<f32x4*>(dv), a.groups, per4, n4);
    }
    return hipGetLastError();
}

}  // namespace mc
