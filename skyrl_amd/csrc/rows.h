// What the products of a few rows (rows_product.hip, normed_product.hip) share: their operands and what becomes of the sums.
#pragma once
#include "gate.h"
#include "stream.h"

namespace skyrl {

enum Mode { kRound, kParts, kGated, kCapped };

struct RowsProduct {
    const uint16_t* x;
    int64_t ldx;
    int n, K;
    const uint16_t* w;
    int64_t ldw;
    int N;  // output columns; kGated: gate rows, the up rows follow
    const uint16_t* bias;
    Gate gate;
    int turn0, turn1;  // kRound: columns whose rounded values go through tanh
    float cap;         // kCapped: the rounded values between -cap and cap by tanh, f32 (0: as they are)
    void* out;
    int64_t ldo, ldsplit;
    int row_blocks;  // gridDim.z = batch row_blocks
    int64_t x_batch, w_batch, out_batch;
};

template <int MODE, int NT>
constexpr int out_cols() {  // of a workgroup
    return MODE == kGated ? 8 * NT : 16 * NT;
}

// What follows a product and moves little stands here instead of in a launch of its own (3 to 6 us of a decode step each): the
// logits' cap and the tanh of a low-rank product's inputs, on the rounded values as those launches had them.
template <int MODE, class St, int WK>
__device__ __forceinline__ void put_rows(const uint16_t* smem, const RowsProduct& p, int n0, int m0, int batch) {
    constexpr int BM = St::BM, OC = MODE == kGated ? St::BN / 2 : St::BN;
    const int tid = threadIdx.x;
    const bool four = p.N % 4 == 0 && p.ldo % 4 == 0 && p.out_batch % 4 == 0 && (reinterpret_cast<uintptr_t>(p.out) & 7) == 0;
    for (int i = tid; i < BM * (OC / 4); i += WK * kWave) {
        const int m = i / (OC / 4), n = i % (OC / 4) * 4, col = n0 + n;
        if (m0 + m >= p.n || col >= p.N) continue;
        f32x4 y = St::total(smem, m, n);
        if constexpr (MODE == kGated) {
            const f32x4 u = St::total(smem, m, OC + n);
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = gated(y[j], u[j], p.gate);
        } else if (p.bias && blockIdx.y == 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] += ld(p.bias + min(col + j, p.N - 1));
        }
        if constexpr (MODE == kRound) {
            if (col + 3 >= p.turn0 && col < p.turn1) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (col + j >= p.turn0 && col + j < p.turn1) y[j] = tanhf(bf16_to_f32(f32_to_bf16(y[j])));
            }
        }
        if constexpr (MODE == kCapped) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float v = bf16_to_f32(f32_to_bf16(y[j]));
                y[j] = p.cap > 0.f ? p.cap * tanhf(v / p.cap) : v;
            }
        }
        if constexpr (MODE == kParts || MODE == kCapped) {
            float* o = reinterpret_cast<float*>(p.out) + (MODE == kParts ? blockIdx.y * p.ldsplit : 0) + (m0 + m) * p.ldo + col;
            if (four) st4(o, make_float4(y[0], y[1], y[2], y[3]));
            else
                for (int j = 0; j < 4 && col + j < p.N; ++j) st(o + j, y[j]);
        } else {
            uint16_t* o = reinterpret_cast<uint16_t*>(p.out) + batch * p.out_batch + (m0 + m) * p.ldo + col;
            if (four) st4(o, make_float4(y[0], y[1], y[2], y[3]));
            else
                for (int j = 0; j < 4 && col + j < p.N; ++j) st(o + j, y[j]);
        }
    }
}

// NT 16-row weight tiles (kGated: half of each matrix) and MT 16-row tiles of x per workgroup, the depth in `splits` * WK shares;
// blocks of MT tiles and products of a batch along z.
template <int MODE, int NT, int MT, int WK, int S, bool ONCE = true, bool EXACT = false>
__device__ __forceinline__ void rows_block(const RowsProduct& p, uint16_t* smem, int bx, int by, int bz, int splits) {
    using St = Stream<NT, MT, WK, S, false, ONCE, EXACT>;
    constexpr int BM = St::BM, OC = out_cols<MODE, NT>();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = bx * OC, batch = bz / p.row_blocks, m0 = bz % p.row_blocks * BM;
    const int steps = (p.K + 63) / 64, shares = splits * WK, share = by * WK + wave;
    const int s0 = (int)((int64_t)steps * share / shares), nk = (int)((int64_t)steps * (share + 1) / shares) - s0;
    f32x4 acc[MT][NT];
    St::run(
        smem, p.K, s0, nk,
        [&](int r) {  // rows past the last: the last
            const int row = MODE == kGated && r >= OC ? p.N + min(n0 + r - OC, p.N - 1) : min(n0 + r, p.N - 1);
            return p.w + batch * p.w_batch + row * p.ldw;
        },
        [&](int r) { return p.x + batch * p.x_batch + min(m0 + r, p.n - 1) * p.ldx; }, acc);
    St::store(smem, acc);
    put_rows<MODE, St, WK>(smem, p, n0, m0, batch);
}

}  // namespace skyrl
