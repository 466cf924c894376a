// Products of a few activation rows with a weight matrix, y[n, N] = x[n, K] w[N, K]^T (decode steps; include/skyrl_layers.h).
//
// Bound: the weights' bytes. At 1 to 128 rows a weight matrix is read once and used little, and what the time went on
// before was how it was read: the library's tiles for these shapes leave most CUs idle or few loads in flight. Here:
//   one row   a wave per weight row (or gate and up row), lanes along the depth, so that every load is 1 KB of one row.
//   more      a wave owns 16 NT weight rows and a share of the depth alone: it fetches its pieces (64 deep, whole 128-byte
//             lines, chunks xor-swizzled by the row) with direct loads into LDS of its own, S of them in flight, and
//             never meets the other waves until the sums of the shares are joined. Few weight rows are cut into
//             `splits` shares of the depth across workgroups too, each with f32 sums of its own that the next norm adds.
// Measured on one MI355X, weights from HBM, us (GB/s of weights) against the library's:
//   N, K            1 row            16 rows          32 rows          64 rows
//   2048, 2048      3.8 / 11.0       4.1 / 11.1       4.4 / 11.3       5.3 / 11.8
//   2048, 6144      6.5 / 12.0       7.4 / 12.2       7.8 / 16.8       9.7 / 19.7
//   3648, 2048      4.9 / 12.1       5.5 / 12.0       6.5 / 11.8       8.5 / 12.2   (no splits)
//   12288, 2048     10.6 / 16.7      12.7 / 16.6      13.1 / 16.8      16.3 / 18.3  (no splits; 4.8 TB/s at one row)
//   32768, 2048     23.6 / 35.0      26.3 / 34.5      29.5 / 36.8      30.3 / 37.1  (no splits; 5.7 TB/s at one row)
// Batches (a head's up-projections of latent attention, 512 x 128 and 128 x 512): 16 heads, 1 / 64 rows, both products with the
// copy that the library's needed: 15.4 / 17.1 us, here 5.9 / 7.6 us.
#include "gate.h"

namespace skyrl {
namespace {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void gbl_void;

enum Mode { kRound, kParts, kGated };

struct RowsProduct {
    const uint16_t* x;
    int64_t ldx;
    int n, K;
    const uint16_t* w;
    int64_t ldw;
    int N;  // output columns; kGated: gate rows, the up rows follow
    const uint16_t* bias;
    Gate gate;
    void* out;
    int64_t ldo, ldsplit;
    int row_blocks;  // gridDim.z = batch row_blocks
    int64_t x_batch, w_batch, out_batch;
};

template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void lds_read(s16x8& v, uint32_t at, int offset) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(offset));
}
__device__ const uint4 kZero16 = {0u, 0u, 0u, 0u};

// One row: R consecutive outputs per wave (kGated: R pairs), C loads of every weight row in flight.
template <int MODE, int C, int NWV>
__global__ __launch_bounds__(NWV* kWave) void one_row_kernel(RowsProduct p) {
    constexpr int R = MODE == kGated ? 2 : 1;
    const int lane = threadIdx.x & 63, n = blockIdx.x * NWV + (threadIdx.x >> 6);
    if (n >= p.N) return;
    const uint16_t* w[R];
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        w[r] = p.w + (int64_t)(n + r * p.N) * p.ldw;
        acc[r] = 0.f;
    }
    for (int k = lane * 8; k < p.K; k += 512 * C) {
        uint4 wv[R][C], xv[C];
#pragma unroll
        for (int j = 0; j < C; ++j) {
            const int at = min(k + j * 512, p.K - 8);
#pragma unroll
            for (int r = 0; r < R; ++r) wv[r][j] = *reinterpret_cast<const uint4*>(w[r] + at);
            xv[j] = *reinterpret_cast<const uint4*>(p.x + at);
        }
#pragma unroll
        for (int j = 0; j < C; ++j) {
            if (k + j * 512 >= p.K) break;
            float x[8];
            unpack8(xv[j], x);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float v[8];
                unpack8(wv[r][j], v);
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[r] = fmaf(v[i], x[i], acc[r]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = wave_sum(acc[r]);
    if (lane) return;
    float y = acc[0];
    if constexpr (MODE == kGated) y = gated(y, acc[1], p.gate);
    else if (p.bias) y += ld(p.bias + n);
    if constexpr (MODE == kParts) st(reinterpret_cast<float*>(p.out) + n, y);
    else st(reinterpret_cast<uint16_t*>(p.out) + n, y);
}

// NT 16-row weight tiles (kGated: half of each matrix) and MT 16-row tiles of x per workgroup, the depth in gridDim.y * WK shares;
// blocks of MT tiles and products of a batch along z.
template <int MODE, int NT, int MT, int WK, int S>
__global__ __launch_bounds__(WK* kWave) void rows_product_kernel(RowsProduct p) {
    constexpr int BN = 16 * NT, BM = 16 * MT, WP = 2 * NT, XP = 2 * MT, L = WP + XP;  // 1 KB pieces: 8 rows, 64 deep
    constexpr int OC = MODE == kGated ? BN / 2 : BN;  // output columns
    constexpr int kStage = (BN + BM) * 64;            // elements
    constexpr int LR = BN + 4;                        // a row of a share's sums
    constexpr int kSums = WK * BM * LR * 2, kPieces = WK * S * kStage;
    static_assert(MODE != kGated || NT % 2 == 0, "gate and up rows");
    static_assert(S <= 4, "the waits below");
    __shared__ __attribute__((aligned(16))) uint16_t smem[kPieces > kSums ? kPieces : kSums];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * OC, batch = blockIdx.z / p.row_blocks, m0 = blockIdx.z % p.row_blocks * BM;
    const int steps = (p.K + 63) / 64, shares = gridDim.y * WK, share = blockIdx.y * WK + wave;
    const int s0 = (int)((int64_t)steps * share / shares), nk = (int)((int64_t)steps * (share + 1) / shares) - s0;
    uint16_t* own = smem + wave * (S * kStage);
    // this lane's 16 bytes of every piece: row lane / 8, chunk (lane % 8) ^ row, so that 16 rows read at a time lie in
    // different banks; rows past the last are the last again and are not stored
    const int r8 = lane >> 3, ch = ((lane & 7) ^ r8) * 8;
    const uint16_t *ws[WP], *xs[XP];
#pragma unroll
    for (int i = 0; i < WP; ++i) {
        const int r = i * 8 + r8;
        const int row = MODE == kGated && r >= OC ? p.N + min(n0 + r - OC, p.N - 1) : min(n0 + r, p.N - 1);
        ws[i] = p.w + batch * p.w_batch + row * p.ldw + s0 * 64 + ch;
    }
#pragma unroll
    for (int i = 0; i < XP; ++i) xs[i] = p.x + batch * p.x_batch + min(m0 + i * 8 + r8, p.n - 1) * p.ldx + s0 * 64 + ch;
    auto fetch = [&](int t) {
        uint16_t* dst = own + (t % S) * kStage;
        const bool in = (s0 + t) * 64 + ch < p.K;  // K is a multiple of 8
#pragma unroll
        for (int i = 0; i < WP; ++i) {
            const void* src = in ? (const void*)(ws[i] + t * 64) : (const void*)&kZero16;
            __builtin_amdgcn_global_load_lds((gbl_void*)src, (lds_void*)(dst + i * 512), 16, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            const void* src = in ? (const void*)(xs[i] + t * 64) : (const void*)&kZero16;
            __builtin_amdgcn_global_load_lds((gbl_void*)src, (lds_void*)(dst + (WP + i) * 512), 16, 0, 0);
        }
    };
    f32x4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < S; ++t)
        if (t < nk) fetch(t);
    const uint32_t base = (uint32_t)(uintptr_t)(lds_void*)own + c * 128;
    for (int t = 0; t < nk; ++t) {
        const int left = nk - 1 - t;  // pieces after this one; at most S - 1 of them are under way
        if (left >= S - 1) wait_loads<(S - 1) * L>();
        else if (S > 3 && left == 2) wait_loads<2 * L>();
        else if (S > 2 && left == 1) wait_loads<L>();
        else wait_loads<0>();
        // The reads are not the compiler's: it would wait for every load into LDS under way before one. They are waited
        // for at once, and their registers tied past the wait.
        s16x8 wf[2][NT], xf[2][MT];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t at = base + (t % S) * kStage * 2 + ((h * 4 + g) ^ (c & 7)) * 16;
#pragma unroll
            for (int n = 0; n < NT; ++n) lds_read(wf[h][n], at, n * 2048);
#pragma unroll
            for (int m = 0; m < MT; ++m) lds_read(xf[h][m], at, (NT + m) * 2048);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int n = 0; n < NT; ++n) asm volatile("" : "+v"(wf[h][n]));
#pragma unroll
            for (int m = 0; m < MT; ++m) asm volatile("" : "+v"(xf[h][m]));
        }
        if (t + S < nk) fetch(t + S);  // over the piece that has been read
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][n], xf[h][m], acc[m][n], 0, 0, 0);
    }
    __syncthreads();  // nothing is under way any more: the sums take the pieces' place
    float* sums = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
            *reinterpret_cast<f32x4*>(sums + (wave * BM + m * 16 + c) * LR + n * 16 + 4 * g) = acc[m][n];
    __syncthreads();
    auto total = [&](int m, int n) {
        f32x4 s = *reinterpret_cast<f32x4*>(sums + m * LR + n);
#pragma unroll
        for (int k = 1; k < WK; ++k) s += *reinterpret_cast<f32x4*>(sums + (k * BM + m) * LR + n);
        return s;
    };
    const bool four = p.N % 4 == 0 && p.ldo % 4 == 0 && p.out_batch % 4 == 0 && (reinterpret_cast<uintptr_t>(p.out) & 7) == 0;
    for (int i = tid; i < BM * (OC / 4); i += WK * kWave) {
        const int m = i / (OC / 4), n = i % (OC / 4) * 4, col = n0 + n;
        if (m0 + m >= p.n || col >= p.N) continue;
        f32x4 y = total(m, n);
        if constexpr (MODE == kGated) {
            const f32x4 u = total(m, OC + n);
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = gated(y[j], u[j], p.gate);
        } else if (p.bias && blockIdx.y == 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] += ld(p.bias + min(col + j, p.N - 1));
        }
        if constexpr (MODE == kParts) {
            float* o = reinterpret_cast<float*>(p.out) + blockIdx.y * p.ldsplit + (m0 + m) * p.ldo + col;
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

constexpr int kWide = 8192;       // output columns from which wider tiles still fill the chip and read x less often
constexpr int kFill = 256;        // workgroups that a split product is cut into
constexpr int kManyRowsCols = 4096;

bool rows_fit(int n, int K, int N, bool gated) {
    // Above 64 rows the library's tiles are as fast on wide matrices (128 rows, 12288 x 2048: 21.0 against 20.7 us) and
    // slower on narrow ones (2048 x 2048: 6.9 against 11.5 us, 2048 x 6144: 13.6 against 18.2 us, in parts).
    return n > 0 && K > 0 && N > 0 && K % 8 == 0 && (n <= 64 || (n <= 128 && N <= kManyRowsCols && !gated));
}

int splits_for(int n, int K, int N) {
    if (n == 1) return 1;
    const int bn = n <= 16 ? 16 : 32, tiles = (N + bn - 1) / bn, most = K / 64 / 4;  // a piece per wave at least
    int s = (kFill + tiles / 2) / tiles;
    if (s > most) s = most;
    return s < 1 ? 1 : s > 8 ? 8 : s;
}

template <int MODE, int NT, int MT, int WK, int S>
void launch_rows(RowsProduct p, int splits, hipStream_t s, int batch = 1) {
    constexpr int OC = MODE == kGated ? 8 * NT : 16 * NT;
    p.row_blocks = (p.n + 16 * MT - 1) / (16 * MT);
    hipLaunchKernelGGL((rows_product_kernel<MODE, NT, MT, WK, S>), dim3((p.N + OC - 1) / OC, splits, p.row_blocks * batch),
                       dim3(WK * kWave), 0, s, p);
}

}  // namespace
}  // namespace skyrl

using namespace skyrl;

extern "C" int32_t skyrl_rows_product_fits(int32_t n, int32_t K, int32_t N, int32_t gated) {
    return rows_fit(n, K, N, gated != 0);
}

extern "C" int32_t skyrl_rows_product_splits(int32_t n, int32_t K, int32_t N) { return splits_for(n, K, N); }

extern "C" int skyrl_rows_product(const void* x, int64_t ldx, int32_t n, int32_t K, const void* w, int64_t ldw, int32_t N,
                                  const void* bias, int32_t act, float alpha, float limit, int32_t splits, void* out,
                                  int64_t ldo, void* stream) {
    const bool gate = act >= 0;
    SKYRL_REQUIRE(rows_fit(n, K, N, gate), "rows_product: sizes that the library takes");
    SKYRL_REQUIRE(x && w && out, "rows_product: null pointer");
    SKYRL_REQUIRE(aligned16(x) && aligned16(w) && ldx % 8 == 0 && ldw % 8 == 0 && ldw >= K && (n == 1 || ldx >= K),
                  "rows_product: rows must be 16-byte aligned");
    SKYRL_REQUIRE((reinterpret_cast<uintptr_t>(out) & (splits ? 3 : 1)) == 0 && (n == 1 || ldo >= N), "rows_product: bad output");
    SKYRL_REQUIRE(!gate || (!bias && splits == 0 && (act == SKYRL_ACT_SILU || act == SKYRL_ACT_GELU_TANH || act == SKYRL_ACT_CLAMPED)),
                  "rows_product: a gated product has an activation, no bias and no splits");
    SKYRL_REQUIRE(splits == 0 || splits == splits_for(n, K, N), "rows_product: splits are skyrl_rows_product_splits'");
    const RowsProduct p{reinterpret_cast<const uint16_t*>(x), ldx, n, K, reinterpret_cast<const uint16_t*>(w), ldw, N,
                        reinterpret_cast<const uint16_t*>(bias), Gate{act, alpha, limit}, out, ldo, (int64_t)n * ldo, 1, 0, 0, 0};
    hipStream_t s = as_stream(stream);
    if (n == 1) {  // 4 loads of a row: 2048 deep at a time
        const dim3 grid((N + 3) / 4), block(4 * kWave);
        if (gate) hipLaunchKernelGGL((one_row_kernel<kGated, 4, 4>), grid, block, 0, s, p);
        else if (splits) hipLaunchKernelGGL((one_row_kernel<kParts, 4, 4>), grid, block, 0, s, p);
        else hipLaunchKernelGGL((one_row_kernel<kRound, 4, 4>), grid, block, 0, s, p);
        return check_launch("one_row_kernel");
    }
    // Wide tiles where there are columns enough, since every workgroup reads x again; else 16 rows of weights, so that
    // the chip is full (3648 x 2048 at 64 rows: 8.5 us with 16, 9.4 with 32).
    if (gate) {
        if (n <= 16) launch_rows<kGated, 2, 1, 4, 2>(p, 1, s);
        else if (n <= 32) launch_rows<kGated, 4, 2, 4, 2>(p, 1, s);
        else launch_rows<kGated, 4, 4, 2, 2>(p, 1, s);
    } else if (splits) {
        if (n <= 16) launch_rows<kParts, 1, 1, 4, 4>(p, splits, s);
        else if (n <= 32) launch_rows<kParts, 2, 2, 4, 2>(p, splits, s);
        else if (n <= 64) launch_rows<kParts, 2, 4, 4, 2>(p, splits, s);
        else launch_rows<kParts, 2, 8, 4, 1>(p, splits, s);
    } else if (N >= kWide) {
        if (n <= 16) launch_rows<kRound, 2, 1, 4, 2>(p, 1, s);
        else if (n <= 32) launch_rows<kRound, 4, 2, 4, 2>(p, 1, s);
        else launch_rows<kRound, 4, 4, 2, 2>(p, 1, s);
    } else {
        if (n <= 16) launch_rows<kRound, 1, 1, 4, 4>(p, 1, s);
        else if (n <= 32) launch_rows<kRound, 1, 2, 4, 3>(p, 1, s);
        else if (n <= 64) launch_rows<kRound, 1, 4, 4, 2>(p, 1, s);
        else launch_rows<kRound, 1, 8, 4, 2>(p, 1, s);
    }
    return check_launch("rows_product_kernel");
}

extern "C" int skyrl_rows_batch(const void* x, int64_t ldx, int64_t x_batch, int32_t n, int32_t K, const void* w, int64_t ldw,
                                int64_t w_batch, int32_t N, int32_t batch, void* out, int64_t ldo, int64_t out_batch,
                                void* stream) {
    SKYRL_REQUIRE(n >= 0 && K > 0 && N > 0 && K % 8 == 0 && batch > 0 && (int64_t)batch * ((n + 63) / 64) <= 65535,
                  "rows_batch: bad sizes");
    if (n == 0) return SKYRL_OK;
    SKYRL_REQUIRE(x && w && out, "rows_batch: null pointer");
    SKYRL_REQUIRE(aligned16(x) && aligned16(w) && ldx % 8 == 0 && ldw % 8 == 0 && x_batch % 8 == 0 && w_batch % 8 == 0 &&
                      ldw >= K && (reinterpret_cast<uintptr_t>(out) & 1) == 0,
                  "rows_batch: rows must be 16-byte aligned");
    const RowsProduct p{reinterpret_cast<const uint16_t*>(x), ldx, n, K, reinterpret_cast<const uint16_t*>(w), ldw, N, nullptr,
                        Gate{-1, 0.f, 0.f}, out, ldo, 0, 1, x_batch, w_batch, out_batch};
    hipStream_t s = as_stream(stream);
    // A head's matrix is small: all its pieces are under way at once. Shallow ones (the queries' up-projection) take two
    // waves a workgroup and 32 columns, deep ones (the outputs') four waves and 16 columns.
    if (K <= 256) {
        if (n <= 16) launch_rows<kRound, 2, 1, 2, 2>(p, 1, s, batch);
        else if (n <= 32) launch_rows<kRound, 2, 2, 2, 2>(p, 1, s, batch);
        else launch_rows<kRound, 2, 4, 2, 1>(p, 1, s, batch);
    } else {
        if (n <= 16) launch_rows<kRound, 1, 1, 4, 2>(p, 1, s, batch);
        else if (n <= 32) launch_rows<kRound, 1, 2, 4, 2>(p, 1, s, batch);
        else launch_rows<kRound, 1, 4, 4, 2>(p, 1, s, batch);
    }
    return check_launch("rows_product_kernel");
}
