// Products of many bf16 rows, y[n, N] = x[n, K] w[N, K]^T rounded once (skyrl_dense_product): the tiles of 256 of wide.h, and smaller
// ones where those would leave the chip partly idle. Each form sums a result in one chain of 32-deep products along the depth, from 0 but
// for kOnce, which begins at a depth of the columns' own and goes round.
#include "wide.h"

namespace skyrl {
namespace {

struct Dense {
    const uint16_t *x, *w;
    int64_t ldx, ldw;
    int n, K, N;
    uint16_t* out;
};

// As product(), with the sums in vector registers.
__device__ __forceinline__ void product_v(f32x4& a, const s16x8& w, const s16x8& x) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(a) : "v"(w), "v"(x));
}

// TM rows x TN columns a workgroup, two by two waves, S stages of 64 deep. A wave's loads of a stage are waited for when those of the S - 1
// behind it are under way; the operands of one 32-deep half are read while the other half's products run. Bound: the loads into LDS, 80
// to 90 GB/s a CU whatever the stages (64 x 32, 256 rows of 2048 x 2048: 8.4 us with 12 stages, 7.9 with 6, 8.0 with the operands of two
// stages read ahead of two others' products); the sums stay in vector registers, since the compiler's form copied them on every turn.
template <int TM, int TN, int S>
__global__ __launch_bounds__(256) void dense_kernel(Dense p) {
    constexpr int BK = 64, WM = 2, WN = 2, NWV = WM * WN, MT = TM / WM / 16, NT = TN / WN / 16;
    constexpr int XL = TM / 8 / NWV, WL = TN / 8 / NWV, L = XL + WL;  // 1 KB pieces of 8 rows a wave and stage
    constexpr uint32_t STAGE = (TM + TN) * BK * 2;
    constexpr int LO = TN + 8;  // a row of the results in LDS
    static_assert(XL * 8 * NWV == TM && WL * 8 * NWV == TN && TM * LO * 2 <= (int)(S * STAGE) && S >= 3 && (S - 1) * L < 64, "tile");
    __shared__ __attribute__((aligned(16))) uint16_t smem[S * STAGE / 2];
    const int ntm = (p.n + TM - 1) / TM, ntn = (p.N + TN - 1) / TN;
    // An XCD takes a run of tiles, the rows of one column of them behind each other: they read the same weights.
    const int64_t tiles = (int64_t)ntm * ntn;
    const int xcd = blockIdx.x % 8;
    const int64_t tile = tiles * xcd / 8 + blockIdx.x / 8;
    if (tile >= tiles * (xcd + 1) / 8) return;
    const int m0 = (int)(tile % ntm) * TM, n0 = (int)(tile / ntm) * TN;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4, wm = wave / WN, wn = wave % WN;
    const int nk = p.K / BK;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void*)smem;
    const __amdgpu_buffer_rsrc_t x_all = whole_buffer(p.x), w_all = whole_buffer(p.w);
    // This lane's 16 bytes of a piece, in bytes from the first row: chunk (lane % 8) ^ (row / 2 % 8), so that the 16 rows that are read at
    // a time lie in different banks. Rows past the last: the last one, not stored.
    uint32_t xo[XL], wo[WL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int r = (wave * XL + i) * 8 + lane / 8;
        xo[i] = (min(m0 + r, p.n - 1) * (uint32_t)p.ldx + (lane % 8 ^ r / 2 % 8) * 8) * 2;
    }
#pragma unroll
    for (int i = 0; i < WL; ++i) {
        const int r = (wave * WL + i) * 8 + lane / 8;
        wo[i] = (min(n0 + r, p.N - 1) * (uint32_t)p.ldw + (lane % 8 ^ r / 2 % 8) * 8) * 2;
    }
    auto fetch = [&](int t, uint32_t at) __attribute__((always_inline)) {  // stage t (the last again past the end) to place `at`
        const int k0 = min(t, nk - 1) * (BK * 2);
        const uint32_t dst = lds0 + at;
#pragma unroll
        for (int i = 0; i < WL; ++i)
            buffer_to_lds(w_all, wo[i], k0, dst + TM * BK * 2 + (wave * WL + i) * 1024);
#pragma unroll
        for (int i = 0; i < XL; ++i)
            buffer_to_lds(x_all, xo[i], k0, dst + (wave * XL + i) * 1024);
    };
    f32x4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    // The operands' reads are not the compiler's: it would wait for every load into LDS under way before one.
    s16x8 xf[2][MT], wf[2][NT];
    const uint32_t xat = lds0 + (wm * MT * 16 + c) * BK * 2, wat = lds0 + (TM + wn * NT * 16 + c) * BK * 2;
    const uint32_t half[2] = {(uint32_t)(g ^ c / 2) * 16, (uint32_t)((4 + g) ^ c / 2) * 16};
    auto operands = [&](uint32_t at, int ks) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < NT; ++n) lds_read(wf[ks][n], wat + at + half[ks], n * 16 * BK * 2);
#pragma unroll
        for (int m = 0; m < MT; ++m) lds_read(xf[ks][m], xat + at + half[ks], m * 16 * BK * 2);
    };
    auto hold = [&](int ks) __attribute__((always_inline)) {  // the operands' registers are in use up to here
#pragma unroll
        for (int n = 0; n < NT; ++n) asm volatile("" : "+v"(wf[ks][n]));
#pragma unroll
        for (int m = 0; m < MT; ++m) asm volatile("" : "+v"(xf[ks][m]));
    };
    auto ready = [&](int ks) __attribute__((always_inline)) {  // all but the reads of the other half have returned
        asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(MT + NT < 15 ? MT + NT : 15) : "memory");
        hold(ks);
    };
    auto products = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n)
                product_v(acc[m][n], wf[ks][n], xf[ks][m]);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int t = 0; t < S; ++t) fetch(t, t * STAGE);
    wait_loads<(S - 1) * L>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    operands(0, 0);
    uint32_t at = 0;
    for (int t = 0; t < nk; ++t) {
        const uint32_t next = at + STAGE == S * STAGE ? 0 : at + STAGE;
        operands(at, 1);
        ready(0);
        products(0);
        wait_loads<(S - 2) * L>();     // this wave's loads of stage t + 1 have landed, its reads of stage t too
        __builtin_amdgcn_s_barrier();  // and everyone's
        asm volatile("" ::: "memory");
        hold(1);
        fetch(t + S, at);
        operands(next, 0);
        products(1);
        at = next;
    }
    wait_loads<0>();  // nothing is under way, into LDS or into the registers of the last reads
    hold(0);
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last products are in their registers
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) asm volatile("" : "+v"(acc[m][n]));
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
            *reinterpret_cast<uint2*>(&smem[((wm * MT + m) * 16 + c) * LO + (wn * NT + n) * 16 + 4 * g]) =
                make_uint2(pack_bf16x2(acc[m][n][0], acc[m][n][1]), pack_bf16x2(acc[m][n][2], acc[m][n][3]));
    __syncthreads();
    for (int i = tid; i < TM * (TN / 8); i += 256) {
        const int r = i / (TN / 8), col = i % (TN / 8) * 8;
        if (m0 + r < p.n && n0 + col < p.N)
            *reinterpret_cast<uint4*>(p.out + (int64_t)(m0 + r) * p.N + n0 + col) = *reinterpret_cast<const uint4*>(&smem[r * LO + col]);
    }
}

template <int TM, int TN, int S>
void launch_dense(const Dense& p, hipStream_t s) {
    const int64_t tiles = (int64_t)((p.n + TM - 1) / TM) * ((p.N + TN - 1) / TN);
    hipLaunchKernelGGL((dense_kernel<TM, TN, S>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(256), 0, s, p);
}

enum Form { kOnce, k64x32, k64x64, k64x128, k128x128, kWide192, kWide256 };
int64_t tiles_of(int n, int N, int tm, int tn) { return (int64_t)((n + tm - 1) / tm) * ((N + tn - 1) / tn); }

// Rounds of whole tiles of 256 that the wide form with tiles of `rows` takes, in hundredths: a tile of 192 is 82 of them, half of
// the columns of one 62 %, 70 where all are halves (their loads have less time to land).
int64_t wide_rounds(int n, int N, int rows) {
    const int64_t tiles = tiles_of(n, N, rows, 256), left = (tiles + 7) / 8, over = left % (kCUs / 8), whole = rows == 256 ? 100 : 82;
    if (2 * tiles <= kCUs) return whole * 70 / 100;
    return left / (kCUs / 8) * whole + (over == 0 ? 0 : 2 * over <= kCUs / 8 ? whole * 62 / 100 : whole);
}

// The form, and whether it is the faster one beside the library's. Up to some 1000 rows the smallest tiles that are one round
// of workgroups (64 x 32 to 64 x 64 fit a CU twice, and 64 x 128 do, so that half a round more costs little): a CU's loads bound
// them, 80 to 90 GB/s, and the library's tiles leave CUs idle. Above, the wide form, beside the library's tiles of 256 x 256.
// us, here / the library's, weights from HBM, both in a captured graph:
//   N, K            256 rows       512            1024           1563           3000          5637          8192
//   2048, 2048      8.2 / 10.8     10.0 / 12.3    14.3 / 16.3    -              -             -             -
//   3408, 2048      9.9 / 12.4     14.0 / 16.5    21.4 / 24.4    -              39.8 / 49.3   73 / 84       94 / 115
//   12352, 2048     25.4 / 29.0    -              48.2 / 56.4    75.5 / 80.0    121 / 141     216 / 298     320 / 378
//   3072, 768       6.1 / 8.6      8.1 / 10.5     -              -              -             31 / 47       38 / 46
//   2048, 512       4.7 / 6.8      5.5 / 8.6      7.0 / 9.7      9.3 / 11.4     12.8 / 14.2   17.5 / 27.9   21.5 / 23.2
//   24640, 4096     -              -              -              267 / 374      456 / 515     837 / 929     1149 / 1218
// One tile of 128 or 256 rows and columns for the whole chip (logits): the wide form, in which weights go past the caches and neighbouring
// columns begin at another depth (wide.h's depth_start; with several tiles of rows they would read x at as many depths):
//   N, K            65 rows       128           256
//   32768, 2048     28.2 / 37.6   30.4 / 40.5   42.3 / 46.2
//   28672, 2048     -             28.7 / 34.2   42.0 / 45.3   (192 pieces of 128 columns of 4096 deep: 60.0 / 57.4, 84.8 / 72.0)
//   40000, 2048     -             40.6 / 51.2   54.5 / 59.5
//   65536, 4096     -             -             121 / 162
//   151936, 2048    -             124 / 175     161 / 219
// Where a line lies: of 2500 sizes (65 to 8192 rows, 8 to 152000 columns, 64 to 12288 deep) those that it takes are 1.29 times as fast as
// the library's (geometric mean; one in a hundred is more than 3 % slower, the worst, 273 x 1280, 10880, 10 %), those that it leaves 0.93
// times. Left, rows x K, N:
//   64 x 32, few of them along a long depth, which the library cuts: 256 x 6144, 24 15.0 / 7.8; 65 x 2048, 512 7.4 / 6.3; 512 x 4096,
//     512 12.0 / 11.4; 65 x 4096, 2560 11.9 / 11.1. With more than half of the CUs, 256 x 4096, 1264 1.20 times as fast. As 64 x 64: 65 x
//     4096, 5120 19.7 / 17.7, and past 4096 deep where rows fill its tiles (256 x 6144, 3072 31.1 / 28.7; 192 x 6144, 4096 is 1.5 times as fast).
//   64 x 128: 384 x 6144, 3072 46 / 36, 512 x 4096, 2560 22.4 / 21.6 (240 of 256 tiles: 1.07); 1400 x 2048, 2048 21.3 / 19.2, whose 352 tiles are 1 3/8 rounds.
//   128 x 128 with up to 192 of the CUs: 1500 x 2048, 1024 20.1 / 14.3, 1563 x 1536, 1536 17.1 / 16.0 (1563 x 2048, 2048, 208 tiles: 20.8 / 20.6
//     alone, and in a step between other launches 22 / 25); 768 x 1536, 4096 17.4 / 16.4, 384 x 1536, 8192 17.8 / 16.2; shallow
//     ones of several rounds where the library's tiles fit: 1024 x 512, 16384 29.5 / 22.7 (1024 x 512, 9280 is even, 1400 x 384, 3408 1.3 times as fast).
//   Shallow and narrow, from 2049 rows: 3000 x 256, 512 7.5 / 6.4, 2049 x 512, 1536 12.5 / 10.1 (4096 x 512, 1536 1.16 times as fast).
//   Columns a multiple of 256, as many rounds as the library: 7091 x 1536, 2048 41 / 38, 6270 x 3072, 2560 81 / 72; past 2048 deep also where
//     a third less: 5637 x 6144, 2048 127 / 113, 6405 x 3072, 7680 0.91 times (5432 x 3072, 3072, 1.33 rounds for 2: 96 / 111). Other columns
//     past 6144 deep: 2844 x 10048, 12160 0.85 times.
Form form_of(int n, int K, int N, bool& faster) {
    faster = true;
    if (n > 64 && n <= 256 && N >= 28672) return kOnce;
    const bool columns = N % 256 != 0;  // that the library's tiles do not fit
    if (n <= 1400 && K <= 6144 && (n <= 1024 || K <= 2048)) {
        const int64_t least = K <= 3072 || n > 96 ? kCUs / 2 : kCUs * 5 / 8;
        int64_t t = tiles_of(n, N, 64, 32);
        if (t <= kCUs) {
            faster = K <= 1024 || t > (K <= 2048 ? kCUs / 8 : least);
            return k64x32;
        }
        if ((t = tiles_of(n, N, 64, 64)) <= kCUs) {
            faster = (K <= 2048 || t > least) && (K <= 4096 || (n > 96 && n <= 192));
            return k64x64;
        }
        t = tiles_of(n, N, 64, 128);
        if ((K <= 2048 || N < 4096) && (t <= kCUs || (K <= 2048 && n > 512 && t <= kCUs * (K <= 1024 ? 22 : 21) / 16))) {
            faster = K <= 3072 || (K <= 4096 && t > kCUs * 3 / 4);
            return k64x128;
        }
        if (K <= 2048 && (t = tiles_of(n, N, 128, 128)) <= kCUs) {
            faster = n <= 256 || columns || K < 1024 || t > kCUs * 7 / 8;
            return k128x128;
        }
    }
    if (K <= 512 && n <= 2048) {
        const bool one = tiles_of(n, N, 64, 128) <= 2 * kCUs;
        faster = one ? N > 32 : columns;
        return one ? k64x128 : k128x128;
    }
    if (n <= 2048 && K <= 2048 && tiles_of(n, N, 128, 128) <= kCUs) {
        faster = tiles_of(n, N, 128, 128) > kCUs * 3 / 4;
        return k128x128;
    }
    const int64_t r256 = wide_rounds(n, N, 256), r192 = wide_rounds(n, N, 192), rounds = r192 < r256 ? r192 : r256;
    const int64_t whole = (tiles_of(n, N, 256, 256) + kCUs - 1) / kCUs * 100;  // the library's
    if (K <= 512) faster = N >= 2048 || (N >= 1536 && (columns || n >= 4096));
    else if ((int64_t)n * N * 100 < 70 * rounds * 256 * 256 * kCUs / 100) faster = false;
    else if (columns) faster = n >= 800 && K <= 6144;
    else if (n < 4096 || (n % 256 == 0 && (n < 5000 || K > 1024))) faster = false;
    else faster = K <= 1024 ? rounds < whole || whole > 100 : K <= 2048 ? rounds < whole : K <= 3072 && 3 * rounds <= 2 * whole;
    return r192 < r256 ? kWide192 : kWide256;
}

}  // namespace
}  // namespace skyrl

using namespace skyrl;

extern "C" int32_t skyrl_dense_product_fits(int32_t n, int32_t K, int32_t N) {
    bool faster = false;
    if (n > 0 && N > 0 && N % 8 == 0 && K > 0 && K % 64 == 0) form_of(n, K, N, faster);
    return faster;
}

extern "C" int skyrl_dense_product(const void* x, int64_t ldx, int32_t n, int32_t K, const void* w, int64_t ldw, int32_t N, void* out,
                                   void* stream) {
    SKYRL_REQUIRE(n > 0 && N > 0 && N % 8 == 0 && K > 0 && K % 64 == 0, "dense_product: K must be a multiple of 64, N of 8");
    SKYRL_REQUIRE(x && w && out, "dense_product: null pointer");
    SKYRL_REQUIRE(aligned16(x) && aligned16(w) && aligned16(out) && ldx % 8 == 0 && ldw % 8 == 0 && ldw >= K && (n == 1 || ldx >= K),
                  "dense_product: rows must be 16-byte aligned");
    SKYRL_REQUIRE(n * ldx < (1ll << 31) && N * ldw < (1ll << 31), "dense_product: operands of less than 4 GB");
    const uint16_t *x_ = reinterpret_cast<const uint16_t*>(x), *w_ = reinterpret_cast<const uint16_t*>(w);
    uint16_t* o_ = reinterpret_cast<uint16_t*>(out);
    hipStream_t s = as_stream(stream);
    const Dense d{x_, w_, ldx, ldw, n, K, N, o_};
    bool faster;
    const Form form = form_of(n, K, N, faster);
    SKYRL_REQUIRE(tiles_of(n, N, 64, 32) < (1ll << 30), "dense_product: too many rows in one call");
    const Wide one{x_, w_, o_, K, N, ldx, ldw, 1, nullptr, nullptr, 1, 0, 0, nullptr, n, n <= 128 ? 128 : 256, Gate{}};
    if (form == kOnce) return n <= 128 ? launch_wide<kDense, SKYRL_ACT_SILU, true, 128>(one, s) : launch_wide<kDense, SKYRL_ACT_SILU, true>(one, s);
    if (form == k64x32) launch_dense<64, 32, 6>(d, s);
    else if (form == k64x64) launch_dense<64, 64, 4>(d, s);
    else if (form == k64x128) launch_dense<64, 128, 3>(d, s);
    else if (form == k128x128) launch_dense<128, 128, 3>(d, s);
    else {
        const int rows = form == kWide256 ? 256 : 192;
        return launch_wide<kDense>(Wide{x_, w_, o_, K, N, ldx, ldw, (n + rows - 1) / rows, nullptr, nullptr, 1, 0, 0, nullptr, n, rows, Gate{}}, s);
    }
    return check_launch("dense_kernel");
}

