// Products of a few activation rows with a weight matrix, y[n, N] = x[n, K] w[N, K]^T (decode steps; include/skyrl_layers.h).
//
// Bound: the weights' bytes. At 1 to 128 rows a weight matrix is read once and used little, and what the time went on
// before was how it was read: the library's tiles for these shapes leave most CUs idle or few loads in flight. Here a wave has a
// share of the depth to itself (stream.h). Few weight rows are cut into `splits` shares of the depth across workgroups too, each
// with f32 sums of its own that the next norm adds. One row takes the same form, with that row in all 16 places: a wave per
// weight row, lanes along the depth, took 5.6, 11.6, 6.2, 12.8 and 27.0 us for the five matrices below (its sums start when the
// whole row is there).
// Measured on one MI355X, weights from HBM and past the caches (stream.h), us, here / the library's:
//   N, K            1 row            16 rows          32 rows          64 rows
//   2048, 2048      3.9 / 10.9       4.1 / 11.0       4.4 / 11.2       5.5 / 11.7
//   2048, 6144      6.9 / 11.1       7.2 / 11.2       7.5 / 16.5       9.6 / 19.4
//   3648, 2048      4.8 / 11.8       5.5 / 11.7       6.5 / 11.6       8.4 / 12.1   (no splits)
//   12288, 2048     11.5 / 16.6      11.8 / 15.2      12.7 / 15.2      15.5 / 16.3  (no splits; 4.4 TB/s at one row)
//   24576, 2048     20.6 / 40.0      21.7 / 40.1      23.6 / 29.3      29.7 / 30.2  (gated: 12288 pairs of rows)
//   32768, 2048     24.1 / 35.1      24.6 / 32.9      27.5 / 35.3      27.9 / 35.7  (no splits; 5.6 TB/s at one row)
// At 64 rows a workgroup's x is as many bytes as its weights, over the same 64 bytes a clock into LDS: 12288 x 2048 gated took,
// in 192 workgroups of 64 rows of weights, 16.4 us, 13.4 without x, 7.3 without the weights, 5.3 without either; leaving out the products
// changed it by 0.4. In 256 of 48 it takes 15.0.
// Batches (a head's up-projections of latent attention, 512 x 128 and 128 x 512): 16 heads, 1 / 64 rows, both products with the
// copy that the library's needed: 15.4 / 17.1 us, here 5.9 / 7.6 us.
#include "rows.h"

namespace skyrl {
namespace {

template <int MODE, int NT, int MT, int WK, int S, bool ONCE, bool EXACT>
__global__ __launch_bounds__(WK* kWave) void rows_product_kernel(RowsProduct p) {
    __shared__ __attribute__((aligned(16))) uint16_t smem[Stream<NT, MT, WK, S>::kLds];
    rows_block<MODE, NT, MT, WK, S, ONCE, EXACT>(p, smem, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.y);
}

constexpr int kWide = 8192;       // output columns from which wider tiles still fill the chip and read x less often
constexpr int kFill = 256;        // one workgroup a CU: what a split product is cut into
constexpr int kManyRowsCols = 4096;

enum Form { kFormRound, kFormGated, kFormParts };

// What the kernels compute.
bool rows_take(int n, int K, int N, int form) {
    return n > 0 && K > 0 && N > 0 && K % 8 == 0 && (n <= 64 || (n <= 128 && N <= kManyRowsCols && form == kFormParts));
}

// Where they are the faster form; us, here / the library's. Above 64 rows its tiles are as fast on wide matrices and slower on narrow
// ones only against parts (128 rows, 2048 x 2048 7.2 / 11.1, 2048 x 6144 12.9 / 17.6). Depths above 2048 give them more to pipeline:
//   up to 16 rows  until a matrix is both deep and large: 4096 x 4096 8.4 / 15.5, 30720 x 4096 43.3 / 59.3, 4096 x 6144 in parts
//                  12.9 / 23.0 (one row: 11.0 / 22.9), 2048 x 8192 8.5 / 13.1 (7.6 / 12.7); 4096 x 8192 16.1 / 16.2 (15.5 / 15.8), and
//                  past it little between them (4096 x 12288 20.9 / 22.1): the line is where they were equal with cached weights.
//   more rows      in parts, up to 8192 columns (32 rows: 4096 x 12288 21.7 / 26.9, 8192 x 4096 14.3 / 16.9; 64 rows: 27.6 /
//                  37.4, 17.7 / 19.3); rounded or gated, narrow ones (64 rows, 4096 x 4096 13.7 / 15.0, but 6144 x 4096 23.7 /
//                  18.0) and up to 32 rows of wide ones 4096 deep (32768 x 4096 50.2 / 66.7, gated 24576 x 4096 44.5 / 54.0;
//                  64 rows: 68.2 / 64.9, 52.3 / 54.4).
//   past 16384     at any number of rows (4096 x 18432: 26.9 / 51.6, 42.2 / 123.0, 53.6 / 131.8 at 1, 32, 64 rows).
bool rows_fit(int n, int K, int N, int form) {
    if (!rows_take(n, K, N, form)) return false;
    if (n > 64 || K <= 2048 || K > (1 << 14)) return true;
    const bool parts = form == kFormParts;
    const int64_t rows = form == kFormGated ? 2ll * N : N;
    if (n <= 16) return K <= 4096 || rows * K < (parts ? 1 << 25 : 1 << 24);
    if (rows <= kWide) return parts || (K <= 4096 && rows <= kManyRowsCols);
    return n <= 32 && K >= 4096;
}

int splits_for(int n, int K, int N) {
    const int bn = n <= 16 ? 16 : 32, tiles = (N + bn - 1) / bn, most = K / 64 / 4;  // a piece per wave at least
    int s = (kFill + tiles / 2) / tiles;
    if (s > most) s = most;
    return s < 1 ? 1 : s > 8 ? 8 : s;
}

template <int MODE, int NT, int MT, int WK, int S, bool ONCE = true, bool EXACT = false>
void launch_rows(RowsProduct p, int splits, hipStream_t s, int batch = 1) {
    constexpr int OC = MODE == kGated ? 8 * NT : 16 * NT;
    p.row_blocks = (p.n + 16 * MT - 1) / (16 * MT);
    hipLaunchKernelGGL((rows_product_kernel<MODE, NT, MT, WK, S, ONCE, EXACT>), dim3((p.N + OC - 1) / OC, splits, p.row_blocks * batch),
                       dim3(WK * kWave), 0, s, p);
}

// From 17 rows of x on, the fewest rows of weights a workgroup of which one a CU holds all: 16 (rounded ones), 32 (with gated ones both
// matrices'), 48, else 64. With more, CUs stood idle: 6144 pairs are 192 workgroups of 64 and 256 of 48. us at 32 / 64 rows of x with 64 rows of weights, 48, 32:
//   768 pairs x 2048     10.2 / 13.3   9.1 / 11.9    8.3 / 9.6
//   4096 pairs x 2048    12.7 / 15.9   11.8 / 14.8   10.5 / 12.4
//   6144 pairs x 2048    14.1 / 16.3   12.9 / 15.0   15.4 / 19.7
//   6144 pairs x 4096    23.8 / 29.4   21.5 / 26.3   26.7 / -
//   8192 x 2048          12.7 / 16.6   11.6 / 14.7   9.9 / 13.3
//   12288 x 2048         14.4 / 17.6   12.8 / 16.7   15.1 / 19.8
//   12352 x 2048         14.2 / 18.0   16.6 / 19.4   15.2 / -   (64 rows of x with four waves for two, up to one workgroup a CU: 15.6)
// with 16 rows of weights and 32: 2048 x 2048 64 rows 8.4, 9.6; 4608 x 2048 10.4 / 13.7, 9.2 / 10.4; 8184 x 2048 64 rows 15.2, 12.4.
// Four waves share the depth, two where 64 rows of x take several rounds of 64 rows of weights.
int weight_tiles(int rows) { return rows <= 16 * kFill ? 1 : rows <= 32 * kFill ? 2 : rows <= 48 * kFill ? 3 : 4; }

// Up to 16 rows of x, 16 rows of weights a workgroup up to 512 workgroups of these, 48 or 64 up to one workgroup a CU, then 32; us at
// 1 / 16 rows of x with 16, 32 and 64 rows of weights:
//   8192 x 2048    7.5 / 8.4     7.7 / 8.0     8.7 / 9.6
//   8192 x 4096    13.3 / 14.9   13.8 / 14.3   16.9 / 19.2
//   10240 x 2048   9.9 / 11.2    10.1 / 11.5   9.5 / 10.2
//   12288 x 2048   -             -             11.8 / 12.4  (48 rows: 11.4 / 11.8)
//   16640 x 2048   15.6 / 16.1   15.6 / 16.0   17.5 / 18.3
//   24576 x 4096   34.1 / 38.1   34.2 / 35.0   37.1 / 40.0
template <int MODE>
void launch_rounded(const RowsProduct& p, hipStream_t s) {
    const int nt = weight_tiles(p.N);
    if (p.n <= 16) {
        if (p.N <= kWide) launch_rows<MODE, 1, 1, 4, 4>(p, 1, s);
        else if (nt == 3) launch_rows<MODE, 3, 1, 4, 2>(p, 1, s);
        else if (p.N <= 2 * kWide) launch_rows<MODE, 4, 1, 4, 2>(p, 1, s);
        else launch_rows<MODE, 2, 1, 4, 2>(p, 1, s);
    } else if (p.n <= 32) {
        if (nt == 1) launch_rows<MODE, 1, 2, 4, 3>(p, 1, s);
        else if (nt == 2) launch_rows<MODE, 2, 2, 4, 2>(p, 1, s);
        else if (nt == 3) launch_rows<MODE, 3, 2, 4, 2>(p, 1, s);
        else launch_rows<MODE, 4, 2, 4, 2>(p, 1, s);
    } else {
        if (nt == 1) launch_rows<MODE, 1, 4, 4, 2>(p, 1, s);
        else if (nt == 2) launch_rows<MODE, 2, 4, 4, 2>(p, 1, s);
        else if (nt == 3) launch_rows<MODE, 3, 4, 4, 2>(p, 1, s);
        else if (p.N <= 64 * kFill) launch_rows<MODE, 4, 4, 4, 2>(p, 1, s);
        else launch_rows<MODE, 4, 4, 2, 2>(p, 1, s);
    }
}

// Gated, a pair of rows is two rows of weights. Up to 16 rows of x, 32 rows of weights, but 64 where 32 were more than one workgroup
// a CU and 64 are not, unless the depth makes up for it, or 48 where these are (4608 pairs x 1536, one row: 9.4 -> 8.6); us at 1 / 16 rows of x with 32 and 64 rows of weights:
//   2048 pairs x 2048    6.1 / 7.0     9.5 / 9.9
//   4096 pairs x 2048    8.7 / 8.3     11.1 / 10.2
//   6144 pairs x 2048    12.2 / 12.3   11.7 / 11.1
//   6144 pairs x 4096    20.4 / 23.3   24.7 / 25.1
//   12288 pairs x 2048   19.4 / 20.0   20.6 / 21.4
// Above, weight_tiles. At 33 to 64 rows of x and 64 rows of weights two waves, two workgroups a CU, where these are one round and four waves would be two; us at 64 rows with two
// and four waves: 6144 x 2048 17.9, 15.7; 8448 x 2048 25.0, 27.4; 16384 x 2048 30.0, 33.0; 24576 x 2048 53.2, 47.7.
void launch_gated(const RowsProduct& p, hipStream_t s) {
    const int tiles = (p.N + 31) / 32, nt = weight_tiles(2 * p.N);  // of 64 rows
    if (p.n <= 16) {
        if (nt == 3 && p.K <= 3072) launch_rows<kGated, 3, 1, 4, 3>(p, 1, s);
        else if (tiles > kFill / 2 && tiles <= kFill && p.K <= 3072) launch_rows<kGated, 4, 1, 2, 4>(p, 1, s);
        else launch_rows<kGated, 2, 1, 4, 3>(p, 1, s);
    } else if (p.n <= 32) {
        if (nt <= 2) launch_rows<kGated, 2, 2, 4, 2>(p, 1, s);
        else if (nt == 3) launch_rows<kGated, 3, 2, 4, 2>(p, 1, s);
        else launch_rows<kGated, 4, 2, 4, 2>(p, 1, s);
    } else if (nt <= 2) {
        launch_rows<kGated, 2, 4, 4, 2>(p, 1, s);
    } else if (nt == 3) {
        launch_rows<kGated, 3, 4, 4, 2>(p, 1, s);
    } else if (tiles > kFill && tiles <= 2 * kFill) {
        launch_rows<kGated, 4, 4, 2, 2>(p, 1, s);
    } else {
        launch_rows<kGated, 4, 4, 4, 2>(p, 1, s);
    }
}

}  // namespace
}  // namespace skyrl

using namespace skyrl;

extern "C" int32_t skyrl_rows_product_fits(int32_t n, int32_t K, int32_t N, int32_t form) {
    return rows_fit(n, K, N, form);
}

extern "C" int32_t skyrl_rows_product_splits(int32_t n, int32_t K, int32_t N) { return splits_for(n, K, N); }

namespace {

// capped: f32 [n, N], the rounded product between -cap and cap; turn0, turn1: columns of a rounded one that go through tanh.
int rows_product(const void* x, int64_t ldx, int32_t n, int32_t K, const void* w, int64_t ldw, int32_t N, const void* bias,
                 int32_t act, float alpha, float limit, int32_t splits, void* out, int64_t ldo, bool capped, float cap, int32_t turn0,
                 int32_t turn1, void* stream) {
    const bool gate = act >= 0;
    SKYRL_REQUIRE(rows_take(n, K, N, gate ? kFormGated : splits ? kFormParts : kFormRound), "rows_product: sizes that the library takes");
    SKYRL_REQUIRE(x && w && out, "rows_product: null pointer");
    SKYRL_REQUIRE(aligned16(x) && aligned16(w) && ldx % 8 == 0 && ldw % 8 == 0 && ldw >= K && (n == 1 || ldx >= K),
                  "rows_product: rows must be 16-byte aligned");
    SKYRL_REQUIRE((reinterpret_cast<uintptr_t>(out) & (splits || capped ? 3 : 1)) == 0 && (n == 1 || ldo >= N), "rows_product: bad output");
    SKYRL_REQUIRE(!gate || (!bias && splits == 0 && (act == SKYRL_ACT_SILU || act == SKYRL_ACT_GELU_TANH || act == SKYRL_ACT_CLAMPED)),
                  "rows_product: a gated product has an activation, no bias and no splits");
    SKYRL_REQUIRE(splits == 0 || splits == splits_for(n, K, N), "rows_product: splits are skyrl_rows_product_splits'");
    const RowsProduct p{reinterpret_cast<const uint16_t*>(x), ldx, n, K, reinterpret_cast<const uint16_t*>(w), ldw, N,
                        reinterpret_cast<const uint16_t*>(bias), Gate{act, alpha, limit}, turn0, turn1, cap, out, ldo, (int64_t)n * ldo, 1, 0, 0, 0};
    hipStream_t s = as_stream(stream);
    // Wide tiles where there are columns enough, since every workgroup reads x again; else 16 rows of weights, so that
    // the chip is full (3648 x 2048 at 64 rows: 8.5 us with 16, 9.4 with 32).
    if (gate) {
        launch_gated(p, s);
    } else if (splits) {
        if (n == 1) launch_rows<kParts, 1, 1, 4, 4, true, true>(p, splits, s);
        else if (n <= 16) launch_rows<kParts, 1, 1, 4, 4>(p, splits, s);
        else if (n <= 32) launch_rows<kParts, 2, 2, 4, 2>(p, splits, s);
        else if (n <= 64) launch_rows<kParts, 2, 4, 4, 2>(p, splits, s);
        else launch_rows<kParts, 2, 8, 4, 1>(p, splits, s);
    } else if (capped) {
        launch_rounded<kCapped>(p, s);
    } else {
        launch_rounded<kRound>(p, s);
    }
    return check_launch("rows_product_kernel");
}

}  // namespace

extern "C" int skyrl_rows_product(const void* x, int64_t ldx, int32_t n, int32_t K, const void* w, int64_t ldw, int32_t N,
                                  const void* bias, int32_t act, float alpha, float limit, int32_t splits, void* out,
                                  int64_t ldo, void* stream) {
    return rows_product(x, ldx, n, K, w, ldw, N, bias, act, alpha, limit, splits, out, ldo, false, 0.f, 0, 0, stream);
}

extern "C" int skyrl_rows_product_tanh(const void* x, int64_t ldx, int32_t n, int32_t K, const void* w, int64_t ldw, int32_t N,
                                       const void* bias, int32_t first, int32_t last, void* out, int64_t ldo, void* stream) {
    SKYRL_REQUIRE(first >= 0 && first <= last && last <= N, "rows_product_tanh: bad columns");
    return rows_product(x, ldx, n, K, w, ldw, N, bias, -1, 0.f, 0.f, 0, out, ldo, false, 0.f, first, last, stream);
}

extern "C" int skyrl_rows_product_capped(const void* x, int64_t ldx, int32_t n, int32_t K, const void* w, int64_t ldw, int32_t N,
                                         float cap, float* out, int64_t ldo, void* stream) {
    return rows_product(x, ldx, n, K, w, ldw, N, nullptr, -1, 0.f, 0.f, 0, out, ldo, true, cap, 0, 0, stream);
}

namespace {

int rows_batch(const void* x, int64_t ldx, int64_t x_batch, int32_t n, int32_t K, const void* w, int64_t ldw, int64_t w_batch,
               int32_t N, int32_t batch, void* out, int64_t ldo, int64_t out_batch, bool in_order, void* stream) {
    SKYRL_REQUIRE(n >= 0 && K > 0 && N > 0 && K % 8 == 0 && batch > 0 && (int64_t)batch * ((n + 63) / 64) <= 65535,
                  "rows_batch: bad sizes");
    if (n == 0) return SKYRL_OK;
    SKYRL_REQUIRE(x && w && out, "rows_batch: null pointer");
    SKYRL_REQUIRE(aligned16(x) && aligned16(w) && ldx % 8 == 0 && ldw % 8 == 0 && x_batch % 8 == 0 && w_batch % 8 == 0 &&
                      ldw >= K && (reinterpret_cast<uintptr_t>(out) & 1) == 0,
                  "rows_batch: rows must be 16-byte aligned");
    const RowsProduct p{reinterpret_cast<const uint16_t*>(x), ldx, n, K, reinterpret_cast<const uint16_t*>(w), ldw, N, nullptr,
                        Gate{-1, 0.f, 0.f}, 0, 0, 0.f, out, ldo, 0, 1, x_batch, w_batch, out_batch};
    hipStream_t s = as_stream(stream);
    // A head's matrix is small: all its pieces are under way at once. Shallow ones (the queries' up-projection) take two
    // waves a workgroup and 32 columns, deep ones (the outputs') four waves and 16 columns. In order: one wave, which has the
    // whole depth (16 heads, 256 rows: 12.4 and 15.0 us, in shares 12.2 and 13.5, the library 22.8 and 35.6 with its copy).
    // Past 64 rows the blocks of 64 share a head's matrix: the forms of more than 32 rows leave it in the caches.
    if (in_order) {
        if (K <= 256) launch_rows<kRound, 2, 4, 1, 2, false>(p, 1, s, batch);
        else launch_rows<kRound, 1, 4, 1, 3, false>(p, 1, s, batch);
    } else if (K <= 256) {
        if (n <= 16) launch_rows<kRound, 2, 1, 2, 2>(p, 1, s, batch);
        else if (n <= 32) launch_rows<kRound, 2, 2, 2, 2>(p, 1, s, batch);
        else launch_rows<kRound, 2, 4, 2, 1, false>(p, 1, s, batch);
    } else {
        if (n <= 16) launch_rows<kRound, 1, 1, 4, 2>(p, 1, s, batch);
        else if (n <= 32) launch_rows<kRound, 1, 2, 4, 2>(p, 1, s, batch);
        else launch_rows<kRound, 1, 4, 4, 2, false>(p, 1, s, batch);
    }
    return check_launch("rows_product_kernel");
}

}  // namespace

extern "C" int skyrl_rows_batch(const void* x, int64_t ldx, int64_t x_batch, int32_t n, int32_t K, const void* w, int64_t ldw,
                                int64_t w_batch, int32_t N, int32_t batch, void* out, int64_t ldo, int64_t out_batch,
                                void* stream) {
    return rows_batch(x, ldx, x_batch, n, K, w, ldw, w_batch, N, batch, out, ldo, out_batch, false, stream);
}

extern "C" int skyrl_rows_batch_in_order(const void* x, int64_t ldx, int64_t x_batch, int32_t n, int32_t K, const void* w,
                                         int64_t ldw, int64_t w_batch, int32_t N, int32_t batch, void* out, int64_t ldo,
                                         int64_t out_batch, void* stream) {
    return rows_batch(x, ldx, x_batch, n, K, w, ldw, w_batch, N, batch, out, ldo, out_batch, true, stream);
}
