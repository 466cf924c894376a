// The norm ahead of a product and the product of one row in one launch (decode steps; include/skyrl_layers.h).
//
// Bound: the weights' bytes, as in rows_product.hip. A step of one row is a chain of launches of a few us each, and every second
// one was the norm of a single row (4 to 5.5 us, one workgroup on the chip): now each of the product's workgroups (about 200)
// forms the row for itself, from 24 to 60 KB of which its L2 has most, while its first pieces of the weights are on their way: four
// waves stream, four form the row (a wave that did both would wait for its weights with its row). Sums are in the order and the
// roundings of add_norm_kernel and gate_norm_add_kernel: the same bits. The first workgroup leaves the new residual, in another
// buffer, since the rest still read the old one, and the normed row where a later launch reads it too.
// The first row of a step is read from the embedding's table in the same way (a step of one row 5.5 us less).
// Measured, us in a step's profile, both launches before and the one now (2048 deep): 3648 rows 4.4 + 5.0, 6.8; 12352 rows 4.3 +
// 10.8, 10.9; gated 12288 rows 4.3 + 11.0, 11.3; two shares of 2112 rows 4.7 + 5.5, 6.2; behind 8 experts' rows, 12352 rows
// 6.1 + 11.8, 11.9. Eight pieces of 16 rows (four of 64) under way: all of 2048 (half of it).
#include "normed.h"

namespace skyrl {
namespace {

constexpr int kNT = kFormers;
constexpr int kLongest = 4096;  // of a row
constexpr int kShares = 4, kRows = 8;  // of a product, of a token, that are summed: all are loaded ahead of the weights

__device__ __forceinline__ float4 four(uint2 v) {
    return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                       __uint_as_float(v.y & 0xffff0000u));
}

// Eight values as they are stored: what is loaded ahead is converted, and waited for, where it is used.
template <typename T>
struct Eight {
    uint4 v[sizeof(T) / 2];
    __device__ __forceinline__ void load(const T* p) {
#pragma unroll
        for (int i = 0; i < (int)sizeof(T) / 2; ++i) v[i] = reinterpret_cast<const uint4*>(p)[i];
    }
    __device__ __forceinline__ void get(float (&o)[8]) const {
        if constexpr (sizeof(T) == 2) {
            unpack8(v[0], o);
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                o[4 * i] = __uint_as_float(v[i].x);
                o[4 * i + 1] = __uint_as_float(v[i].y);
                o[4 * i + 2] = __uint_as_float(v[i].z);
                o[4 * i + 3] = __uint_as_float(v[i].w);
            }
        }
    }
};

// residual += the sum of `parts` rows (0: nothing), += step; norm (add_norm_kernel).
struct AddNorm {
    static constexpr bool kBeforeGated = true, kBeforeParts = false;
    const float* delta;
    int parts;
    const float* h;
    const uint16_t *step, *w;
    float base;
    int H;
    float eps;
    int kind;
    float* h_out;
    uint16_t* out;
    const int64_t* tokens;  // the residual is a row of table times scale (NULL: h)
    const uint16_t* table;
    float scale;

    template <int MAXK>  // groups of four a thread
    struct Row {
        float4 h[MAXK], d[kShares][MAXK], kept[MAXK];
        uint2 s[MAXK], w[MAXK], y[MAXK], e[MAXK];
        __device__ __forceinline__ void load(const AddNorm& p) {
            const int nv = p.H / 4;
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                const int v = min((int)threadIdx.x % kNT + k * kNT, nv - 1);
                h[k] = make_float4(0.f, 0.f, 0.f, 0.f);
                e[k] = make_uint2(0u, 0u);
                if (p.tokens) e[k] = *reinterpret_cast<const uint2*>(p.table + p.tokens[0] * p.H + 4 * v);
                else h[k] = ld4(p.h + 4 * v);
                w[k] = *reinterpret_cast<const uint2*>(p.w + 4 * v);
                s[k] = make_uint2(0u, 0u);
                if (p.step) s[k] = *reinterpret_cast<const uint2*>(p.step + 4 * v);
            }
#pragma unroll
            for (int i = 0; i < kShares; ++i)
#pragma unroll
                for (int k = 0; k < MAXK; ++k) {
                    d[i][k] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (i < p.parts) d[i][k] = ld4(p.delta + i * p.H + 4 * min((int)threadIdx.x % kNT + k * kNT, nv - 1));
                }
        }
        static __device__ __forceinline__ int barriers(const AddNorm& p) { return p.kind == SKYRL_NORM_LAYER ? 2 : 1; }  // of form
        // the normed row into LDS at x
        __device__ __forceinline__ void form(const AddNorm& p, uint32_t x, int, uint32_t red) {
            const int nv = p.H / 4;
            float sum = 0.f, ss = 0.f;
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                const int v = threadIdx.x % kNT + k * kNT;
                if (v >= nv) continue;
                if (p.tokens) {
                    const float4 x = four(e[k]);
                    h[k] = make_float4(x.x * p.scale, x.y * p.scale, x.z * p.scale, x.w * p.scale);
                }
#pragma unroll
                for (int i = 1; i < kShares; ++i) {
                    d[0][k].x += d[i][k].x; d[0][k].y += d[i][k].y; d[0][k].z += d[i][k].z; d[0][k].w += d[i][k].w;
                }
                if (p.parts) { h[k].x += d[0][k].x; h[k].y += d[0][k].y; h[k].z += d[0][k].z; h[k].w += d[0][k].w; }
                if (p.step) {
                    const float4 e = four(s[k]);
                    h[k].x += e.x; h[k].y += e.y; h[k].z += e.z; h[k].w += e.w;
                }
                kept[k] = h[k];
                sum += h[k].x; sum += h[k].y; sum += h[k].z; sum += h[k].w;
            }
            const float mean = p.kind == SKYRL_NORM_LAYER ? total(sum, red) / (float)p.H : 0.f;
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                if ((int)threadIdx.x % kNT + k * kNT >= nv) continue;
                h[k].x -= mean; h[k].y -= mean; h[k].z -= mean; h[k].w -= mean;
                ss += h[k].x * h[k].x; ss += h[k].y * h[k].y; ss += h[k].z * h[k].z; ss += h[k].w * h[k].w;
            }
            const float r = 1.f / sqrtf(total(ss, red + 16) / (float)p.H + p.eps);
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                const int v = threadIdx.x % kNT + k * kNT;
                if (v >= nv) continue;
                const float4 e = four(w[k]);
                y[k] = make_uint2(pack_bf16x2(h[k].x * r * (p.base + e.x), h[k].y * r * (p.base + e.y)),
                                  pack_bf16x2(h[k].z * r * (p.base + e.z), h[k].w * r * (p.base + e.w)));
                lds_put2(x + 8 * v, y[k]);
            }
        }
        __device__ __forceinline__ void leave(const AddNorm& p) const {
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                const int v = threadIdx.x % kNT + k * kNT;
                if (v >= p.H / 4) continue;
                st4(p.h_out + 4 * v, kept[k]);
                if (p.out) *reinterpret_cast<uint2*>(p.out + 4 * v) = y[k];
            }
        }
    };
    template <int H_>
    using RowOf = Row<H_ / 4 / kNT>;
};

// A sublayer's result, gated, normed in equal parts and added, and the next norm (gate_norm_add_kernel): A f32, `parts` shares of
// it, and gate logits bf16; or A bf16, `parts` rows that are summed, and gate logits in z_parts shares.
template <typename A, typename Z>
struct GateNorm {
    static constexpr bool kBeforeGated = false, kBeforeParts = sizeof(A) == 4;
    const A* a;
    int parts;
    const Z* z;
    int z_parts;
    int64_t z_part_stride;
    const float* zb;
    const uint16_t* w;
    int groups, L;
    float eps, mult;
    const float* h;
    const uint16_t* wn;
    int H;
    float* h_out;
    uint16_t* out;
    const int64_t* tokens;  // the row of a, with no gate and a residual that starts at 0 (NULL: neither)

    template <int MAXK>  // groups of eight a thread
    struct Row {
        static constexpr int NA = sizeof(A) == 4 ? kShares : kRows, NZ = sizeof(Z) == 4 ? kShares : 1;
        Eight<A> a[NA][MAXK];
        Eight<Z> z[NZ][MAXK];
        Eight<float> b[MAXK], hh[MAXK];
        Eight<uint16_t> w[MAXK], wn[MAXK];
        float y[MAXK][8], h[MAXK][8], r[MAXK];
        __device__ __forceinline__ void load(const GateNorm& p) {
            const int nv = p.H / 8;
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                const int v = 8 * min((int)threadIdx.x % kNT + k * kNT, nv - 1);
                hh[k] = Eight<float>{};
                if (!p.tokens) {
                    hh[k].load(p.h + v);
                    b[k].load(p.zb + v);
                }
                w[k].load(p.w + v);
                wn[k].load(p.wn + v);
#pragma unroll
                for (int i = 0; i < NZ; ++i) {
                    z[i][k] = Eight<Z>{};
                    if (i < p.z_parts) z[i][k].load(p.z + i * p.z_part_stride + v);
                }
#pragma unroll
                for (int i = 0; i < NA; ++i) {
                    a[i][k] = Eight<A>{};
                    if (i < p.parts) a[i][k].load(p.a + (p.tokens ? p.tokens[0] + i : i) * p.H + v);
                }
            }
        }
        __device__ __forceinline__ void scales(const GateNorm& p, uint32_t red) {
            const int nv = p.H / 8, per = nv / p.groups, sums = per / p.L;
            const float len = (float)(p.H / p.groups);
            if (p.groups == 1) {  // a wave's 64 groups of eight at a time, as that kernel has them
#pragma unroll
                for (int k = 0; k < MAXK; ++k) {
                    const float t = wave_total(r[k]);
                    if ((threadIdx.x & 63) == 0) lds_put(red + (k * kNT / kWave + (threadIdx.x % kNT >> 6)) * 4, t);
                }
                lds_barrier();
                float one = 0.f;
#pragma unroll
                for (int k = 0; k < MAXK; ++k) {
                    const f32x4 t = lds_get4(red + k * kNT / kWave * 4);
#pragma unroll
                    for (int i = 0; i < 4; ++i) one += t[i];
                }
                one = 1.f / sqrtf(one / len + p.eps);
#pragma unroll
                for (int k = 0; k < MAXK; ++k) r[k] = one;
                return;
            }
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                if (p.L > 1) r[k] = lane_add<1>(r[k]);
                if (p.L > 2) r[k] = lane_add<2>(r[k]);
                if (p.L > 4) r[k] = lane_add<4>(r[k]);
                if (p.L > 8) r[k] = lane_add<8>(r[k]);
                if (p.L > 16) r[k] = lane_add<16>(r[k]);
                if (p.L > 32) r[k] = lane_add<32>(r[k]);
            }
            if (sums > 1) {
#pragma unroll
                for (int k = 0; k < MAXK; ++k) {
                    const int v = threadIdx.x % kNT + k * kNT;
                    if (v < nv && v % p.L == 0) lds_put(red + v / p.L * 4, r[k]);
                }
                lds_barrier();
#pragma unroll
                for (int k = 0; k < MAXK; ++k) {
                    const int v = threadIdx.x % kNT + k * kNT;
                    if (v >= nv) continue;
                    float s = 0.f;
                    for (int i = 0; i < sums; ++i) s += lds_get(red + (v / per * sums + i) * 4);
                    r[k] = s;
                }
            }
#pragma unroll
            for (int k = 0; k < MAXK; ++k) r[k] = 1.f / sqrtf(r[k] / len + p.eps);
        }
        static __device__ __forceinline__ int barriers(const GateNorm& p) {
            return p.groups == 1 || p.H / 8 / p.groups > p.L ? 2 : 0;
        }
        __device__ __forceinline__ void form(const GateNorm& p, uint32_t x, int, uint32_t red) {
            const int nv = p.H / 8;
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                r[k] = 0.f;
                if ((int)threadIdx.x % kNT + k * kNT >= nv) continue;
                float zz[8], x[8];
                a[0][k].get(y[k]);
                z[0][k].get(zz);
                hh[k].get(h[k]);
#pragma unroll
                for (int i = 1; i < NA; ++i) {
                    a[i][k].get(x);
#pragma unroll
                    for (int j = 0; j < 8; ++j) y[k][j] += x[j];
                }
#pragma unroll
                for (int i = 1; i < NZ; ++i) {
                    z[i][k].get(x);
#pragma unroll
                    for (int j = 0; j < 8; ++j) zz[j] += x[j];
                }
                if (!p.tokens) {
                    b[k].get(x);
#pragma unroll
                    for (int j = 0; j < 8; ++j) y[k][j] *= sigmoid_<uint16_t>(zz[j] + x[j]);
                }
                r[k] = squares(y[k]);
            }
            scales(p, red);
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                const int v = threadIdx.x % kNT + k * kNT;
                const float rk = r[k];
                r[k] = 0.f;
                if (v >= nv) continue;
                float x[8];
                w[k].get(x);
#pragma unroll
                for (int j = 0; j < 8; ++j) h[k][j] += p.mult * (y[k][j] * rk * x[j]);
                r[k] = squares(h[k]);
            }
            scales(p, red + kLongest / 8 * 4);
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                const int v = threadIdx.x % kNT + k * kNT;
                if (v >= nv) continue;
                float x8[8];
                wn[k].get(x8);
#pragma unroll
                for (int j = 0; j < 8; ++j) y[k][j] = h[k][j] * (r[k] * x8[j]);
                lds_put2(x + 16 * v, make_uint2(pack_bf16x2(y[k][0], y[k][1]), pack_bf16x2(y[k][2], y[k][3])));
                lds_put2(x + 16 * v + 8, make_uint2(pack_bf16x2(y[k][4], y[k][5]), pack_bf16x2(y[k][6], y[k][7])));
            }
        }
        __device__ __forceinline__ void leave(const GateNorm& p) const {
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                const int v = threadIdx.x % kNT + k * kNT;
                if (v >= p.H / 8) continue;
                st8(p.h_out + 8 * v, h[k]);
                if (p.out) st8(p.out + 8 * v, y[k]);
            }
        }
    };
    template <int H_>
    using RowOf = Row<H_ / 8 / kNT>;
};

constexpr int kRed = 2 * kLongest / 8;

// As rows_product_kernel with four waves, the row in all 16 places. LONG: rows up to this length.
template <int MODE, int NT, int S, int LONG, class Pre>
__global__ __launch_bounds__(2 * kNT) void normed_product_kernel(RowsProduct p, Pre pre) {
    __shared__ __attribute__((aligned(16))) uint16_t smem[formed_lds<NT, S, LONG, 1, kRed>()];
    formed_product<MODE, NT, S, LONG, 1, kRed>(p, pre, smem, 0, blockIdx.x == 0 && blockIdx.y == 0);
}

constexpr int kWideCols = 8192;  // as in rows_product.hip
// Pairs up to which 48 rows of weights a workgroup are at most one a CU: 64 leave CUs idle (us a launch, 64 / 48: 6144 x 2048 10.95 / 10.68,
// 4608 x 1536 9.12 / 8.50, 4096 x 2048 10.06 / 9.46; in a step of one row with four such products within its noise; rounded ones of
// 8192 to 12288 columns: no change).
constexpr int kPairs = 24 * 256;

template <int LONG, class Pre>
void launch(const RowsProduct& p, const Pre& pre, bool gate, int splits, hipStream_t s) {
#define LAUNCH(MODE, NT, S)                                                                                                 \
    hipLaunchKernelGGL((normed_product_kernel<MODE, NT, S, LONG, Pre>), dim3((p.N + out_cols<MODE, NT>() - 1) / out_cols<MODE, NT>(), \
                       splits ? splits : 1), dim3(2 * kNT), 0, s, p, pre)
    if (gate) {
        if constexpr (Pre::kBeforeGated) {
            if (p.N <= kPairs) LAUNCH(kGated, 3, 5);
            else LAUNCH(kGated, 4, 4);
        }
    } else if (splits) {
        if constexpr (Pre::kBeforeParts) LAUNCH(kParts, 1, 4);
    } else if (p.N >= kWideCols) LAUNCH(kRound, 4, 4);
    else LAUNCH(kRound, 1, 8);  // all of 2048 deep
#undef LAUNCH
}

template <class Pre>
int run(const RowsProduct& p, const Pre& pre, bool gate, int splits, hipStream_t s) {
    // what no decoder has: a gated product behind a gated result, shares behind experts' rows
    SKYRL_REQUIRE((!gate || Pre::kBeforeGated) && (!splits || Pre::kBeforeParts), "normed_product: no such product behind this norm");
    if (p.K <= kLongest / 2) launch<kLongest / 2>(p, pre, gate, splits, s);
    else launch<kLongest>(p, pre, gate, splits, s);
    return check_launch("normed_product_kernel");
}

bool aligned(const void* p) { return !p || aligned16(p); }

// The product's operands; an error's text, or NULL.
const char* bad_product(const skyrl_normed_product* q) {
    if (!q || !q->w || !q->out || !q->h_out || (q->tokens ? !q->table : !q->h)) return "normed_product: null pointer";
    if (q->K <= 0 || q->K > kLongest || q->K % 8 != 0 || q->N <= 0 || q->ldw < q->K || q->ldw % 8 != 0)
        return "normed_product: bad sizes";
    if (q->h == q->h_out) return "normed_product: the residual must leave in another buffer";
    const bool gate = q->act >= 0;
    if (gate && (q->bias || q->splits || !(q->act == SKYRL_ACT_SILU || q->act == SKYRL_ACT_GELU_TANH || q->act == SKYRL_ACT_CLAMPED)))
        return "normed_product: a gated product has an activation, no bias and no splits";
    if (q->splits && q->splits != skyrl_rows_product_splits(1, q->K, q->N))
        return "normed_product: splits are skyrl_rows_product_splits'";
    if (!aligned16(q->w) || !aligned(q->h) || !aligned(q->table) || !aligned16(q->h_out) || !aligned(q->x_out) ||
        (reinterpret_cast<uintptr_t>(q->out) & (q->splits ? 3 : 1)))
        return "normed_product: rows must be 16-byte aligned";
    return nullptr;
}

RowsProduct product(const skyrl_normed_product* q) {
    RowsProduct p{};
    p.n = 1;
    p.K = q->K;
    p.w = reinterpret_cast<const uint16_t*>(q->w);
    p.ldw = q->ldw;
    p.N = q->N;
    p.bias = reinterpret_cast<const uint16_t*>(q->bias);
    p.gate = Gate{q->act, q->alpha, q->limit};
    p.turn0 = q->turn0;
    p.turn1 = q->turn1;
    p.out = q->out;
    p.ldo = p.ldsplit = q->N;
    p.row_blocks = 1;
    return p;
}

}  // namespace
}  // namespace skyrl

using namespace skyrl;

extern "C" int32_t skyrl_normed_product_fits(int32_t K, int32_t shares, int32_t rows) {
    return K > 0 && K <= kLongest && K % 8 == 0 && shares <= kShares && rows <= kRows;
}

extern "C" int skyrl_add_norm_product(const skyrl_normed_product* q, const float* delta, int32_t parts, const void* step,
                                      const void* weight, float w_base, float eps, int32_t kind, void* stream) {
    const char* bad = bad_product(q);
    SKYRL_REQUIRE(!bad, bad);
    SKYRL_REQUIRE(kind == SKYRL_NORM_LAYER || kind == SKYRL_NORM_RMS, "add_norm_product: unknown norm kind");
    SKYRL_REQUIRE(weight && parts >= 0 && parts <= kShares && (parts == 0 || delta), "add_norm_product: null pointer, or more shares than are taken");
    SKYRL_REQUIRE(aligned(delta) && aligned(step) && aligned16(weight), "add_norm_product: rows must be 16-byte aligned");
    const AddNorm pre{delta, parts, q->h, reinterpret_cast<const uint16_t*>(step), reinterpret_cast<const uint16_t*>(weight), w_base,
                      q->K, eps, kind, q->h_out, reinterpret_cast<uint16_t*>(q->x_out), q->tokens,
                      reinterpret_cast<const uint16_t*>(q->table), q->scale};
    return run(product(q), pre, q->act >= 0, q->splits, as_stream(stream));
}

extern "C" int skyrl_gate_norm_product(const skyrl_normed_product* q, const void* a, int32_t a_shares, int32_t parts, const void* gate,
                                       int32_t gate_shares, int64_t gate_stride, const float* gate_bias, const void* weight,
                                       int32_t groups, float eps, float mult, const void* next, void* stream) {
    const char* bad = bad_product(q);
    SKYRL_REQUIRE(!bad, bad);
    if (q->tokens) {
        a = q->table;
        a_shares = 0, parts = 1, gate = gate_bias = nullptr, gate_shares = 1, gate_stride = q->K;
    }
    SKYRL_REQUIRE(a && weight && next && (q->tokens || (gate && gate_bias)), "gate_norm_product: null pointer");
    SKYRL_REQUIRE(groups > 0 && q->K % groups == 0 && q->K / groups % 8 == 0, "gate_norm_product: groups must be multiples of 8");
    SKYRL_REQUIRE((a_shares > 0) != (gate_shares > 0) && parts > 0 && (a_shares == 0 || parts == 1) &&
                      a_shares <= kShares && gate_shares <= kShares && parts <= kRows && (gate_shares == 0 || gate_stride >= q->K) &&
                      gate_stride % 4 == 0,
                  "gate_norm_product: either the rows or the gate's logits are a product's shares");
    SKYRL_REQUIRE(aligned16(a) && aligned(gate) && aligned(gate_bias) && aligned16(weight) && aligned16(next),
                  "gate_norm_product: rows must be 16-byte aligned");
    int L = 1;
    while (L < kWave && q->K / 8 / groups % (2 * L) == 0) L <<= 1;
    const uint16_t *w = reinterpret_cast<const uint16_t*>(weight), *wn = reinterpret_cast<const uint16_t*>(next);
    uint16_t* x = reinterpret_cast<uint16_t*>(q->x_out);
    if (a_shares)
        return run(product(q), GateNorm<float, uint16_t>{reinterpret_cast<const float*>(a), a_shares, reinterpret_cast<const uint16_t*>(gate),
                   1, 0, gate_bias, w, groups, L, eps, mult, q->h, wn, q->K, q->h_out, x, nullptr}, q->act >= 0, q->splits, as_stream(stream));
    return run(product(q), GateNorm<uint16_t, float>{reinterpret_cast<const uint16_t*>(a), parts, reinterpret_cast<const float*>(gate),
               q->tokens ? 0 : gate_shares, gate_stride, gate_bias, w, groups, L, eps, mult, q->h, wn, q->K, q->h_out, x, q->tokens}, q->act >= 0, q->splits,
               as_stream(stream));
}
