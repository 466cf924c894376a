// Latent attention (low-rank shared keys/values) over a paged latent cache.
//
// Per token only the normed latent c (rank) and one rotated key part (rot_dim) shared by every head
// are cached. A head's score against token j is q_n . (W_uk c_j) + q_r . kr_j, its value W_uv c_j.
//
// Decode form (latent_attend): the up-projections are moved to the query and the output, so that all
// heads share one key row [c | kr] and one value row c: q_n . (W_uk c) = (W_uk^T q_n) . c, and the sum
// over keys of p_j W_uv c_j = W_uv (sum p_j c_j). The cache is streamed once for up to 16 heads.
// A workgroup takes a share of a token's pages, four pages (64 keys) at a time: each wave scores one
// page, S^T[token x head] = K[16 x row] . Q^T[row x 16] (mfma_f32_16x16x32_bf16, K straight from HBM to
// registers, the next tile's loads in flight), scores and latents go to LDS, and each wave sums a quarter of the rank over all 64 keys, O^T[rank x head] +=
// C^T[rank x keys] . P^T[keys x head], C^T by transposing LDS reads.
//
// Prompt form (latent_gather + two library products + latent_prefill): a long portion pays the
// up-projection once per key instead of once per query, and the scores cost dim + rot_dim instead of
// rank + rot_dim per pair. latent_prefill is a windowed flash-style kernel: four waves share a K and
// a V^T tile of 64 keys in LDS, each wave owns 32 queries of one head.
#include <type_traits>

#include "normed.h"

namespace skyrl {
namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kBS = 16;  // tokens per cache block
constexpr int kNT = 256;

// Dimension pairs of the rotation: neighbours, or i with i + rot / 2 (halves).
struct Pairs {
    int rot, halves;
    __device__ __forceinline__ int first(int i) const { return halves ? i : 2 * i; }
    __device__ __forceinline__ int second(int i) const { return halves ? i + rot / 2 : 2 * i + 1; }
};

// Parts of a token's row that are there: the rotated parts of `heads` queries at its start, or (q_rank > 0) a query latent that is
// normed in place; the key latent and its rotated part at lat_at (rank > 0).
template <typename T>
struct Write {
    T* proj;
    int64_t stride;
    int heads, dim;
    Pairs pr;
    int q_rank;
    const T* q_norm;
    int rank, lat_at;
    const T* norm_w;
    float eps;
    const int64_t *positions, *slots;
    const float* cos_sin;
    T* cache;
    int row;
};
// A workgroup of NT threads, token t. A row is little and its time is latencies, so what a thread handles first of each part is
// loaded ahead of everything else.
constexpr int kHeld = 4, kPairs = 2;
template <typename T, int NT>
__device__ __forceinline__ void write_row(const Write<T>& w, int t) {
    __shared__ float s_red[NT / kWave];
    struct Held {
        T x[kHeld], w[kHeld];
    };
    const int tid = threadIdx.x;
    T* p = w.proj + (int64_t)t * w.stride;
    const Pairs pr = w.pr;
    const int rot = pr.rot, qd = w.dim + rot, h2 = rot / 2, turns = w.heads * h2;
    const T* lat = p + w.lat_at;
    Held q, k;
    auto load = [&](Held& h, const T* x, const T* weight, int n) {
#pragma unroll
        for (int j = 0; j < kHeld; ++j) {
            const int i = min(tid + j * NT, n - 1);
            h.x[j] = x[i];
            h.w[j] = weight[i];
        }
    };
    auto factor = [&](const Held& h, const T* x, int n) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < kHeld; ++j) {
            const float v = tid + j * NT < n ? ld(&h.x[j]) : 0.f;
            ss += v * v;
        }
        for (int i = tid + kHeld * NT; i < n; i += NT) {
            const float v = ld(x + i);
            ss += v * v;
        }
        return 1.f / sqrtf(block_total<NT>(ss, s_red) / (float)n + w.eps);
    };
    auto put = [&](const Held& h, const T* x, const T* weight, T* to, int n, float r) {
#pragma unroll
        for (int j = 0; j < kHeld; ++j)
            if (tid + j * NT < n) st(to + tid + j * NT, ld(&h.x[j]) * r * ld(&h.w[j]));
        for (int i = tid + kHeld * NT; i < n; i += NT) st(to + i, ld(x + i) * r * ld(weight + i));
    };
    struct Turned {
        T u, v;
        float c, s;
    };
    const float* cs = w.cos_sin + w.positions[t] * rot;
    auto pair = [&](const T* x, int i) { return Turned{x[pr.first(i)], x[pr.second(i)], cs[i], cs[h2 + i]}; };
    // Which of the two products is rounded is said here: left to the compiler it changes with the code around it, and one rotated
    // bf16 value in some 200,000 with it.
    auto turn = [&](const Turned& e, T* to, int i) {
        const float u = ld(&e.u), v = ld(&e.v);
        st(to + pr.first(i), fmaf(u, e.c, -(v * e.s)));
        st(to + pr.second(i), sizeof(T) == 2 ? fmaf(u, e.s, v * e.c) : fmaf(v, e.c, u * e.s));
    };
    auto head = [&](int e) { return p + (int64_t)(e / h2) * qd + w.dim; };
    if (w.q_rank > 0) load(q, p, w.q_norm, w.q_rank);
    int64_t slot = -1;
    if (w.rank > 0) {
        slot = w.slots[t];
        load(k, lat, w.norm_w, w.rank);
    }
    Turned key{}, qs[kPairs] = {};
    if (w.rank > 0 && h2 > 0) key = pair(lat + w.rank, min(tid, h2 - 1));
    if (turns > 0) {
#pragma unroll
        for (int j = 0; j < kPairs; ++j) {
            const int e = min(tid + j * NT, turns - 1);
            qs[j] = pair(head(e), e % h2);
        }
    }
    if (w.q_rank > 0) put(q, p, w.q_norm, p, w.q_rank, factor(q, p, w.q_rank));
    if (w.rank > 0) {
        const float r = factor(k, lat, w.rank);
        if (slot >= 0) {
            T* c = w.cache + slot * w.row;
            put(k, lat, w.norm_w, c, w.rank, r);
            if (tid < h2) turn(key, c + w.rank, tid);
            for (int i = tid + NT; i < h2; i += NT) turn(pair(lat + w.rank, i), c + w.rank, i);
        }
    }
    if (turns > 0) {
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
            if (tid + j * NT < turns) turn(qs[j], head(tid + j * NT), (tid + j * NT) % h2);
        for (int e = tid + kPairs * NT; e < turns; e += NT) turn(pair(head(e), e % h2), head(e), e % h2);
    }
}

template <typename T>
__global__ __launch_bounds__(kNT) void latent_write_kernel(Write<T> w) {
    write_row<T, kNT>(w, blockIdx.x);
}

// What ends a head's softmax: a learned sink in the denominator and a sigmoid gate on the output, each optional.
template <typename T>
struct HeadEnd {
    const float* sinks;  // [heads]
    const T* gate;       // logits [token][head]
    int64_t gate_stride;
    __device__ __forceinline__ float sink(int h) const { return sinks ? sinks[h] : -INFINITY; }
    __device__ __forceinline__ float gated(int t, int h) const {
        return gate ? sigmoidf_(ld(gate + (int64_t)t * gate_stride + h)) : 1.f;
    }
};
// Factor of the value sums with running maximum m and denominator l, all in powers of two; sink in the same units.
__device__ __forceinline__ float sum_factor(float m, float l, float sink) {
    const float mm = fmaxf(m, sink), a = fast_exp2(m - mm);
    return a / (l * a + fast_exp2(sink - mm));
}

// ---- decode form, plain: one workgroup per (token, head), any rank up to 2048, f32 or bf16 ----
template <typename T>
__global__ __launch_bounds__(kNT) void latent_attend_plain_kernel(
    const T* __restrict__ qa, const T* __restrict__ q_rot, int64_t q_stride, int64_t q_head,
    const T* __restrict__ cache, int row, const int32_t* __restrict__ tables, int64_t bt_stride,
    const int32_t* __restrict__ bt_row, const int64_t* __restrict__ positions, int ntok, int heads, int rank, int rot,
    float scale, int window, HeadEnd<T> end, T* __restrict__ out) {
    extern __shared__ float s_q[];  // rank + rot
    __shared__ float s_p[kWave];
    constexpr int kAcc = 8;
    const int h = blockIdx.x, t = blockIdx.y;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int pos = (int)positions[t];
    const int lo = window > 0 ? max(0, pos - window + 1) : 0;
    const int32_t* bt = tables + (int64_t)bt_row[t] * bt_stride;
    const int n = rank + rot;
    for (int i = threadIdx.x; i < n; i += kNT)
        s_q[i] = i < rank ? ld(qa + ((int64_t)h * ntok + t) * rank + i)
                          : ld(q_rot + (int64_t)t * q_stride + (int64_t)h * q_head + (i - rank));
    __syncthreads();
    float acc[kAcc], m = -INFINITY, l = 0.f;
#pragma unroll
    for (int k = 0; k < kAcc; ++k) acc[k] = 0.f;
    for (int j0 = lo; j0 <= pos; j0 += kWave) {
        const int nk = min(kWave, pos + 1 - j0);
        for (int jj = wave; jj < nk; jj += kNT / kWave) {
            const int j = j0 + jj;
            const T* key = cache + ((int64_t)bt[j / kBS] * kBS + j % kBS) * row;
            float s = 0.f;
            for (int i = lane; i < n; i += kWave) s += s_q[i] * ld(key + i);
            s = wave_sum(s);
            if (lane == 0) s_p[jj] = s * scale;
        }
        __syncthreads();
        const float sv = lane < nk ? s_p[lane] : -INFINITY;
        const float mn = fmaxf(m, wave_max(sv));
        const float alpha = expf(m - mn);
        const float p = lane < nk ? expf(sv - mn) : 0.f;
        l = l * alpha + wave_sum(p);
        m = mn;
        __syncthreads();
        if (threadIdx.x < kWave) s_p[threadIdx.x] = p;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kAcc; ++k) acc[k] *= alpha;
        for (int jj = 0; jj < nk; ++jj) {
            const int j = j0 + jj;
            const T* key = cache + ((int64_t)bt[j / kBS] * kBS + j % kBS) * row;
            const float pj = s_p[jj];
#pragma unroll
            for (int k = 0; k < kAcc; ++k) {
                const int d = threadIdx.x + k * kNT;
                if (d < rank) acc[k] += pj * ld(key + d);
            }
        }
        __syncthreads();
    }
    const float sink = end.sink(h), mm = fmaxf(m, sink), a = expf(m - mm);
    const float f = a / (l * a + expf(sink - mm)) * end.gated(t, h);
#pragma unroll
    for (int k = 0; k < kAcc; ++k) {
        const int d = threadIdx.x + k * kNT;
        if (d < rank) st(out + ((int64_t)h * ntok + t) * rank + d, acc[k] * f);
    }
}

// Pages [p0, p0 + np) of a token's context cut into shares of `per` pages; parts = number of shares.
struct PageSplit {
    int p0, per, parts, np;
};
__device__ __forceinline__ PageSplit page_split(int lo, int pos, int part_min, int nparts) {
    PageSplit s;
    s.p0 = lo / kBS;
    s.np = pos / kBS - s.p0 + 1;
    s.per = max((s.np + nparts - 1) / nparts, part_min / kBS);
    s.parts = (s.np + s.per - 1) / s.per;
    return s;
}

// Transposing LDS read: within each group of 16 lanes, lane 4 k + q supplies the address of row k's
// elements 4 q .. 4 q + 3, and lane i receives element i of the four rows.
__device__ __forceinline__ s16x4 lds_read_tr(const uint16_t* p) {
    typedef __attribute__((address_space(3))) s16x4* lds_ptr;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)p);
}

// ---- decode form, MFMA ------------------------------------------------------------------------
// grid (nparts, ceil(heads / (16 HG)), tokens), four waves per group of 16 heads. A tile is four pages, staged
// through registers into LDS in whole 1 KB pieces (a page is contiguous; row-by-row operand loads from
// HBM ran at half the rate), one page per wave, the next tile's loads in flight. Each wave scores one
// page for its head group; for the values it takes a quarter of the rank over all 64 keys. With HG = 2
// two head groups share the tile and each stages half of it. NV: 16-wide tiles of the rank,
// NK: 32-wide steps of the cache row; EXACT when both equal the shape's own.
template <int NV, int NK, bool EXACT, int HG>
__global__ __launch_bounds__(kNT * HG) __attribute__((amdgpu_waves_per_eu(1, 2))) void latent_attend_mfma_kernel(
    const uint16_t* __restrict__ qa, const uint16_t* __restrict__ q_rot, int64_t q_stride, int64_t q_head,
    const uint16_t* __restrict__ cache, int row, const int32_t* __restrict__ tables, int64_t bt_stride,
    const int32_t* __restrict__ bt_row, const int64_t* __restrict__ positions, int ntok, int heads, int rank, int rot,
    float scale_log2, int window, int part_min, int nparts, HeadEnd<uint16_t> end, uint16_t* __restrict__ out,
    float* __restrict__ ws_o, float* __restrict__ ws_ml) {
    constexpr int LDR = NK * 32 + 8;  // padded LDS row
    constexpr int LDS_ = 64 + 4, NW = NV / 4, NT = kNT * HG;
    constexpr int NL = (NK + HG - 1) / HG;  // 16-byte pieces of its page per lane
    __shared__ __attribute__((aligned(16))) uint16_t s_c[64 * LDR];  // first the query, then the tile
    __shared__ __attribute__((aligned(16))) float s_scores[HG * 16 * LDS_];  // scores [head][key of the tile]
    const int t = blockIdx.z;
    const int near_row = bt_row[min(max(t - 1 + min((int)threadIdx.x & 63, 2), 0), ntok - 1)];
    const int pos = (int)positions[t];
    const int lo = window > 0 ? max(0, pos - window + 1) : 0;
    const PageSplit sp = page_split(lo, pos, part_min, nparts);
    const int part = blockIdx.x;
    if (part >= sp.parts) return;
    const int nk = EXACT ? NK : row / 32;
    const int nv = EXACT ? NV : (rank + 15) / 16;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3, hg = __builtin_amdgcn_readfirstlane(tid >> 8);
    const int c = lane & 15, g = lane >> 4;
    const int h0 = blockIdx.y * 16 * HG;  // the workgroup's first head
    float* s_s = s_scores + hg * 16 * LDS_;

    const int first = sp.p0 + part * sp.per;
    const int np = min(sp.per, sp.np - part * sp.per);
    const int32_t* bt = tables + (int64_t)bt_row[t] * bt_stride + first;
    // Pages come in windows of 64, whose block ids a wave holds by lane (no table load ahead of a page's).
    // Pages that a workgroup has alone go past the caches (non-temporal), since the step's weights put them out before the next step:
    // up to 32 heads, and where the neighbouring tokens' page in the place of its first is another one, which it is not for tokens
    // of one sequence or for sequences that share a prompt. 512 + 64, 16 / 32 heads, us with the caches swept before each launch (all
    // cached; all past): 64 rows 41.5 / 34 (52 / 46; 41.5 / 34), 256 rows 80 / 66 (112 / 105; 80 / 65), 256 rows on 32 prompts 71 / 59
    // (72 / 60; 73 / 66), 64 sequences of 4 tokens 73 / 61 (74 / 61; 83 / 64); 48 heads, 64 sequences of 4 tokens 111 (110; 127).
    // Loads are unconditional, the last page again past the end: a branch around them would turn every
    // wait into one for all loads in flight. Both ways of the one in load_page issue the same number.
    const int rc = EXACT ? NK * 4 : nk * 4;  // pieces per row
    auto piece = [&](int k) { return min(lane + 64 * (hg + HG * k), 16 * rc - 1); };
    int lds_at[NL];
#pragma unroll
    for (int k = 0; k < NL; ++k) {
        const int e = piece(k), r = e / rc;
        lds_at[k] = (16 * wave + r) * LDR + (e - r * rc) * 8;
    }
    s16x8 st_[NL];
    int tbl = 0, npw = 0;
    auto window_at = [&](int w0) {
        npw = min(64, np - w0);
        tbl = bt[w0 + min(lane, npw - 1)];
    };
    window_at(0);
    const int near = tables[(int64_t)near_row * bt_stride + first];  // by lane: the first page here of tokens t - 1, t, t + 1
    bool alone = false;
    auto load_page = [&](int j) {
        const uint16_t* p = cache + (int64_t)__builtin_amdgcn_readlane(tbl, min(j, npw - 1)) * kBS * row;
        auto load = [&](auto once) {
            asm volatile("; pages %0" ::"n"(once.value));  // else the compiler takes both ways' loads for the same, ordinary ones
#pragma unroll
            for (int k = 0; k < NL; ++k) {
                const s16x8* src = reinterpret_cast<const s16x8*>(p + piece(k) * 8);
                if constexpr (once.value) st_[k] = __builtin_nontemporal_load(src);
                else st_[k] = *src;
            }
            asm volatile("; pages %0" ::"n"(once.value));
        };
        if (alone) load(std::true_type{});
        else load(std::false_type{});
    };
    // The query rows of this head group, [latent | rotated | 0], through LDS into MFMA operands. Loads return in order: those of
    // whole 16-byte pieces go ahead of the pages', all at once, and land while the block table is read (16 heads, 512 + 64,
    // context 1024, us with the merge, against a loop of loads behind the first pages': 1 row 12.3 against 18.0, 64 rows 23.7
    // against 28.8, 256 rows 60.5 against 67.1, over and over on one cache, part of which stays on chip; in engine passes 64 rows
    // take 24.5, 256 rows 58.5, the cache's 302 MB at 5.2 TB/s).
    constexpr int QP = HG * 16 * NK * 4, QL = (QP + NT - 1) / NT;
    const bool pieces = rank % 8 == 0 && rot % 8 == 0 && q_stride % 8 == 0 && q_head % 8 == 0 &&
                        (reinterpret_cast<uintptr_t>(q_rot) & 15) == 0;
    auto query = [&](int e, int& d, int& h) {
        const int hh = e / (NK * 4);
        d = (e - hh * (NK * 4)) * 8;
        h = h0 + hh;
        return &s_c[hh * LDR + d];
    };
    s16x8 q_[QL];
    if (pieces) {
#pragma unroll
        for (int i = 0; i < QL; ++i) {  // past the end, past the heads and past the row: another piece, not used
            int d, h;
            query(min(tid + NT * i, QP - 1), d, h);
            h = min(h, heads - 1);
            const bool latent = d < rank || rot == 0;
            const int64_t at = latent ? ((int64_t)h * ntok + t) * rank + min(d, rank - 8)
                                      : (int64_t)t * q_stride + (int64_t)h * q_head + min(d - rank, rot - 8);
            q_[i] = *reinterpret_cast<const s16x8*>((latent ? qa : q_rot) + at);
        }
    }
    const int mine = __builtin_amdgcn_readlane(near, 1);
    alone = gridDim.y == 1 && (t == 0 || __builtin_amdgcn_readlane(near, 0) != mine) &&
            (t == ntok - 1 || __builtin_amdgcn_readlane(near, 2) != mine);
    load_page(wave);
    if (pieces) {
#pragma unroll
        for (int i = 0; i < QL; ++i) {
            int d, h;
            uint16_t* at = query(min(tid + NT * i, QP - 1), d, h);
            if (h >= heads || d >= rank + rot) q_[i] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (tid + NT * i < QP) *reinterpret_cast<s16x8*>(at) = q_[i];
        }
    } else {
        const bool vec = rank % 8 == 0;
        for (int e = tid; e < QP; e += NT) {
            int d, h;
            uint16_t* at = query(e, d, h);
            s16x8 f = {0, 0, 0, 0, 0, 0, 0, 0};
            if (h < heads && d < row) {
                const uint16_t* qrow = qa + ((int64_t)h * ntok + t) * rank;
                const uint16_t* rrow = q_rot + (int64_t)t * q_stride + (int64_t)h * q_head;
                if (vec && d + 8 <= rank) {
                    f = *reinterpret_cast<const s16x8*>(qrow + d);
                } else {
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const int dd = d + j;
                        const uint16_t* src = dd < rank ? qrow + dd : dd < rank + rot ? rrow + (dd - rank) : qrow;
                        const uint16_t x = *src;
                        f[j] = (short)(dd < rank + rot ? x : 0);
                    }
                }
            }
            *reinterpret_cast<s16x8*>(at) = f;
        }
    }
    __syncthreads();
    s16x8 qf[NK];
#pragma unroll
    for (int s = 0; s < NK; ++s) qf[s] = *reinterpret_cast<const s16x8*>(&s_c[(16 * hg + c) * LDR + 32 * s + 8 * g]);

    f32x4 o[NW];
#pragma unroll
    for (int n = 0; n < NW; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    auto tile = [&](int w0, int j0) {
        const int tb = (first + w0 + j0 + wave) * kBS;  // this wave's page
        const bool edge = j0 + wave >= npw || tb < lo || tb + kBS - 1 > pos;
        if (edge) {  // a masked slot may hold anything: 0 * NaN must not reach the sums
#pragma unroll
            for (int k = 0; k < NL; ++k) {
                const int tok = tb + piece(k) / rc;
                if (!(j0 + wave < npw && tok >= lo && tok <= pos)) st_[k] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
            }
        }
        __syncthreads();  // the query operands, or the previous tile, are consumed
#pragma unroll
        for (int k = 0; k < NL; ++k) *reinterpret_cast<s16x8*>(&s_c[lds_at[k]]) = st_[k];
        load_page(j0 + 4 + wave);
        __syncthreads();
        f32x4 sa = {0.f, 0.f, 0.f, 0.f}, sb = sa;
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            if (EXACT || s < nk) {
                const s16x8 kf = *reinterpret_cast<const s16x8*>(&s_c[(16 * wave + c) * LDR + 32 * s + 8 * g]);
                if (s & 1) sb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[s], sb, 0, 0, 0);
                else sa = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[s], sa, 0, 0, 0);
            }
        }
        f32x4 sv = (sa + sb) * scale_log2;  // token tb + 4 g + i, head c
        if (edge) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int tok = tb + 4 * g + i;
                if (!(j0 + wave < npw && tok >= lo && tok <= pos)) sv[i] = -INFINITY;
            }
        }
        *reinterpret_cast<f32x4*>(&s_s[c * LDS_ + 16 * wave + 4 * g]) = sv;
        __syncthreads();
        // every wave: weights of all 64 keys, the lane's own 16 in the order of the MFMA operand
        f32x4 x[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) x[w] = *reinterpret_cast<const f32x4*>(&s_s[c * LDS_ + 16 * w + 4 * g]);
        float bm = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; ++w) bm = fmaxf(bm, fmaxf(fmaxf(x[w][0], x[w][1]), fmaxf(x[w][2], x[w][3])));
        bm = lane_max<32>(lane_max<16>(bm));
        const float mn = fmaxf(m, bm);
        const float alpha = fast_exp2(m - mn);  // first tile: m = -inf, 0; every share starts with a visible key
        float sum = 0.f;
        s16x8 pf[2];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            uint32_t pk[4];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                float p[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    p[i] = fast_exp2(x[2 * kk + b][i] - mn);
                    sum += p[i];
                }
                pk[2 * b] = pack_bf16x2(p[0], p[1]);
                pk[2 * b + 1] = pack_bf16x2(p[2], p[3]);
            }
            pf[kk] = __builtin_bit_cast(s16x8, make_uint4(pk[0], pk[1], pk[2], pk[3]));
        }
        l = l * alpha + sum;
        m = mn;
#pragma unroll
        for (int n = 0; n < NW; ++n) {
            const int vt = wave * NW + n;
            if (EXACT || vt < nv) {
                o[n] = o[n] * alpha;
#pragma unroll
                for (int kk = 0; kk < 2; ++kk) {
                    const uint16_t* vp = &s_c[(32 * kk + 4 * g + (c >> 2)) * LDR + 16 * vt + 4 * (c & 3)];
                    const s16x4 a = lds_read_tr(vp), b = lds_read_tr(vp + 16 * LDR);
                    const s16x8 vf = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
                    o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[kk], o[n], 0, 0, 0);
                }
            }
        }
    };
    for (int w0 = 0; w0 < np; w0 += 64) {
        if (w0 > 0) {
            window_at(w0);
            load_page(wave);
        }
        for (int j0 = 0; j0 < npw; j0 += 4) tile(w0, j0);
    }
    l = lane_add<32>(lane_add<16>(l));  // the sum over all keys, the same in every wave
    const int h = h0 + 16 * hg + c;
    if (h >= heads) return;
    if (sp.parts == 1) {
        const float inv = sum_factor(m, l, end.sink(h) * kLog2e) * end.gated(t, h);
        uint16_t* orow = out + ((int64_t)h * ntok + t) * rank;
#pragma unroll
        for (int n = 0; n < NW; ++n) {
            const int d = 16 * (wave * NW + n) + 4 * g;
            if (EXACT || (rank % 4 == 0 && d + 4 <= rank)) {
                *reinterpret_cast<uint2*>(orow + d) =
                    make_uint2(pack_bf16x2(o[n][0] * inv, o[n][1] * inv), pack_bf16x2(o[n][2] * inv, o[n][3] * inv));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (d + i < rank) orow[d + i] = f32_to_bf16(o[n][i] * inv);
            }
        }
    } else {
        const int64_t rec = ((int64_t)t * heads + h) * nparts + part;
        float* wo = ws_o + rec * (((rank + 15) / 16) * 16);
#pragma unroll
        for (int n = 0; n < NW; ++n)
            if (EXACT || wave * NW + n < nv) *reinterpret_cast<f32x4*>(wo + 16 * (wave * NW + n) + 4 * g) = o[n];
        if (wave == 0 && g == 0) {
            ws_ml[rec * 2] = m;
            ws_ml[rec * 2 + 1] = l;
        }
    }
}

// Merge of the shares of one (token, head): grid (heads, tokens), one wave per 256 dimensions.
__global__ __launch_bounds__(kWave * 2) void latent_merge_kernel(const float* __restrict__ ws_o,
                                                                 const float* __restrict__ ws_ml,
                                                                 const int64_t* __restrict__ positions, int ntok,
                                                                 int heads, int rank, int window, int part_min,
                                                                 int nparts, HeadEnd<uint16_t> end,
                                                                 uint16_t* __restrict__ out) {
    const int h = blockIdx.x, t = blockIdx.y, lane = threadIdx.x & 63;
    const int pos = (int)positions[t];
    const int lo = window > 0 ? max(0, pos - window + 1) : 0;
    const PageSplit sp = page_split(lo, pos, part_min, nparts);
    if (sp.parts == 1) return;
    const int64_t rec = ((int64_t)t * heads + h) * nparts;
    const int rp = ((rank + 15) / 16) * 16;
    float M = -INFINITY;
    for (int p = lane; p < sp.parts; p += kWave) M = fmaxf(M, ws_ml[(rec + p) * 2]);
    M = wave_largest(M);
    float L = 0.f;
    for (int p = lane; p < sp.parts; p += kWave) L += fast_exp2(ws_ml[(rec + p) * 2] - M) * ws_ml[(rec + p) * 2 + 1];
    const float inv = sum_factor(M, wave_total(L), end.sink(h) * kLog2e) * end.gated(t, h);
    uint16_t* orow = out + ((int64_t)h * ntok + t) * rank;
    for (int d = threadIdx.x * 4; d < rp; d += kWave * 8) {
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
        for (int p = 0; p < sp.parts; ++p) {
            const float w = fast_exp2(ws_ml[(rec + p) * 2] - M) * inv;
            const float4 x = ld4(ws_o + (rec + p) * rp + d);
            acc.x += w * x.x; acc.y += w * x.y; acc.z += w * x.z; acc.w += w * x.w;
        }
        if (rank % 4 == 0 && d + 4 <= rank) {
            st4(orow + d, acc);
        } else {
            const float v[4] = {acc.x, acc.y, acc.z, acc.w};
            for (int i = 0; i < 4; ++i)
                if (d + i < rank) orow[d + i] = f32_to_bf16(v[i]);
        }
    }
}

// ---- steps of few rows: what stands between the large products and the attention -----------------
// Each of these is a launch of a few us that waits for the one before; what does not depend on each other shares one.

// A row's write, and the up-projection of its queries' unrotated parts, which the write leaves alone: the first workgroups write a
// token each, the others take the product (rows_batch's form of up to 256 deep). 16 heads, us: one row 4.2 + 3.7 before, now
// 4.9; 64 rows 5.6 + 5.5, a step of two such layers 11 less.
template <int MT>
__global__ __launch_bounds__(kNT) void latent_lift_kernel(Write<uint16_t> w, int ntok, RowsProduct p, int cols) {
    __shared__ __attribute__((aligned(16))) uint16_t smem[Stream<2, MT, kNT / kWave, 1>::kLds];
    int b = blockIdx.x;
    if (b < ntok) return write_row<uint16_t, kNT>(w, b);
    b -= ntok;
    rows_block<kRound, 2, MT, kNT / kWave, 1>(p, smem, b % cols, 0, b / cols, 1);
}

// The row of one query latent, normed (write_row).
struct LatentNorm {
    const uint16_t *x, *w;
    int n;
    float eps;
    template <int MAXK>
    struct Row {
        uint16_t x[MAXK], w[MAXK];
        __device__ __forceinline__ void load(const LatentNorm& p) {
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                const int i = min((int)threadIdx.x % kFormers + k * kFormers, p.n - 1);
                x[k] = p.x[i];
                w[k] = p.w[i];
            }
        }
        static __device__ __forceinline__ int barriers(const LatentNorm&) { return 1; }
        __device__ __forceinline__ void form(const LatentNorm& p, uint32_t to, int, uint32_t red) {
            float ss = 0.f;
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                const float v = bf16_to_f32(x[k]);
                if ((int)threadIdx.x % kFormers + k * kFormers < p.n) ss += v * v;
            }
            const float r = 1.f / sqrtf(total(ss, red) / (float)p.n + p.eps);
#pragma unroll
            for (int k = 0; k < MAXK; ++k) {
                const int i = threadIdx.x % kFormers + k * kFormers;
                if (i < p.n) lds_put16(to + 2 * i, f32_to_bf16(bf16_to_f32(x[k]) * r * bf16_to_f32(w[k])));
            }
        }
        __device__ __forceinline__ void leave(const LatentNorm&) const {}
    };
    template <int LONG>
    using RowOf = Row<LONG / kFormers>;
};

// One token's query latent, normed, and the product behind it; the last workgroup writes the key latent. Rank 768, 16 heads of 192:
// 5.6 + 3.8 us before, now 5.0.
constexpr int kQueryRank = 2048;
__global__ __launch_bounds__(2 * kFormers) void latent_query_kernel(Write<uint16_t> w, RowsProduct p, LatentNorm pre) {
    __shared__ __attribute__((aligned(16))) uint16_t smem[formed_lds<1, 4, kQueryRank, 1, 8>()];
    if (blockIdx.x == gridDim.x - 1) {  // as latent_write: its 256 threads' sums (barriers are not waited for by waves that have ended)
        if (threadIdx.x < kNT) write_row<uint16_t, kNT>(w, 0);
        return;
    }
    formed_product<kRound, 1, 4, kQueryRank, 1, 8>(p, pre, smem, 0, false);
}

// The shares of up to kMergeRows tokens' contexts, merged (latent_merge_kernel) for a head, blockIdx.z.
constexpr int kMergeRows = 4, kMergeRank = 512, kMergeParts = 256;
struct Merge {
    const float *ws_o, *ws_ml;
    const int64_t* positions;
    int ntok, heads, rank, window, part_min, nparts;
    HeadEnd<uint16_t> end;
    const uint16_t* out;  // of a token whose context is one share
    // Everything is loaded at once, ahead of the number of shares (those past it hold anything and are left out).
    struct Row {
        static constexpr int kAhead = 24;
        float2 v[kAhead];  // of the thread's first two dimensions
        float2 ml;         // of the wave's first token
        int pos, mine;     // positions of the tokens of these
        float sink, gate;
        static __device__ __forceinline__ int parts(const Merge& m, int pos) {
            return page_split(m.window > 0 ? max(0, pos - m.window + 1) : 0, pos, m.part_min, m.nparts).parts;
        }
        static __device__ __forceinline__ int64_t record(const Merge& m, int t) {
            return ((int64_t)t * m.heads + blockIdx.z) * m.nparts;
        }
        __device__ __forceinline__ void load(const Merge& m) {
            const int tid = threadIdx.x % kFormers, half = m.rank / 2, e = min(tid, m.ntok * half - 1), t = e / half;
            const int own = min(tid >> 6, m.ntok - 1), rp = (m.rank + 15) / 16 * 16;
            mine = (int)m.positions[own];
            pos = (int)m.positions[t];
            ml = reinterpret_cast<const float2*>(m.ws_ml)[record(m, own) + min(tid & 63, m.nparts - 1)];
            sink = m.end.sink(blockIdx.z) * kLog2e;
            gate = m.end.gated(own, blockIdx.z);
            const float* src = m.ws_o + record(m, t) * rp + (e - t * half) * 2;
#pragma unroll
            for (int p = 0; p < kAhead; ++p) v[p] = *reinterpret_cast<const float2*>(src + min(p, m.nparts - 1) * rp);
        }
        static __device__ __forceinline__ int barriers(const Merge&) { return 1; }
        __device__ __forceinline__ void form(const Merge& m, uint32_t x, int pitch, uint32_t red) {
            typedef __attribute__((address_space(3))) const float lds_float;
            const int tid = threadIdx.x % kFormers, lane = tid & 63, rp = (m.rank + 15) / 16 * 16, half = m.rank / 2;
            const int own = tid >> 6;
            static_assert(kMergeRows <= kFormers / kWave, "a wave per token");
            if (own < m.ntok) {  // its shares' weights
                const int n = parts(m, mine);
                const float2* rest = reinterpret_cast<const float2*>(m.ws_ml) + record(m, own);
                float M = lane < n ? ml.x : -INFINITY, L = 0.f;
                for (int p = lane + kWave; p < n; p += kWave) M = fmaxf(M, rest[p].x);
                M = wave_largest(M);
                if (lane < n) L = fast_exp2(ml.x - M) * ml.y;
                for (int p = lane + kWave; p < n; p += kWave) L += fast_exp2(rest[p].x - M) * rest[p].y;
                const float inv = sum_factor(M, wave_total(L), sink) * gate;
                if (lane < n) lds_put(red + (own * kMergeParts + lane) * 4, fast_exp2(ml.x - M) * inv);
                for (int p = lane + kWave; p < n; p += kWave)
                    lds_put(red + (own * kMergeParts + p) * 4, fast_exp2(rest[p].x - M) * inv);
            }
            lds_barrier();
            auto place = [&](int e, int& t, int& d) {
                t = e / half;
                d = (e - t * half) * 2;
            };
            auto merged = [&](int t, int d, int n, int from, float2 acc) {
                lds_float* wt = (lds_float*)(uintptr_t)(red + t * kMergeParts * 4);
                const float* src = m.ws_o + record(m, t) * rp + d;
#pragma unroll 8
                for (int p = from; p < n; ++p) {
                    const float w = wt[p];
                    const float2 u = *reinterpret_cast<const float2*>(src + (int64_t)p * rp);
                    acc.x += w * u.x;
                    acc.y += w * u.y;
                }
                // one share: the row is there
                const uint32_t y = n == 1 ? *reinterpret_cast<const uint32_t*>(m.out + ((int64_t)blockIdx.z * m.ntok + t) * m.rank + d)
                                          : pack_bf16x2(acc.x, acc.y);
                lds_put32(x + t * pitch + d * 2, y);
            };
            int t, d;
            place(min(tid, m.ntok * half - 1), t, d);  // threads past the last do the last one's again
            const int n = parts(m, pos);
            lds_float* wt = (lds_float*)(uintptr_t)(red + t * kMergeParts * 4);
            float2 acc = make_float2(0.f, 0.f);
#pragma unroll
            for (int p = 0; p < kAhead; ++p) {
                const float w = wt[p];
                acc.x = p < n ? acc.x + w * v[p].x : acc.x;
                acc.y = p < n ? acc.y + w * v[p].y : acc.y;
            }
            merged(t, d, n, kAhead, acc);
            for (int e = tid + kFormers; e < m.ntok * half; e += kFormers) {
                place(e, t, d);
                merged(t, d, parts(m, (int)m.positions[t]), 0, make_float2(0.f, 0.f));
            }
        }
        __device__ __forceinline__ void leave(const Merge&) const {}
    };
    template <int>
    using RowOf = Row;
};

// The merge and the outputs' up-projection: grid (columns / 16, 1, heads), each workgroup merges its head's rows. 16 heads, one row
// of 17 shares: 4.5 + 3.7 us before, now 5.5.
__global__ __launch_bounds__(2 * kFormers) void latent_merge_up_kernel(RowsProduct p, Merge pre) {
    constexpr int kRed = kMergeRows * kMergeParts;
    __shared__ __attribute__((aligned(16))) uint16_t smem[formed_lds<1, 2, kMergeRank, kMergeRows, kRed>()];
    formed_product<kRound, 1, 2, kMergeRank, kMergeRows, kRed>(p, pre, smem, blockIdx.z, false);
}

// ---- prompt form --------------------------------------------------------------------------------
// grid (ceil(max rows / 16), nseg): 16 packed rows per workgroup; rows past the segment's count up to the next
// multiple of 64 are zeroed.
template <typename T>
__global__ __launch_bounds__(kNT) void latent_gather_kernel(const T* __restrict__ cache, int row,
                                                            const int32_t* __restrict__ tables, int64_t bt_stride,
                                                            const int32_t* __restrict__ seg, int rank, int rot,
                                                            T* __restrict__ latent, T* __restrict__ k_rot) {
    const int32_t* sg = seg + 4 * blockIdx.y;
    const int count = sg[2], padded = (count + 63) / 64 * 64;
    const int r0 = blockIdx.x * 16;
    if (r0 >= padded) return;
    const int32_t* bt = tables + (int64_t)sg[0] * bt_stride;
    const int n = rank + rot;
    if (rank % 4 == 0 && rot % 4 == 0) {
        const int n4 = n / 4;
        for (int e = threadIdx.x; e < 16 * n4; e += kNT) {
            const int rr = e / n4, d = (e - rr * n4) * 4, r = r0 + rr;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (r < count) {
                const int p = sg[1] + r;
                v = ld4(cache + ((int64_t)bt[p / kBS] * kBS + p % kBS) * row + d);
            }
            const int64_t dst = sg[3] + r;
            if (d < rank) st4(latent + dst * rank + d, v);
            else st4(k_rot + dst * rot + (d - rank), v);
        }
        return;
    }
    for (int e = threadIdx.x; e < 16 * n; e += kNT) {
        const int rr = e / n, d = e - rr * n, r = r0 + rr;
        float v = 0.f;
        if (r < count) {
            const int p = sg[1] + r;
            v = ld(cache + ((int64_t)bt[p / kBS] * kBS + p % kBS) * row + d);
        }
        const int64_t dst = sg[3] + r;
        if (d < rank) st(latent + dst * rank + d, v);
        else st(k_rot + dst * rot + (d - rank), v);
    }
}

constexpr int kKT = 64;   // keys per LDS tile

// 8 consecutive elements starting at column d of a key row assembled from [nope | rot | 0].
template <bool VEC>
__device__ __forceinline__ s16x8 key_chunk(const uint16_t* nope, const uint16_t* rotp, int d, int dim, int rot) {
    s16x8 f = {0, 0, 0, 0, 0, 0, 0, 0};
    if constexpr (VEC) {
        if (d < dim) f = *reinterpret_cast<const s16x8*>(nope + d);
        else if (d < dim + rot) f = *reinterpret_cast<const s16x8*>(rotp + (d - dim));
        return f;
    }
    const uint16_t* none = dim > 0 ? nope : rotp;
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // loads without a branch
        const int dd = d + j;
        const uint16_t x = *(dd < dim ? nope + dd : dd < dim + rot ? rotp + (dd - dim) : none);
        f[j] = (short)(dd < dim + rot ? x : 0);
    }
    return f;
}

// LDS reads that the compiler does not know as such: it would have them wait for every direct load under way. They are waited for
// by count, and their registers tied past the wait.
__device__ __forceinline__ void lds_read(s16x8& v, uint32_t at, int offset) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(offset));
}
__device__ __forceinline__ void lds_wait(s16x8& v, int left) {  // left: of the reads behind it that may be under way
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(v) : "n"(left) : "memory");
}
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void gbl_void;
__device__ const uint4 kNoKey = {0u, 0u, 0u, 0u};

// QT: 16-query tiles per wave, 128 queries per workgroup. VEC: every row piece is 16-byte aligned.
// A tile of 64 keys is in pieces of 1 KB: 8 key rows of 64 columns or 8 value rows (of V^T) of 64 keys, whole 128-byte lines, by
// direct loads into one of two buffers while the other is worked on: one barrier a tile, and at dk = 192, vdim = 128 two workgroups
// fill a CU's LDS. In the scores' product row r of 16-row tile t is key 32 (t / 2) + 8 (r / 4) + 4 (t % 2) + r % 4, so that a lane's
// weights are of 8 keys in a row, which one 16-byte read of V^T gives; 16-byte chunks are swizzled for both reads. Bound: the
// matrix cores', the LDS reads' and the vector units' time, of which two waves a SIMD overlap a part. 16 heads, dk 192, vdim 128,
// window 1024, us: one prompt of 8192 109, eight of 341 to 1024 51, three of 300 to 700 25.5; dk 256, vdim 256, one of 1500 49.5. (Tiles
// staged through 40 registers a lane in lines cut in two, two barriers a tile, operands read where they were used, masks formed for
// every tile: 150, 70, 35.5, 84. Without exponentials 98, with all tiles in L2 99, without the scores' products 85.)
template <int NK, int NV, int QT, bool VEC>
__global__ __launch_bounds__(512 / QT) __attribute__((amdgpu_waves_per_eu(2))) void latent_prefill_kernel(
    const uint16_t* __restrict__ q, int64_t q_stride, const uint16_t* __restrict__ k_nope, int64_t k_stride,
    const uint16_t* __restrict__ k_rot, const uint16_t* __restrict__ v_t, int64_t vt_stride,
    const int32_t* __restrict__ tiles, int heads, int dim, int rot, int vdim, float scale_log2, int window,
    HeadEnd<uint16_t> end, uint16_t* __restrict__ out, int64_t out_stride) {
    constexpr int NT = 512 / QT, NW = NT / kWave, QW = 16 * QT;
    constexpr int KG = NK / 2, KB = KG * kKT * 128, VB = NV * 16 * 128, BUF = KB + VB;  // 64-column groups; bytes
    constexpr int KPW = KG * 8 / NW, VPW = NV * 2 / NW;                                  // pieces per wave
    static_assert(NK % 2 == 0 && KG * 8 % NW == 0 && NV * 2 % NW == 0 && kKT == 64, "whole pieces");
    static_assert(2 * BUF <= 160 * 1024 && BUF <= 65536, "LDS; offsets of the reads");
    __shared__ __attribute__((aligned(16))) char smem[2 * BUF];
    const int h = blockIdx.x % heads;  // one head's tiles stay on one XCD when heads is a multiple of 8
    const int32_t* tl = tiles + 8 * (blockIdx.x / heads);
    const int tok0 = tl[0], ntok = tl[1], pos0 = tl[2], seg_row = tl[3], seg_pos = tl[4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, g = lane >> 4;
    const int dk = dim + rot;
    const int w = window > 0 ? window : 0x3fffffff;

    // this wave's queries: QW * wave + 16 qq + c
    s16x8 qf[QT][NK];
    int qpos[QT];
#pragma unroll
    for (int qq = 0; qq < QT; ++qq) {
        const int qi = QW * wave + 16 * qq + c;
        const bool ok = qi < ntok;
        qpos[qq] = pos0 + qi;
        const uint16_t* qr = q + (int64_t)(tok0 + (ok ? qi : 0)) * q_stride + (int64_t)h * dk;
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            s16x8 f = {0, 0, 0, 0, 0, 0, 0, 0};
            if (ok) f = key_chunk<VEC>(qr, qr + dim, 32 * s + 8 * g, dim, rot);
            if (!(scale_log2 > 0.f)) {  // the largest score is the largest product's: a scale below 0 turns the queries instead
#pragma unroll
                for (int i = 0; i < 8; ++i) f[i] = scale_log2 < 0.f ? f[i] ^ (short)0x8000 : scale_log2 == 0.f ? (short)0 : f[i];
            }
            qf[qq][s] = f;
        }
    }
    scale_log2 = scale_log2 == 0.f ? 1.f : fabsf(scale_log2);
    f32x4 o[NV][QT];
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
        for (int qq = 0; qq < QT; ++qq) o[n][qq] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m[QT], l[QT];
#pragma unroll
    for (int qq = 0; qq < QT; ++qq) {
        m[qq] = -INFINITY;
        l[qq] = 0.f;
    }

    const int lo = max(0, pos0 - w + 1);
    const int j0 = (lo - seg_pos) / kKT, j1 = (pos0 + ntok - 1 - seg_pos) / kKT;
    const int wq0 = pos0 + QW * wave;                                // the wave's first query
    const int wq1 = min(wq0 + QW - 1, pos0 + ntok - 1);                  // and its last

    // Pieces: this lane's 16 bytes of row lane / 8. Key row r has its chunk x at x ^ key_swizzle(r), value row d at x ^ d % 8.
    const int r8 = lane >> 3;
    auto key_swizzle = [](int r) { return ((r & 3) >> 1) | ((r >> 3 & 3) << 1); };
    auto piece = [&](int i) { return wave + NW * i; };  // the wave's i-th: of keys 8-row group % 8, column group / 8
    s16x8 kr[VEC ? 1 : KPW];
    auto fetch = [&](int j) {
        char* dst = smem + (j - j0 & 1) * BUF;
        const int64_t r0 = seg_row + (int64_t)j * kKT;
        int own = lane;
        // else the addresses and limits of all unaligned pieces' elements stay in registers from tile to tile, and most of them in
        // memory: 164 and 408 bytes a lane at dk of 128 and 192, now none and 12
        if (!VEC) asm volatile("" : "+v"(own));
#pragma unroll
        for (int i = 0; i < KPW; ++i) {
            const int at = piece(i) % 8 * 8 + (own >> 3), d = 64 * (piece(i) / 8) + 8 * ((own & 7) ^ key_swizzle(at));
            const int64_t row = r0 + at;
            const uint16_t *kp = k_nope + row * k_stride + (int64_t)h * dim, *rp = k_rot + row * rot;
            if constexpr (VEC) {
                const void* src = d < dim ? (const void*)(kp + d) : d < dk ? (const void*)(rp + (d - dim)) : (const void*)&kNoKey;
                __builtin_amdgcn_global_load_lds((gbl_void*)src, (lds_void*)(dst + piece(i) * 1024), 16, 0, 0);
            } else {
                kr[i] = key_chunk<false>(kp, rp, d, dim, rot);
            }
        }
        const uint16_t* vp = v_t + (int64_t)h * vdim * vt_stride + r0 + 8 * ((lane & 7) ^ r8);
#pragma unroll
        for (int i = 0; i < VPW; ++i) {  // rows past the last: the last, whose sums nothing reads
            const int d = min(piece(i) * 8 + r8, vdim - 1);
            __builtin_amdgcn_global_load_lds((gbl_void*)(vp + d * vt_stride), (lds_void*)(dst + KB + piece(i) * 1024), 16, 0, 0);
        }
    };
    const uint32_t lds = (uint32_t)(uintptr_t)(lds_void*)smem;
    const int krow = 8 * (c >> 2) + (c & 3);  // of tile t: + 32 (t / 2) + 4 (t % 2)
    const uint32_t ka[2] = {lds + krow * 128 + ((g ^ key_swizzle(krow)) * 16), lds + krow * 128 + (((4 + g) ^ key_swizzle(krow)) * 16)};
    const uint32_t va[2] = {lds + KB + c * 128 + ((g ^ (c & 7)) * 16), lds + KB + c * 128 + (((4 + g) ^ (c & 7)) * 16)};
    fetch(j0);
    for (int j = j0; j <= j1; ++j) {
        const uint32_t buf = (j - j0 & 1) * BUF;
        if constexpr (!VEC) {
#pragma unroll
            for (int i = 0; i < KPW; ++i) *reinterpret_cast<s16x8*>(smem + buf + piece(i) * 1024 + lane * 16) = kr[i];
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();  // this tile is there, the one before consumed
        if (j < j1) fetch(j + 1);
        const int kp0 = seg_pos + j * kKT, kp1 = kp0 + kKT - 1;
        if (kp0 > wq1 || kp1 < wq0 - w + 1 || wq0 > wq1) continue;  // no key of this tile for this wave
        const bool edge = kp1 > wq0 || kp0 < wq1 - w + 1 || wq1 != wq0 + QW - 1;
        // key rows are read AHEAD products ahead, the first value rows while the scores become weights
        constexpr int AHEAD = QT == 1 ? 8 : 5, VAHEAD = 3;
        f32x4 sc[4][QT];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int qq = 0; qq < QT; ++qq) sc[tt][qq] = f32x4{0.f, 0.f, 0.f, 0.f};
        s16x8 kf[AHEAD + 1], vf[VAHEAD + 1][2];
        auto key = [&](int f) {  // step f / 4, tile f % 4
            lds_read(kf[f % (AHEAD + 1)], ka[f / 4 & 1] + buf, (f / 8) * (kKT * 128) + (f % 4 / 2) * 4096 + (f & 1) * 512);
        };
        auto values = [&](int n) {
            lds_read(vf[n % (VAHEAD + 1)][0], va[0] + buf, n * 2048);
            lds_read(vf[n % (VAHEAD + 1)][1], va[1] + buf, n * 2048);
        };
#pragma unroll
        for (int f = 0; f < AHEAD; ++f) key(f);
#pragma unroll
        for (int f = 0; f < 4 * NK; ++f) {
            s16x8& k = kf[f % (AHEAD + 1)];
            if (f + AHEAD < 4 * NK) {
                key(f + AHEAD);
                lds_wait(k, AHEAD);
            } else {
                lds_wait(k, 4 * NK - 1 - f);
            }
#pragma unroll
            for (int qq = 0; qq < QT; ++qq)
                sc[f % 4][qq] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, qf[qq][f / 4], sc[f % 4][qq], 0, 0, 0);
        }
#pragma unroll
        for (int n = 0; n < VAHEAD; ++n) values(n);
        s16x8 pf[QT][2];  // [query tile][32-key step]
        float alpha[QT];
        auto weights = [&](auto masked) {  // masked: some key of the tile is after a query or too far back
#pragma unroll
            for (int qq = 0; qq < QT; ++qq) {
                float bm = -INFINITY;
                const unsigned dist = qpos[qq] - kp0 - 8 * g;  // to the lane's first key
#pragma unroll
                for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (decltype(masked)::value && dist - (32 * (tt / 2) + 4 * (tt % 2) + i) >= (unsigned)w) sc[tt][qq][i] = -INFINITY;
                        bm = fmaxf(bm, sc[tt][qq][i]);
                    }
                bm = lane_max<32>(lane_max<16>(bm)) * scale_log2;
                const float mn = fmaxf(m[qq], bm);
                const float base = mn == -INFINITY ? 0.f : mn;  // no key seen yet: every weight is 0
                alpha[qq] = fast_exp2(m[qq] - base);
                float sum = 0.f;
#pragma unroll
                for (int kk = 0; kk < 2; ++kk) {
                    uint32_t pk[4];
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        float p[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            p[i] = fast_exp2(fmaf(sc[2 * kk + b][qq][i], scale_log2, -base));
                            sum += p[i];
                        }
                        pk[2 * b] = pack_bf16x2(p[0], p[1]);
                        pk[2 * b + 1] = pack_bf16x2(p[2], p[3]);
                    }
                    pf[qq][kk] = __builtin_bit_cast(s16x8, make_uint4(pk[0], pk[1], pk[2], pk[3]));
                }
                l[qq] = l[qq] * alpha[qq] + sum;
                m[qq] = mn;
            }
        };
        if (edge) weights(std::true_type{});
        else weights(std::false_type{});
        bool same = true;  // no maximum has moved: factors of 1
#pragma unroll
        for (int qq = 0; qq < QT; ++qq) same &= alpha[qq] == 1.f;
        if (!__all(same)) {
#pragma unroll
            for (int n = 0; n < NV; ++n)
#pragma unroll
                for (int qq = 0; qq < QT; ++qq) o[n][qq] = o[n][qq] * alpha[qq];
        }
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            s16x8(&v)[2] = vf[n % (VAHEAD + 1)];
            if (n + VAHEAD < NV) values(n + VAHEAD);
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                lds_wait(v[kk], 2 * (min(n + VAHEAD, NV - 1) - n) + 1 - kk);
#pragma unroll
                for (int qq = 0; qq < QT; ++qq)
                    o[n][qq] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[kk], pf[qq][kk], o[n][qq], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int qq = 0; qq < QT; ++qq) {
        float s = l[qq];
        s = lane_add<32>(lane_add<16>(s));
        const int qi = QW * wave + 16 * qq + c;
        if (qi >= ntok) continue;
        const float inv = sum_factor(m[qq], s, end.sink(h) * kLog2e) * end.gated(tok0 + qi, h);
        uint16_t* orow = out + (int64_t)(tok0 + qi) * out_stride + (int64_t)h * vdim;
        const bool ovec = vdim % 4 == 0 && out_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            const int d = 16 * n + 4 * g;
            if (ovec && d + 4 <= vdim) {
                *reinterpret_cast<uint2*>(orow + d) = make_uint2(pack_bf16x2(o[n][qq][0] * inv, o[n][qq][1] * inv),
                                                                 pack_bf16x2(o[n][qq][2] * inv, o[n][qq][3] * inv));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (d + i < vdim) orow[d + i] = f32_to_bf16(o[n][qq][i] * inv);
            }
        }
    }
}


}  // namespace
}  // namespace skyrl

using namespace skyrl;

namespace {

const char* bad_write(const void* proj, int64_t proj_stride, int32_t T_, int32_t heads, int32_t dim, int32_t rot_dim, int32_t q_rank,
                      const void* q_norm, int32_t rank, int32_t latent_at, const void* norm_weight, const int64_t* positions,
                      const int64_t* slots, const float* cos_sin, const void* cache, int32_t row) {
    if (!(T_ >= 0 && heads >= 0 && dim >= 0 && rot_dim >= 0 && rot_dim % 2 == 0 && rank >= 0 && q_rank >= 0))
        return "latent_write: bad sizes";
    if (!(heads == 0 || q_rank == 0)) return "latent_write: queries or their latent, not both";
    if (!(rank == 0 || (row % 32 == 0 && row >= rank + rot_dim)))
        return "latent_write: row must be a multiple of 32 >= rank + rot_dim";
    const int64_t qw = q_rank > 0 ? q_rank : (int64_t)heads * (dim + rot_dim);
    if (!(proj_stride >= qw && (rank == 0 || (latent_at >= qw && proj_stride >= (int64_t)latent_at + rank + rot_dim))))
        return "latent_write: proj_stride";
    if (T_ > 0 && !(proj && positions && cos_sin && (q_rank == 0 || q_norm) && (rank == 0 || (norm_weight && slots && cache))))
        return "latent_write: null pointer";
    return nullptr;
}

template <typename T>
Write<T> write_of(void* proj, int64_t proj_stride, int32_t heads, int32_t dim, int32_t rot_dim, int32_t halves, int32_t q_rank,
                  const void* q_norm, int32_t rank, int32_t latent_at, const void* norm_weight, float eps,
                  const int64_t* positions, const int64_t* slots, const float* cos_sin, void* cache, int32_t row) {
    return Write<T>{reinterpret_cast<T*>(proj), proj_stride, heads, dim, Pairs{rot_dim, halves}, q_rank,
                    reinterpret_cast<const T*>(q_norm), rank, latent_at, reinterpret_cast<const T*>(norm_weight), eps, positions,
                    slots, cos_sin, reinterpret_cast<T*>(cache), row};
}

}  // namespace

extern "C" int skyrl_latent_write(void* proj, int64_t proj_stride, int32_t T_, int32_t heads, int32_t dim,
                                  int32_t rot_dim, int32_t halves, int32_t q_rank, const void* q_norm, int32_t rank,
                                  int32_t latent_at, const void* norm_weight, float eps, const int64_t* positions,
                                  const int64_t* slots, const float* cos_sin, void* cache, int32_t row, int32_t dtype,
                                  void* stream) {
    SKYRL_REQUIRE_T(dtype, "latent_write");
    const char* bad = bad_write(proj, proj_stride, T_, heads, dim, rot_dim, q_rank, q_norm, rank, latent_at, norm_weight, positions,
                                slots, cos_sin, cache, row);
    SKYRL_REQUIRE(!bad, bad);
    if (T_ == 0) return SKYRL_OK;
    SKYRL_DISPATCH_T(dtype, {
        hipLaunchKernelGGL((latent_write_kernel<T>), dim3(T_), dim3(kNT), 0, as_stream(stream),
                           write_of<T>(proj, proj_stride, heads, dim, rot_dim, halves, q_rank, q_norm, rank, latent_at, norm_weight,
                                       eps, positions, slots, cos_sin, cache, row));
    })
    return check_launch("latent_write_kernel");
}

extern "C" int skyrl_latent_lift(void* proj, int64_t proj_stride, int32_t T_, int32_t heads, int32_t dim, int32_t rot_dim,
                                 int32_t halves, int32_t rank, const void* norm_weight, float eps, const int64_t* positions,
                                 const int64_t* slots, const float* cos_sin, void* cache, int32_t row, const void* up,
                                 int32_t up_rank, void* qa, void* stream) {
    const int latent_at = heads * (dim + rot_dim);
    const char* bad = bad_write(proj, proj_stride, T_, heads, dim, rot_dim, 0, nullptr, rank, latent_at, norm_weight, positions, slots,
                                cos_sin, cache, row);
    SKYRL_REQUIRE(!bad, bad);
    SKYRL_REQUIRE(T_ <= 64 && heads > 0 && dim > 0 && dim <= 256 && dim % 8 == 0 && up_rank > 0, "latent_lift: bad sizes");
    if (T_ == 0) return SKYRL_OK;
    SKYRL_REQUIRE(up && qa && aligned16(proj) && aligned16(up) && aligned16(qa) && proj_stride % 8 == 0 && (dim + rot_dim) % 8 == 0,
                  "latent_lift: rows must be 16-byte aligned");
    const auto w = write_of<uint16_t>(proj, proj_stride, heads, dim, rot_dim, halves, 0, nullptr, rank, latent_at, norm_weight, eps,
                                      positions, slots, cos_sin, cache, row);
    RowsProduct p{};
    p.x = reinterpret_cast<const uint16_t*>(proj);
    p.ldx = proj_stride;
    p.n = T_;
    p.K = dim;
    p.w = reinterpret_cast<const uint16_t*>(up);
    p.ldw = dim;
    p.N = up_rank;
    p.out = qa;
    p.ldo = up_rank;
    p.row_blocks = 1;
    p.x_batch = dim + rot_dim;
    p.w_batch = (int64_t)up_rank * dim;
    p.out_batch = (int64_t)T_ * up_rank;
    const int cols = (up_rank + 31) / 32;
    const dim3 grid(T_ + cols * heads), block(kNT);
    hipStream_t s = as_stream(stream);
    if (T_ <= 16) hipLaunchKernelGGL(latent_lift_kernel<1>, grid, block, 0, s, w, T_, p, cols);
    else if (T_ <= 32) hipLaunchKernelGGL(latent_lift_kernel<2>, grid, block, 0, s, w, T_, p, cols);
    else hipLaunchKernelGGL(latent_lift_kernel<4>, grid, block, 0, s, w, T_, p, cols);
    return check_launch("latent_lift_kernel");
}

extern "C" int skyrl_latent_query(void* proj, int64_t proj_stride, int32_t rot_dim, int32_t halves, int32_t q_rank, const void* q_norm,
                                  int32_t rank, const void* norm_weight, float eps, const int64_t* positions,
                                  const int64_t* slots, const float* cos_sin, void* cache, int32_t row, const void* wuq, int32_t N,
                                  void* q, void* stream) {
    const char* bad = bad_write(proj, proj_stride, 1, 0, 0, rot_dim, q_rank, q_norm, rank, q_rank, norm_weight, positions, slots, cos_sin,
                                cache, row);
    SKYRL_REQUIRE(!bad, bad);
    SKYRL_REQUIRE(q_rank > 0 && q_rank <= kQueryRank && q_rank % 8 == 0 && N > 0, "latent_query: bad sizes");
    SKYRL_REQUIRE(wuq && q && aligned16(wuq) && (reinterpret_cast<uintptr_t>(q) & 1) == 0, "latent_query: rows must be 16-byte aligned");
    const auto w = write_of<uint16_t>(proj, proj_stride, 0, 0, rot_dim, halves, 0, nullptr, rank, q_rank, norm_weight, eps, positions,
                                      slots, cos_sin, cache, row);
    RowsProduct p{};
    p.n = 1;
    p.K = q_rank;
    p.w = reinterpret_cast<const uint16_t*>(wuq);
    p.ldw = q_rank;
    p.N = N;
    p.out = q;
    p.ldo = N;
    p.row_blocks = 1;
    hipLaunchKernelGGL(latent_query_kernel, dim3((N + 15) / 16 + 1), dim3(2 * kFormers), 0, as_stream(stream), w, p,
                       LatentNorm{reinterpret_cast<const uint16_t*>(proj), reinterpret_cast<const uint16_t*>(q_norm), q_rank, eps});
    return check_launch("latent_query_kernel");
}

extern "C" int skyrl_latent_attend_mfma(int32_t rank, int32_t rot_dim, int32_t row, int32_t dtype) {
    return dtype == SKYRL_BF16 && rank > 0 && rot_dim >= 0 && rank <= 512 && row % 32 == 0 && row >= rank + rot_dim &&
           row <= 640;
}

extern "C" size_t skyrl_latent_attend_workspace_bytes(int32_t T_, int32_t heads, int32_t rank, int32_t nparts) {
    const size_t recs = (size_t)(T_ > 0 ? T_ : 0) * heads * nparts;
    return recs * ((size_t)((rank + 15) / 16) * 16 + 2) * sizeof(float) + 16;
}

#define LAUNCH_ATTEND_(NV, NK, EX, HG)                                                                               \
    hipLaunchKernelGGL((latent_attend_mfma_kernel<NV, NK, EX, HG>), dim3(nparts, (heads + 16 * HG - 1) / (16 * HG), T_), \
                       dim3(kNT * HG), 0, s, q_, r_, q_stride, q_head, c_, row, block_tables, bt_stride, bt_row,     \
                       positions, T_, heads, rank, rot_dim, scale * kLog2e, window, part_min, nparts, end_, o_,  \
                       ws_o, ws_ml)
#define LAUNCH_ATTEND(NV, NK, EX)                    \
    if (heads > 16) LAUNCH_ATTEND_(NV, NK, EX, 2);   \
    else LAUNCH_ATTEND_(NV, NK, EX, 1)

namespace {

int latent_attend(const void* qa, const void* q_rot, int64_t q_stride, int64_t q_head, const void* cache, int32_t row,
                  const int32_t* block_tables, int64_t bt_stride, const int32_t* bt_row, const int64_t* positions, int32_t T_,
                  int32_t heads, int32_t rank, int32_t rot_dim, float scale, int32_t window, int32_t part_min, int32_t nparts,
                  const float* sinks, const void* gate, int64_t gate_stride, void* out, void* workspace, int32_t dtype,
                  const RowsProduct* up, void* stream) {
    SKYRL_REQUIRE_T(dtype, "latent_attend");
    SKYRL_REQUIRE(!gate || gate_stride >= heads, "latent_attend: gate_stride");
    SKYRL_REQUIRE(T_ >= 0 && T_ <= 65535 && heads > 0 && rank > 0 && rank <= 2048 && rot_dim >= 0,
                  "latent_attend: bad sizes (T <= 65535, rank <= 2048)");
    SKYRL_REQUIRE(row % 32 == 0 && row >= rank + rot_dim, "latent_attend: row must be a multiple of 32 >= rank + rot_dim");
    if (T_ == 0) return SKYRL_OK;
    SKYRL_REQUIRE(qa && q_rot && cache && block_tables && bt_row && positions && out, "latent_attend: null pointer");
    hipStream_t s = as_stream(stream);
    if (!skyrl_latent_attend_mfma(rank, rot_dim, row, dtype)) {
        SKYRL_DISPATCH_T(dtype, {
            hipLaunchKernelGGL((latent_attend_plain_kernel<T>), dim3(heads, T_), dim3(kNT),
                               (rank + rot_dim) * sizeof(float), s, reinterpret_cast<const T*>(qa),
                               reinterpret_cast<const T*>(q_rot), q_stride, q_head, reinterpret_cast<const T*>(cache),
                               row, block_tables, bt_stride, bt_row, positions, T_, heads, rank, rot_dim, scale,
                               window, HeadEnd<T>{sinks, reinterpret_cast<const T*>(gate), gate_stride},
                               reinterpret_cast<T*>(out));
        })
        return check_launch("latent_attend_plain_kernel");
    }
    SKYRL_REQUIRE(nparts >= 1 && part_min >= kBS && part_min % kBS == 0,
                  "latent_attend: nparts >= 1 and part_min a positive multiple of 16");
    SKYRL_REQUIRE(nparts == 1 || workspace, "latent_attend: nparts > 1 needs a workspace");
    SKYRL_REQUIRE(aligned16(qa) && aligned16(cache) && aligned16(workspace), "latent_attend: 16-byte alignment");
    const uint16_t* q_ = reinterpret_cast<const uint16_t*>(qa);
    const uint16_t* r_ = reinterpret_cast<const uint16_t*>(q_rot);
    const uint16_t* c_ = reinterpret_cast<const uint16_t*>(cache);
    uint16_t* o_ = reinterpret_cast<uint16_t*>(out);
    const HeadEnd<uint16_t> end_{sinks, reinterpret_cast<const uint16_t*>(gate), gate_stride};
    float* ws_o = reinterpret_cast<float*>(workspace);
    float* ws_ml = ws_o ? ws_o + (size_t)T_ * heads * nparts * (((rank + 15) / 16) * 16) : nullptr;
    const int nk = row / 32, nv = (rank + 15) / 16;
    if (nv <= 4 && nk <= 4) {
        LAUNCH_ATTEND(4, 4, false);
    } else if (nv <= 8 && nk <= 6) {
        LAUNCH_ATTEND(8, 6, false);
    } else if (nv <= 16 && nk <= 10) {
        LAUNCH_ATTEND(16, 10, false);
    } else if (rank == 512 && nk == 18) {
        LAUNCH_ATTEND(32, 18, true);
    } else {
        LAUNCH_ATTEND(32, 20, false);
    }
    int rc = check_launch("latent_attend_mfma_kernel");
    if (rc != SKYRL_OK || nparts == 1) return rc;
    if (up) {
        hipLaunchKernelGGL(latent_merge_up_kernel, dim3((up->N + 15) / 16, 1, heads), dim3(2 * kFormers), 0, s, *up,
                           Merge{ws_o, ws_ml, positions, T_, heads, rank, window, part_min, nparts, end_, o_});
        return check_launch("latent_merge_up_kernel");
    }
    hipLaunchKernelGGL(latent_merge_kernel, dim3(heads, T_), dim3(kWave * 2), 0, s, ws_o, ws_ml, positions, T_, heads, rank,
                       window, part_min, nparts, end_, o_);
    return check_launch("latent_merge_kernel");
}

}  // namespace

extern "C" int skyrl_latent_attend(const void* qa, const void* q_rot, int64_t q_stride, int64_t q_head,
                                   const void* cache, int32_t row, const int32_t* block_tables, int64_t bt_stride,
                                   const int32_t* bt_row, const int64_t* positions, int32_t T_, int32_t heads,
                                   int32_t rank, int32_t rot_dim, float scale, int32_t window, int32_t part_min,
                                   int32_t nparts, const float* sinks, const void* gate, int64_t gate_stride, void* out,
                                   void* workspace, int32_t dtype, void* stream) {
    return latent_attend(qa, q_rot, q_stride, q_head, cache, row, block_tables, bt_stride, bt_row, positions, T_, heads, rank, rot_dim,
                         scale, window, part_min, nparts, sinks, gate, gate_stride, out, workspace, dtype, nullptr, stream);
}

extern "C" int32_t skyrl_latent_attend_up_fits(int32_t T_, int32_t rank, int32_t rot_dim, int32_t row, int32_t nparts) {
    return T_ > 0 && T_ <= kMergeRows && nparts > 1 && nparts <= kMergeParts && rank % 8 == 0 && rank <= kMergeRank &&
           skyrl_latent_attend_mfma(rank, rot_dim, row, SKYRL_BF16);
}

extern "C" int skyrl_latent_attend_up(const void* qa, const void* q_rot, int64_t q_stride, int64_t q_head,
                                      const void* cache, int32_t row, const int32_t* block_tables, int64_t bt_stride,
                                      const int32_t* bt_row, const int64_t* positions, int32_t T_, int32_t heads,
                                      int32_t rank, int32_t rot_dim, float scale, int32_t window, int32_t part_min,
                                      int32_t nparts, const float* sinks, const void* gate, int64_t gate_stride, void* out,
                                      void* workspace, const void* up, int32_t vdim, void* y, int64_t y_token, int64_t y_head,
                                      void* stream) {
    SKYRL_REQUIRE(skyrl_latent_attend_up_fits(T_, rank, rot_dim, row, nparts), "latent_attend_up: sizes that it does not take");
    SKYRL_REQUIRE(up && y && vdim > 0 && aligned16(up) && (reinterpret_cast<uintptr_t>(y) & 1) == 0,
                  "latent_attend_up: rows must be 16-byte aligned");
    RowsProduct p{};
    p.n = T_;
    p.K = rank;
    p.w = reinterpret_cast<const uint16_t*>(up);
    p.ldw = rank;
    p.N = vdim;
    p.out = y;
    p.ldo = y_token;
    p.row_blocks = 1;
    p.w_batch = (int64_t)vdim * rank;
    p.out_batch = y_head;
    return latent_attend(qa, q_rot, q_stride, q_head, cache, row, block_tables, bt_stride, bt_row, positions, T_, heads, rank, rot_dim,
                         scale, window, part_min, nparts, sinks, gate, gate_stride, out, workspace, SKYRL_BF16, &p, stream);
}

extern "C" int skyrl_latent_gather(const void* cache, int32_t row, const int32_t* block_tables, int64_t bt_stride,
                                   const int32_t* seg, int32_t nseg, int32_t max_count, int32_t rank, int32_t rot_dim,
                                   void* latent, void* k_rot, int32_t dtype, void* stream) {
    SKYRL_REQUIRE_T(dtype, "latent_gather");
    SKYRL_REQUIRE(nseg >= 0 && nseg <= 65535 && max_count > 0 && rank > 0 && rot_dim >= 0 && row >= rank + rot_dim &&
                      row % 32 == 0,
                  "latent_gather: bad sizes");
    if (nseg == 0) return SKYRL_OK;
    SKYRL_REQUIRE(cache && block_tables && seg && latent && k_rot, "latent_gather: null pointer");
    SKYRL_DISPATCH_T(dtype, {
        hipLaunchKernelGGL((latent_gather_kernel<T>), dim3((max_count + 63) / 64 * 4, nseg), dim3(kNT), 0,
                           as_stream(stream), reinterpret_cast<const T*>(cache), row, block_tables, bt_stride, seg,
                           rank, rot_dim, reinterpret_cast<T*>(latent), reinterpret_cast<T*>(k_rot));
    })
    return check_launch("latent_gather_kernel");
}

#define LAUNCH_PREFILL(NK, NV, QT)                                                                                    \
    if (vec) LAUNCH_PREFILL_(NK, NV, QT, true);                                                                       \
    else LAUNCH_PREFILL_(NK, NV, QT, false)
#define LAUNCH_PREFILL_(NK, NV, QT, VEC)                                                                              \
    hipLaunchKernelGGL((latent_prefill_kernel<NK, NV, QT, VEC>), dim3((unsigned)ntiles * heads), dim3(512 / QT), 0,   \
                       as_stream(stream), reinterpret_cast<const uint16_t*>(q), q_stride,                             \
                       reinterpret_cast<const uint16_t*>(k_nope), k_stride, reinterpret_cast<const uint16_t*>(k_rot), \
                       reinterpret_cast<const uint16_t*>(v_t), vt_stride, tiles, heads, dim, rot_dim, vdim,           \
                       scale * kLog2e, window, end_, reinterpret_cast<uint16_t*>(out), out_stride)

extern "C" int skyrl_latent_prefill(const void* q, int64_t q_stride, const void* k_nope, int64_t k_stride,
                                    const void* k_rot, const void* v_t, int64_t vt_stride, const int32_t* tiles,
                                    int32_t ntiles, int32_t heads, int32_t dim, int32_t rot_dim, int32_t vdim,
                                    float scale, int32_t window, const float* sinks, const void* gate,
                                    int64_t gate_stride, void* out, int64_t out_stride, void* stream) {
    SKYRL_REQUIRE(ntiles >= 0 && heads > 0 && dim >= 0 && rot_dim >= 0 && dim + rot_dim > 0 && dim + rot_dim <= 256 &&
                      vdim > 0 && vdim <= 256,
                  "latent_prefill: dim + rot_dim and vdim must be in [1, 256]");
    SKYRL_REQUIRE((int64_t)ntiles * heads < (1 << 30), "latent_prefill: grid too large");
    SKYRL_REQUIRE(vt_stride % 64 == 0, "latent_prefill: vt_stride must be a multiple of 64");
    if (ntiles == 0) return SKYRL_OK;
    SKYRL_REQUIRE(q && k_nope && k_rot && v_t && tiles && out, "latent_prefill: null pointer");
    SKYRL_REQUIRE(aligned16(k_nope) && aligned16(k_rot) && aligned16(v_t), "latent_prefill: 16-byte alignment");
    SKYRL_REQUIRE(!gate || gate_stride >= heads, "latent_prefill: gate_stride");
    const HeadEnd<uint16_t> end_{sinks, reinterpret_cast<const uint16_t*>(gate), gate_stride};
    const int nk = (dim + rot_dim + 31) / 32, nv = (vdim + 15) / 16;
    const bool vec = dim % 8 == 0 && rot_dim % 8 == 0 && k_stride % 8 == 0 && q_stride % 8 == 0 && aligned16(q);
    if (nk <= 2 && nv <= 8) {
        LAUNCH_PREFILL(2, 8, 2);
    } else if (nk <= 4 && nv <= 8) {
        LAUNCH_PREFILL(4, 8, 2);
    } else if (nk <= 6 && nv <= 8) {
        LAUNCH_PREFILL(6, 8, 2);
    } else {
        LAUNCH_PREFILL(8, 16, 1);
    }
    return check_launch("latent_prefill_kernel");
}
