// Products of many bf16 rows on the matrix instructions, two of them gated (moe.hip, gated_product.hip).
#pragma once
#include <type_traits>

#include "gate.h"
#include "stream.h"

namespace skyrl {

// All but the N latest loads have landed, all LDS reads have returned.
template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void lds_read(s16x8& v, uint32_t at, int offset) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(offset));
}

// The gated product of one pair of f32 sums where it is rounded to 16 bits at once: gated()'s forms with the bare exponential and
// reciprocal, whose error (1e-6 at arguments of 20) is lost in that rounding. Against 64 bits, relative 2-norm, depths 1536 to
// 4096: 0.00166 for every activation, 0.0028 to 0.0031 by the library's products, rounded to 16 bits, and gated(). Where the
// products are exact and the activation alone errs, both are off by the same seven digits, and results that are not the nearest
// are 8e-6 to 3e-5 (silu; gated() 0 to 1e-5) and 1e-5 to 6e-3 (gelu; gated() 2e-5 to 0.19, from 1 + tanh). gated() in its place:
// 8192 x 2048, 6144: 412 against 385 us (gelu), 366 against 342 (silu).
template <int ACT>
__device__ __forceinline__ float gated16(float g, float u, const Gate& f) {
    if constexpr (ACT == SKYRL_ACT_SILU) return g * sigmoid_<uint16_t>(g) * u;
    if constexpr (ACT == SKYRL_ACT_CLAMPED) {
        g = fminf(g, f.limit);
        u = fminf(fmaxf(u, -f.limit), f.limit);
        return g * sigmoid_<uint16_t>(f.alpha * g) * (u + 1.f);
    }
    return gelu_tanh_<uint16_t>(g) * u;
}

enum WideKind { kGateUp, kDown, kGated };
constexpr int kCUs = 256;  // a multiple of the 8 XCDs
struct Wide {
    const uint16_t *x, *w;
    uint16_t* out;
    int K, N;  // depth, output columns
    int64_t ldx, ldw;
    int ntiles;  // routed: at most, those in use in tile_expert[ntiles]
    // routed
    const int32_t *order, *tile_expert;
    int row_div;          // kGateUp: row of x of a pair: pair / row_div
    const float* weight;  // kDown: of the pair, NULL: 1
    // kGated
    int n;
    Gate gate;
};

// a += w x on 16 x 16 x 32, in the accumulator's own registers (the compiler's form may take others and copy them back on
// every turn of a loop). Before anything but a product reads them, the caller lets 16 cycles pass.
__device__ __forceinline__ void product(f32x4& a, const s16x8& w, const s16x8& x) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(a) : "v"(w), "v"(x));
}

// Whether an expert's tiles, which follow each other, are this one alone.
__device__ __forceinline__ bool one_tile(const int32_t* tile_expert, int tile, int ntiles, int e) {
    return (tile == 0 || tile_expert[tile - 1] != e) && (tile + 1 == ntiles || tile_expert[tile + 1] != e);
}

// Tiles of 256 rows (prompts): 256 weight rows per workgroup of four waves, 128 x 128 results and a SIMD each. A wave has nobody
// to hide behind, so its reads of the next operands and the loads of later stages are placed between the products, one every
// few. With 128 x 64 a wave (eight of them) the operands' reads alone took as many LDS cycles as the products took matrix cycles.
// Stages of 64 deep go round a ring of LDS slots of 64 rows, 19 for two stages of 8 and the first three of a third: with two
// stages alone a stage's loads started when the one before was released and either met all at once (64 bytes a cycle and CU)
// or had too little time to land.
// A workgroup per CU goes through its XCD's run of items (a tile and 256 weight rows): the next one's first stages are loaded
// while the results leave, 16 rows at a time through a piece of LDS of the wave's own.
// A tile's rows are spread over the two rows of waves by sixteens, and products past its last 64 used rows are left out (700
// pairs per expert: a sixth of the rows is padding). The depth is a multiple of 64, the columns of the item's.
//   kGateUp, kDown  routed experts (moe.hip): rows by the pairs' order. kGateUp takes a row of x per token and leaves one per
//                   place, silu(gate) up; kDown takes one per place and leaves one per pair, weighted.
//   kGated          one matrix of N gate and N up rows, x and the output row by row, any activation (gated_product.hip).
// Bound: the products; in the loop they run at 1.5 PFLOP/s over all CUs, the rate of a large product of the library, the clock
// being at 1.75 to 1.9 GHz then. Measured, 64 experts of 768 x 2048, 8 per token, gate_up / down, us (before: eight waves, a
// workgroup per tile and columns, two stages): 2048 tokens 153 / 85 (174 / 94), 5637 tokens 273 / 170 (305 / 189), 8192 tokens
// 380 / 255 (434 / 275).
// ONCE: weights of an expert with one tile go past the caches (non-temporal), those of an expert with several, which read them from
// there, do not: 64 experts of 768 x 2048, both products, us (all cached / all past): 1563 tokens 185 (195 / 186), unevenly loaded 192
// (196 / 202), 2048 tokens 260 (259 / 275). The loops for both are one inlined body each: as calls they kept their captures in scratch.
template <int KIND, int ACT, bool ONCE>
__global__ __launch_bounds__(256) void wide_kernel(Wide p) {
    constexpr bool GATED = KIND != kDown, ROUTED = KIND != kGated, GATHER = KIND != kDown;
    const int ncols = p.N / (GATED ? 128 : 256);
    constexpr int TM = 256, BK = 64, NT = 8, L = 8;       // results: NT 16-wide tiles of columns a wave; L loads each of x, w
    constexpr int kSlot = 64 * BK, RING = 19;              // 64 rows; slots of a stage: four of x, four of w
    constexpr int OC = GATED ? 128 : 256, WC = OC / 2;     // output columns, a wave's
    constexpr int LR = WC / 8, SI = LR / 4, LO = WC + 8;   // lanes per row as it leaves, stores of 16 rows, row in LDS
    constexpr int E1 = 3, E2 = 3, F3 = 5;                  // a stage's loads in the groups of products: early, from the release on
    __shared__ __attribute__((aligned(16))) uint16_t smem[RING * kSlot];
    uint16_t* const s_out = smem + 16 * kSlot;             // free between items, as the first stages go to slots 0 .. 13
    static_assert(4 * 16 * LO <= 3 * kSlot && E1 + E2 == 6, "ring");
    __shared__ int s_row[2][TM], s_rows[2][4];  // of the output, or -1; the last in use
    __shared__ float s_wt[2][TM];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4, wm = wave >> 1, wn = wave & 1;
    const int ntiles = ROUTED ? p.tile_expert[p.ntiles] : p.ntiles;
    const int64_t items = (int64_t)ntiles * ncols;
    const int xcd = blockIdx.x % 8, stride = gridDim.x / 8;
    const int end = (int)(items * (xcd + 1) / 8);
    int item = (int)(items * xcd / 8) + blockIdx.x / 8;
    if (item >= end) return;
    const int nk = p.K / BK;

    // An XCD's workgroups read few tiles' rows and few columns' weights at a time. Routed: a tile's columns follow each other
    // (an expert has about as many tiles as its weights have columns here). kGated: blocks of four tiles, column by column.
    auto place = [&](int it, int& tile, int& col) {
        if constexpr (ROUTED) {
            tile = it / ncols;
            col = it % ncols;
        } else {
            const int block = it / (4 * ncols), in = it - block * 4 * ncols, high = min(4, ntiles - 4 * block);
            col = in / high;
            tile = 4 * block + in - col * high;
        }
    };
    // the item after this one: its rows' pairs are read an item ahead
    int next_e = 0, next_pair = 0, next_rows[L];
    bool next_once = false, once = false;  // the item's
    auto peek = [&](int it) __attribute__((always_inline)) {
        if constexpr (ROUTED) {
            int tile, col;
            place(it, tile, col);
            const int32_t* order = p.order + (int64_t)tile * TM;
            next_e = p.tile_expert[tile];
            if constexpr (ONCE) next_once = one_tile(p.tile_expert, tile, p.ntiles, next_e);
            next_pair = order[tid];
            if constexpr (GATHER)
#pragma unroll
                for (int i = 0; i < L; ++i) next_rows[i] = order[i / 2 * 64 + wave * 16 + i % 2 * 8 + lane / 8];
        }
    };
    // A slot is loaded by all waves, two pieces of 8 rows each. Global sources of this lane's 16 bytes: chunk (lane % 8) ^ (row
    // / 2 % 8), so that the 16 rows a matrix operand reads at a time lie in different banks. Rows of w follow each other.
    const int chunk[2] = {(lane % 8 ^ lane / 16) * 8, (lane % 8 ^ (lane / 16 + 4)) * 8};  // even, odd piece
    const uint16_t *xs[GATHER ? L : 2], *ws[2];
    auto wrap = [](int slot) { return slot >= RING ? slot - RING : slot; };
    auto fetch = [&](auto nt, int t, int base, int i) __attribute__((always_inline)) {  // load i of stage t (the last again past the end), whose first slot is base
        uint16_t* dst = smem + wrap(base + i / 2) * kSlot + (wave * 2 + i % 2) * 512;
        const int64_t k0 = min(t, nk - 1) * BK;
        const int64_t row = (i % L) / 2 * 64 + (GATED && i >= L + L / 2 ? p.N - OC : 0);
        const uint16_t* src = i >= L ? ws[i % 2] + (k0 + row * p.ldw) : GATHER ? xs[i % L] + k0 : xs[i % 2] + (k0 + row * p.ldx);
        if (nt.value && i >= L) __builtin_amdgcn_global_load_lds((gbl_void*)src, (lds_void*)dst, 16, 0, 2);
        else __builtin_amdgcn_global_load_lds((gbl_void*)src, (lds_void*)dst, 16, 0, 0);
    };
    int n0, q = 0;
    const double per_row = KIND == kGateUp ? 1.0 / p.row_div : 0.0;
    auto open = [&](int it) __attribute__((always_inline)) {  // start on the item that was peeked at
        const int r0 = wave * 16 + lane / 8;
        int tile, nb;
        place(it, tile, nb);
        n0 = nb * OC;
        const uint16_t* we = p.w + (ROUTED ? (int64_t)max(next_e, 0) * (GATED ? 2 : 1) * p.N * p.ldw : 0);
        we += (n0 + r0) * p.ldw;
        ws[0] = we + chunk[0], ws[1] = we + 8 * p.ldw + chunk[1];
        if constexpr (KIND == kGated) {
#pragma unroll
            for (int i = 0; i < L; ++i)  // rows past the last: the last one, not stored
                xs[i] = p.x + min(tile * TM + i / 2 * 64 + i % 2 * 8 + r0, p.n - 1) * p.ldx + chunk[i % 2];
        } else if constexpr (KIND == kGateUp) {
#pragma unroll
            for (int i = 0; i < L; ++i) {
                const int pair = max(next_rows[i], 0);  // places without a pair: row 0, not stored
                const int d = (int)(pair * per_row), rest = pair - d * p.row_div;  // pair / row_div, one off at most
                xs[i] = p.x + (d + (rest >= p.row_div) - (rest < 0)) * p.ldx + chunk[i % 2];
            }
        } else {
            const uint16_t* xt = p.x + (tile * TM + r0) * p.ldx;
            xs[0] = xt + chunk[0], xs[1] = xt + 8 * p.ldx + chunk[1];
        }
        auto first = [&](auto nt) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 2 * L; ++i) fetch(nt, 0, 0, i);
#pragma unroll
            for (int i = 0; i < E1 + E2 + F3; ++i) fetch(nt, 1, 8, i);
        };
        once = next_once;
        if (ONCE && once) first(std::true_type{});
        else first(std::false_type{});
        if constexpr (KIND == kGated) next_pair = tile * TM + tid < p.n ? tile * TM + tid : -1;
        s_row[q][tid] = GATED && next_pair >= 0 ? tile * TM + tid : next_pair;
        if constexpr (!GATED) s_wt[q][tid] = p.weight && next_pair >= 0 ? p.weight[next_pair] : 1.f;
        const uint64_t in = __ballot(next_pair >= 0);
        if (lane == 0) s_rows[q][wave] = in ? 64 * wave + 64 - __builtin_clzll(in) : 0;
    };
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void*)smem;
    uint32_t xat[2], wat[2];  // of the lane in a slot, by half of the depth
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        wat[ks] = lds0 + c * BK * 2 + ((ks * 4 + g) ^ (c / 2)) * 16;
        xat[ks] = wat[ks] + wm * 16 * BK * 2;
    }
    const int w0 = 4 + (GATED ? wn : 2 * wn), w1 = GATED ? w0 + 2 : w0 + 1;  // the wave's slots of w
    const uint32_t oat = lds0 + (16 * kSlot + wave * 16 * LO) * 2;

    // A step's products in four groups: half of the depth ks, half h of the 2 MH tiles of rows that are in use.
    auto run = [&](auto mh_, auto nt, bool more) __attribute__((always_inline)) {
        constexpr int MH = mh_, M = MH * NT;
        f32x4 acc[2 * MH][NT];
#pragma unroll
        for (int m = 0; m < 2 * MH; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
        s16x8 wf[2][NT], xf[2][MH];
        // The operands' reads are not the compiler's: it would wait for every load into LDS under way before one. Their
        // registers are tied past the wait that ends the group they are in.
        auto read_w = [&](int base, int ks, int n) {
            lds_read(wf[ks][n], wat[ks] + wrap(base + (n < NT / 2 ? w0 : w1)) * (kSlot * 2), n % (NT / 2) * 16 * BK * 2);
        };
        auto read_x = [&](int base, int ks, int h, int i) {
            const int m = h * MH + i;
            lds_read(xf[h][i], xat[ks] + wrap(base + m / 2) * (kSlot * 2), m % 2 * 32 * BK * 2);
        };
        auto landed = [&]() {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
                for (int n = 0; n < NT; ++n) asm volatile("" : "+v"(wf[ks][n]));
#pragma unroll
                for (int i = 0; i < MH; ++i) asm volatile("" : "+v"(xf[ks][i]));
            }
        };
        // the products of (ks, h) with `jobs` calls of job spread between them
        auto group = [&](auto ks_, auto h_, auto jobs_, auto job) __attribute__((always_inline)) {
            constexpr int ks = ks_, h = h_, J = jobs_;
#pragma unroll
            for (int i = 0; i < M; ++i) {
                const int m = i / NT, n = i % NT;
                product(acc[h * MH + m][n], wf[ks][n], xf[h][m]);
#pragma unroll
                for (int j = 0; j < J; ++j)
                    if (j * M / J == i) job(j);
                __builtin_amdgcn_sched_barrier(0);
            }
            landed();
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
#pragma unroll
        for (int n = 0; n < NT; ++n) read_w(0, 0, n), read_w(0, 1, n);
#pragma unroll
        for (int i = 0; i < MH; ++i) read_x(0, 0, 0, i), read_x(0, 0, 1, i);
        landed();
        for (int t = 0, b0 = 0; t < nk; ++t) {
            const int b1 = wrap(b0 + 8), b2 = wrap(b1 + 8);  // of the next stages
            group(I0{}, I0{}, std::integral_constant<int, MH + 2 * L - E1 - E2 - F3>{}, [&](int j) {
                if (j < MH) read_x(b0, 0, 1, j);
                else fetch(nt, t + 1, b1, E1 + E2 + F3 + j - MH);
            });
            group(I0{}, I1{}, std::integral_constant<int, NT + MH + E1>{}, [&](int j) {
                if (j < NT) read_w(b0, 1, j);
                else if (j < NT + MH) read_x(b0, 1, 0, j - NT);
                else fetch(nt, t + 2, b2, j - NT - MH);
            });
            group(I1{}, I0{}, std::integral_constant<int, MH + E2>{}, [&](int j) {
                if (j < MH) read_x(b0, 1, 1, j);
                else fetch(nt, t + 2, b2, E1 + j - MH);
            });
            wait_loads<E1 + E2>();         // this wave's loads of stage t + 1 have landed, its reads of stage t too
            __builtin_amdgcn_s_barrier();  // and everyone's
            asm volatile("" ::: "memory");
            group(I1{}, I1{}, std::integral_constant<int, NT + MH + F3>{}, [&](int j) {
                if (j < NT) read_w(b1, 0, j);
                else if (j < NT + MH) read_x(b1, 0, 0, j - NT);
                else fetch(nt, t + 2, b2, E1 + E2 + j - NT - MH);
            });
            b0 = b1;
        }
        wait_loads<0>();
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last products are in their registers
        __syncthreads();
        const int o = q;
        uint16_t* to = p.out + n0 + wn * WC + lane % LR * 8;
        float scale[2 * MH];
        if constexpr (!GATED)
#pragma unroll
            for (int m = 0; m < 2 * MH; ++m) scale[m] = s_wt[o][(2 * m + wm) * 16 + c];
        if (more) {
            q ^= 1;
            open(item + stride);
        }
        uint4 v[2][SI];
        auto gather = [&](int m, uint4 (&y)[SI]) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < NT; ++n) asm volatile("" : "+a"(acc[m][n]));  // in the accumulators' registers until here
#pragma unroll
            for (int n = 0; n < (GATED ? NT / 2 : NT); ++n) {
                float z[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if constexpr (GATED) z[i] = gated16<ACT>(acc[m][n][i], acc[m][n + NT / 2][i], p.gate);
                    else z[i] = acc[m][n][i] * scale[m];
                }
                *reinterpret_cast<uint2*>(&s_out[wave * 16 * LO + c * LO + n * 16 + 4 * g]) =
                    make_uint2(pack_bf16x2(z[0], z[1]), pack_bf16x2(z[2], z[3]));
            }
            asm volatile("" ::: "memory");
            s16x8 b[SI];
#pragma unroll
            for (int k = 0; k < SI; ++k) lds_read(b[k], oat + (lane / LR * LO + lane % LR * 8) * 2, k * (64 / LR) * LO * 2);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int k = 0; k < SI; ++k) {
                asm volatile("" : "+v"(b[k]));
                y[k] = *reinterpret_cast<const uint4*>(&b[k]);
            }
        };
        auto leave = [&](int m, const uint4 (&y)[SI]) __attribute__((always_inline)) {
            int row[SI];
#pragma unroll
            for (int k = 0; k < SI; ++k) row[k] = s_row[o][(2 * m + wm) * 16 + k * (64 / LR) + lane / LR];
#pragma unroll
            for (int k = 0; k < SI; ++k)
                if (row[k] >= 0) *reinterpret_cast<uint4*>(to + (int64_t)row[k] * p.N) = y[k];
        };
        gather(0, v[0]);
        gather(1, v[1]);
        wait_loads<0>();  // the next item's first stages, before stores are under way too
        leave(0, v[0]);
        leave(1, v[1]);
#pragma unroll
        for (int m = 2; m < 2 * MH; ++m) {
            gather(m, v[m & 1]);
            leave(m, v[m & 1]);
        }
    };
    peek(item);
    open(item);
    wait_loads<0>();
    for (; item < end; item += stride) {
        __syncthreads();
        const int* sr = s_rows[q];
        const int rows = max(max(sr[0], sr[1]), max(sr[2], sr[3]));
        const bool more = item + stride < end;
        if (more) peek(item + stride);
        auto all = [&](auto nt) __attribute__((always_inline)) {
            if (rows > 192) run(std::integral_constant<int, 4>{}, nt, more);
            else if (rows > 128) run(std::integral_constant<int, 3>{}, nt, more);
            else if (rows > 64) run(std::integral_constant<int, 2>{}, nt, more);
            else run(std::integral_constant<int, 1>{}, nt, more);
        };
        if (ONCE && once) all(std::bool_constant<ONCE>{});
        else all(std::false_type{});
    }
}

// Items one each for up to three rounds of workgroups, which then go to the CUs as these get free; with more, a workgroup per
// CU (gate_up as above, 2048 tokens: 161 us against 171; 8192: 395 against 380).
inline bool wide_fits(int K, int N, bool gated) { return K > 0 && K % 64 == 0 && N % (gated ? 128 : 256) == 0; }
template <int KIND, int ACT = SKYRL_ACT_SILU, bool ONCE = false>
int launch_wide(const Wide& p, hipStream_t s) {
    const int64_t items = (int64_t)(p.N / (KIND == kDown ? 256 : 128)) * p.ntiles;
    SKYRL_REQUIRE(items < (1ll << 31) && p.ntiles < (1 << 23), "wide products: too many rows in one call");
    const unsigned grid = (unsigned)(items > 3 * kCUs ? kCUs : (items + 7) / 8 * 8);
    hipLaunchKernelGGL((wide_kernel<KIND, ACT, ONCE>), dim3(grid), dim3(256), 0, s, p);
    return check_launch("wide_kernel");
}

}  // namespace skyrl
