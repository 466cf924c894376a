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
__device__ __forceinline__ void lds_read(uint32_t& v, uint32_t at, int offset) {
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(offset));
}
__device__ __forceinline__ void lds_write(uint32_t at, uint32_t v) {
    asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(v) : "memory");
}
__device__ __forceinline__ void lds_write(uint32_t at, uint2 v) {
    asm volatile("ds_write_b64 %0, %1" ::"v"(at), "v"(v) : "memory");
}
// 16 bytes a lane into LDS from `offset` bytes past what `all` begins with and the lane's own. Operands of less than 4 GB: a uniform
// step of the depth costs no vector instruction, and an address one register.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t whole_buffer(const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0xffffffff, 0x00027000);
}
template <int POLICY = 0>
__device__ __forceinline__ void buffer_to_lds(__amdgpu_buffer_rsrc_t all, uint32_t own, int offset, uint32_t to) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(all, (lds_void*)(uintptr_t)to, 16, own, offset, 0, POLICY);
}
// 16 bytes from the lanes whose row is not negative, without a way round the store. NT: past the caches, with the weights (64 experts
// of 768 x 2048, gate_up / down, us: 800 tokens 76 / 48 -> 70 / 45, 1563 tokens 93 / 58 -> 91 / 55; with weights that stay, 5637 tokens 239 /
// 150 -> 240 / 149).
template <bool NT>
__device__ __forceinline__ void store_row(uint16_t* to, s16x8 v, int row) {
    uint64_t all;
    if constexpr (NT)
        asm volatile(
            "v_cmp_lt_i32 vcc, -1, %3\n\t"
            "s_and_saveexec_b64 %0, vcc\n\t"
            "global_store_dwordx4 %1, %2, off nt\n\t"
            "s_mov_b64 exec, %0"
            : "=&s"(all)
            : "v"(to), "v"(v), "v"(row)
            : "vcc", "scc", "memory");
    else
        asm volatile(
            "v_cmp_lt_i32 vcc, -1, %3\n\t"
            "s_and_saveexec_b64 %0, vcc\n\t"
            "global_store_dwordx4 %1, %2, off\n\t"
            "s_mov_b64 exec, %0"
            : "=&s"(all)
            : "v"(to), "v"(v), "v"(row)
            : "vcc", "scc", "memory");
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

enum WideKind { kGateUp, kDown, kGated, kDense };
constexpr int kCUs = 256;  // a multiple of the 8 XCDs
struct Wide {
    const uint16_t *x, *w;
    uint16_t* out;
    int K, N;  // depth, output columns
    int64_t ldx, ldw;
    int ntiles;  // routed: at most, those in use in tile_expert[ntiles]
    // routed
    const int32_t *order, *tile_expert;
    int row_div;          // kGateUp: row of x of a pair: pair / row_div, by div_mul and div_shift
    uint32_t div_mul;
    int div_shift;
    const float* weight;  // kDown: of the pair, NULL: 1
    // kGated, kDense
    int n, tile_rows;  // rows of a tile: 64 to 256 by 64
    Gate gate;
};

// n / d for 0 <= n < 2^31, 1 < d <= 2^31: the upper half of n ceil(2^(32 + s) / d), shifted by s = ceil(log2 d) - 1. The multiplier
// is less than d <= 2^(s + 1) parts of 2^(32 + s) / d too large, n times which is less than one part of d.
inline void set_division(Wide& p) {
    int s = 0;
    while ((2ll << s) < p.row_div) ++s;
    p.div_shift = s;
    p.div_mul = p.row_div > 1 ? (uint32_t)(((1ull << (32 + s)) + p.row_div - 1) / p.row_div) : 0;
}

// a += w x on 16 x 16 x 32, in the accumulator's own registers (the compiler's form may take others and copy them back on
// every turn of a loop). Before anything but a product reads them, the caller lets 16 cycles pass.
__device__ __forceinline__ void product(f32x4& a, const s16x8& w, const s16x8& x) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(a) : "v"(w), "v"(x));
}

__device__ __forceinline__ void first_product(f32x4& a, const s16x8& w, const s16x8& x) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(a) : "v"(w), "v"(x));
}

// A uniform value that no store of this launch changes, by a scalar load.
__device__ __forceinline__ int32_t uniform(const int32_t* p) {
    return *reinterpret_cast<const __attribute__((address_space(4))) int32_t*>(reinterpret_cast<uintptr_t>(p));
}

// The step of the depth that an expert's products begin with; past the last one they go on at the first. Workgroups run about in
// step, and at a row stride of 4 KB the same depth of all rows lies in the same few of the memory's channels: weights from HBM
// came at 5.2 TB/s where all experts began at 0, at 6.2 where each begins elsewhere (64 experts of 768 x 2048, gate_up, us: 256 tokens
// 79 -> 63, 700 tokens in tiles of 128 90 -> 75; down, rows of 1536 bytes, 40.7 -> 39.4). One start for an expert: its tiles, and
// a tile's columns, share what they read (a start for each column: 5637 tokens 265 us, 243 with this). kDense with ONCE, where all
// columns read the same few rows: a start for each half of an item's columns. Which items are halved follows from the columns alone there,
// so a row's sums do not depend on its place. kGated has one call's items of a column whole and halved: all from 0, as its tiles of 256
// (128 x 2048, 6144 gated 22.1 us, 21.1 with a start for each half, by which equal rows of different tiles had different bits).
__device__ __forceinline__ int depth_start(int e, int K) {
    return K % 256 == 0 ? (int)__umulhi((uint32_t)e * 0x9E3779B9u, (uint32_t)K / 64) : 0;
}

// A workgroup's items: of an XCD's run, one in `stride`, and of what is left over behind the whole rounds halves of the columns where
// there are workgroups for both.
struct Share {
    int first, stride, at, rounds, mine;
    bool halve;
    __host__ __device__ Share(int64_t items, int grid, int block) : stride(grid / 8), at(block / 8) {
        const int xcd = block % 8;
        first = (int)(items * xcd / 8);
        const int left = (int)(items * (xcd + 1) / 8) - first, over = left % stride;
        rounds = left / stride, halve = 2 * over <= stride;
        mine = rounds + (at < (halve ? 2 * over : over));
    }
    // The i-th of them, and whether it is one half of its columns or the other (1, 2).
    __host__ __device__ int nth(int i) const { return first + i * stride + (halve && i == rounds ? at / 2 : at); }
    __host__ __device__ int half_of(int i) const { return halve && i == rounds ? 1 + at % 2 : 0; }
};
// A workgroup per CU, or as many as every XCD needs to halve all of its items.
inline int wide_grid(int64_t items) { return (int)(items > kCUs / 2 ? kCUs : (items + 7) / 8 * 16); }

// Whether an expert's tiles, which follow each other, are this one alone.
__device__ __forceinline__ bool one_tile(const int32_t* tile_expert, int tile, int ntiles, int e) {
    return (tile == 0 || tile_expert[tile - 1] != e) && (tile + 1 == ntiles || tile_expert[tile + 1] != e);
}

// Tiles of TM rows, 256 (prompts) or, routed, 64 and 128: 256 weight rows per workgroup of four waves, 128 x 128 results and a SIMD each. A wave has nobody
// to hide behind, so its reads of the next operands and the loads of later stages are placed between the products, one every
// few. With 128 x 64 a wave (eight of them) the operands' reads alone took as many LDS cycles as the products took matrix cycles.
// Stages of 64 deep go round a ring of LDS slots of 64 rows, 19 for two stages of 8 and the first three of a third: with two
// stages alone a stage's loads started when the one before was released and either met all at once (64 bytes a cycle and CU)
// or had too little time to land. With tiles of 64 a stage is five slots, three stages are ahead.
// A workgroup per CU goes through its XCD's run of items (a tile and 256 weight rows). The ring does not stop between them: an
// item's last two steps load the next one's first two stages, which land while the results leave, 16 rows at a time through a piece
// of LDS of the wave's own. The next item's rows and weights of pairs go to LDS by direct loads, too, since a load into a register
// would be waited for with everything under way. The first step of an item does not wait for the stores ahead of it, and starts the sums.
// What is left over behind the whole rounds is cut into halves of the columns where there are workgroups for both (1500 x 2048,
// 6144 gated: 288 items, 93 us in two whole rounds, 74 in one and a half). Cut by rows, both halves would read the weights.
// A tile's rows are spread over the two rows of waves by sixteens, and products past its last 64 used rows are left out (700
// pairs per expert: a sixth of the rows is padding), their loads are not: tiles of 64 and 128 where most experts have no more. The depth is a multiple of 64, the columns of the item's.
//   kGateUp, kDown  routed experts (moe.hip): rows by the pairs' order. kGateUp takes a row of x per token and leaves one per
//                   place, silu(gate) up; kDown takes one per place and leaves one per pair, weighted.
// kDense with ONCE: the weights of one tile of rows, all past the caches.
//   kGated, kDense  one matrix, x and the output row by row in tiles of tile_rows (gated_product.hip): of N gate and N up rows,
//                   any activation; of N rows, a multiple of 8, as they are.
// Bound: the products at the power limit (weights of zeros: 8192 x 2048, 6144 gated in 226 us, random ones in 297, 1.39 PFLOP/s, the
// clock at 1.8 to 1.9 GHz); kDown: its loads, 12 stages an item and 128 KB of results. What the ring and the direct loads gave alone, all
// experts from depth 0 (before: an item's loads start when the one before has left, addresses in the ring by compare and select; 64 experts of
// 768 x 2048, 8 per token, gate_up / down, us): 1000 tokens 96 / 53 (111 / 58), 1563 tokens 103 / 58 (119 / 65), 3000 tokens 154 / 98
// (162 / 106), 5637 tokens 247 / 152 (265 / 166), 8192 tokens 356 / 230 (379 / 260); with depth_start and store_row as they are 1563 tokens take
// 91 / 55, 5637 239 / 150. gated: 8192 x 2048, 6144 297 (321), 4000 x 2048, 6144 150 (161).
// Where the loads of an item's last steps were cases in the loop's body, its branches took more than all this gave (324).
// ONCE: weights of an expert with one tile go past the caches (non-temporal), those of an expert with several, which read them from
// there, do not: both products, us (all cached / all past), before: 1563 tokens 185 (195 / 186), unevenly loaded 192 (196 / 202), 2048
// tokens 260 (259 / 275). The loops for both are one inlined body each: as calls they kept their captures in scratch.
template <int KIND, int ACT, bool ONCE, int TM>
__global__ __launch_bounds__(256) void wide_kernel(Wide p) {
    constexpr bool GATED = KIND == kGateUp || KIND == kGated, ROUTED = KIND == kGateUp || KIND == kDown, GATHER = KIND != kDown;
    const int ncols = KIND == kDense ? (p.N + 255) / 256 : p.N / (GATED ? 128 : 256);
    constexpr int BK = 64, XS = TM / 64;                   // slots of x
    constexpr int LW = 8, LX = 2 * XS, L = LX + LW;        // loads of w, of x, of a stage
    constexpr int SS = 4 + XS;                             // slots of a stage
    constexpr int AHEAD = XS == 1 ? 3 : 2;                 // stages under way
    // 64 rows, bytes. Slots of a stage: four of x, four of w, those ahead that are loaded ahead: weights that come from HBM, which
    // have the longer way (1563 tokens 103 / 58 us, behind the rows 106 / 60), else the rows (5637 tokens 247 / 152, 250 / 153).
    constexpr uint32_t SLOT = 64 * BK * 2, RING = 19;
    constexpr bool WF = ONCE;
    constexpr int OC = GATED ? 128 : 256;                  // output columns
    constexpr int REST = XS == 4 ? 5 : 0;                  // of a stage's loads, the last ones
    constexpr int kOut = XS == 4 ? 5 : 2;                  // of a stage's slots, the first where results pass through LDS
    __shared__ __attribute__((aligned(16))) uint16_t smem[RING * SLOT / 2];
    __shared__ int s_rows[2][4];  // of 64 rows each: the last in use; kAll: all are
    constexpr uint32_t kAll = 1 << 16;
    __shared__ int s_row[ROUTED ? 2 : 1][TM];        // the pairs of this item's and the next one's rows, or -1
    __shared__ float s_wt[KIND == kDown ? 2 : 1][TM];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4, wm = wave >> 1, wn = wave & 1;
    const int ntiles = ROUTED ? uniform(p.tile_expert + p.ntiles) : p.ntiles;
    const Share share((int64_t)ntiles * ncols, gridDim.x, blockIdx.x);
    const int mine = share.mine;
    if (mine == 0) return;
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
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void*)smem, rows_at = (uint32_t)(uintptr_t)(lds_void*)&s_rows[0][0],
                   row_at = (uint32_t)(uintptr_t)(lds_void*)&s_row[0][0], wt_at = (uint32_t)(uintptr_t)(lds_void*)&s_wt[0][0];
    // The item after this one: what it needs of its tile is on its way an item ahead.
    int next_tile = 0, next_n0 = 0, next_half = 0, next_e = 0, e_before = 0, e_after = 0;
    auto peek = [&](int i, int qn) __attribute__((always_inline)) {
        int col;
        place(share.nth(i), next_tile, col);
        next_half = share.half_of(i);
        next_n0 = col * OC;
        if constexpr (ROUTED) {
            if (XS == 4 || wave < XS)
                __builtin_amdgcn_global_load_lds((gbl_void*)(p.order + ((int64_t)next_tile * TM + tid)), (lds_void*)&s_row[qn][wave * kWave], 4, 0, 0);
            next_e = uniform(p.tile_expert + next_tile);
            if constexpr (ONCE) {
                e_before = next_tile > 0 ? uniform(p.tile_expert + next_tile - 1) : -1;
                e_after = next_tile + 1 < p.ntiles ? uniform(p.tile_expert + next_tile + 1) : -1;
            }
        }
    };
    // A slot is loaded by all waves, two pieces of 8 rows each. Global sources of this lane's 16 bytes: chunk (lane % 8) ^ (row
    // / 2 % 8), so that the 16 rows a matrix operand reads at a time lie in different banks. Rows of w follow each other.
    const int chunk[2] = {(lane % 8 ^ lane / 16) * 8, (lane % 8 ^ (lane / 16 + 4)) * 8};  // even, odd piece
    const uint16_t *xs[GATHER ? LX : 2], *ws[2];
    uint32_t xo[LX] = {}, wo[LW] = {};  // kDense: in bytes from the first row
    const __amdgpu_buffer_rsrc_t x_all = whole_buffer(p.x), w_all = whole_buffer(p.w);
    int64_t wslot[4] = {};  // what a slot's rows of w are past the item's first; those of a half are the first slots'
    auto wrap = [](uint32_t at) { return min(at, at - RING * SLOT); };  // of less than two rings
    int k_start = 0;        // of the item whose loads are under way
    constexpr bool TURNED = ROUTED || ONCE;
    auto depth = [&](int k) { return TURNED && k + k_start >= p.K ? k + k_start - p.K : k + k_start; };
    auto fetch = [&](auto nt, int k0, uint32_t base, int i) __attribute__((always_inline)) {  // load i at depth k0 of the stage at base
        const bool is_w = WF ? i < LW : i >= LX;
        const int u = WF ? (is_w ? i : i - LW) : is_w ? i - LX : i;
        const uint32_t to = lds0 + wrap(base + i / 2 * SLOT + wave * (SLOT / 4)) + u % 2 * (SLOT / 8);
        lds_void* dst = (lds_void*)(uintptr_t)to;
        if constexpr (KIND == kDense) {
            if (nt.value && is_w) buffer_to_lds<2>(w_all, wo[u], k0 * 2, to);
            else buffer_to_lds(is_w ? w_all : x_all, is_w ? wo[u] : xo[u], k0 * 2, to);
        } else {
            const uint16_t* src = is_w ? ws[u % 2] + (k0 + wslot[u / 2]) : GATHER ? xs[u] + k0 : xs[u % 2] + (k0 + u / 2 * 64 * p.ldx);
            if (nt.value && is_w) __builtin_amdgcn_global_load_lds((gbl_void*)src, dst, 16, 0, 2);
            else __builtin_amdgcn_global_load_lds((gbl_void*)src, dst, 16, 0, 0);
        }
    };
    int n0 = 0, q = 0, tile = 0, half = 0;  // the item's
    bool once = false;
    // Turn to the item that was peeked at: from here on its stages are loaded. What is written to LDS and read of it is not the
    // compiler's, which would wait for every load into LDS under way.
    auto turn = [&](int qn) __attribute__((always_inline)) {
        const int r0 = wave * 16 + lane / 8;
        uint32_t pair = 0, rows[LX] = {};
        if constexpr (ROUTED) lds_read(pair, row_at + (qn * TM + tid % TM) * 4, 0);
        if constexpr (KIND == kGateUp)
#pragma unroll
            for (int i = 0; i < LX; ++i) lds_read(rows[i], row_at + (qn * TM + r0) * 4, (i / 2 * 64 + i % 2 * 8) * 4);
        const int flip = next_half == 2 ? OC / 2 : 0;
        if constexpr (KIND == kDense) {
#pragma unroll
            for (int i = 0; i < LW; ++i)  // rows past the last: the last one, its columns not stored
                wo[i] = (min(next_n0 + (i / 2 * 64 ^ flip) + i % 2 * 8 + r0, p.N - 1) * (uint32_t)p.ldw + chunk[i % 2]) * 2;
        } else {
            const uint16_t* we = p.w + (ROUTED ? (int64_t)max(next_e, 0) * (GATED ? 2 : 1) * p.N * p.ldw : 0);
            we += (next_n0 + r0) * p.ldw;
            ws[0] = we + chunk[0], ws[1] = we + 8 * p.ldw + chunk[1];
#pragma unroll
            for (int j = 0; j < 4; ++j) wslot[j] = ((j * 64 ^ flip) + (GATED && j >= 2 ? p.N - OC : 0)) * p.ldw;
        }
        if constexpr (TURNED) k_start = depth_start(ROUTED ? next_e : next_n0 / (OC / 2) + (next_half == 2), p.K) * BK;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        asm volatile("" : "+v"(pair));
        if constexpr (!ROUTED) {
            const int row0 = next_tile * p.tile_rows;
#pragma unroll
            for (int i = 0; i < LX; ++i) {  // rows past the last: the last one, not stored
                const int row = min(row0 + i / 2 * 64 + i % 2 * 8 + r0, p.n - 1);
                if constexpr (KIND == kDense) xo[i] = (row * (uint32_t)p.ldx + chunk[i % 2]) * 2;
                else xs[i] = p.x + row * p.ldx + chunk[i % 2];
            }
            pair = tid < p.tile_rows && row0 + tid < p.n ? 0 : -1;
        } else if constexpr (KIND == kGateUp) {
#pragma unroll
            for (int i = 0; i < LX; ++i) {
                asm volatile("" : "+v"(rows[i]));
                const uint32_t row = max((int)rows[i], 0);  // places without a pair: row 0, not stored
                xs[i] = p.x + (p.row_div > 1 ? __umulhi(row, p.div_mul) >> p.div_shift : row) * p.ldx + chunk[i % 2];
            }
        } else {
            const uint16_t* xt = p.x + (next_tile * TM + r0) * p.ldx;
            xs[0] = xt + chunk[0], xs[1] = xt + 8 * p.ldx + chunk[1];
            if (XS == 4 || wave < XS) {
                if (p.weight) __builtin_amdgcn_global_load_lds((gbl_void*)(p.weight + max((int)pair, 0)), (lds_void*)&s_wt[qn][wave * kWave], 4, 0, 0);
                else lds_write(wt_at + (qn * TM + tid) * 4, __float_as_uint(1.f));
            }
        }
        if (XS < 4 && wave >= XS) pair = -1;
        const uint64_t in = __ballot((int)pair >= 0);
        if (lane == 0)
            lds_write(rows_at + (qn * 4 + wave) * 4, (uint32_t)(in ? 64 * wave + 64 - __builtin_clzll(in) : 0) | (~in ? 0u : kAll));
    };
    auto turned = [&]() __attribute__((always_inline)) {  // the item's output and tile
        tile = next_tile, half = next_half;
        n0 = next_n0 + (half == 2 ? OC / 2 : 0);
        once = ONCE && (!ROUTED || (e_before != next_e && e_after != next_e));
    };
    const bool chain = nk > 2 * AHEAD - 2;  // an item's last steps load the next one's first stages; its rows have landed then
    uint32_t b0 = 0;            // where the next stage starts in the ring
    auto prime = [&](int i) __attribute__((always_inline)) {
        peek(i, q);
        wait_loads<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        turn(q);
        turned();
#pragma unroll
        for (int j = 0; j < AHEAD; ++j)
#pragma unroll
            for (int i = 0; i < L; ++i) fetch(std::false_type{}, depth(min(j, nk - 1) * BK), wrap(b0 + j * SS * SLOT), i);
        wait_loads<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    uint32_t xat[2], wat[2];  // of the lane in a slot, by half of the depth
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        wat[ks] = lds0 + c * BK * 2 + ((ks * 4 + g) ^ (c / 2)) * 16;
        xat[ks] = wat[ks] + wm * 16 * BK * 2;
    }
    // The last item had all rows and, in this wave, columns: every store had a lane and is counted. Whether one without any is, nothing
    // here depends on.
    bool whole = false;

    // A step's products in four groups: half of the depth ks, half h of the 2 MH tiles of rows that are in use.
    // HALF: of one half of the item's columns, a workgroup's last.
    auto run = [&](auto mh_, auto half_, auto nt, int rows, bool all_rows, bool more) __attribute__((always_inline)) {
        constexpr bool HALF = half_;
        constexpr int MH = mh_, NT = HALF ? 4 : 8, M = MH * NT;     // NT 16-wide tiles of columns a wave
        constexpr int WC = OC / (HALF ? 4 : 2);                   // output columns a wave
        constexpr int LR = WC / 8, SI = LR / 4;                   // lanes per row as it leaves, stores of 16 rows
        constexpr int HW = HALF ? LW / 2 : LW;                    // loads of w a stage
        // A stage's loads in the groups of products: early, from the release on, in the next step.
        constexpr int E1 = XS == 4 ? (HALF ? 2 : 3) : HW / 2, E2 = E1, F3 = XS == 4 ? 5 : LX, F1 = HW + LX - E1 - E2 - F3;
        static_assert(4 * 16 * WC * 2 <= 2 * SLOT && (HALF || F1 == REST) && AHEAD * SS + (E1 + E2) / 2 <= (int)RING, "ring");
        const bool chained = !HALF && more && chain;
        // load i of the run's: half of the columns is two slots' rows of w, with GATED the gate's and the other matrix' first
        auto stage = [&](int k0, uint32_t base, int i) __attribute__((always_inline)) {
            const int before = WF ? 0 : LX, u = i - before;  // of w's loads
            const bool is_w = u >= 0 && u < HW;
            fetch(nt, k0, base, is_w ? before + (HALF && GATED && u >= 2 ? u + 2 : u) : WF ? i - HW + LW : i);
        };
        // the wave's slots of w and its rows in them
        const uint32_t w0 = ((WF ? 0 : XS) + (GATED ? (HALF ? 0 : wn) : HALF ? wn : 2 * wn)) * SLOT, w1 = w0 + (GATED ? 2 : HALF ? 0 : 1) * SLOT;
        constexpr int WT = GATED || !HALF ? NT / 2 : NT;          // tiles of a slot
        const uint32_t wrow = GATED && HALF ? wn * 32 * BK * 2 : 0;
        // Results pass through LDS, 16 rows of WC columns a wave, 16-byte chunks xor-swizzled by the row.
        auto mix = [](int row) { return row / (16 / LR); };
        f32x4 acc[2 * MH][NT];
        s16x8 wf[2][NT], xf[2][MH];
        // The operands' reads are not the compiler's either. Their registers are tied past the wait that ends the group they are in.
        auto read_w = [&](uint32_t base, int ks, int n) {
            lds_read(wf[ks][n], wat[ks] + wrow + wrap(base + (n < WT ? w0 : w1)), n % WT * 16 * BK * 2);
        };
        auto read_x = [&](uint32_t base, int ks, int h, int i) {
            const int m = h * MH + i;
            lds_read(xf[h][i], xat[ks] + wrap(base + ((WF ? 4 : 0) + m / 2) * SLOT), m % 2 * 32 * BK * 2);
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
        auto group = [&](auto first, auto ks_, auto h_, auto jobs_, auto job) __attribute__((always_inline)) {
            constexpr int ks = ks_, h = h_, J = jobs_;
#pragma unroll
            for (int i = 0; i < M; ++i) {
                const int m = i / NT, n = i % NT;
                if constexpr (first.value) first_product(acc[h * MH + m][n], wf[ks][n], xf[h][m]);
                else product(acc[h * MH + m][n], wf[ks][n], xf[h][m]);
#pragma unroll
                for (int j = 0; j < J; ++j)
                    if (j * M / J == i) job(j);
                __builtin_amdgcn_sched_barrier(0);
            }
            landed();
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using Later = std::false_type;
        int k2 = 0;  // depth of the loads under way
        // A step, whose loads are two stages ahead, at depth k; with `turning`, the next item's from here on.
        auto step = [&](auto first, auto turning, int k) __attribute__((always_inline)) {
            // of the next stage, of the one to load and the one before that
            const uint32_t b1 = wrap(b0 + SS * SLOT), bl = wrap(b0 + (AHEAD - 1) * SS * SLOT), b2 = wrap(bl + SS * SLOT);
            constexpr int G1 = first.value ? 0 : F1;        // the first step's stand ahead of the last item's stores
            group(first, I0{}, I0{}, std::integral_constant<int, MH + G1>{}, [&](int j) {
                if (j < MH) read_x(b0, 0, 1, j);
                else stage(k2, bl, E1 + E2 + F3 + j - MH);
            });
            if constexpr (turning.value)
                if (chained) turn(q ^ 1);
            k2 = depth(k);
            group(first, I0{}, I1{}, std::integral_constant<int, NT + MH + E1>{}, [&](int j) {
                if (j < NT) read_w(b0, 1, j);
                else if (j < NT + MH) read_x(b0, 1, 0, j - NT);
                else stage(k2, b2, j - NT - MH);
            });
            group(Later{}, I1{}, I0{}, std::integral_constant<int, MH + E2>{}, [&](int j) {
                if (j < MH) read_x(b0, 1, 1, j);
                else stage(k2, b2, E1 + j - MH);
            });
            // this wave's loads of stage t + 1 have landed, its reads of stage t too
            constexpr int LATER = (AHEAD - 2) * (HW + LX) + E1 + E2;
            if (first.value && whole) wait_loads<LATER + OC / 8>();
            else wait_loads<LATER>();
            __builtin_amdgcn_s_barrier();  // and everyone's
            asm volatile("" ::: "memory");
            group(Later{}, I1{}, I1{}, std::integral_constant<int, NT + MH + F3>{}, [&](int j) {
                if (j < NT) read_w(b1, 0, j);
                else if (j < NT + MH) read_x(b1, 0, 0, j - NT);
                else stage(k2, b2, E1 + E2 + j - NT - MH);
            });
            b0 = b1;
        };
#pragma unroll
        for (int n = 0; n < NT; ++n) read_w(b0, 0, n);
#pragma unroll
        for (int i = 0; i < MH; ++i) read_x(b0, 0, 0, i);
        landed();
        // Past the item's last stage the loads are the next item's, or the last stage's again. The steps around that are copies of
        // their own: as cases of the loop's body they cost it 7 %.
        const int last = (nk - 1) * BK;
        step(std::true_type{}, Later{}, min(AHEAD * BK, last));
        if constexpr (HALF) {
            for (int t = 1; t < nk; ++t) step(Later{}, Later{}, min((t + AHEAD) * BK, last));
        } else {
            for (int t = 1; t < nk - AHEAD; ++t) step(Later{}, Later{}, (t + AHEAD) * BK);
            if (nk > AHEAD) step(Later{}, std::true_type{}, chained ? 0 : last);
#pragma unroll
            for (int j = 1; j < AHEAD; ++j)
                if (nk > AHEAD - j) step(Later{}, Later{}, chained ? j * BK : last);
            if (chained)
#pragma unroll
                for (int i = L - REST; i < L; ++i) fetch(nt, k2, wrap(b0 + (AHEAD - 1) * SS * SLOT), i);  // what remains of the next item's
        }
        uint16_t* const to = p.out + n0 + wn * WC + lane % LR * 8;
        const int own = tile * (ROUTED ? TM : p.tile_rows);
        const bool in = KIND != kDense || n0 + wn * WC + lane % LR * 8 < p.N, any = KIND != kDense || n0 + wn * WC < p.N;  // this lane's columns, some lane's
        // The last products are in their registers 16 cycles on. The item's last stage is read: two of its slots, the ones that
        // nothing is loaded into before the next barrier, are the results' way.
        uint32_t scale[2 * MH];
        if constexpr (KIND == kDown) {
#pragma unroll
            for (int m = 0; m < 2 * MH; ++m) lds_read(scale[m], wt_at + q * TM * 4 + (wm * 16 + c) * 4, m * 128);
        }
        if (chained) turned();
        asm volatile("s_nop 15\n\ts_nop 15\n\ts_waitcnt lgkmcnt(0)" ::: "memory");
        if constexpr (KIND == kDown)
#pragma unroll
            for (int m = 0; m < 2 * MH; ++m) asm volatile("" : "+v"(scale[m]));
        const uint32_t out_at = lds0 + wrap(wrap(b0 + (RING - SS) * SLOT) + (kOut + wave / 2) * SLOT);
        uint32_t put_at[WC / 16], get_at[SI];
        int l = lane;
        asm volatile("" : "+v"(l));  // formed here: as values of the whole launch they were put out to memory
#pragma unroll
        for (int n = 0; n < WC / 16; ++n)
            put_at[n] = out_at + (wave % 2 * 16 * WC + l % 16 * WC) * 2 + ((2 * n + l / 32) ^ mix(l % 16)) * 16 + l / 16 % 2 * 8;
#pragma unroll
        for (int k = 0; k < SI; ++k) {
            const int row = k * (64 / LR) + l / LR;
            get_at[k] = out_at + (wave % 2 * 16 * WC + row * WC) * 2 + ((l % LR) ^ mix(row)) * 16;
        }
        auto put = [&](int m) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < NT; ++n) asm volatile("" : "+a"(acc[m][n]));  // in the accumulators' registers until here
#pragma unroll
            for (int n = 0; n < WC / 16; ++n) {
                float z[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if constexpr (GATED) z[i] = gated16<ACT>(acc[m][n][i], acc[m][n + NT / 2][i], p.gate);
                    else if constexpr (KIND == kDown) z[i] = acc[m][n][i] * __uint_as_float(scale[m]);
                    else z[i] = acc[m][n][i];
                }
                lds_write(put_at[n], make_uint2(pack_bf16x2(z[0], z[1]), pack_bf16x2(z[2], z[3])));
            }
        };
        s16x8 y[2][SI];
        uint32_t row[2][SI];
        // A wave's LDS accesses are in order: the reads of 16 rows follow their writes and go ahead of the next ones'.
        auto get = [&](int m) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < SI; ++k) {
                if constexpr (KIND == kDown)
                    lds_read(row[m & 1][k], row_at + q * TM * 4 + (wm * 16 + lane / LR) * 4, (m * 32 + k * (64 / LR)) * 4);
                lds_read(y[m & 1][k], get_at[k], 0);
            }
        };
        auto leave = [&](int m) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < SI; ++k) {
                asm volatile("" : "+v"(y[m & 1][k]));
                int64_t to_row;
                int on;
                if constexpr (KIND == kDown) {
                    asm volatile("" : "+v"(row[m & 1][k]));
                    on = (int)row[m & 1][k];
                    to_row = row[m & 1][k];
                } else {
                    const int r = (2 * m + wm) * 16 + k * (64 / LR) + lane / LR;
                    on = in ? rows - 1 - r : -1;
                    to_row = own + r;
                }
                store_row<ONCE && ROUTED>(to + to_row * p.N, y[m & 1][k], on);
            }
        };
        put(0);
        get(0);
#pragma unroll
        for (int m = 0; m < 2 * MH; ++m) {
            if (m + 1 < 2 * MH) {
                put(m + 1);
                asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(WC / 16) : "memory");
                get(m + 1);
            } else {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            }
            leave(m);
        }
        whole = MH == 4 && all_rows && any && nk > AHEAD + 1;  // with fewer stages the next item's rows are needed right behind the first step
    };
    prime(0);
    for (int i = 0;; ++i) {
        uint32_t r4[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) lds_read(r4[j], rows_at + q * 16, j * 4);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(r4[j]));
        int rows = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) rows = max(rows, (int)(r4[j] & (kAll - 1)));
        rows = __builtin_amdgcn_readfirstlane(rows);
        const bool all_rows = __builtin_amdgcn_readfirstlane(r4[0] & r4[1] & r4[2] & r4[3]) & kAll, more = i + 1 < mine;
        if (more && chain) peek(i + 1, q ^ 1);
        auto all = [&](auto half_, auto nt) __attribute__((always_inline)) {
            const auto of = [&](auto mh) __attribute__((always_inline)) { run(mh, half_, nt, rows, all_rows, more); };
            if constexpr (XS == 4)
                if (rows > 192) return of(std::integral_constant<int, 4>{});
            if constexpr (XS == 4)
                if (rows > 128) return of(std::integral_constant<int, 3>{});
            if constexpr (XS >= 2)
                if (rows > 64) return of(std::integral_constant<int, 2>{});
            of(std::integral_constant<int, 1>{});
        };
        if (half) {
            if (ONCE && once) all(std::true_type{}, std::bool_constant<ONCE>{});
            else all(std::true_type{}, std::false_type{});
        } else {
            if (ONCE && once) all(std::false_type{}, std::bool_constant<ONCE>{});
            else all(std::false_type{}, std::false_type{});
        }
        if (!more) break;
        q ^= 1;
        __builtin_amdgcn_s_barrier();  // everyone's results have left LDS
        asm volatile("" ::: "memory");
        if (!chain) {
            wait_loads<0>();
            prime(i + 1);
        }
    }
    wait_loads<0>();  // into LDS that is another workgroup's next
}

inline bool wide_fits(int K, int N, bool gated) { return K > 0 && K % 64 == 0 && N % (gated ? 128 : 256) == 0; }
template <int KIND, int ACT = SKYRL_ACT_SILU, bool ONCE = false, int TM = 256>
int launch_wide(Wide p, hipStream_t s) {
    set_division(p);
    const int64_t items = (int64_t)(KIND == kDense ? (p.N + 255) / 256 : p.N / (KIND == kDown ? 256 : 128)) * p.ntiles;
    SKYRL_REQUIRE(items < (1ll << 31) && p.ntiles < (1 << 23), "wide products: too many rows in one call");
    hipLaunchKernelGGL((wide_kernel<KIND, ACT, ONCE, TM>), dim3((unsigned)wide_grid(items)), dim3(256), 0, s, p);
    return check_launch("wide_kernel");
}

}  // namespace skyrl
