// Products of few bf16 rows with streamed weight rows on the matrix instructions (rows_product.hip, moe.hip). A wave fetches its
// own share of the depth, in pieces of 64, with direct loads into LDS of its own: whole 128-byte lines, 16-byte chunks
// xor-swizzled by the row, S pieces under way. Waves meet when the shares' sums are joined, not before.
#pragma once
#include "elem.h"

namespace skyrl {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void gbl_void;

__device__ const uint4 kZero16 = {0u, 0u, 0u, 0u};

// NT 16-row weight tiles, MT 16-row tiles of x, WK waves. HELD: the rows of x lie in LDS whole and are not streamed. ONCE: no
// other workgroup reads these weight rows (moe_stream_kernel has both, by tile), so they go past the caches (non-temporal): a
// step's weights, several times the last-level cache, put out what is read again and wait for its lines to be put out (32768 x
// 2048: 16 rows 28.0 -> 24.6 us, 64 rows 30.1 -> 27.9; in a step's place, eight of 64 experts of 768 x 2048 for 64 rows 74.8 + 39.3
// -> 59.7 + 34.3).
// EXACT: the pieces' sums are added in 64 bits, for one row whose results leave in f32. One chain of f32 sums a wave rounds more than
// the lanes of a wave per weight row did: error / result against 64 bits 0.95e-7, 1.90e-7, 1.65e-7 at 2048, 4096, 6144 deep (2048,
// 4096, 2048 columns), where those had 0.75e-7, 0.85e-7, 0.91e-7, and this has 0.64e-7 at all (3.9, 8.1, 6.8 us; 4.0, 8.2, 6.9).
template <int NT, int MT, int WK, int S, bool HELD = false, bool ONCE = true, bool EXACT = false>
struct Stream {
    static constexpr int kPolicy = ONCE ? 2 : 0;  // the load's cache policy bits: 2 is nt
    static constexpr int BN = 16 * NT, BM = 16 * MT, WP = 2 * NT, XP = HELD ? 0 : 2 * MT, L = WP + XP;  // 1 KB pieces: 8 rows, 64 deep
    static constexpr int kStage = (BN + (HELD ? 0 : BM)) * 64;  // elements
    static constexpr int LR = BN + 4;              // a row of a share's sums
    static constexpr int kSums = WK * BM * LR * 2, kPieces = WK * S * kStage;
    static constexpr int kLds = kPieces > kSums ? kPieces : kSums;  // elements
    static_assert(S <= 8 && (S - 1) * L < 64, "the waits below");

    template <int N>
    static __device__ __forceinline__ void wait_loads() {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
    }
    static __device__ __forceinline__ void lds_read(s16x8& v, uint32_t at, int offset) {
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(offset));
    }

    // acc[m][n]: lane (c, g) has x row 16 m + c, weight rows 16 n + 4 g .. + 3. wrow(r), xrow(r): start of the tile's row r, valid
    // for every r (rows past the last: any row, not stored). K a multiple of 8, the wave's pieces s0 .. s0 + nk - 1 of 64.
    // HELD: between(), called when the first pieces are under way, returns the LDS address of the row in this lane's place, readable
    // up to a multiple of 64 with numbers in it; xrow is not called.
    struct Streamed {
        __device__ uint32_t operator()() const { return 0; }
    };
    template <class WRow, class XRow, class Between = Streamed>
    static __device__ __forceinline__ void run(uint16_t* smem, int K, int s0, int nk, WRow wrow, XRow xrow, f32x4 (&acc)[MT][NT],
                                               Between between = Between{}) {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int c = lane & 15, g = lane >> 4;
        uint16_t* own = smem + wave * (S * kStage);
        // this lane's 16 bytes of every piece: row lane / 8, chunk (lane % 8) ^ row, so that 16 rows read at a time lie in
        // different banks
        const int r8 = lane >> 3, ch = ((lane & 7) ^ r8) * 8;
        static_assert(!HELD || MT == 1, "one tile of held rows");
        const uint16_t *ws[WP], *xs[XP ? XP : 1];
#pragma unroll
        for (int i = 0; i < WP; ++i) ws[i] = wrow(i * 8 + r8) + s0 * 64 + ch;
#pragma unroll
        for (int i = 0; i < XP; ++i) xs[i] = xrow(i * 8 + r8) + s0 * 64 + ch;
        auto fetch = [&](int t) {
            uint16_t* dst = own + (t % S) * kStage;
            const bool in = (s0 + t) * 64 + ch < K;
#pragma unroll
            for (int i = 0; i < WP; ++i) {
                const void* src = in ? (const void*)(ws[i] + t * 64) : (const void*)&kZero16;
                __builtin_amdgcn_global_load_lds((gbl_void*)src, (lds_void*)(dst + i * 512), 16, 0, kPolicy);
            }
#pragma unroll
            for (int i = 0; i < XP; ++i) {
                const void* src = in ? (const void*)(xs[i] + t * 64) : (const void*)&kZero16;
                __builtin_amdgcn_global_load_lds((gbl_void*)src, (lds_void*)(dst + (WP + i) * 512), 16, 0, 0);
            }
        };
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < S; ++t)
            if (t < nk) fetch(t);
        double sums[EXACT ? MT : 1][EXACT ? NT : 1][4] = {};
        const uint32_t base = (uint32_t)(uintptr_t)(lds_void*)own + c * 128;
        const uint32_t held = HELD ? between() + s0 * 128 + g * 16 : 0;
        for (int t = 0; t < nk; ++t) {
            const int left = nk - 1 - t;  // pieces after this one; at most S - 1 of them are under way
            if (left >= S - 1) wait_loads<(S - 1) * L>();
            else if (S > 7 && left == 6) wait_loads<(S > 7 ? 6 * L : 0)>();
            else if (S > 6 && left == 5) wait_loads<(S > 6 ? 5 * L : 0)>();
            else if (S > 5 && left == 4) wait_loads<(S > 5 ? 4 * L : 0)>();
            else if (S > 4 && left == 3) wait_loads<(S > 4 ? 3 * L : 0)>();
            else if (S > 3 && left == 2) wait_loads<(S > 3 ? 2 * L : 0)>();
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
                for (int m = 0; m < MT; ++m) {
                    if constexpr (HELD) lds_read(xf[h][m], held + t * 128, h * 64);
                    else lds_read(xf[h][m], at, (NT + m) * 2048);
                }
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
            if constexpr (EXACT) {
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int n = 0; n < NT; ++n) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) sums[m][n][j] += (double)acc[m][n][j];
                        acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
            }
        }
        if constexpr (EXACT) {
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[m][n][j] = (float)sums[m][n][j];
        }
    }

    // The waves' sums side by side in LDS, in the pieces' place; total() then adds them.
    static __device__ __forceinline__ void store(uint16_t* smem, const f32x4 (&acc)[MT][NT]) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
        float* sums = reinterpret_cast<float*>(smem);
        __syncthreads();  // nothing is under way any more
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n)
                *reinterpret_cast<f32x4*>(sums + (wave * BM + m * 16 + c) * LR + n * 16 + 4 * g) = acc[m][n];
        __syncthreads();
    }
    // x row m, weight rows n .. n + 3
    static __device__ __forceinline__ f32x4 total(const uint16_t* smem, int m, int n) {
        const float* sums = reinterpret_cast<const float*>(smem);
        f32x4 s = *reinterpret_cast<const f32x4*>(sums + m * LR + n);
#pragma unroll
        for (int k = 1; k < WK; ++k) s += *reinterpret_cast<const f32x4*>(sums + (k * BM + m) * LR + n);
        return s;
    }
};

}  // namespace skyrl
