// A product of a few rows that are formed ahead of it in the same launch (normed_product.hip, latent.hip): four waves of a workgroup
// form them in LDS while the other four have their first weights on the way (a wave that did both would wait for its weights with
// its rows).
#pragma once
#include "rows.h"

namespace skyrl {

constexpr int kFormers = 256;  // threads that form the rows; as many stream

// LDS by hand, since the barriers are.
__device__ __forceinline__ uint32_t lds_at(const void* p) { return (uint32_t)(uintptr_t)(lds_void*)p; }
__device__ __forceinline__ void lds_put(uint32_t at, float v) { asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(v) : "memory"); }
__device__ __forceinline__ void lds_put32(uint32_t at, uint32_t v) { asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(v) : "memory"); }
__device__ __forceinline__ void lds_put16(uint32_t at, uint32_t v) { asm volatile("ds_write_b16 %0, %1" ::"v"(at), "v"(v) : "memory"); }
__device__ __forceinline__ float lds_get(uint32_t at) {
    float v;
    asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(at) : "memory");
    return v;
}
__device__ __forceinline__ f32x4 lds_get4(uint32_t at) {
    f32x4 v;
    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(at) : "memory");
    return v;
}
__device__ __forceinline__ void lds_put2(uint32_t at, uint2 v) {
    const uint64_t w = (uint64_t)v.y << 32 | v.x;
    asm volatile("ds_write_b64 %0, %1" ::"v"(at), "v"(w) : "memory");
}
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// Sum over the block, in every thread; red: four floats of LDS, free again after the next barrier.
__device__ __forceinline__ float total(float v, uint32_t red) {
    v = wave_total(v);
    if ((threadIdx.x & 63) == 0) lds_put(red + (threadIdx.x % kFormers >> 6) * 4, v);
    lds_barrier();
    const f32x4 s = lds_get4(red);
    return ((0.f + s[0]) + s[1]) + s[2] + s[3];
}

// Pre: RowOf<LONG> with load(pre), form(pre, x, pitch, red): the rows into LDS at x, `pitch` bytes apart, red: kRed floats of
// scratch; barriers(pre): lds_barrier calls of form; leave(pre): what else becomes of the rows, called in the first workgroup.
// n rows, at most ROWS, of up to LONG: one each in the first places, the last one in the others of 16; four shares of the depth a
// workgroup, of its gridDim.y-th.
template <int MODE, int NT, int S, int LONG, int ROWS, int kRed, class Pre>
__device__ __forceinline__ void formed_product(const RowsProduct& p, const Pre& pre, uint16_t* smem, int batch, bool first) {
    constexpr int WK = kFormers / kWave, kPitch = LONG * 2 + (ROWS > 1 ? 16 : 0);  // bytes
    using St = Stream<NT, 1, WK, S, true, true, MODE == kParts>;
    using Row = typename Pre::template RowOf<LONG>;
    constexpr int OC = out_cols<MODE, NT>();
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * OC;
    const uint32_t x = lds_at(smem + St::kLds);
    if (wave >= WK) {
        __builtin_amdgcn_s_setprio(2);
        Row row;
        row.load(pre);
        row.form(pre, x, kPitch, x + ROWS * kPitch);
        const int end = tid - kFormers, left = (64 - p.K % 64) % 64 / 4;  // the last piece's end
        if (left && end < ROWS * left) lds_put2(x + end / left * kPitch + p.K * 2 + end % left * 8, make_uint2(0u, 0u));
        lds_barrier();
        __builtin_amdgcn_s_setprio(0);
        if (first) row.leave(pre);
        __syncthreads();  // those of St::store
        __syncthreads();
    } else {
        const int steps = (p.K + 63) / 64, shares = gridDim.y * WK, share = blockIdx.y * WK + wave;
        const int s0 = (int)((int64_t)steps * share / shares), nk = (int)((int64_t)steps * (share + 1) / shares) - s0;
        f32x4 acc[1][NT];
        St::run(
            smem, p.K, s0, nk,
            [&](int r) {
                const int at = MODE == kGated && r >= OC ? p.N + min(n0 + r - OC, p.N - 1) : min(n0 + r, p.N - 1);
                return p.w + batch * p.w_batch + at * p.ldw;
            },
            [&](int) { return (const uint16_t*)nullptr; }, acc,
            [&]() {
                for (int i = Row::barriers(pre); i >= 0; --i) lds_barrier();
                return x + (ROWS > 1 ? min(tid & 15, p.n - 1) * kPitch : 0);
            });
        St::store(smem, acc);
    }
    put_rows<MODE, St, 2 * WK>(smem, p, n0, 0, batch);
}
template <int NT, int S, int LONG, int ROWS, int kRed>
constexpr int formed_lds() {  // elements
    return Stream<NT, 1, kFormers / kWave, S, true>::kLds + ROWS * (LONG + (ROWS > 1 ? 8 : 0)) + 2 * kRed;
}

}  // namespace skyrl
