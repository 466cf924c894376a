// Gated delta rule: a recurrent layer with a [dim x vdim] matrix state per head
// (include/skyrl_layers.h has the equations and the tensor layouts).
//
// Token form (delta_scan): one workgroup per (sequence, head). The state is read once into registers,
// carried over the sequence's tokens and written once, so a decode step costs one read and one write
// of the state. Convolution, unit norms, gates, recurrence, output norm and output gate are one pass.
// Both products with the state are taken before the update, S^T k and S^T q, in one sweep:
// o = (g S + k u^T)^T q = g S^T q + (k . q) u.
//
// Prompt form (conv, chunk, chain, out): chunks of 64 tokens. Unrolling the recurrence over a chunk
// with G_i the summed log decays up to token i gives
//   u_i = beta_i (v_i - e^{G_i} S0^T k_i - sum_{j<i} e^{G_i - G_j} (k_i . k_j) u_j),
// i.e. (I + A) U = diag(beta) V - diag(beta e^G) K S0 with A_ij = beta_i e^{G_i - G_j} k_i . k_j below
// the diagonal. delta_chunk solves it for both right-hand sides, all chunks at once: U0 = (I + A)^-1
// diag(beta) V and W = (I + A)^-1 diag(beta e^G) K, and forms P_ij = e^{G_i - G_j} q_i . k_j (j <= i).
// delta_chain then walks a sequence's chunks with a 16-column slice of S per workgroup:
//   U = U0 - W S,   O = diag(e^G) Q S + P U,   S <- e^{G_n} S + K^T diag(e^{G_n - G}) U.
// Everything is f32, the products on the f32 matrix instructions (v_mfma_f32_16x16x4_f32): a lane's
// four consecutive k values of a 16-step feed four instructions, the same permutation of k on both sides.
#include <type_traits>

#include "conv.h"

namespace skyrl {
namespace {

constexpr int kNT = 256;
constexpr int kMaxTaps = 64;
constexpr int kC = 64;       // tokens per chunk
constexpr int kWin = 4;      // taps of a convolution that are loaded ahead

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct Dims {
    int H, K, D, V, taps;
    float eps;
    __host__ __device__ int vpad() const { return (V + 3) / 4 * 4; }
    __host__ __device__ int d16() const { return (D + 15) / 16 * 16; }
    __host__ __device__ int v16() const { return (V + 15) / 16 * 16; }
    __host__ __device__ int channels() const { return 2 * K * D + H * V; }
};

template <typename T>
__device__ __forceinline__ float conv_silu(const T* __restrict__ proj, int64_t stride, const T* __restrict__ w,
                                           const T* __restrict__ ring, int channels, int taps, int ch, int t, int t0,
                                           int pos, int r) {
    return siluf_(short_conv(proj, stride, w, ring, channels, taps, ch, t, t0, pos, r));
}

// ---- token form -------------------------------------------------------------------------------
// One workgroup per (sequence, head), the state in registers. A decode step is bound by the state, read and written once. The
// first token is a copy of the loop's body of its own (AHEAD: at most kWin taps, a channel per thread), so that nothing but
// the products waits for the state: 32 heads of 128 x 128, one token each: 64 rows 62.6 us (4.3 TB/s) against 79.8, 1 row 9.0
// against 11.7. The state goes past the caches both ways (non-temporal): left there it is put out before the next step by the
// weights, and what is written is in their way (64 rows 59.4 -> 57.3 us; with the latent pages, which go the same way, four small
// products of the step 27.5 -> 18.4 us).
// A value as it is stored, in a register of its own: what is loaded ahead is converted, and waited for, where it is used.
template <typename T>
using Raw = std::conditional_t<sizeof(T) == 2, uint32_t, T>;
template <typename T>
__device__ __forceinline__ float of_raw(Raw<T> x) {
    if constexpr (sizeof(T) == 2) return __uint_as_float(x << 16);
    else return x;
}

// NT threads, RPT state rows per thread: thread (cg, rg) holds columns 4 cg .. 4 cg + 3 of rows rg, rg + RG, ...
template <typename T, int NT, int RPT, bool AHEAD>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void delta_scan_kernel(Dims d, const T* __restrict__ proj, int64_t stride,
                                                         const T* __restrict__ conv_w, const float* __restrict__ a_log,
                                                         const float* __restrict__ dt_bias,
                                                         const T* __restrict__ norm_w, const int32_t* __restrict__ cu,
                                                         const int32_t* __restrict__ rows,
                                                         const int64_t* __restrict__ positions,
                                                         float* __restrict__ state, T* __restrict__ conv_state,
                                                         int save_conv, T* __restrict__ out, int64_t out_stride) {
    extern __shared__ float smem[];
    const int h = blockIdx.x, s = blockIdx.y;
    const int row = rows[s];
    if (row < 0) return;
    const int t0 = cu[s], t1 = cu[s + 1];
    if (t0 >= t1) return;
    const int D = d.D, V = d.V, VP = d.vpad(), NC = VP / 4, RG = NT / NC;
    const int ch_all = d.channels();
    const int kh = h / (d.H / d.K);
    float* s_q = smem;             // D
    float* s_k = s_q + D;          // D
    float* s_v = s_k + D;          // VP
    float* s_o = s_v + VP;         // VP
    float* s_red = s_o + VP;       // RG * VP * 2
    float* s_n = s_red + RG * VP * 2;  // 4 scalars
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int cg = tid % NC, rg = tid / NC;
    const bool act = rg < RG;
    const bool fold = NC <= kWave && (NC & (NC - 1)) == 0;  // a wave holds whole row groups
    const int nrec = fold ? NT / kWave : RG;
    const int64_t pos0 = positions[t0];
    T* ring = conv_state + (int64_t)row * d.taps * ch_all;
    float* st_ = state + ((int64_t)row * d.H + h) * D * VP;
    const int qoff = kh * D, koff = (d.K + kh) * D, voff = 2 * d.K * D + h * V;
    auto channel = [&](int e) { return e < D ? qoff + e : e < 2 * D ? koff + e - D : voff + min(e - 2 * D, V - 1); };
    // What the first token needs ahead of the state is loaded ahead of it, since loads return in order: its convolutions,
    // norms and gates then run while the state is on its way. Addresses are clamped and not branched around.
    Raw<T> cx[kWin], cf[kWin];
    if constexpr (AHEAD) {
        const int ch = channel(min(tid, 2 * D + VP - 1)), slot = (int)(pos0 % d.taps);
#pragma unroll
        for (int back = 0; back < kWin; ++back) {
            const int b = min(back, d.taps - 1), at = slot - b < 0 ? slot - b + d.taps : slot - b;
            const T* src = b == 0 ? proj + (int64_t)t0 * stride : ring + (int64_t)at * ch_all;
            cx[back] = Raw<T>(src[ch]);
            cf[back] = Raw<T>(conv_w[(int64_t)ch * d.taps + d.taps - 1 - b]);
        }
    }
    const T* p0 = proj + (int64_t)t0 * stride;
    const int goff = ch_all + h * V, boff = ch_all + d.H * V + h, aoff = boff + d.H;
    const Raw<T> b0 = p0[boff], a0 = p0[aoff], gate0 = p0[goff + min(tid, V - 1)], nw0 = norm_w[min(tid, V - 1)];
    const float rate = a_log[h], dt = dt_bias[h];
    float S[RPT][4];
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const float4 v = ld4_once(st_ + (int64_t)min(rg + i * RG, D - 1) * VP + 4 * cg);
        S[i][0] = v.x; S[i][1] = v.y; S[i][2] = v.z; S[i][3] = v.w;
    }
    const float neg_rate = -expf(rate);
    const float qscale = 1.f / sqrtf((float)D);
    auto step = [&](auto first_, int t) {
        constexpr bool first = first_;
        const int pos = (int)pos0 + (t - t0);
        const T* p = proj + (int64_t)t * stride;
        const int slot = pos % d.taps;
        const float b_raw = first ? of_raw<T>(b0) : ld(p + boff), a_raw = first ? of_raw<T>(a0) : ld(p + aoff);
        const float gate = first ? of_raw<T>(gate0) : ld(p + goff + min(tid, V - 1)), nw = of_raw<T>(nw0);
        if (AHEAD && first) {
            float y = 0.f;
#pragma unroll
            for (int back = 0; back < kWin; ++back) y += back < d.taps && back <= pos ? of_raw<T>(cx[back]) * of_raw<T>(cf[back]) : 0.f;
            if (tid < 2 * D + VP) smem[tid] = tid < 2 * D + V ? siluf_(y) : 0.f;
        } else {
            for (int e = tid; e < 2 * D + VP; e += NT)  // s_q | s_k | s_v are contiguous
                smem[e] = e < 2 * D + V ? conv_silu(proj, stride, conv_w, ring, ch_all, d.taps, channel(e), t, t0, pos, slot) : 0.f;
        }
        __syncthreads();
        if (wave < 3) {  // |q|^2, |k|^2, q . k of the raw vectors
            const float* a = wave == 1 ? s_k : s_q;
            const float* b = wave == 0 ? s_q : s_k;
            float x = 0.f;
            for (int i = lane; i < D; i += kWave) x += a[i] * b[i];
            x = wave_total(x);
            if (lane == 0) s_n[wave] = x;
        }
        __syncthreads();
        const float rq = qscale / sqrtf(s_n[0] + 1e-6f), rk = 1.f / sqrtf(s_n[1] + 1e-6f);
        const float kq = s_n[2] * rq * rk;
        const float beta = sigmoidf_(b_raw);
        const float g = expf(neg_rate * softplusf_(a_raw + dt));
        if (first && pos0 <= 0)
#pragma unroll
            for (int i = 0; i < RPT; ++i) S[i][0] = S[i][1] = S[i][2] = S[i][3] = 0.f;
        float a[4] = {0.f, 0.f, 0.f, 0.f}, b[4] = {0.f, 0.f, 0.f, 0.f};
        if (act) {
#pragma unroll
            for (int i = 0; i < RPT; ++i) {
                const int r = rg + i * RG;
                if (r < D) {
                    const float kr = s_k[r] * rk, qr = s_q[r] * rq;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        a[j] += S[i][j] * kr;
                        b[j] += S[i][j] * qr;
                    }
                }
            }
            if (fold)  // the wave's own row groups first
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    a[j] = lanes_add_from(a[j], NC);
                    b[j] = lanes_add_from(b[j], NC);
                }
            if (!fold || lane < NC) {
                const int rec = fold ? wave : rg;
                st4(s_red + (rec * 2) * VP + 4 * cg, make_float4(a[0], a[1], a[2], a[3]));
                st4(s_red + (rec * 2 + 1) * VP + 4 * cg, make_float4(b[0], b[1], b[2], b[3]));
            }
        }
        __syncthreads();
        if (act) {
            float4 A = make_float4(0.f, 0.f, 0.f, 0.f), B = A;
            for (int r = 0; r < nrec; ++r) {
                const float4 x = ld4(s_red + (r * 2) * VP + 4 * cg), y = ld4(s_red + (r * 2 + 1) * VP + 4 * cg);
                A.x += x.x; A.y += x.y; A.z += x.z; A.w += x.w;
                B.x += y.x; B.y += y.y; B.z += y.z; B.w += y.w;
            }
            const float4 v = ld4(s_v + 4 * cg);
            const float u[4] = {beta * (v.x - g * A.x), beta * (v.y - g * A.y), beta * (v.z - g * A.z),
                                beta * (v.w - g * A.w)};
#pragma unroll
            for (int i = 0; i < RPT; ++i) {
                const int r = rg + i * RG;
                if (r < D) {
                    const float kr = s_k[r] * rk;
#pragma unroll
                    for (int j = 0; j < 4; ++j) S[i][j] = g * S[i][j] + kr * u[j];
                }
            }
            if (rg == 0)
                st4(s_o + 4 * cg,
                    make_float4(g * B.x + kq * u[0], g * B.y + kq * u[1], g * B.z + kq * u[2], g * B.w + kq * u[3]));
        }
        __syncthreads();
        if (wave * kWave < V) {
            float x = 0.f;
            for (int i = lane; i < V; i += kWave) x += s_o[i] * s_o[i];
            x = wave_total(x);
            const float r = 1.f / sqrtf(x / (float)V + d.eps);
            T* dst = out + (int64_t)t * out_stride + h * V;
            if (tid < V) st(dst + tid, s_o[tid] * r * nw * siluf_(gate));
            for (int i = tid + NT; i < V; i += NT) st(dst + i, s_o[i] * r * ld(norm_w + i) * siluf_(ld(p + goff + i)));
        }
        // s_q/s_k/s_v are rewritten only after every thread passed the barrier above; s_o not before the next two
    };
    step(std::true_type{}, t0);
    for (int t = t0 + 1; t < t1; ++t) step(std::false_type{}, t);
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const int r = rg + i * RG;
        if (act && r < D) st4_once(st_ + (int64_t)r * VP + 4 * cg, make_float4(S[i][0], S[i][1], S[i][2], S[i][3]));
    }
    if (save_conv) {  // one token: its slot is not among those the convolutions read
        const T* p = proj + (int64_t)t0 * stride;
        T* dst = ring + (int64_t)(pos0 % d.taps) * ch_all;
        for (int e = tid; e < V; e += NT) dst[voff + e] = p[voff + e];
        if (h % (d.H / d.K) == 0)
            for (int e = tid; e < D; e += NT) {
                dst[qoff + e] = p[qoff + e];
                dst[koff + e] = p[koff + e];
            }
    }
}

// ---- prompt form ------------------------------------------------------------------------------
struct SeqRef {
    const int32_t* chunk;  // [nchunks, 4]: first token, tokens, sequence, 0
    const int32_t* cu;
    const int32_t* rows;
    const int64_t* positions;
};

// Operand order: a 16 x 16 tile of a matrix that is read as an operand of the matrix instructions is 256 consecutive numbers,
// lane (c, g)'s four first: row c, columns 4 g .. 4 g + 3. A wave's load is then 1 KB in a piece (64 bytes a cycle); the
// same tile in rows cost four times as long, a cache line per lane. Tokens past a chunk's end are zero.
//   q, k   qk [chunk][key head][q | k][token tile][dim tile]      k transposed   kt [chunk][key head][dim tile][token tile]
//   v transposed  vt [chunk][head][vdim tile][token tile]         W  [chunk][head][token tile][dim tile]
//   P      [chunk][head][token tile][token tile]                  U  as its product leaves it: row 4 g + i, column c, tiles as vt
constexpr int kTile = 256;

// Convolution, silu, unit norms and gates. grid (nchunks, K + ceil(H V / 256)): the first K groups are the
// key heads (q and k), the others 256 value channels each; gates with group 0. A channel's 64 inputs and the TAPS - 1 before
// are all in flight at once (TAPS 0: any number of taps, loaded where they are used; ONCE: a channel per thread in every group,
// otherwise a key head's threads take sixteen inputs of each of their channels at a time). Bound: 470 MB for 8192 tokens of 8192
// channels (100 us at a large copy's rate); 120 us, 190 with both forms in one kernel, whose registers leave half the waves.
template <typename T, int TAPS, bool ONCE>
__global__ __launch_bounds__(kNT) void delta_conv_kernel(Dims d, SeqRef sq, const T* __restrict__ proj, int64_t stride,
                                                         const T* __restrict__ conv_w, const float* __restrict__ a_log,
                                                         const float* __restrict__ dt_bias,
                                                         const T* __restrict__ conv_state, float* __restrict__ qk,
                                                         float* __restrict__ kt, float* __restrict__ vt, float* __restrict__ lg,
                                                         float* __restrict__ beta) {
    extern __shared__ __attribute__((aligned(16))) float smem[];  // [16][2 D + 4] of the key heads
    __shared__ float s_r[32];                                     // their scales
    const int32_t* ck = sq.chunk + 4 * blockIdx.x;
    const int t0 = ck[0], n = ck[1], seq = ck[2];
    const int sfirst = sq.cu[seq];
    const int pos0 = (int)sq.positions[sfirst] + (t0 - sfirst);
    const int ch_all = d.channels(), D = d.D, V = d.V, nd = d.d16() / 16, nv = d.v16() / 16, LK = 2 * D + 4;
    const T* ring = conv_state + (int64_t)sq.rows[seq] * d.taps * ch_all;
    const int tid = threadIdx.x;
    const bool keys = (int)blockIdx.y < d.K;
    const int kh = blockIdx.y;
    if (blockIdx.y == 0) {
        for (int e = tid; e < n * d.H; e += kNT) {
            const int i = e / d.H, h = e - i * d.H;
            const T* p = proj + (int64_t)(t0 + i) * stride + ch_all + d.H * d.V;
            beta[(int64_t)(t0 + i) * d.H + h] = sigmoidf_(ld(p + h));
            lg[(int64_t)(t0 + i) * d.H + h] = -expf(a_log[h]) * softplusf_(ld(p + d.H + h) + dt_bias[h]);
        }
    }
    // input of channel ch at local token i (negative: before the chunk, from the portion or the stored inputs)
    auto input = [&](int ch, int i) -> float {
        if (pos0 + i < 0) return 0.f;
        if (t0 + i >= sfirst) return ld(proj + (int64_t)(t0 + i) * stride + ch);
        return ld(ring + (int64_t)((pos0 + i) % d.taps) * ch_all + ch);
    };
    const int nch = keys ? 2 * D : min(kNT, d.H * V - ((int)blockIdx.y - d.K) * kNT);
    constexpr int kSub = 16, kBack = TAPS > 0 ? TAPS - 1 : 0;
    const bool once = ONCE || nch <= kNT;  // one channel per thread: its inputs stay in registers
    float x[kBack + kC], w[TAPS > 0 ? TAPS : 1];
    auto channel = [&](int e) {
        return !keys ? 2 * d.K * D + ((int)blockIdx.y - d.K) * kNT + e : e < D ? kh * D + e : (d.K + kh) * D + (e - D);
    };
    auto fetch = [&](int ch, int from, int to) {  // inputs [from, to) of the channel's, in the unrolled loops
#pragma unroll
        for (int j = 0; j < TAPS; ++j)
            w[j] = j >= TAPS - d.taps ? ld(conv_w + (int64_t)ch * d.taps + j - (TAPS - d.taps)) : 0.f;
#pragma unroll
        for (int i = 0; i < kC; ++i)
            if (kBack + i >= from && kBack + i < to) x[kBack + i] = ld(proj + (int64_t)(t0 + min(i, n - 1)) * stride + ch);
#pragma unroll
        for (int j = 0; j < kBack; ++j)
            if (j >= from) x[j] = j > kBack - d.taps ? input(ch, j - kBack) : 0.f;
    };
    if constexpr (TAPS > 0)
        if (once && tid < nch) fetch(channel(tid), 0, kBack + kC);
#pragma unroll
    for (int sub = 0; sub < kC / kSub; ++sub) {
        const int i0 = sub * kSub;
        for (int e = tid; e < nch; e += kNT) {
            const int ch = channel(e);
            if constexpr (TAPS > 0)
                if (!once) fetch(ch, i0, i0 + kBack + kSub);
            float y[kSub];
#pragma unroll
            for (int i = 0; i < kSub; ++i) {
                y[i] = 0.f;
                if constexpr (TAPS > 0) {
#pragma unroll
                    for (int j = 0; j < TAPS; ++j) y[i] += x[i0 + i + j] * w[j];
                } else if (i0 + i < n) {
                    for (int j = 0; j < d.taps; ++j)
                        y[i] += input(ch, i0 + i - (d.taps - 1) + j) * ld(conv_w + (int64_t)ch * d.taps + j);
                }
                y[i] = i0 + i < n ? siluf_(y[i]) : 0.f;
                if (keys) smem[i * LK + e] = y[i];
            }
            if (keys) continue;
            const int col = ((int)blockIdx.y - d.K) * kNT + e, h = col / V, c = col - h * V;
            float* dst = vt + ((((int64_t)blockIdx.x * d.H + h) * nv + c / 16) * 4 + sub) * kTile + c % 16 * 4;
#pragma unroll
            for (int g = 0; g < 4; ++g) st4(dst + g * 64, make_float4(y[4 * g], y[4 * g + 1], y[4 * g + 2], y[4 * g + 3]));
        }
        if (!keys) continue;
        __syncthreads();
        {  // eight threads per (token, q or k)
            const int i = tid >> 4, which = (tid >> 3) & 1, part = tid & 7;
            const float* src = smem + i * LK + which * D;
            float ss = 0.f;
            for (int k = part; k < D; k += 8) ss += src[k] * src[k];
#pragma unroll
            for (int o = 1; o < 8; o <<= 1) ss += __shfl_xor(ss, o, kWave);
            float r = 1.f / sqrtf(ss + 1e-6f);
            if (which == 0) r *= 1.f / sqrtf((float)D);
            if (part == 0) s_r[2 * i + which] = r;
        }
        __syncthreads();
        const int64_t head = (int64_t)blockIdx.x * d.K + kh;
        for (int e = tid; e < nd * 3 * kWave; e += kNT) {
            const int l = e & 63, tile = (e >> 6) % nd, form = (e >> 6) / nd, c = l & 15, g = l >> 4;
            float y[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = form < 2 ? c : 4 * g + j, k = 16 * tile + (form < 2 ? 4 * g + j : c);
                y[j] = k < D ? smem[i * LK + (form > 0 ? D : 0) + k] * s_r[2 * i + (form > 0)] : 0.f;
            }
            float* dst = form < 2 ? qk + (((head * 2 + form) * 4 + sub) * nd + tile) * kTile
                                  : kt + ((head * nd + tile) * 4 + sub) * kTile;
            st4(dst + l * 4, make_float4(y[0], y[1], y[2], y[3]));
        }
        __syncthreads();
    }
}

__device__ __forceinline__ f32x4 mma4(const float4& a, const float4& b, f32x4 acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc, 0, 0, 0);
}
__device__ __forceinline__ float4 as_float4(const f32x4& v) { return make_float4(v[0], v[1], v[2], v[3]); }

// One workgroup per (chunk, head). The 64 x 64 system is solved in 16 x 16 blocks: each wave inverts one
// diagonal block by substitution, the blocks below follow diagonal by diagonal from
// T_rb = -T_rr sum_k A_rk T_kb, and T then multiplies both right-hand sides. A 16 x 16 result's registers
// (rows 4 g + i, column c) are the next product's right operand as they are, and a transposed product's are its operand order.
// Bound: 600 MB of HBM and the f32 products, about as long (8192 tokens of 32 heads of 128 x 128: 75 us each); the next slab and
// the next right-hand side are loaded while one is worked on: 158 us, where each was loaded when it was due 176.
__global__ __launch_bounds__(kNT) __attribute__((amdgpu_waves_per_eu(4))) void delta_chunk_kernel(Dims d, const int32_t* __restrict__ chunk,
                                                          const float* __restrict__ qk, const float* __restrict__ kt,
                                                          const float* __restrict__ vt, const float* __restrict__ lg, const float* __restrict__ beta,
                                                          float* __restrict__ W, float* __restrict__ U,
                                                          float* __restrict__ P, float* __restrict__ G) {
    constexpr int LD = kC + 4;
    __shared__ __attribute__((aligned(16))) float s_k[kC * LD];  // a 64-wide slab of K; then A
    __shared__ __attribute__((aligned(16))) float s_q[kC * LD];  // a slab of Q; then T = (I + A)^-1
    __shared__ __attribute__((aligned(16))) float s_g[kC], s_b[kC], s_w[kC];
    const int h = blockIdx.x % d.H, ci = blockIdx.x / d.H;
    const int32_t* ck = chunk + 4 * ci;
    const int t0 = ck[0], n = ck[1];
    const int kh = h / (d.H / d.K), D16 = d.d16(), V16 = d.v16();
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int64_t ch = (int64_t)ci * d.H + h;
    if (wave == 0) {  // inclusive sums of the log decays; tokens past the chunk's end have beta 0 and decay 1
        float x = lane < n ? lg[(int64_t)(t0 + lane) * d.H + h] : 0.f;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const float y = __shfl_up(x, o, kWave);
            if (lane >= o) x += y;
        }
        const float be = lane < n ? beta[(int64_t)(t0 + lane) * d.H + h] : 0.f;
        s_g[lane] = x;
        s_b[lane] = be;
        s_w[lane] = be * expf(x);
        const float last = __shfl(x, kWave - 1, kWave);
        G[ch * 2 * kC + lane] = expf(x);
        G[ch * 2 * kC + kC + lane] = expf(last - x);
    }
    // K K^T and Q K^T on the ten blocks at and below the diagonal: 20 block products, five per wave
    f32x4 acc[5];
    int br[5], bc[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int item = (wave + 4 * k) % 10;  // (0,0) (1,0) (1,1) (2,0) ...
        br[k] = item >= 6 ? 3 : item >= 3 ? 2 : item >= 1 ? 1 : 0;
        bc[k] = item - br[k] * (br[k] + 1) / 2;
    }
    const int nd = D16 / 16;
    const float* qp = qk + ((int64_t)ci * d.K + kh) * 2 * 4 * nd * kTile;
    float4 slab[2][4];  // of q and k: four dim tiles of every token tile, the next ones while these are worked on
    auto load_slab = [&](int d0) {
        const int w = min(4, nd - d0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // token tile i; tiles past the last: the last again
            const int x = min(tid, w * kWave - 1);
            const float* src = qp + (i * nd + d0) * kTile + x * 4;
            slab[0][i] = ld4(src);
            slab[1][i] = ld4(src + 4 * nd * kTile);
        }
    };
    static_assert(kNT == 4 * kWave, "a token tile's four dim tiles by one pass of the threads");
    load_slab(0);
    for (int d0 = 0; d0 < nd; d0 += 4) {
        const int w = min(4, nd - d0);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            st4(&s_q[(i * kNT + tid) * 4], slab[0][i]);
            st4(&s_k[(i * kNT + tid) * 4], slab[1][i]);
        }
        if (d0 + 4 < nd) load_slab(d0 + 4);
        __syncthreads();
        for (int s = 0; s < w; ++s) {
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                const bool own = wave + 4 * k < 10;  // K K^T; otherwise (Q K^T)^T
                const float* right = own ? s_k : s_q;
                acc[k] = mma4(ld4(&s_k[((own ? br[k] : bc[k]) * 4 + s) * kTile + lane * 4]),
                              ld4(&right[((own ? bc[k] : br[k]) * 4 + s) * kTile + lane * 4]), acc[k]);
            }
        }
    }
    __syncthreads();
    // the right-hand sides, a tile ahead of their use
    const int nv = V16 / 16;
    float4 ahead[4];
    auto load_x = [&](int tile) {  // past the last: the last again
        tile = min(tile, nd + nv - 1);
        const bool isw = tile < nd;
        const int vtile = tile - nd;
        const float* src = (isw ? kt + (((int64_t)ci * d.K + kh) * nd + tile) * 4 * kTile : vt + (ch * nv + vtile) * 4 * kTile) + lane * 4;
#pragma unroll
        for (int s = 0; s < 4; ++s) ahead[s] = ld4(src + s * kTile);
    };
    load_x(wave);
    float *s_a = s_k, *s_t = s_q;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        if (wave + 4 * k < 10) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 16 * br[k] + 4 * g + i, cc = 16 * bc[k] + c;
                s_a[r * LD + cc] = cc < r ? s_b[r] * expf(s_g[r] - s_g[cc]) * acc[k][i] : 0.f;
            }
        } else {
            const int r = 16 * br[k] + c;
            float y[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int cc = 16 * bc[k] + 4 * g + i;
                y[i] = cc <= r ? expf(s_g[r] - s_g[cc]) * acc[k][i] : 0.f;
            }
            st4(P + ((ch * 4 + br[k]) * 4 + bc[k]) * kTile + lane * 4, make_float4(y[0], y[1], y[2], y[3]));
        }
    }
    __syncthreads();
    {  // diagonal block `wave`: column c of its inverse
        float x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float r = i == c ? 1.f : 0.f;
#pragma unroll
            for (int j4 = 0; j4 < (i + 3) / 4; ++j4) {
                const float4 a = ld4(&s_a[(16 * wave + i) * LD + 16 * wave + 4 * j4]);
                r -= a.x * x[4 * j4];
                if (4 * j4 + 1 < i) r -= a.y * x[4 * j4 + 1];
                if (4 * j4 + 2 < i) r -= a.z * x[4 * j4 + 2];
                if (4 * j4 + 3 < i) r -= a.w * x[4 * j4 + 3];
            }
            x[i] = r;
        }
        if (g == 0) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s_t[(16 * wave + i) * LD + 16 * wave + c] = x[i];
        }
    }
#pragma unroll
    for (int lev = 1; lev < 4; ++lev) {
        __syncthreads();
        if (wave + lev < 4) {
            const int b = wave, r = wave + lev;
            f32x4 m = {0.f, 0.f, 0.f, 0.f}, tt = m;
            for (int k = b; k < r; ++k) {
                const float* tk = &s_t[(16 * k + 4 * g) * LD + 16 * b + c];
                m = mma4(ld4(&s_a[(16 * r + c) * LD + 16 * k + 4 * g]),
                         make_float4(tk[0], tk[LD], tk[2 * LD], tk[3 * LD]), m);
            }
            tt = mma4(ld4(&s_t[(16 * r + c) * LD + 16 * r + 4 * g]), as_float4(m), tt);
#pragma unroll
            for (int i = 0; i < 4; ++i) s_t[(16 * r + 4 * g + i) * LD + 16 * b + c] = -tt[i];
        }
    }
    __syncthreads();
    // T times [diag(beta e^G) K | diag(beta) V], 16 columns at a time; the first transposed
    for (int tile = wave; tile < nd + nv; tile += 4) {
        const bool isw = tile < nd;
        const int vtile = tile - nd;
        const bool on = isw || 16 * vtile + c < d.V;  // columns past vdim hold nothing
        float4 x[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) x[s] = on ? ahead[s] : make_float4(0.f, 0.f, 0.f, 0.f);
        load_x(tile + 4);
        f32x4 o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float4 sc = ld4((isw ? s_w : s_b) + 16 * s + 4 * g);
            const float4 bv = make_float4(x[s].x * sc.x, x[s].y * sc.y, x[s].z * sc.z, x[s].w * sc.w);
#pragma unroll
            for (int r = s; r < 4; ++r) {
                const float4 t = ld4(&s_t[(16 * r + c) * LD + 16 * s + 4 * g]);
                o[r] = isw ? mma4(bv, t, o[r]) : mma4(t, bv, o[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
            st4((isw ? W + ((ch * 4 + r) * nd + tile) * kTile : U + ((ch * nv + vtile) * 4 + r) * kTile) + lane * 4, as_float4(o[r]));
    }
}

// One workgroup per (sequence, head, 16 columns of S). NS: 16-wide steps of dim (EXACT: dim = 16 NS); DT
// 16-row tiles of S per wave; SETS: register sets of operands. With two (dim up to 128) a chunk's operands are under way for
// the whole chunk before. Only U = U0 - W S and the update of S are a chain, which four waves walk; four others, one beside each
// on its SIMD, form the outputs, so that the matrix unit has work while a chain's wave waits for LDS or for the others.
// Operands come from HBM and each is read by all slices of S: a slice's threads touch their share of the lines two chunks ahead,
// else all of them ask for a line that is still on its way (418 us against 370 below).
// Bound: the f32 matrix rate (178 us for 8192 tokens of 32 heads of 128 x 128). Measured there: 712 us with operands in rows,
// loaded half a chunk ahead, and products in the order of the equations; 418 us with one set of waves for both, products that end
// in the output where the others' results go through LDS; 328 us this way, 298 with operands that are in L2.
template <int NS, bool EXACT, int SETS>
__global__ __launch_bounds__(2 * kNT) __attribute__((amdgpu_waves_per_eu(2))) void delta_chain_kernel(
    Dims d, SeqRef sq, const int32_t* __restrict__ seq_chunks, int seq0, int nseq, const float* __restrict__ qk,
    const float* __restrict__ kt, const float* __restrict__ W, const float* __restrict__ U, const float* __restrict__ P,
    const float* __restrict__ G, float* __restrict__ state, float* __restrict__ o) {
    constexpr int LS = NS * 16 + 4, LU = kC + 4, DT = (NS + 3) / 4;
    __shared__ __attribute__((aligned(16))) float s_s[2][16 * LS];   // S^T slice, by turns
    __shared__ __attribute__((aligned(16))) float s_u[2][16 * LU];   // U^T, by turns
    __shared__ __attribute__((aligned(16))) float s_d[16 * LU];      // decayed
    const int V16 = d.v16(), D16 = EXACT ? NS * 16 : d.d16(), VP = d.vpad(), nt = V16 / 16;
    // the slices of one (sequence, head) read the same W, Q, K and P, neighbouring heads the same Q and K: on one XCD
    const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8, grp = xcd * ((nseq * d.H + 7) / 8) + slot / nt;
    if (grp >= nseq * d.H) return;
    const int vt = slot % nt, h = grp % d.H, si = grp / d.H;
    const int seq = seq0 + si, row = sq.rows[seq];
    if (row < 0) return;
    const int64_t pos0 = sq.positions[sq.cu[seq]];
    const int kh = h / (d.H / d.K);
    const int tid = threadIdx.x % kNT, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool outputs = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) != 0;
    const int c = lane & 15, g = lane >> 4;
    const int ns = EXACT ? NS : D16 / 16;
    const int c0 = seq_chunks[si], c1 = seq_chunks[si + 1];
    if (c0 >= c1) return;
    const int vcol = 16 * vt + c, goff = 16 * wave + 4 * g, woff = wave * ns * kTile + 4 * lane;
    // What is the same in every lane stays a vector load, which is waited for a step later with the others: a scalar one is waited
    // for with the next LDS read, and a value that the compiler knows to be uniform is moved to a scalar at once.
    int zero;
    asm("v_mov_b32 %0, 0" : "=v"(zero));
    auto read_s = [&](int B, float4 (&b)[NS]) {
#pragma unroll
        for (int s = 0; s < NS; ++s)
            if (EXACT || s < ns) b[s] = ld4(&s_s[B][c * LS + 16 * s + 4 * g]);
    };
    // The loop has both turns or none: with a way from the first to itself past the second, even one that is never taken, it would
    // wait for all its loads at once, as nothing is known to be behind them. The last chunk's loads are its own again: loads
    // without a branch.
    auto walk = [&](auto step) {
        int ci = c0;
        for (; ci + 1 < c1; ci += 2) {
            step(std::integral_constant<int, 0>{}, ci);
            step(std::integral_constant<int, 1>{}, ci + 1);
        }
        if (ci < c1) step(std::integral_constant<int, 0>{}, ci);
    };
    if (outputs) {
        struct Operands {
            float4 q[NS], eg;
        } in[SETS];
        float4 p[4], ul[4];
        int t0 = 0, n = 0, t1, n1;  // first token, tokens (any chunk may be short): of the outputs under way, of p's chunk
        // Lines of 128 bytes of a chunk's W, q and k transposed (ns * 4 KB, ns * 32 lines each) and P (16 KB).
        const int per = ns * 32, line = vt * kNT + tid, sec = line / per;
        const char* ahead = sec == 0   ? reinterpret_cast<const char*>(W + (int64_t)h * 4 * ns * kTile) + line * 128
                            : sec == 1 ? reinterpret_cast<const char*>(qk + (int64_t)kh * 8 * ns * kTile) + (line - per) * 128
                            : sec == 2 ? reinterpret_cast<const char*>(kt + (int64_t)kh * 4 * ns * kTile) + (line - 2 * per) * 128
                                       : reinterpret_cast<const char*>(P + (int64_t)h * 16 * kTile) + min(line - 3 * per, 127) * 128;
        const int64_t ahead_step = (int64_t)(sec == 0 ? d.H * 4 * ns : sec == 1 ? d.K * 8 * ns : sec == 2 ? d.K * 4 * ns : d.H * 16) * kTile * 4;
        int touched = 0;
        const int ostep = d.H * d.V;
        auto load_q = [&](Operands& x, int ci, int s) {
            if (EXACT || s < ns) x.q[s] = ld4(qk + ((int64_t)ci * d.K + kh) * 8 * ns * kTile + woff + s * kTile);
        };
        auto load_eg = [&](Operands& x, int ci) { x.eg = ld4(G + ((int64_t)ci * d.H + h) * 2 * kC + goff); };
        auto load_p = [&](int ci) {
            const int64_t ch = (int64_t)ci * d.H + h;
#pragma unroll
            for (int s = 0; s < 4; ++s)  // lower triangular: the blocks above are loaded, not used
                p[s] = ld4(P + ((ch * 4 + wave) * 4 + s) * kTile + 4 * lane);
            const int2 at = *reinterpret_cast<const int2*>(sq.chunk + 4 * ci + zero);
            t1 = at.x;
            n1 = at.y;
        };
        // A chunk's outputs are a phase behind the chain: diag(e^G) Q S while it updates S, mostly, and P U while it forms the
        // next U. What is read of LDS is read a phase ahead.
        f32x4 ao = {0.f, 0.f, 0.f, 0.f};
        auto finish = [&]() {
#pragma unroll
            for (int s = 0; s < 4; ++s) {  // the blocks above the diagonal as zeros: behind a branch their loads would be, too
                const bool in = s <= wave;
                ao = mma4(make_float4(in ? p[s].x : 0.f, in ? p[s].y : 0.f, in ? p[s].z : 0.f, in ? p[s].w : 0.f), ul[s], ao);
            }
            t0 = t1, n = n1;
            float* op = o + ((int64_t)t0 * d.H + h) * d.V;
            if (vcol < d.V) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (goff + i < n) op[(goff + i) * ostep + vcol] = ao[i];
            }
        };
        load_eg(in[0], c0);
#pragma unroll
        for (int s = 0; s < NS; ++s) load_q(in[0], c0, s);
#pragma unroll
        for (int s = 0; s < 4; ++s) p[s] = ul[s] = make_float4(0.f, 0.f, 0.f, 0.f);
        t1 = n1 = 0;
        walk([&](auto turn, int ci) {
            constexpr int B = decltype(turn)::value, EARLY = NS / 4;
            Operands &x = in[B % SETS], &next = in[(B + 1) % SETS];
            const int cn = min(ci + 1, c1 - 1);
            __syncthreads();  // S^T of the chunk before is in LDS
            float4 b[NS];
            read_s(B, b);
            finish();  // the chunk before; at the first, nothing
            load_p(ci);
            if (SETS > 1) load_eg(next, cn);
            asm volatile("" ::"v"(touched));
            touched = *reinterpret_cast<const int*>(ahead + min(ci + 2, c1 - 1) * ahead_step);
            ao = f32x4{0.f, 0.f, 0.f, 0.f};
            auto product = [&](int s) {  // a load a product: a burst of them would hold the products up
                if (EXACT || s < ns) ao = mma4(x.q[s], b[s], ao);
                if (SETS > 1) load_q(next, cn, s);
                __builtin_amdgcn_sched_barrier(0);
            };
#pragma unroll
            for (int s = 0; s < EARLY; ++s) product(s);
            __syncthreads();  // U^T is
#pragma unroll
            for (int s = 0; s < 4; ++s) ul[s] = ld4(&s_u[B][c * LU + 16 * s + 4 * g]);
#pragma unroll
            for (int s = EARLY; s < NS; ++s) product(s);
            ao[0] *= x.eg.x;
            ao[1] *= x.eg.y;
            ao[2] *= x.eg.z;
            ao[3] *= x.eg.w;
            if constexpr (SETS == 1) {
                load_eg(next, cn);
#pragma unroll
                for (int s = 0; s < NS; ++s) load_q(next, cn, s);
            }
        });
        finish();
        return;
    }
    float* st_ = state + ((int64_t)row * d.H + h) * d.D * VP;
    // this wave's rows of S: tiles wave, wave + 4, ...; element i: dim 16 tile + 4 g + i, column c
    f32x4 S[DT];
#pragma unroll
    for (int k = 0; k < DT; ++k) {
        const int tile = wave + 4 * k;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int dd = 16 * tile + 4 * g + i;
            S[k][i] = (pos0 > 0 && dd < d.D && vcol < VP) ? st_[(int64_t)dd * VP + vcol] : 0.f;
        }
        if (EXACT || tile < ns) *reinterpret_cast<f32x4*>(&s_s[0][c * LS + 16 * tile + 4 * g]) = S[k];
    }
    struct Operands {
        float4 w[NS], kk[DT][4], u0, er;
        float decay;
    } in[SETS];
    auto load_w = [&](Operands& x, int ci, int s) {
        if (EXACT || s < ns) x.w[s] = ld4(W + ((int64_t)ci * d.H + h) * 4 * ns * kTile + woff + s * kTile);
    };
    auto load_ends = [&](Operands& x, int ci) {
        const int64_t ch = (int64_t)ci * d.H + h;
        x.u0 = ld4(U + ((ch * nt + vt) * 4 + wave) * kTile + 4 * lane);
        x.er = ld4(G + ch * 2 * kC + kC + goff);
        x.decay = G[ch * 2 * kC + kC - 1 + zero];
    };
    auto load_k = [&](Operands& x, int ci, int s) {
#pragma unroll
        for (int k = 0; k < DT; ++k)
            if (EXACT || wave + 4 * k < ns)
                x.kk[k][s] = ld4(kt + (((int64_t)ci * d.K + kh) * ns + wave + 4 * k) * 4 * kTile + s * kTile + 4 * lane);
    };
    load_ends(in[0], c0);
#pragma unroll
    for (int s = 0; s < NS; ++s) load_w(in[0], c0, s);
    if constexpr (SETS > 1) {
#pragma unroll
        for (int s = 0; s < 4; ++s) load_k(in[0], c0, s);
    }
    __builtin_amdgcn_s_setprio(1);  // ahead of the outputs' waves
    walk([&](auto turn, int ci) {
        constexpr int B = decltype(turn)::value;
        Operands &x = in[B % SETS], &next = in[(B + 1) % SETS];
        const int cn = min(ci + 1, c1 - 1);
        if constexpr (SETS == 1) {
#pragma unroll
            for (int s = 0; s < 4; ++s) load_k(x, ci, s);
        }
        __syncthreads();  // S^T of the chunk before is in LDS
        float4 b[NS];
        read_s(B, b);
        const float decay = x.decay;  // with one set the next chunk's takes its place
        f32x4 aw = {0.f, 0.f, 0.f, 0.f};
        if constexpr (SETS > 1) load_ends(next, cn);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (EXACT || s < ns) aw = mma4(x.w[s], b[s], aw);
            if (SETS > 1) load_w(next, cn, s);
            __builtin_amdgcn_sched_barrier(0);
        }
        const float4 u = make_float4(x.u0.x - aw[0], x.u0.y - aw[1], x.u0.z - aw[2], x.u0.w - aw[3]);
        st4(&s_u[B][c * LU + goff], u);
        st4(&s_d[c * LU + goff], make_float4(u.x * x.er.x, u.y * x.er.y, u.z * x.er.z, u.w * x.er.w));
#pragma unroll
        for (int k = 0; k < DT; ++k) S[k] = S[k] * decay;
        __syncthreads();  // U^T is
        float4 ud[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) ud[s] = ld4(&s_d[c * LU + 16 * s + 4 * g]);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int k = 0; k < DT; ++k)
                if (EXACT || wave + 4 * k < ns) S[k] = mma4(x.kk[k][s], ud[s], S[k]);
            if (SETS > 1) load_k(next, cn, s);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (SETS == 1) {
            load_ends(next, cn);
#pragma unroll
            for (int s = 0; s < NS; ++s) load_w(next, cn, s);
        }
#pragma unroll
        for (int k = 0; k < DT; ++k)
            if (EXACT || wave + 4 * k < ns)
                *reinterpret_cast<f32x4*>(&s_s[1 - B][c * LS + 16 * (wave + 4 * k) + 4 * g]) = S[k];
    });
#pragma unroll
    for (int k = 0; k < DT; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int dd = 16 * (wave + 4 * k) + 4 * g + i;
            if (dd < d.D && vcol < VP) st_[(int64_t)dd * VP + vcol] = S[k][i];
        }
}

// Output norm and gate of tokens [first, T). LG lanes share a (token, head), four values a lane (VEC: vdim
// a multiple of 4, at most 4 LG); otherwise a wave takes one and strides over vdim.
template <typename T, bool VEC>
__global__ __launch_bounds__(kNT) void delta_out_kernel(Dims d, const float* __restrict__ o, const T* __restrict__ proj,
                                                        int64_t stride, const T* __restrict__ norm_w, int first, int LG,
                                                        int64_t items, T* __restrict__ out, int64_t out_stride) {
    const int lane = threadIdx.x & 63;
    if constexpr (VEC) {
        const int per = kNT / LG, sub = threadIdx.x % LG, i = 4 * sub;
        constexpr int kIt = 4;
        const int64_t e0 = (int64_t)blockIdx.x * per * kIt + threadIdx.x / LG;
        float4 x[kIt], gt[kIt];
#pragma unroll
        for (int k = 0; k < kIt; ++k) {
            const int64_t e = min(e0 + (int64_t)k * per, items - 1), t = first + e / d.H;
            const int h = (int)(e % d.H), ii = min(i, d.V - 4);
            x[k] = ld4(o + (t * d.H + h) * d.V + ii);
            const T* gp = proj + t * stride + d.channels() + h * d.V + ii;
            gt[k] = make_float4(ld(gp), ld(gp + 1), ld(gp + 2), ld(gp + 3));
        }
        const int ii = min(i, d.V - 4);
        const float4 w = make_float4(ld(norm_w + ii), ld(norm_w + ii + 1), ld(norm_w + ii + 2), ld(norm_w + ii + 3));
#pragma unroll
        for (int k = 0; k < kIt; ++k) {
            float ss = i < d.V ? x[k].x * x[k].x + x[k].y * x[k].y + x[k].z * x[k].z + x[k].w * x[k].w : 0.f;
            for (int q = 1; q < LG; q <<= 1) ss += __shfl_xor(ss, q, kWave);
            const float r = 1.f / sqrtf(ss / (float)d.V + d.eps);
            const int64_t e = e0 + (int64_t)k * per;
            if (e < items && i < d.V) {
                T* dst = out + (first + e / d.H) * out_stride + (e % d.H) * d.V + i;
                st(dst, x[k].x * r * w.x * siluf_(gt[k].x));
                st(dst + 1, x[k].y * r * w.y * siluf_(gt[k].y));
                st(dst + 2, x[k].z * r * w.z * siluf_(gt[k].z));
                st(dst + 3, x[k].w * r * w.w * siluf_(gt[k].w));
            }
        }
        return;
    }
    const int64_t e = (int64_t)blockIdx.x * (kNT / kWave) + (threadIdx.x >> 6);
    if (e >= items) return;
    const int64_t t = first + e / d.H;
    const int h = (int)(e % d.H);
    const float* src = o + (t * d.H + h) * d.V;
    const T* gate = proj + t * stride + d.channels() + h * d.V;
    float ss = 0.f;
    for (int i = lane; i < d.V; i += kWave) ss += src[i] * src[i];
    const float r = 1.f / sqrtf(wave_sum(ss) / (float)d.V + d.eps);
    for (int i = lane; i < d.V; i += kWave)
        st(out + t * out_stride + h * d.V + i, src[i] * r * ld(norm_w + i) * siluf_(ld(gate + i)));
}

int scan_rows_per_thread(const Dims& d, int nt) {
    const int RG = nt / (d.vpad() / 4);
    return (d.D + RG - 1) / RG;
}

const char* bad_shape(const skyrl_delta_shape* sh) {
    if (!sh) return "delta: null shape";
    if (sh->heads <= 0 || sh->kv_heads <= 0 || sh->heads % sh->kv_heads) return "delta: heads must be a multiple of kv_heads";
    if (sh->dim <= 0 || sh->vdim <= 0 || sh->dim > 1024 || sh->vdim > 1024) return "delta: dim and vdim must be in [1, 1024]";
    if (sh->taps <= 0 || sh->taps > kMaxTaps) return "delta: taps must be in [1, 64]";
    return nullptr;
}
Dims dims_of(const skyrl_delta_shape* sh) {
    return Dims{sh->heads, sh->kv_heads, sh->dim, sh->vdim, sh->taps, sh->eps};
}
int64_t proj_width(const Dims& d) { return d.channels() + (int64_t)d.H * d.V + 2 * d.H; }

}  // namespace
}  // namespace skyrl

using namespace skyrl;

#define LAUNCH_SCAN(NT, R)                                                                                         \
    hipLaunchKernelGGL((d.taps <= kWin && 2 * d.D + d.vpad() <= NT ? delta_scan_kernel<T, NT, R, true>             \
                                                                   : delta_scan_kernel<T, NT, R, false>),          \
                       dim3(d.H, nseq), dim3(NT), lds, as_stream(stream), d,                                       \
                       reinterpret_cast<const T*>(proj), proj_stride, reinterpret_cast<const T*>(conv_w), a_log,   \
                       dt_bias, reinterpret_cast<const T*>(norm_w), cu, rows, positions, state,                    \
                       reinterpret_cast<T*>(conv_state), save_conv, reinterpret_cast<T*>(out), out_stride)

extern "C" int skyrl_delta_scan(const skyrl_delta_shape* shape, const void* proj, int64_t proj_stride,
                                const void* conv_w, const float* a_log, const float* dt_bias, const void* norm_w,
                                const int32_t* cu, const int32_t* rows, const int64_t* positions, int32_t nseq,
                                float* state, void* conv_state, int32_t save_conv, void* out, int64_t out_stride,
                                int32_t dtype, void* stream) {
    SKYRL_REQUIRE_T(dtype, "delta_scan");
    const char* bad = bad_shape(shape);
    SKYRL_REQUIRE(!bad, bad);
    const Dims d = dims_of(shape);
    SKYRL_REQUIRE(nseq >= 0 && nseq <= 65535, "delta_scan: nseq must be in [0, 65535]");
    SKYRL_REQUIRE(proj_stride >= proj_width(d), "delta_scan: proj_stride");
    SKYRL_REQUIRE(out_stride >= (int64_t)d.H * d.V, "delta_scan: out_stride");
    if (nseq == 0) return SKYRL_OK;
    SKYRL_REQUIRE(proj && conv_w && a_log && dt_bias && norm_w && cu && rows && positions && state && conv_state && out,
                  "delta_scan: null pointer");
    const int nt = scan_rows_per_thread(d, 256) <= 8 ? 256 : scan_rows_per_thread(d, 512) <= 8 ? 512 : 1024;
    const int rpt = scan_rows_per_thread(d, nt), RG = nt / (d.vpad() / 4);
    SKYRL_REQUIRE(rpt <= 16, "delta_scan: dim * vdim too large for one workgroup's registers (at most 65536)");
    const size_t lds = (size_t)(2 * d.D + 2 * d.vpad() + 2 * RG * d.vpad() + 4) * sizeof(float);
    SKYRL_DISPATCH_T(dtype, {
        if (nt == 256 && rpt <= 4) LAUNCH_SCAN(256, 4);
        else if (nt == 256) LAUNCH_SCAN(256, 8);
        else if (nt == 512) LAUNCH_SCAN(512, 8);
        else if (rpt <= 8) LAUNCH_SCAN(1024, 8);
        else LAUNCH_SCAN(1024, 16);
    })
    return check_launch("delta_scan_kernel");
}

extern "C" int skyrl_delta_conv(const skyrl_delta_shape* shape, const void* proj, int64_t proj_stride,
                                const void* conv_w, const float* a_log, const float* dt_bias, const int32_t* chunk,
                                int32_t nchunks, const int32_t* cu, const int32_t* rows, const int64_t* positions,
                                const void* conv_state, float* qk, float* kt, float* vt, float* lg, float* beta,
                                int32_t dtype, void* stream) {
    SKYRL_REQUIRE_T(dtype, "delta_conv");
    const char* bad = bad_shape(shape);
    SKYRL_REQUIRE(!bad, bad);
    const Dims d = dims_of(shape);
    SKYRL_REQUIRE(nchunks >= 0 && proj_stride >= proj_width(d), "delta_conv: bad sizes");
    if (nchunks == 0) return SKYRL_OK;
    SKYRL_REQUIRE(proj && conv_w && a_log && dt_bias && chunk && cu && rows && positions && conv_state && qk && kt && vt &&
                      lg && beta,
                  "delta_conv: null pointer");
    SKYRL_DISPATCH_T(dtype, {
#define LAUNCH_CONV(TAPS)                                                                                                 \
    hipLaunchKernelGGL((2 * d.D <= kNT ? delta_conv_kernel<T, TAPS, true> : delta_conv_kernel<T, TAPS, false>),            \
                       dim3(nchunks, d.K + (d.H * d.V + kNT - 1) / kNT), dim3(kNT), 16 * (2 * d.D + 4) * sizeof(float),       \
                       as_stream(stream), d, SeqRef{chunk, cu, rows, positions}, reinterpret_cast<const T*>(proj),         \
                       proj_stride, reinterpret_cast<const T*>(conv_w), a_log, dt_bias,                                    \
                       reinterpret_cast<const T*>(conv_state), qk, kt, vt, lg, beta)
        if (d.taps <= 4) LAUNCH_CONV(4);
        else if (d.taps <= kConvWindow) LAUNCH_CONV(kConvWindow);
        else LAUNCH_CONV(0);
    })
    return check_launch("delta_conv_kernel");
}

extern "C" int skyrl_delta_chunk(const skyrl_delta_shape* shape, const int32_t* chunk, int32_t nchunks,
                                 const float* qk, const float* kt, const float* vt, const float* lg, const float* beta,
                                 float* W, float* U, float* P, float* G, void* stream) {
    const char* bad = bad_shape(shape);
    SKYRL_REQUIRE(!bad, bad);
    const Dims d = dims_of(shape);
    SKYRL_REQUIRE(nchunks >= 0 && (int64_t)nchunks * d.H < (1 << 30), "delta_chunk: bad sizes");
    if (nchunks == 0) return SKYRL_OK;
    SKYRL_REQUIRE(chunk && qk && kt && vt && lg && beta && W && U && P && G, "delta_chunk: null pointer");
    hipLaunchKernelGGL(delta_chunk_kernel, dim3(nchunks * d.H), dim3(kNT), 0, as_stream(stream), d, chunk, qk, kt, vt,
                       lg, beta, W, U, P, G);
    return check_launch("delta_chunk_kernel");
}

#define LAUNCH_CHAIN(NS, EXACT, SETS)                                                                           \
    hipLaunchKernelGGL((delta_chain_kernel<NS, EXACT, SETS>),                                                           \
                       dim3((unsigned)(nseq * d.H + 7) / 8 * 8 * (d.v16() / 16)), dim3(2 * kNT), 0, as_stream(stream), \
                       d, SeqRef{chunk, cu, rows, positions}, seq_chunks, seq0, nseq, qk, kt, W, U, P, G, state, o)

extern "C" int skyrl_delta_chain(const skyrl_delta_shape* shape, const int32_t* chunk, const int32_t* seq_chunks,
                                 int32_t seq0, int32_t nseq, const int32_t* cu, const int32_t* rows,
                                 const int64_t* positions, const float* qk, const float* kt, const float* W,
                                 const float* U, const float* P, const float* G, float* state, float* o, void* stream) {
    const char* bad = bad_shape(shape);
    SKYRL_REQUIRE(!bad, bad);
    const Dims d = dims_of(shape);
    SKYRL_REQUIRE(d.D <= 256, "delta_chain: dim must be at most 256");
    SKYRL_REQUIRE(nseq >= 0 && seq0 >= 0 && (int64_t)nseq * d.H * (d.v16() / 16) < (1 << 30), "delta_chain: bad sizes");
    if (nseq == 0) return SKYRL_OK;
    SKYRL_REQUIRE(chunk && seq_chunks && cu && rows && positions && qk && kt && W && U && P && G && state && o,
                  "delta_chain: null pointer");
    if (d.D == 64) LAUNCH_CHAIN(4, true, 2);
    else if (d.D < 64) LAUNCH_CHAIN(4, false, 2);
    else if (d.D == 128) LAUNCH_CHAIN(8, true, 2);
    else if (d.D < 128) LAUNCH_CHAIN(8, false, 2);
    else LAUNCH_CHAIN(16, false, 1);
    return check_launch("delta_chain_kernel");
}

extern "C" int skyrl_delta_out(const skyrl_delta_shape* shape, const float* o, const void* proj, int64_t proj_stride,
                               const void* norm_w, int32_t first, int32_t T_, void* out, int64_t out_stride,
                               int32_t dtype, void* stream) {
    SKYRL_REQUIRE_T(dtype, "delta_out");
    const char* bad = bad_shape(shape);
    SKYRL_REQUIRE(!bad, bad);
    const Dims d = dims_of(shape);
    SKYRL_REQUIRE(first >= 0 && T_ >= first && proj_stride >= proj_width(d) && out_stride >= (int64_t)d.H * d.V,
                  "delta_out: bad sizes");
    const int64_t items = (int64_t)(T_ - first) * d.H;
    if (items == 0) return SKYRL_OK;
    SKYRL_REQUIRE(o && proj && norm_w && out, "delta_out: null pointer");
    SKYRL_DISPATCH_T(dtype, {
        int LG = 1;
        while (4 * LG < d.V) LG <<= 1;
        const T* p = reinterpret_cast<const T*>(proj);
        const T* w = reinterpret_cast<const T*>(norm_w);
        T* dst = reinterpret_cast<T*>(out);
        if (d.V % 4 == 0 && LG <= kWave) {
            const int64_t per = (int64_t)kNT / LG * 4;
            hipLaunchKernelGGL((delta_out_kernel<T, true>), dim3((unsigned)((items + per - 1) / per)), dim3(kNT), 0,
                               as_stream(stream), d, o, p, proj_stride, w, first, LG, items, dst, out_stride);
        } else {
            hipLaunchKernelGGL((delta_out_kernel<T, false>), dim3((unsigned)((items + 3) / 4)), dim3(kNT), 0,
                               as_stream(stream), d, o, p, proj_stride, w, first, LG, items, dst, out_stride);
        }
    })
    return check_launch("delta_out_kernel");
}
