// HBM-bound row and elementwise kernels: basic.tl softmax (:10-17),
// rmsnorm (:20-26) and add (:3-7); llm.tl embed (:10-16), rmsnorm (:19-25),
// rmsnorm_rows (:175-182), rope_q (:78-88) and kv_write (:93-112).
//
// A row is owned by one 64-lane wavefront (short rows, and enough of them) or
// by a workgroup of 256 to 1024 threads: it is read once with 16-byte loads at
// any alignment into registers, reduced (DPP within wavefronts, LDS between
// them) and written once, so each element crosses HBM once each way. Rows longer
// than the register budget take a second, cache-resident pass.
#include "common.h"

#include <climits>
#include <type_traits>

namespace {

constexpr int ROWS_PER_WG = 4;  // one wavefront per row, 4 per workgroup
constexpr float LOG2E_F = 1.4426950408889634f;

// softmax and basic.rmsnorm rows are read once and their outputs are not
// read back by the same kernel: nontemporal loads and stores (4096^2, rows
// from HBM: rmsnorm 14.0 -> 13.2 us, softmax 27.1 -> 25.6 us, with softmax's
// division as DivBy).
template <class T>
TSL_DEV T load_once(const T* p) { return __builtin_nontemporal_load(p); }
template <class T>
TSL_DEV void store_out(T v, T* p) { __builtin_nontemporal_store(v, p); }

// Vectors at element alignment: rows of any length start at any element, and
// gfx950's wide global accesses need no more (odd row lengths had one load per
// element: measured at the kernels below). Functions, not templates over the
// vector: a template argument drops the alignment.
typedef float4v float4u __attribute__((aligned(4)));
typedef u32x4 u32x4u __attribute__((aligned(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef u32x2 u32x2u __attribute__((aligned(2)));
TSL_DEV float4v load_once4(const float* p) { return __builtin_nontemporal_load(reinterpret_cast<const float4u*>(p)); }
TSL_DEV u32x4 load_once8(const u16* p) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4u*>(p)); }
TSL_DEV void store_out4(float4v v, float* p) { __builtin_nontemporal_store(v, reinterpret_cast<float4u*>(p)); }
TSL_DEV void store_out8(u32x4 v, u16* p) { __builtin_nontemporal_store(v, reinterpret_cast<u32x4u*>(p)); }
TSL_DEV void store_out4h(u32x2 v, u16* p) { __builtin_nontemporal_store(v, reinterpret_cast<u32x2u*>(p)); }
TSL_DEV float4v load4(const float* p) { return *reinterpret_cast<const float4u*>(p); }
TSL_DEV u32x4 load8(const u16* p) { return *reinterpret_cast<const u32x4u*>(p); }
TSL_DEV u32x2 load4h(const u16* p) { return *reinterpret_cast<const u32x2u*>(p); }

// Largest / sum of x over the workgroup's NT threads, every thread receiving
// it (the wavefronts' results in order; red: NT / 64 floats, free again
// after the next barrier).
template <int NT, bool MAX>
TSL_DEV float wg_reduce(float x, float* red) {
    x = MAX ? wave_max(x) : wave_sum(x);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
    __syncthreads();
    if constexpr (!MAX && NT >= 512) {  // (8 and 16 sums pairwise: a chain of 16 rounds the total by an ulp)
        float p[NT / 64];
#pragma unroll
        for (int w = 0; w < NT / 64; w++) p[w] = red[w];
#pragma unroll
        for (int h = 1; h < NT / 64; h *= 2)
#pragma unroll
            for (int w = 0; w < NT / 64; w += 2 * h) p[w] += p[w + h];
        return p[0];
    }
    float r = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++) r = MAX ? fmaxf(r, red[w]) : r + red[w];
    return r;
}

// ---------------------------------------------------------------- softmax
// Y[r, c] = exp(x - max) / sum(exp(x - max)) over the first ncols = min(BC, C)
// columns; columns past C read -inf (kernels/basic.tl:13), so they add 0.
template <int NV, int RPW = ROWS_PER_WG>
__global__ __launch_bounds__(64 * RPW) void softmax_kernel(const float* __restrict__ X, float* __restrict__ Y, int R, int C,
                                                      int ncols) {
    const int lane = threadIdx.x & 63, row = blockIdx.x * RPW + (threadIdx.x >> 6);
    if (row >= R) return;
    const float* x = X + (size_t)row * C;
    float* y = Y + (size_t)row * C;
    // FULL: every chunk of every lane lies inside the row (a uniform branch,
    // so the common shape runs without per-chunk tests).
    auto body = [&](auto full) {
        constexpr bool FULL = decltype(full)::value;
        float v[NV][4];
        float m = -INFINITY;
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int c = i * 256 + lane * 4;
            if (FULL || c + 4 <= ncols) {
                float4v t = load_once4(x + c);
                for (int e = 0; e < 4; e++) v[i][e] = t[e];
            } else {
                for (int e = 0; e < 4; e++) v[i][e] = (c + e < ncols) ? x[c + e] : -INFINITY;
            }
            for (int e = 0; e < 4; e++) m = fmaxf(m, v[i][e]);
        }
        m = wave_max(m);
        // exp(x - m) as exp2((x - m) log2(e)): one v_exp_f32 and two operations
        // per element where expf expands to ~12 (its range reduction and
        // overflow/underflow selects); x - m <= 0, so exp2's argument is in
        // range, and its rounding adds (m - x) 2^-24 relative (1e-6 at a
        // probability of e^-16). 4096^2 from HBM: 25.6 -> 23.8 us.
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < NV; i++)
            for (int e = 0; e < 4; e++) {
                v[i][e] = __builtin_amdgcn_exp2f((v[i][e] - m) * LOG2E_F);
                s += v[i][e];
            }
        const DivBy by_s(wave_sum(s));  // s >= 1: the row's max contributes exp(0)
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int c = i * 256 + lane * 4;
            if (FULL || c + 4 <= ncols) {
                float4v t;
                for (int e = 0; e < 4; e++) t[e] = by_s(v[i][e]);
                store_out4(t, y + c);
            } else {
                for (int e = 0; e < 4; e++)
                    if (c + e < ncols) y[c + e] = by_s(v[i][e]);
            }
        }
    };
    if (ncols == NV * 256) body(std::true_type{});
    else body(std::false_type{});
}

// exp(d) for d <= 0 (NaN for NaN) to about an ulp, rounded below the smallest
// normal, for rows longer than 4096 columns: n + f = d log2(e) with n whole and f
// from the unrounded product (log2(e) in two parts), 2^f by v_exp_f32, scaled by
// 2^n. (As exp2(d log2(e)) the product's one rounding costs a probability of
// 1e-30 5e-6 of itself, and v_exp_f32 flushes results below 2^-126: 256 x 32000
// took 12.6 us so and takes 14.0, 2000 x 8192 22.6 and 22.8.)
TSL_DEV float exp_neg(float d) {
    constexpr float LOG2E_LO = 1.9259629911e-8f;  // log2(e) - LOG2E_F
    const float n = fmaxf(__builtin_rintf(d * LOG2E_F), -200.0f);  // (0 from -151 on; -inf stays out of n)
    const float f = __builtin_fmaf(d, LOG2E_LO, __builtin_fmaf(d, LOG2E_F, -n));
    return __builtin_ldexpf(__builtin_amdgcn_exp2f(f), (int)n);
}

// One workgroup of NT threads per row (up to 4 NT NV columns): thread t holds
// chunks t, t + NT, .. of 4 columns, all loaded at once, so a row crosses
// memory once each way and a few long rows still use 256 to 1024 lanes each.
// Many rows are bound by HBM (inputs rotated past the last-level cache: 2000 x
// 8192 5.7 TB/s), a row per CU by its chain of load, exponentials and store (256 x
// 32000 4.7 TB/s). Against one wavefront per row with scalar loads in two
// serial passes, calls back to back over the same rows: 256 x 32000 361 -> 13.3
// us, 19 x 25587 160 -> 7.5, 2000 x 8192 114 -> 22.5; up to 4096 columns against
// one wavefront with 16 chunks, 48 x 2816 4.6 -> 3.9, 1000 x 2813 7.1 -> 5.3, 8192 x
// 2500 31.8 -> 28.1.
template <int NT, int NV>
__global__ __launch_bounds__(NT) void softmax_wg_kernel(const float* __restrict__ X, float* __restrict__ Y, int C,
                                                        int ncols) {
    constexpr bool EXACT = 4 * NT * NV > 4096;  // (up to 4096 columns the exponential of softmax_kernel)
    __shared__ float red[2][NT / 64];
    TSL_POISON(red);
    const int t = threadIdx.x;
    const float* x = X + (size_t)blockIdx.x * C;
    float* y = Y + (size_t)blockIdx.x * C;
    float v[NV][4];
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = (i * NT + t) * 4;
        if (c + 4 <= ncols) {
            const float4v q = load_once4(x + c);
            for (int e = 0; e < 4; e++) v[i][e] = q[e];
        } else {
            for (int e = 0; e < 4; e++) v[i][e] = c + e < ncols ? x[c + e] : -INFINITY;
        }
    }
#pragma unroll
    for (int i = 0; i < NV; i++)
        for (int e = 0; e < 4; e++) m = fmaxf(m, v[i][e]);
    m = wg_reduce<NT, true>(m, red[0]);
    float s[4] = {};  // (long rows: a sum per column of the chunks, so a thread's 32 terms round in 8s)
#pragma unroll
    for (int i = 0; i < NV; i++)
        for (int e = 0; e < 4; e++) {
            v[i][e] = EXACT ? exp_neg(v[i][e] - m) : __builtin_amdgcn_exp2f((v[i][e] - m) * LOG2E_F);
            s[EXACT ? e : 0] += v[i][e];
        }
    const DivBy by_s(wg_reduce<NT, false>((s[0] + s[1]) + (s[2] + s[3]), red[1]));  // s >= 1: the row's max contributes exp(0)
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = (i * NT + t) * 4;
        if (c + 4 <= ncols) {
            float4v q;
            for (int e = 0; e < 4; e++) q[e] = by_s(v[i][e]);
            store_out4(q, y + c);
        } else {
            for (int e = 0; e < 4; e++)
                if (c + e < ncols) y[c + e] = by_s(v[i][e]);
        }
    }
}

// Rows longer than softmax_wg_kernel's registers: a workgroup per row, a
// running max and sum per thread, then a second, cache-resident pass for the
// writes.
constexpr int SML_THREADS = 1024;
__global__ __launch_bounds__(SML_THREADS) void softmax_long_kernel(const float* __restrict__ X, float* __restrict__ Y,
                                                                   int C, int ncols) {
    __shared__ float red[2][SML_THREADS / 64];
    TSL_POISON(red);
    const float* x = X + (size_t)blockIdx.x * C;
    float* y = Y + (size_t)blockIdx.x * C;
    auto load = [&](int c) {
        if (c + 4 <= ncols) return load4(x + c);
        float4v q;
        for (int e = 0; e < 4; e++) q[e] = c + e < ncols ? x[c + e] : -INFINITY;
        return q;
    };
    float m = -INFINITY, s = 0.0f;
    for (int c = threadIdx.x * 4; c < ncols; c += SML_THREADS * 4) {
        const float4v q = load(c);
        const float m2 = fmaxf(m, fmaxf(fmaxf(q[0], q[1]), fmaxf(q[2], q[3])));
        // (while every column so far is -inf there is nothing to rescale;
        // NaN columns still reach the sum)
        const float mm = m2 == -INFINITY ? 0.0f : m2;
        s *= exp_neg(m == -INFINITY ? 0.0f : m - mm);
        for (int e = 0; e < 4; e++) s += exp_neg(q[e] - mm);
        m = m2;
    }
    const float mw = wg_reduce<SML_THREADS, true>(m, red[0]);
    s *= exp_neg(m == -INFINITY ? 0.0f : m - mw);
    const DivBy by_s(wg_reduce<SML_THREADS, false>(s, red[1]));
    for (int c = threadIdx.x * 4; c < ncols; c += SML_THREADS * 4) {
        const float4v q = load(c);
        float4v o;
        for (int e = 0; e < 4; e++) o[e] = by_s(exp_neg(q[e] - mw));
        if (c + 4 <= ncols) {
            *reinterpret_cast<float4u*>(y + c) = o;
        } else {
            for (int e = 0; e < 4; e++)
                if (c + e < ncols) y[c + e] = o[e];
        }
    }
}

// ---------------------------------------------------------------- rmsnorm
// y = x * (1 / sqrt(sum(x^2 over BC columns) / n + eps)) * w, over the
// first ncols = min(BC, C) columns (columns past C read 0). XT is f16
// (basic.tl) or f32 (llm.tl); `rows` (rmsnorm_rows) gathers the input row.

// 8 packed columns c .. c + 7 of a row of ncols (zeros past them), and their store.
TSL_DEV u32x4 load8_edge(const u16* p, int c, int ncols) {
    uint32_t h[8];
    for (int e = 0; e < 8; e++) h[e] = c + e < ncols ? p[c + e] : 0;
    return u32x4{h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16)};
}

// The 8 outputs f16(x rs w) of a packed chunk.
TSL_DEV u32x4 rms_scale8(u32x4 x, float rs, u32x4 w) {
    u32x4 o;
    for (int p = 0; p < 4; p++) {
        const u16 lo = f2h(h2f((u16)(x[p] & 0xffff)) * rs * h2f((u16)(w[p] & 0xffff)));
        const u16 hi = f2h(h2f((u16)(x[p] >> 16)) * rs * h2f((u16)(w[p] >> 16)));
        o[p] = (uint32_t)lo | ((uint32_t)hi << 16);
    }
    return o;
}
TSL_DEV float sum_squares8(u32x4 x, float ss) {
    for (int e = 0; e < 8; e++) {
        const float v = h2f((u16)(x[e >> 1] >> (16 * (e & 1))));
        ss += v * v;
    }
    return ss;
}

// f16 rows of any length up to 8 NT NV columns: NT threads per row (64: a
// wavefront each, 4 rows per workgroup; else a workgroup each), the row and
// its weights held packed and loaded together before the reduction. Bound by
// memory, short calls by latency. Calls back to back over the same rows (in part
// from the last-level cache), against rows unpacked to floats, with one load
// per element at lengths not a multiple of 8: 4096 x 1001 13.1 -> 5.4 us,
// 4096 x 3001 33.1 -> 10.8, and against two serial passes of scalar loads
// past 4096 columns, 24 x 6528 38.6 -> 3.6, 2048 x 8192 91 -> 13.2.
template <int NT, int NV>
__global__ __launch_bounds__(NT < 256 ? 256 : NT) void rmsnorm_f16_kernel(const u16* __restrict__ X,
                                                                          const u16* __restrict__ W,
                                                                          u16* __restrict__ Y, int R, int C, int ncols,
                                                                          float n, float eps) {
    constexpr int RPB = NT < 256 ? 256 / NT : 1;
    __shared__ float red[NT / 64];
    TSL_POISON(red);
    const int t = threadIdx.x % NT, row = blockIdx.x * RPB + threadIdx.x / NT;
    if (row >= R) return;
    const u16* x = X + (size_t)row * C;
    u16* y = Y + (size_t)row * C;
    u32x4 xv[NV], wv[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = (i * NT + t) * 8;
        if (c + 8 <= ncols) {
            xv[i] = load_once8(x + c);
            wv[i] = load8(W + c);
        } else {
            xv[i] = load8_edge(x, c, ncols);
            wv[i] = load8_edge(W, c, ncols);
        }
    }
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; i++) ss = sum_squares8(xv[i], ss);
    if constexpr (NT == 64) ss = wave_sum(ss);
    else ss = wg_reduce<NT, false>(ss, red);
    const float rs = 1.0f / sqrtf(ss / n + eps);
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = (i * NT + t) * 8;
        const u32x4 o = rms_scale8(xv[i], rs, wv[i]);
        if (c + 8 <= ncols) {
            store_out8(o, y + c);
        } else {
            for (int e = 0; e < 8; e++)
                if (c + e < ncols) y[c + e] = (u16)(o[e >> 1] >> (16 * (e & 1)));
        }
    }
}

// basic.rmsnorm over f16 rows whose every 16-byte chunk is present (ncols ==
// C == 512 NV): the row and its NV weight chunks stay packed (4 registers a
// chunk each, not 8 floats), so the weight loads are issued with the row's,
// before the reduction, and the wavefront waits on one memory round trip
// instead of two with all 4096 wavefronts of a 4096^2 call resident. The
// weights come once per workgroup through LDS (each wavefront reading all
// of them from L2 doubled the L2 traffic of a 4096^2 call): 4096^2 from HBM
// 11.23 -> 10.86 us. Same arithmetic, in the same order, as rmsnorm_f16_kernel.
// Wavefronts past R load row R - 1 and leave after the barrier.
template <int NV>
__global__ __launch_bounds__(256) void rmsnorm_f16_full_kernel(const u16* __restrict__ X, const u16* __restrict__ W,
                                                               u16* __restrict__ Y, int R, int C, float n, float eps) {
    const int lane = threadIdx.x & 63, row = blockIdx.x * ROWS_PER_WG + (threadIdx.x >> 6);
    __shared__ u32x4 wl[NV * 64];
    u32x4 xv[NV], wv[NV];
    const u16* x = X + (size_t)min(row, R - 1) * C;
    u16* y = Y + (size_t)row * C;
#pragma unroll
    for (int i = 0; i < NV; i++) xv[i] = load_once(reinterpret_cast<const u32x4*>(x + (i * 64 + lane) * 8));
    for (int c = threadIdx.x; c < NV * 64; c += 256) wl[c] = *reinterpret_cast<const u32x4*>(W + c * 8);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NV; i++) wv[i] = wl[i * 64 + lane];
    if (row >= R) return;
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; i++) ss = sum_squares8(xv[i], ss);
    ss = wave_sum(ss);
    const float rs = 1.0f / sqrtf(ss / n + eps);
#pragma unroll
    for (int i = 0; i < NV; i++)
        store_out(rms_scale8(xv[i], rs, wv[i]), reinterpret_cast<u32x4*>(y + (i * 64 + lane) * 8));
}

// ---- one workgroup per row (llm.tl rmsnorm over f32 rows, and the fused
// residual projection): thread t owns the float4 chunks t, t + 256, ... of
// the row, so a decode-sized batch (a few dozen rows) still spreads its
// loads over 256 lanes per row, all issued before the reduction.
// Loads this thread's chunks of W (zeros past ncols).
template <int NC>
TSL_DEV void rms_wg_weights(const u16* __restrict__ W, int t, int ncols, u32x2 (&w)[NC]) {
#pragma unroll
    for (int i = 0; i < NC; i++) {
        const int c = (i * 256 + t) * 4;
        if (c + 4 <= ncols) {
            w[i] = load4h(W + c);
        } else {
            uint32_t h[4];
            for (int e = 0; e < 4; e++) h[e] = c + e < ncols ? W[c + e] : 0;
            w[i] = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
        }
    }
}

// Given this thread's values v (zero past ncols) and weights, writes
// y[c] = f16(v * rs * w[c]) for the first ncols columns, rs = 1 / sqrt(sum
// of squares of the row / n + eps): per-thread sums in chunk order, then
// the wavefront butterfly, then the 4 wavefronts in order.
template <int NC>
TSL_DEV void rms_wg_finish(const float4v (&v)[NC], const u32x2 (&w)[NC], int t, int ncols, float n, float eps,
                           u16* __restrict__ y, float* red) {
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < NC; i++)
        for (int e = 0; e < 4; e++) ss += v[i][e] * v[i][e];
    ss = wave_sum(ss);
    if ((t & 63) == 0) red[t >> 6] = ss;
    __syncthreads();
    const float rs = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / n + eps);
#pragma unroll
    for (int i = 0; i < NC; i++) {
        const int c = (i * 256 + t) * 4;
        u16 o[4];
        for (int e = 0; e < 4; e++) o[e] = f2h(v[i][e] * rs * h2f((u16)(w[i][e >> 1] >> (16 * (e & 1)))));
        if (c + 4 <= ncols) {
            *reinterpret_cast<u32x2u*>(y + c) = u32x2{o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16)};
        } else {
            for (int e = 0; e < 4; e++)
                if (c + e < ncols) y[c + e] = o[e];
        }
    }
}

// llm.tl rmsnorm / rmsnorm_rows over f32 rows of ncols <= 1024 NC columns;
// idx (rmsnorm_rows) gathers the input row.
template <int NC>
__global__ __launch_bounds__(256) void rmsnorm_wg_kernel(const float* __restrict__ X, const int* __restrict__ idx,
                                                         int xrows, const u16* __restrict__ W, u16* __restrict__ Y,
                                                         int C, int ncols, float n, float eps) {
    __shared__ float red[4];
    TSL_POISON(red);
    const int t = threadIdx.x, row = blockIdx.x;
    const int src = idx ? idx[row] : row;
    const bool rin = src >= 0 && src < xrows;
    const float* x = X + (size_t)(rin ? src : 0) * C;
    float4v v[NC];
    u32x2 w[NC];
#pragma unroll
    for (int i = 0; i < NC; i++) {
        const int c = (i * 256 + t) * 4;
        if (rin && c + 4 <= ncols) {
            v[i] = load4(x + c);
        } else {
            for (int e = 0; e < 4; e++) v[i][e] = rin && c + e < ncols ? x[c + e] : 0.0f;
        }
    }
    rms_wg_weights<NC>(W, t, ncols, w);
    rms_wg_finish<NC>(v, w, t, ncols, n, eps, Y + (size_t)row * C, red);
}

// Rows of ncols <= 256 NV columns that are no multiple of 4: a wavefront each, 4
// rows per workgroup. A workgroup per row leaves most of its lanes without a
// column (400000 x 33 302 us so, 70 here; 100000 x 301 80, 36); rows in fours
// keep rmsnorm_wg_kernel, whose sums the fused residual projections share.
template <int NV>
__global__ __launch_bounds__(256) void rmsnorm_wave_kernel(const float* __restrict__ X, const int* __restrict__ idx,
                                                           int xrows, const u16* __restrict__ W, u16* __restrict__ Y,
                                                           int R, int C, int ncols, float n, float eps) {
    const int lane = threadIdx.x & 63, row = blockIdx.x * ROWS_PER_WG + (threadIdx.x >> 6);
    if (row >= R) return;
    const int src = idx ? idx[row] : row;
    const bool rin = src >= 0 && src < xrows;
    const float* x = X + (size_t)(rin ? src : 0) * C;
    u16* y = Y + (size_t)row * C;
    float4v v[NV];
    u32x2 w[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = (i * 64 + lane) * 4;
        if (c + 4 <= ncols) {
            v[i] = rin ? load4(x + c) : float4v{};
            w[i] = load4h(W + c);
        } else {
            uint32_t h[4];
            for (int e = 0; e < 4; e++) {
                v[i][e] = rin && c + e < ncols ? x[c + e] : 0.0f;
                h[e] = c + e < ncols ? W[c + e] : 0;
            }
            w[i] = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
        }
    }
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; i++)
        for (int e = 0; e < 4; e++) ss += v[i][e] * v[i][e];
    const float rs = 1.0f / sqrtf(wave_sum(ss) / n + eps);
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = (i * 64 + lane) * 4;
        uint32_t o[4];
        for (int e = 0; e < 4; e++) o[e] = f2h(v[i][e] * rs * h2f((u16)(w[i][e >> 1] >> (16 * (e & 1)))));
        if (c + 4 <= ncols) {
            store_out4h(u32x2{o[0] | (o[1] << 16), o[2] | (o[3] << 16)}, y + c);
        } else {
            for (int e = 0; e < 4; e++)
                if (c + e < ncols) y[c + e] = (u16)o[e];
        }
    }
}

// The engine's fused step after a K-split residual projection: R[m] += the
// S slices of part[ks][m], added in slice order as skinny_reduce adds them,
// then Y[m] = rmsnorm(R[m]) W as rmsnorm_wg_kernel computes it, over all C
// columns (C % 4 == 0, C <= 1024 NC): the bits of llm/linear_residual (same
// split) followed by llm/rmsnorm. SU > 0: S == SU, every load of the row
// issued at once; 0: any S.
template <int NC, int SU>
__global__ __launch_bounds__(256) void reduce_rmsnorm_kernel(const float* __restrict__ part, int S,
                                                             float* __restrict__ R, const u16* __restrict__ W,
                                                             u16* __restrict__ Y, int M, int C, float n, float eps) {
    __shared__ float red[4];
    TSL_POISON(red);
    const int t = threadIdx.x, row = blockIdx.x;
    const size_t mc = (size_t)M * C;
    float* r = R + (size_t)row * C;
    const float* pr = part + (size_t)row * C;
    const float4v z = {0.0f, 0.0f, 0.0f, 0.0f};
    float4v old[NC], acc[NC];
    u32x2 w[NC];
#pragma unroll
    for (int i = 0; i < NC; i++) {
        const int c = (i * 256 + t) * 4;
        old[i] = c < C ? *reinterpret_cast<const float4v*>(r + c) : z;
        acc[i] = z;
    }
    rms_wg_weights<NC>(W, t, C, w);
    auto slice = [&](int ks) {
#pragma unroll
        for (int i = 0; i < NC; i++) {
            const int c = (i * 256 + t) * 4;
            if (c < C) acc[i] += *reinterpret_cast<const float4v*>(pr + ks * mc + c);
        }
    };
    if constexpr (SU > 0) {
#pragma unroll
        for (int ks = 0; ks < SU; ks++) slice(ks);
    } else {
        for (int ks = 0; ks < S; ks++) slice(ks);
    }
#pragma unroll
    for (int i = 0; i < NC; i++) {
        const int c = (i * 256 + t) * 4;
        if (c < C) {
            old[i] += acc[i];
            *reinterpret_cast<float4v*>(r + c) = old[i];
        }
    }
    rms_wg_finish<NC>(old, w, t, C, n, eps, Y + (size_t)row * C, red);
}

// Rows longer than the kernels above hold: a workgroup per row, the sum of
// squares, then a second, cache-resident pass for the writes.
constexpr int RML_THREADS = 1024;
template <typename XT>
__global__ __launch_bounds__(RML_THREADS) void rmsnorm_long_kernel(const XT* __restrict__ X,
                                                                   const int* __restrict__ idx, int xrows,
                                                                   const u16* __restrict__ W, u16* __restrict__ Y,
                                                                   int C, int ncols, float n, float eps) {
    __shared__ float red[RML_THREADS / 64];
    TSL_POISON(red);
    const int row = blockIdx.x;
    const int src = idx ? idx[row] : row;
    const bool rin = src >= 0 && src < xrows;
    const XT* x = X + (size_t)(rin ? src : 0) * C;
    u16* y = Y + (size_t)row * C;
    auto ld = [&](int c) -> float {
        if (!rin) return 0.0f;
        if constexpr (sizeof(XT) == 2) return h2f(x[c]);
        else return x[c];
    };
    // Four columns of this thread's chunk at c (zeros past the row).
    auto load = [&](int c, float (&v)[4]) {
        if (rin && c + 4 <= ncols) {
            if constexpr (sizeof(XT) == 2) {
                const u32x2 q = load4h(x + c);
                for (int e = 0; e < 4; e++) v[e] = h2f((u16)(q[e >> 1] >> (16 * (e & 1))));
            } else {
                const float4v q = load4(x + c);
                for (int e = 0; e < 4; e++) v[e] = q[e];
            }
        } else {
            for (int e = 0; e < 4; e++) v[e] = c + e < ncols ? ld(c + e) : 0.0f;
        }
    };
    float ss = 0.0f, v[4];
    for (int c = threadIdx.x * 4; c < ncols; c += RML_THREADS * 4) {
        load(c, v);
        for (int e = 0; e < 4; e++) ss += v[e] * v[e];
    }
    const float rs = 1.0f / sqrtf(wg_reduce<RML_THREADS, false>(ss, red) / n + eps);
    for (int c = threadIdx.x * 4; c < ncols; c += RML_THREADS * 4) {
        load(c, v);
        for (int e = 0; e < 4; e++)
            if (c + e < ncols) y[c + e] = f2h(v[e] * rs * h2f(W[c + e]));
    }
}

// Rows per launch: a launch holds fewer than 2^32 work-items, 1024 a row at most.
constexpr long ROWS_MAX = (1L << 22) - 4;
// go(first row, rows) over R rows.
template <class F>
int by_rows(long R, const char* what, F go) {
    for (long r0 = 0; r0 < R; r0 += ROWS_MAX) {
        go(r0, (int)std::min(ROWS_MAX, R - r0));
        if (int e = TSL_LAUNCHED(what)) return e;
    }
    return 0;
}

template <typename XT>
int run_rmsnorm(const XT* X, const int* idx, int xrows, const u16* W, u16* Y, int R, int C, int ncols, float eps,
                hipStream_t s, const char* what) {
    const float n = (float)C;
    auto x = [&](long r0) { return idx ? X : X + r0 * C; };
    auto ix = [&](long r0) { return idx ? idx + r0 : nullptr; };
    if constexpr (sizeof(XT) == 4) {
        auto go = [&](auto nc) {
            return by_rows(R, what, [&](long r0, int rows) {
                hipLaunchKernelGGL(rmsnorm_wg_kernel<decltype(nc)::value>, dim3(rows), dim3(256), 0, s, x(r0), ix(r0),
                                   xrows, W, Y + r0 * C, C, ncols, n, eps);
            });
        };
        auto wave = [&](auto nv) {
            return by_rows(R, what, [&](long r0, int rows) {
                hipLaunchKernelGGL(rmsnorm_wave_kernel<decltype(nv)::value>, dim3((rows + ROWS_PER_WG - 1) / ROWS_PER_WG),
                                   dim3(256), 0, s, x(r0), ix(r0), xrows, W, Y + r0 * C, rows, C, ncols, n, eps);
            });
        };
        if (C % 4 && ncols <= 256) return wave(std::integral_constant<int, 1>{});
        if (C % 4 && ncols <= 512) return wave(std::integral_constant<int, 2>{});
        if (ncols <= 1024) return go(std::integral_constant<int, 1>{});
        if (ncols <= 2048) return go(std::integral_constant<int, 2>{});
        if (ncols <= 4096) return go(std::integral_constant<int, 4>{});
        if (ncols <= 8192) return go(std::integral_constant<int, 8>{});
    } else {
        using std::integral_constant;
        const bool aligned = ((reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(W) |
                               reinterpret_cast<uintptr_t>(Y)) & 15) == 0;
        if (ncols == C && aligned && (C == 2048 || C == 4096)) {
            auto full = [&](auto nv) {
                return by_rows(R, what, [&](long r0, int rows) {
                    hipLaunchKernelGGL(rmsnorm_f16_full_kernel<decltype(nv)::value>,
                                       dim3((rows + ROWS_PER_WG - 1) / ROWS_PER_WG), dim3(256), 0, s, x(r0), W, Y + r0 * C,
                                       rows, C, n, eps);
                });
            };
            return C == 2048 ? full(integral_constant<int, 4>{}) : full(integral_constant<int, 8>{});
        }
        auto go = [&](auto nt, auto nv) {
            constexpr int NT = decltype(nt)::value, NV = decltype(nv)::value;
            return by_rows(R, what, [&](long r0, int rows) {
                hipLaunchKernelGGL((rmsnorm_f16_kernel<NT, NV>),
                                   dim3(NT == 64 ? (rows + ROWS_PER_WG - 1) / ROWS_PER_WG : rows),
                                   dim3(NT < 256 ? 256 : NT), 0, s, x(r0), W, Y + r0 * C, rows, C, ncols, n, eps);
            });
        };
        if (ncols <= 1024) return go(integral_constant<int, 64>{}, integral_constant<int, 2>{});
        if (ncols <= 2048) return go(integral_constant<int, 64>{}, integral_constant<int, 4>{});
        // (a wavefront per row once the rows fill the chip: 4096 x 3001 13.4 us
        // with a workgroup per row, 10.8 with a wavefront; 2000 x 3000 5.7, 7.0)
        if (ncols <= 4096 && R >= 3000) return go(integral_constant<int, 64>{}, integral_constant<int, 8>{});
        if (ncols <= 4096) return go(integral_constant<int, 256>{}, integral_constant<int, 2>{});
        if (ncols <= 8192) return go(integral_constant<int, 256>{}, integral_constant<int, 4>{});
        if (ncols <= 16384) return go(integral_constant<int, 512>{}, integral_constant<int, 4>{});
        if (ncols <= 32768) return go(integral_constant<int, 1024>{}, integral_constant<int, 4>{});
    }
    return by_rows(R, what, [&](long r0, int rows) {
        hipLaunchKernelGGL((rmsnorm_long_kernel<XT>), dim3(rows), dim3(RML_THREADS), 0, s, x(r0), ix(r0), xrows, W,
                           Y + r0 * C, C, ncols, n, eps);
    });
}

// ---------------------------------------------------------------- add, embed

__global__ __launch_bounds__(256) void add_kernel(const float* __restrict__ X, const float* __restrict__ Y,
                                                  float* __restrict__ Z, long n) {
    long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i + 4 <= n) {
        float4v a = *reinterpret_cast<const float4v*>(X + i), b = *reinterpret_cast<const float4v*>(Y + i);
        *reinterpret_cast<float4v*>(Z + i) = a + b;
    } else {
        for (; i < n; i++) Z[i] = X[i] + Y[i];
    }
}

// X[t, :] = f32(E[tok[t], :]); a token outside [0, V) reads zeros.
__global__ __launch_bounds__(256) void embed_kernel(const int* __restrict__ tok, const u16* __restrict__ E,
                                                    float* __restrict__ X, int T, int V, int Dm) {
    const int t = blockIdx.y;
    const int row = tok[t];
    const bool in = row >= 0 && row < V;
    for (int c = (blockIdx.x * 256 + threadIdx.x) * 8; c < Dm; c += gridDim.x * 256 * 8) {
        float* x = X + (size_t)t * Dm + c;
        if (c + 8 <= Dm && (Dm % 8) == 0) {
            float4v a, b;
            if (in) {
                u32x4 h = *reinterpret_cast<const u32x4*>(E + (size_t)row * Dm + c);
                for (int e = 0; e < 4; e++) a[e] = h2f((u16)(h[e >> 1] >> (16 * (e & 1))));
                for (int e = 0; e < 4; e++) b[e] = h2f((u16)(h[2 + (e >> 1)] >> (16 * (e & 1))));
            } else {
                a = float4v{0, 0, 0, 0};
                b = a;
            }
            *reinterpret_cast<float4v*>(x) = a;
            *reinterpret_cast<float4v*>(x + 4) = b;
        } else {
            for (int e = 0; e < 8 && c + e < Dm; e++) x[e] = in ? h2f(E[(size_t)row * Dm + c + e]) : 0.0f;
        }
    }
}

// ---------------------------------------------------------------- rotary
// rope_q: Q[t, h, i] = x1 c - x2 s and Q[t, h, D2 + i] = x2 c + x1 s with
// x1 = QKV[t, h D + i], x2 = QKV[t, h D + D2 + i], (c, s) at pos[t].
struct RopeArgs {
    const u16* QKV;
    const int *pos, *slot;
    const float *Cs, *Sn;
    u16* Q;
    u16 *Kc, *Vc, *K, *V;
    int T, W, NPOS, D2, H, NS, G, D;
};

// Element e of rope_q's T x H x D2 index space.
TSL_DEV void rope_q_elem(const RopeArgs& a, long e) {
    const int i = e % a.D2, h = (e / a.D2) % a.H, t = e / ((long)a.D2 * a.H);
    const int p = a.pos[t];
    const bool pin = p >= 0 && p < a.NPOS;
    const float c = pin ? a.Cs[(size_t)p * a.D2 + i] : 0.0f, s = pin ? a.Sn[(size_t)p * a.D2 + i] : 0.0f;
    const int c1 = h * a.D + i, c2 = h * a.D + a.D2 + i;
    const float x1 = c1 < a.W ? h2f(a.QKV[(size_t)t * a.W + c1]) : 0.0f;
    const float x2 = c2 < a.W ? h2f(a.QKV[(size_t)t * a.W + c2]) : 0.0f;
    u16* q = a.Q + ((size_t)t * a.H + h) * a.D;
    u16 y1, y2;
    rope_rotate(x1, x2, c, s, y1, y2);
    if (i < a.D) q[i] = y1;
    if (a.D2 + i < a.D) q[a.D2 + i] = y2;
}

// kv_write: the rotated keys and the values of kv head g into the paged
// cache at slot[t] (dropped when outside [0, NS)) and into K, V [T, G, D].
// Element e of its T x G x max(D2, D) index space.
TSL_DEV void kv_write_elem(const RopeArgs& a, long e) {
    const int nd = a.D2 > a.D ? a.D2 : a.D;
    const int i = e % nd, g = (e / nd) % a.G, t = e / ((long)nd * a.G);
    const int p = a.pos[t], at = a.slot[t];
    const bool pin = p >= 0 && p < a.NPOS, ain = at >= 0 && at < a.NS;
    const long k0 = (long)a.W - 2L * a.G * a.D + (long)g * a.D;
    u16* kc = a.Kc + ((size_t)(ain ? at : 0) * a.G + g) * a.D;
    u16* vc = a.Vc + ((size_t)(ain ? at : 0) * a.G + g) * a.D;
    u16* kk = a.K + ((size_t)t * a.G + g) * a.D;
    u16* vv = a.V + ((size_t)t * a.G + g) * a.D;
    if (i < a.D2) {
        const float c = pin ? a.Cs[(size_t)p * a.D2 + i] : 0.0f, s = pin ? a.Sn[(size_t)p * a.D2 + i] : 0.0f;
        const long c1 = k0 + i, c2 = k0 + a.D2 + i;
        const float x1 = (c1 >= 0 && c1 < a.W) ? h2f(a.QKV[(size_t)t * a.W + c1]) : 0.0f;
        const float x2 = (c2 >= 0 && c2 < a.W) ? h2f(a.QKV[(size_t)t * a.W + c2]) : 0.0f;
        u16 y1, y2;
        rope_rotate(x1, x2, c, s, y1, y2);
        if (i < a.D) {
            if (ain) kc[i] = y1;
            kk[i] = y1;
        }
        if (a.D2 + i < a.D) {
            if (ain) kc[a.D2 + i] = y2;
            kk[a.D2 + i] = y2;
        }
    }
    if (i < a.D) {
        const long cv = k0 + (long)a.G * a.D + i;
        const u16 v = (cv >= 0 && cv < a.W) ? a.QKV[(size_t)t * a.W + cv] : (u16)0;
        if (ain) vc[i] = v;
        vv[i] = v;
    }
}

// rope_q and kv_write together, 8 columns per thread: item e = (t, head
// slot hh of the H query, G key and G value heads of QKV's row, chunk c of
// D2 / 8). Query and key slots rotate columns 8c .. 8c+7 with their D2
// partners (16-byte loads and stores, the same rope_rotate arithmetic as
// the element kernels, so the same bits); value slots copy both chunks. For
// D = 2 D2, D2 % 8 == 0, W = (H + 2 G) D and 32-bit indices.
__global__ __launch_bounds__(256) void rope_kv_vec(RopeArgs a, int n) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int nc = a.D2 / 8, slots = a.H + 2 * a.G;
    const int c = e % nc, hh = (e / nc) % slots, t = e / (nc * slots);
    const int i0 = 8 * c;
    const u16* row = a.QKV + (size_t)t * a.W + hh * a.D;
    const u32x4 v1 = *reinterpret_cast<const u32x4*>(row + i0), v2 = *reinterpret_cast<const u32x4*>(row + a.D2 + i0);
    const int at = a.slot ? a.slot[t] : -1;
    const bool ain = at >= 0 && at < a.NS;
    if (hh >= a.H + a.G) {  // a value head: copied
        const int g = hh - a.H - a.G;
        u16* vv = a.V + ((size_t)t * a.G + g) * a.D;
        *reinterpret_cast<u32x4*>(vv + i0) = v1;
        *reinterpret_cast<u32x4*>(vv + a.D2 + i0) = v2;
        if (ain) {
            u16* vc = a.Vc + ((size_t)at * a.G + g) * a.D;
            *reinterpret_cast<u32x4*>(vc + i0) = v1;
            *reinterpret_cast<u32x4*>(vc + a.D2 + i0) = v2;
        }
        return;
    }
    const int p = a.pos[t];
    const bool pin = p >= 0 && p < a.NPOS;
    float cs[8], sn[8];
    if (pin) {
        const float4v* cp = reinterpret_cast<const float4v*>(a.Cs + (size_t)p * a.D2 + i0);
        const float4v* sp = reinterpret_cast<const float4v*>(a.Sn + (size_t)p * a.D2 + i0);
        const float4v c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            cs[j] = c0[j], cs[4 + j] = c1[j];
            sn[j] = s0[j], sn[4 + j] = s1[j];
        }
    } else {
#pragma unroll
        for (int j = 0; j < 8; j++) cs[j] = sn[j] = 0.0f;
    }
    u32x4 y1, y2;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        u16 a1, a2, b1, b2;
        rope_rotate(h2f((u16)(v1[j] & 0xffff)), h2f((u16)(v2[j] & 0xffff)), cs[2 * j], sn[2 * j], a1, a2);
        rope_rotate(h2f((u16)(v1[j] >> 16)), h2f((u16)(v2[j] >> 16)), cs[2 * j + 1], sn[2 * j + 1], b1, b2);
        y1[j] = (uint32_t)a1 | ((uint32_t)b1 << 16);
        y2[j] = (uint32_t)a2 | ((uint32_t)b2 << 16);
    }
    if (hh < a.H) {
        u16* q = a.Q + ((size_t)t * a.H + hh) * a.D;
        *reinterpret_cast<u32x4*>(q + i0) = y1;
        *reinterpret_cast<u32x4*>(q + a.D2 + i0) = y2;
        return;
    }
    const int g = hh - a.H;
    u16* kk = a.K + ((size_t)t * a.G + g) * a.D;
    *reinterpret_cast<u32x4*>(kk + i0) = y1;
    *reinterpret_cast<u32x4*>(kk + a.D2 + i0) = y2;
    if (ain) {
        u16* kc = a.Kc + ((size_t)at * a.G + g) * a.D;
        *reinterpret_cast<u32x4*>(kc + i0) = y1;
        *reinterpret_cast<u32x4*>(kc + a.D2 + i0) = y2;
    }
}

// KIND 0: rope_q, 1: kv_write, 2: both (the engine's fused step; the index
// space of rope_q first, then kv_write's).
template <int KIND>
__global__ __launch_bounds__(256) void rope_kernel(RopeArgs a, long nq, long nkv) {
    const long n = nq + nkv;
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < n; e += (long)gridDim.x * 256) {
        if (KIND == 0 || (KIND == 2 && e < nq)) rope_q_elem(a, e);
        else kv_write_elem(a, e - nq);
    }
}

// ---------------------------------------------------------------- argmax
// out[r] = argmax (src/llm/mod.rs:132-140) of row r of X [B, V]: the index
// the sequential scan `if x[i] > x[best] { best = i }` ends on. So a NaN at
// index 0 is the answer (nothing compares greater), later NaNs never are,
// and otherwise it is the first index of the largest value (+0 and -0 tie).
// A workgroup per row (1024 threads, 8 loads in flight each): each thread
// scans its float4 chunks in ascending order, then (value, index) pairs
// meet in a tree that keeps the larger value, the lower index on ties.

// Keeps the better of (bv, bi) and (v, i): i == INT_MAX is no candidate;
// candidates are never NaN.
TSL_DEV void am_pick(float& bv, int& bi, float v, int i) {
    if (i == INT_MAX) return;
    if (bi == INT_MAX || v > bv || (v == bv && i < bi)) {
        bv = v;
        bi = i;
    }
}

constexpr int AM_THREADS = 1024, AM_UNROLL = 8;  // a 32000-float row in one round of loads
__global__ __launch_bounds__(AM_THREADS) void argmax_kernel(const float* __restrict__ X, int V, int* __restrict__ out) {
    constexpr int NW = AM_THREADS / 64;
    __shared__ float rv[NW];
    __shared__ int ri[NW];
    TSL_POISON(rv); TSL_POISON(ri);
    const int tid = threadIdx.x;
    const float* x = X + (size_t)blockIdx.x * V;
    float bv = 0.0f;
    int bi = INT_MAX;  // no candidate yet
    auto see = [&](float v, int i) {
        if (v == v && (bi == INT_MAX || v > bv)) {  // ascending i: strict > keeps the first
            bv = v;
            bi = i;
        }
    };
    if ((V & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0) {
        const int nc = V / 4;
        for (int c0 = tid; c0 < nc; c0 += AM_THREADS * AM_UNROLL) {
            float4v q[AM_UNROLL];
#pragma unroll
            for (int u = 0; u < AM_UNROLL; u++) {
                const int c = c0 + u * AM_THREADS;
                q[u] = c < nc ? *reinterpret_cast<const float4v*>(x + 4 * c) : float4v{};
            }
#pragma unroll
            for (int u = 0; u < AM_UNROLL; u++) {
                const int c = c0 + u * AM_THREADS;
                if (c < nc)
                    for (int e = 0; e < 4; e++) see(q[u][e], 4 * c + e);
            }
        }
    } else {
        for (int c = tid; c < V; c += AM_THREADS) see(x[c], c);
    }
    // Within each 16-lane row by DPP (value and index moved together), then
    // the four rows by readlane: registers only.
    auto step = [&](auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        const float ov = dpp<C>(bv);
        const int oi = __builtin_amdgcn_mov_dpp(bi, C, 0xf, 0xf, false);
        am_pick(bv, bi, ov, oi);
    };
    step(std::integral_constant<int, DPP_XOR1>{});
    step(std::integral_constant<int, DPP_XOR2>{});
    step(std::integral_constant<int, DPP_HALF_MIRROR>{});
    step(std::integral_constant<int, DPP_MIRROR>{});
    for (int r = 16; r < 64; r += 16)
        am_pick(bv, bi, lane_value(bv, r), __builtin_amdgcn_readlane(bi, r));
    bv = lane_value(bv, 0);  // rows 1..3 were folded into lane 0's pair; every lane takes it
    bi = __builtin_amdgcn_readlane(bi, 0);
    if ((tid & 63) == 0) {
        rv[tid >> 6] = bv;
        ri[tid >> 6] = bi;
    }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < NW; w++) am_pick(bv, bi, rv[w], ri[w]);
        const float x0 = x[0];
        out[blockIdx.x] = (x0 != x0 || bi == INT_MAX) ? 0 : bi;
    }
}

int grid1(long n) {
    long g = (n + 255) / 256;
    return (int)(g < 1 ? 1 : (g > 65535 * 4 ? 65535 * 4 : g));
}

}  // namespace

// ---------------------------------------------------------------- launchers

int launch_softmax(TslKernel& k, const uint64_t* a, hipStream_t s) {
    int R = k.dim("R"), C = k.dim("C");
    int ncols = (int)std::min<int64_t>(k.metav("BC"), C);
    const float* X = P<float>(a[0]);
    float* Y = P<float>(a[1]);
    return by_rows(R, "softmax", [&](long r0, int rows) {
        const float* x = X + r0 * C;
        float* y = Y + r0 * C;
        if (ncols <= 256)  // (with the three chunks past the row 400000 x 33 128 us, 90 without; 100000 x 64 32.6, 18.4)
            hipLaunchKernelGGL((softmax_kernel<1>), dim3((rows + ROWS_PER_WG - 1) / ROWS_PER_WG), dim3(256), 0, s, x, y, rows,
                               C, ncols);
        else if (ncols <= 1024)
            hipLaunchKernelGGL((softmax_kernel<4>), dim3((rows + ROWS_PER_WG - 1) / ROWS_PER_WG), dim3(256), 0, s, x, y, rows,
                               C, ncols);
        else if (ncols == 4096 && R >= 1500)
            // Whole 4096-column rows, enough of them to fill the chip: a wavefront
            // per row, two rows per workgroup (4096^2 from HBM: 1 / 2 / 4 / 8 rows
            // per workgroup 23.3 / 22.9 / 23.3 / 23.5 us).
            hipLaunchKernelGGL((softmax_kernel<16, 2>), dim3((rows + 1) / 2), dim3(128), 0, s, x, y, rows, C, ncols);
        else if (ncols <= 4096)
            hipLaunchKernelGGL((softmax_wg_kernel<256, 4>), dim3(rows), dim3(256), 0, s, x, y, C, ncols);
        else if (ncols <= 8192)
            hipLaunchKernelGGL((softmax_wg_kernel<256, 8>), dim3(rows), dim3(256), 0, s, x, y, C, ncols);
        else if (ncols <= 16384)
            hipLaunchKernelGGL((softmax_wg_kernel<512, 8>), dim3(rows), dim3(512), 0, s, x, y, C, ncols);
        else if (ncols <= 32768)
            hipLaunchKernelGGL((softmax_wg_kernel<1024, 8>), dim3(rows), dim3(1024), 0, s, x, y, C, ncols);
        else
            hipLaunchKernelGGL(softmax_long_kernel, dim3(rows), dim3(SML_THREADS), 0, s, x, y, C, ncols);
    });
}

int launch_rmsnorm_basic(TslKernel& k, const uint64_t* a, hipStream_t s) {
    int R = k.dim("R"), C = k.dim("C");
    int ncols = (int)std::min<int64_t>(k.metav("BC"), C);
    return run_rmsnorm<u16>(P<u16>(a[0]), nullptr, R, P<u16>(a[1]), P<u16>(a[2]), R, C, ncols, arg_f32(a[3]), s,
                            "rmsnorm");
}

int launch_add(TslKernel& k, const uint64_t* a, hipStream_t s) {
    long N = k.dim("N");
    if (N == 0) return 0;
    hipLaunchKernelGGL(add_kernel, dim3((unsigned)((N + 1023) / 1024)), dim3(256), 0, s, P<float>(a[0]),
                       P<float>(a[1]), P<float>(a[2]), N);
    return TSL_LAUNCHED("add");
}

int launch_embed(TslKernel& k, const uint64_t* a, hipStream_t s) {
    int T = k.dim("T"), V = k.dim("V"), Dm = k.dim("Dm");
    if (T == 0) return 0;
    dim3 grid((Dm + 2047) / 2048, T);
    hipLaunchKernelGGL(embed_kernel, grid, dim3(256), 0, s, P<int>(a[0]), P<u16>(a[1]), P<float>(a[2]), T, V, Dm);
    return TSL_LAUNCHED("embed");
}

// For the fused residual projection (gemm.hip): R += the S slices of part,
// then Y = rmsnorm(R) W (C % 4 == 0, C <= 4096; reduce_rmsnorm_kernel).
bool reduce_rmsnorm_fits(int C) { return C > 0 && C % 4 == 0 && C <= 4096; }
int run_reduce_rmsnorm(const float* part, int S, float* R, const u16* W, u16* Y, int M, int C, float eps,
                       hipStream_t s) {
    if (M == 0) return 0;
    auto go = [&](auto nc) {
        constexpr int NC = decltype(nc)::value;
        auto k = [&](auto su) {
            hipLaunchKernelGGL((reduce_rmsnorm_kernel<NC, decltype(su)::value>), dim3(M), dim3(256), 0, s, part, S, R,
                               W, Y, M, C, (float)C, eps);
        };
        switch (S) {
            case 2: k(std::integral_constant<int, 2>{}); break;
            case 3: k(std::integral_constant<int, 3>{}); break;
            case 4: k(std::integral_constant<int, 4>{}); break;
            default: k(std::integral_constant<int, 0>{}); break;
        }
    };
    if (C <= 1024) go(std::integral_constant<int, 1>{});
    else if (C <= 2048) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 4>{});
    return TSL_LAUNCHED("linear_residual_rmsnorm");
}
// llm/rmsnorm over f32 rows, for the fused projection's unsplit path.
int run_rmsnorm_f32(const float* X, const u16* W, u16* Y, int M, int C, int ncols, float eps, hipStream_t s) {
    return run_rmsnorm<float>(X, nullptr, M, W, Y, M, C, ncols, eps, s, "linear_residual_rmsnorm");
}

int launch_llm_rmsnorm(TslKernel& k, const uint64_t* a, hipStream_t s) {
    int T = k.dim("T"), Dm = k.dim("Dm");
    int ncols = (int)std::min<int64_t>(k.metav("BC"), Dm);
    return run_rmsnorm<float>(P<float>(a[0]), nullptr, T, P<u16>(a[1]), P<u16>(a[2]), T, Dm, ncols, arg_f32(a[3]), s,
                              "rmsnorm");
}

int launch_rmsnorm_rows(TslKernel& k, const uint64_t* a, hipStream_t s) {
    int T = k.dim("T"), B = k.dim("B"), Dm = k.dim("Dm");
    int ncols = (int)std::min<int64_t>(k.metav("BC"), Dm);
    return run_rmsnorm<float>(P<float>(a[0]), P<int>(a[1]), T, P<u16>(a[2]), P<u16>(a[3]), B, Dm, ncols,
                              arg_f32(a[4]), s, "rmsnorm_rows");
}

// fused/argmax (the engine's scheduler, not a .tl kernel): X [B, V] -> T [B].
int launch_argmax(TslKernel& k, const uint64_t* a, hipStream_t s) {
    const int B = k.dim("B"), V = k.dim("V");
    if (B == 0) return 0;
    if (V == 0) return tsl_fail(-2, "argmax: rows of 0 values");
    hipLaunchKernelGGL(argmax_kernel, dim3(B), dim3(AM_THREADS), 0, s, P<float>(a[0]), V, P<int>(a[1]));
    return TSL_LAUNCHED("argmax");
}

int launch_rope_q(TslKernel& k, const uint64_t* a, hipStream_t s) {
    RopeArgs r{};
    r.T = k.dim("T"), r.W = k.dim("W"), r.NPOS = k.dim("NPOS"), r.D2 = k.dim("D2"), r.H = k.dim("H"), r.D = k.dim("D");
    r.QKV = P<u16>(a[0]), r.pos = P<int>(a[1]), r.Cs = P<float>(a[2]), r.Sn = P<float>(a[3]), r.Q = P<u16>(a[4]);
    const long nq = (long)r.T * r.H * r.D2;
    if (nq == 0) return 0;
    hipLaunchKernelGGL(rope_kernel<0>, dim3(grid1(nq)), dim3(256), 0, s, r, nq, 0L);
    return TSL_LAUNCHED("rope_q");
}

int launch_kv_write(TslKernel& k, const uint64_t* a, hipStream_t s) {
    RopeArgs r{};
    r.T = k.dim("T"), r.W = k.dim("W"), r.NPOS = k.dim("NPOS"), r.D2 = k.dim("D2"), r.NS = k.dim("NS");
    r.G = k.dim("G"), r.D = k.dim("D");
    r.QKV = P<u16>(a[0]), r.pos = P<int>(a[1]), r.slot = P<int>(a[2]), r.Cs = P<float>(a[3]), r.Sn = P<float>(a[4]);
    r.Kc = P<u16>(a[5]), r.Vc = P<u16>(a[6]), r.K = P<u16>(a[7]), r.V = P<u16>(a[8]);
    const long nkv = (long)r.T * r.G * std::max(r.D2, r.D);
    if (nkv == 0) return 0;
    hipLaunchKernelGGL(rope_kernel<1>, dim3(grid1(nkv)), dim3(256), 0, s, r, 0L, nkv);
    return TSL_LAUNCHED("kv_write");
}

// fused/rope_kv: rope_q and kv_write of the same step in one launch (the
// engine's decode and prefill steps; not a .tl kernel). Arguments: QKV, pos,
// slot, C, S, Q, Kc, Vc, K, V.
int launch_rope_kv(TslKernel& k, const uint64_t* a, hipStream_t s) {
    RopeArgs r{};
    r.T = k.dim("T"), r.W = k.dim("W"), r.NPOS = k.dim("NPOS"), r.D2 = k.dim("D2"), r.H = k.dim("H");
    r.NS = k.dim("NS"), r.G = k.dim("G"), r.D = k.dim("D");
    r.QKV = P<u16>(a[0]), r.pos = P<int>(a[1]), r.slot = P<int>(a[2]), r.Cs = P<float>(a[3]), r.Sn = P<float>(a[4]);
    r.Q = P<u16>(a[5]), r.Kc = P<u16>(a[6]), r.Vc = P<u16>(a[7]), r.K = P<u16>(a[8]), r.V = P<u16>(a[9]);
    const long nq = (long)r.T * r.H * r.D2, nkv = (long)r.T * r.G * std::max(r.D2, r.D);
    if (nq + nkv == 0) return 0;
    const long nvec = (long)r.T * (r.H + 2 * r.G) * (r.D2 / 8);
    const bool aligned = ((reinterpret_cast<uintptr_t>(r.QKV) | reinterpret_cast<uintptr_t>(r.Q) |
                           reinterpret_cast<uintptr_t>(r.Kc) | reinterpret_cast<uintptr_t>(r.Vc) |
                           reinterpret_cast<uintptr_t>(r.K) | reinterpret_cast<uintptr_t>(r.V) |
                           reinterpret_cast<uintptr_t>(r.Cs) | reinterpret_cast<uintptr_t>(r.Sn)) & 15) == 0;
    if (aligned && r.D == 2 * r.D2 && r.D2 % 8 == 0 && r.W == (r.H + 2 * r.G) * r.D && (long)r.T * r.W < (1L << 31) &&
        (long)r.NS * r.G * r.D < (1L << 31) && (long)r.NPOS * r.D2 < (1L << 31)) {
        hipLaunchKernelGGL(rope_kv_vec, dim3((unsigned)((nvec + 255) / 256)), dim3(256), 0, s, r, (int)nvec);
        return TSL_LAUNCHED("rope_kv");
    }
    hipLaunchKernelGGL(rope_kernel<2>, dim3(grid1(nq + nkv)), dim3(256), 0, s, r, nq, nkv);
    return TSL_LAUNCHED("rope_kv");
}
