// LayerNorm forward (saves mean / rstd) and backward.
//
// Replaces torch::nn::LayerNorm as TransformerEncoderLayerImpl builds it
// (reference block/details/transformers/classic.hpp:399-404, final norm :495;
// eps 1e-5, elementwise affine), i.e. ATen native_layer_norm and
// native_layer_norm_backward.
//   forward : x̂ = (x − μ)·rstd, rstd = 1/sqrt(var_biased + eps), y = x̂·γ + β
//   backward: g = dy·γ; dx = rstd·(g − Σg/d − x̂·Σ(g·x̂)/d)
//             dγ = Σ_rows dy·x̂, dβ = Σ_rows dy
// A row of up to 16384 columns belongs to WPR wavefronts (one up to 1024
// columns, more for wider ones, so that a lane holds at most 16 values): its x
// and dy stay in VGPRs, the row sums are DPP wave reductions (and one LDS
// exchange where several waves share a row), and every lane keeps running
// dγ / dβ sums for its columns over the rows it takes.  Blocks write per-block
// column partials; a second kernel reduces them (deterministic order).  Longer
// rows: a block per row, three passes over it, partials per row.
#include "common.hpp"

#include <mutex>

#include <initializer_list>

namespace {

constexpr int kThreads = 256;  // 4 waves
constexpr int kWaves = kThreads / 64;
constexpr int kReduceThreads = 1024;   // column reduction: 16 waves split the partial rows
constexpr int kReduceWaves = kReduceThreads / 64;
constexpr int kReduceUnroll = 32;  // 16 waves x 32 loads cover 512 partial rows in one round

// How a row's columns are dealt to the P = 64·WPR lanes that own it: group g of
// lane t covers columns [(g·P + t)·G, +G).  G is the 16-byte group (4 fp32 / 8
// bf16 elements: a wave access is a 1 KB coalesced run) where every row is
// aligned and whole groups, else 1 (any d, any alignment).
template <typename T, int G> struct Group {
    typedef typename Pack16<T>::Raw Raw;
    static_assert(G == Pack16<T>::N, "a 16-byte group");
    template <bool NT> static __device__ __forceinline__ Raw raw(const T* p) { return Pack16<T>::template raw<NT>(p); }
    static __device__ __forceinline__ void unpack(const Raw& r, float (&v)[G]) { Pack16<T>::unpack(r, v); }
    static __device__ __forceinline__ void st(T* p, const float (&v)[G]) { Pack16<T>::template st<false>(p, v); }
};
template <typename T> struct Group<T, 1> {
    typedef T Raw;
    template <bool NT> static __device__ __forceinline__ Raw raw(const T* p) { return *p; }
    static __device__ __forceinline__ void unpack(const Raw& r, float (&v)[1]) { v[0] = Io<T>::ld(&r, 0); }
    static __device__ __forceinline__ void st(T* p, const float (&v)[1]) { Io<T>::st(p, 0, v[0]); }
};

template <int DPL, int G, int P>
struct Row {
    static constexpr int NG = DPL / G;
    static __device__ __forceinline__ int64_t col(int t, int e) { return ((int64_t)(e / G) * P + t) * G + e % G; }
    // Every lane issues all of its loads unconditionally (columns past d read
    // column 0 and get unpack's `past`), so a row's loads stay in flight
    // together.
    template <typename T, bool NT>
    static __device__ __forceinline__ void load(const T* __restrict__ p, int64_t d, int t,
                                                typename Group<T, G>::Raw (&raw)[NG]) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int64_t c0 = ((int64_t)g * P + t) * G;
            raw[g] = Group<T, G>::template raw<NT>(p + (c0 < d ? c0 : 0));
        }
    }
    template <typename T>
    static __device__ __forceinline__ void unpack(const typename Group<T, G>::Raw (&raw)[NG], int64_t d, int t,
                                                  float (&v)[DPL], float past = 0.f) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int64_t c0 = ((int64_t)g * P + t) * G;
            float x[G];
            Group<T, G>::unpack(raw[g], x);
#pragma unroll
            for (int e = 0; e < G; ++e) v[G * g + e] = c0 < d ? x[e] : past;
        }
    }
    template <typename T, bool NT>
    static __device__ __forceinline__ void load_all(const T* __restrict__ p, int64_t d, int t, float (&v)[DPL]) {
        typename Group<T, G>::Raw raw[NG];
        load<T, NT>(p, d, t, raw);
        unpack<T>(raw, d, t, v);
    }
    template <typename T>
    static __device__ __forceinline__ void store(T* __restrict__ p, int64_t d, int t, const float (&v)[DPL]) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int64_t c0 = ((int64_t)g * P + t) * G;
            float x[G];
#pragma unroll
            for (int e = 0; e < G; ++e) x[e] = v[G * g + e];
            if (c0 < d) Group<T, G>::st(p + c0, x);
        }
    }
};

// Sum over the WPR waves of a row of K values each lane holds.  `red` is this
// use's own LDS, K·WPR floats per row of the block; every thread of the block
// calls it.  Two uses that alternate between two buffers need no other barrier.
template <int WPR, int K>
__device__ __forceinline__ void row_sum(float (&v)[K], float* red) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = wave_sum(v[k]);
    if constexpr (WPR > 1) {
        const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
        float* mine = red + (wid / WPR) * (K * WPR);
        if (lane == 0) {
#pragma unroll
            for (int k = 0; k < K; ++k) mine[k * WPR + wid % WPR] = v[k];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < K; ++k) {
            // pairwise: added one after another, 16 waves' sums made the mean of
            // 16384 columns 1.5 times further from 64 bits
            float s[WPR];
#pragma unroll
            for (int w = 0; w < WPR; ++w) s[w] = mine[k * WPR + w];
#pragma unroll
            for (int n = WPR / 2; n > 0; n /= 2)
#pragma unroll
                for (int w = 0; w < n; ++w) s[w] = s[2 * w] + s[2 * w + 1];
            v[k] = s[0];
        }
    }
}

// s / d given inv = 1 / d: the product, corrected by what it leaves of s (the
// product by itself is up to 1.13 times further from 64 bits in the mean and in
// dx, and a division costs 11% of the forward at 30000 x 64).  Aligned rows of up
// to 1024 columns (SHORT: one wave, 16-byte groups) take the product alone and dy·γ
// rounded; the rest would cost them 4% (30000 x 64 bf16: backward 13.5 against
// 12.9 us).
template <bool SHORT>
__device__ __forceinline__ float over(float s, float d, float inv) {
    const float q = s * inv;
    if constexpr (SHORT) return q;
    const float c = fmaf(fmaf(-q, d, s), inv, q);
    return c == c ? c : q;   // (an infinite sum)
}

// GROUPS rows per block at a time, WPR waves each.  Bound by memory: a call of
// 8192x8192 bf16 46 us (5.9 TB/s), 4096x4096 14.4 us, where three passes of
// single elements per row took 109 and 28.
template <typename T, int DPL, int G, int WPR, int GROUPS>
__global__ __launch_bounds__(64 * WPR * GROUPS) void ln_fwd_kernel(const T* __restrict__ x,
                                                                   const T* __restrict__ gamma,
                                                                   const T* __restrict__ beta, float eps,
                                                                   T* __restrict__ y, float* __restrict__ mean,
                                                                   float* __restrict__ rstd, int64_t rows, int64_t d) {
    constexpr int P = 64 * WPR;
    constexpr bool SHORT = WPR == 1 && G > 1;
    typedef Row<DPL, G, P> R;
    __shared__ float red[2][GROUPS * WPR];
    const int t = threadIdx.x % P, grp = threadIdx.x / P;
    float gm[DPL], bt[DPL];
    R::template load_all<T, false>(gamma, d, t, gm);
    R::template load_all<T, false>(beta, d, t, bt);
    const float fd = (float)d, inv_d = 1.f / fd;
    const int64_t stride = (int64_t)gridDim.x * GROUPS;
    for (int64_t r0 = (int64_t)blockIdx.x * GROUPS; r0 < rows; r0 += stride) {
        const int64_t r = r0 + grp;
        if (WPR == 1 && r >= rows) break;
        const bool in = WPR == 1 || r < rows;
        float v[DPL];
        R::template load_all<T, true>(x + (in ? r : rows - 1) * d, d, t, v);
        float s[1] = {0.f};
#pragma unroll
        for (int e = 0; e < DPL; ++e) s[0] += v[e];
        row_sum<WPR, 1>(s, red[0]);
        const float mu = over<SHORT>(s[0], fd, inv_d);
        s[0] = 0.f;
#pragma unroll
        for (int e = 0; e < DPL; ++e) {
            const float u = R::col(t, e) < d ? v[e] - mu : 0.f;
            s[0] += u * u;
        }
        row_sum<WPR, 1>(s, red[1]);
        const float rs = 1.f / sqrtf(over<SHORT>(s[0], fd, inv_d) + eps);
#pragma unroll
        for (int e = 0; e < DPL; ++e) v[e] = (v[e] - mu) * rs * gm[e] + bt[e];
        if (!in) continue;
        R::template store<T>(y + r * d, d, t, v);
        if (t == 0) {
            mean[r] = mu;
            rstd[r] = rs;
        }
    }
}

// One block per CU, GROUPS rows at a time of WPR waves each, 8 waves in all (16
// past 8192 columns): ordinary loads and stores, with the next row's loads in
// flight while the current row is reduced (measured best at 16384x1024, where
// it streams 5.8 TB/s fp32; wider rows keep the same bytes in flight per CU:
// 4096x4096 bf16 24 us a call, 8192x8192 86 us; past 8192 columns one row at a
// time: 2048x16384 bf16 64 us, fp32 107).  A block per row whose dγ / dβ
// partials were written for every row took 71 and 344 us, and 59 us for 5000x771
// fp32 (19 now).
template <typename T, int DPL, int G, int WPR, int GROUPS>
__global__ __launch_bounds__(64 * WPR * GROUPS) void ln_bwd_kernel(const T* __restrict__ x, const T* __restrict__ dy,
                                                                   const float* __restrict__ mean,
                                                                   const float* __restrict__ rstd,
                                                                   const T* __restrict__ gamma, T* __restrict__ dx,
                                                                   float* __restrict__ partial, int64_t rows,
                                                                   int64_t d) {
    constexpr int P = 64 * WPR, NT = P * GROUPS;
    constexpr bool SHORT = WPR == 1 && G > 1;
    typedef Row<DPL, G, P> R;
    extern __shared__ float lds[];  // [GROUPS][2][d] (one group: unused)
    __shared__ float red[2][GROUPS * WPR * 2];
    // 16 waves leave a lane 128 registers: enough for a row, not for the next one
    // beside it (with it the kernel spilled 19 to 107 registers: 2000 x 10001 bf16
    // 183 us against 39, 2048 x 16384 fp32 174 against 107)
    constexpr bool AHEAD = WPR < 16;
    const int t = threadIdx.x % P, grp = threadIdx.x / P;
    float gm[DPL];
    R::template load_all<T, false>(gamma, d, t, gm);
    float dg[DPL], db[DPL];
#pragma unroll
    for (int e = 0; e < DPL; ++e) dg[e] = db[e] = 0.f;
    const float fd = (float)d, inv_d = 1.f / fd;
    const int64_t stride = (int64_t)gridDim.x * GROUPS;
    // The next row is loaded (raw) while the current one is reduced and
    // stored: two rows' loads per group stay in flight.
    typename Group<T, G>::Raw rx[R::NG], rd[R::NG];
    float nmu = 0.f, nrs = 0.f;
    auto fetch = [&](int64_t r) {
        if (WPR > 1 && GROUPS > 1) r = r < rows ? r : rows - 1;   // (a group past the end re-reads the last row)
        int at = t;
        if constexpr (!AHEAD) asm volatile("" : "+v"(at));   // (its columns are formed here, not kept from row to row)
        R::template load<T, false>(x + r * d, d, at, rx);
        R::template load<T, false>(dy + r * d, d, at, rd);
        nmu = mean[r];
        nrs = rstd[r];
    };
    int buf = 0;
    // A wave that has rows to itself stops with its own last one; waves that share
    // them go on with the block.
    const int64_t own = WPR == 1 ? 0 : grp;   // rows of the block before the one that decides
    const int64_t first = (int64_t)blockIdx.x * GROUPS + grp;
    if (AHEAD && first - own < rows) fetch(first);
    for (int64_t r = first; r - own < rows; r += stride) {
        const bool in = WPR == 1 || r < rows;
        if (!AHEAD) fetch(r);
        float xv[DPL], gv[DPL];
        const float mu = nmu, rs = nrs;
        // columns past d hold the mean: x̂ is 0 there (−μ·rstd may overflow, and
        // times their zero dy it would be a NaN in the row's sums)
        R::template unpack<T>(rx, d, t, xv, mu);
        R::template unpack<T>(rd, d, t, gv);
        if (AHEAD && r + stride - own < rows) fetch(r + stride);
        float s[2] = {0.f, 0.f};
#pragma unroll
        for (int e = 0; e < DPL; ++e) {
            const float xh = (xv[e] - mu) * rs;
            const float dyv = gv[e];
            if (in) {
                dg[e] += dyv * xh;
                db[e] += dyv;
            }
            const float g = dyv * gm[e];
            s[0] += g;
            s[1] += g * xh;
            xv[e] = xh;
            if constexpr (SHORT) gv[e] = g;
        }
        row_sum<WPR, 2>(s, red[buf]);
        buf ^= 1;
        const float sg = over<SHORT>(s[0], fd, inv_d), sgx = over<SHORT>(s[1], fd, inv_d);
#pragma unroll
        for (int e = 0; e < DPL; ++e) {
            float g;
            if constexpr (SHORT) {
                g = gv[e] - sg;
            } else if (WPR == 1 && e == 0 && d == 1) {
                float rounded = gv[e] * gm[e];   // a single column cancels against its own rounded sum
                asm volatile("" : "+v"(rounded));
                g = rounded - sg;
            } else {
                g = fmaf(gv[e], gm[e], -sg);     // dy·γ unrounded
            }
            xv[e] = rs * (g - xv[e] * sgx);
        }
        int at = t;
        if constexpr (!AHEAD) asm volatile("" : "+v"(at));
        if (in) R::template store<T>(dx + r * d, d, at, xv);
    }
    // This block's partial row: layout [which][16-column group][block][16], so
    // that the reduction reads each group's partials as one contiguous run.
    const int64_t ngroups = (d + 15) / 16;
    auto put = [&](int which, int64_t col, float v) {
        partial[((which * ngroups + col / 16) * gridDim.x + blockIdx.x) * 16 + col % 16] = v;
    };
    if constexpr (GROUPS == 1) {
#pragma unroll
        for (int e = 0; e < DPL; ++e) {
            const int64_t col = R::col(t, e);
            if (col < d) {
                put(0, col, dg[e]);
                put(1, col, db[e]);
            }
        }
    } else {
#pragma unroll
        for (int e = 0; e < DPL; ++e) {
            const int64_t col = R::col(t, e);
            if (col < d) {
                lds[(grp * 2 + 0) * d + col] = dg[e];
                lds[(grp * 2 + 1) * d + col] = db[e];
            }
        }
        __syncthreads();
        for (int64_t j = threadIdx.x; j < 2 * d; j += NT) {
            const int which = j >= d;
            const int64_t col = j - which * d;
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < GROUPS; ++w) v += lds[(w * 2 + which) * d + col];
            put(which, col, v);
        }
    }
}

// dgamma / dbeta from ln_bwd_kernel's grouped partials.  One 4-wave block
// per 16-column group of one output: thread = (block row b = tid / 4 mod 64,
// column quad tid % 4), 16-byte loads, kGroupUnroll of them in flight (512
// partial rows in one round), so each wave load reads 1 KB of consecutive
// partials.  Each thread adds its rows in order, the 16 row slots of a wave
// combine by a fixed butterfly and the 4 waves in wave order: the summation
// order does not depend on timing.
constexpr int kGroupUnroll = 8;
__global__ __launch_bounds__(256) void col_reduce_grouped_kernel(const float* __restrict__ partial, int64_t nparts,
                                                                 int64_t d, float* __restrict__ dgamma,
                                                                 float* __restrict__ dbeta, int accumulate) {
    __shared__ f32x4 red[4][4];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int64_t ngroups = (d + 15) / 16;
    const int64_t gi = blockIdx.x;                  // which · ngroups + group
    const int which = gi >= ngroups;
    const int64_t cg = gi - which * ngroups;
    const int q = tid & 3, br = tid >> 2;
    const f32x4* src = reinterpret_cast<const f32x4*>(partial + gi * nparts * 16) + q;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    for (int64_t b0 = 0; b0 < nparts; b0 += 64 * kGroupUnroll) {
        f32x4 t[kGroupUnroll];
#pragma unroll
        for (int u = 0; u < kGroupUnroll; ++u) {
            const int64_t b = b0 + u * 64 + br;
            t[u] = b < nparts ? src[b * 4] : f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int u = 0; u < kGroupUnroll; ++u) s += t[u];
    }
#pragma unroll
    for (int off = 4; off < 64; off <<= 1) {
        s.x += __shfl_xor(s.x, off);
        s.y += __shfl_xor(s.y, off);
        s.z += __shfl_xor(s.z, off);
        s.w += __shfl_xor(s.w, off);
    }
    if (lane < 4) red[wid][lane] = s;
    __syncthreads();
    if (tid >= 4) return;
    s = red[0][q] + red[1][q] + red[2][q] + red[3][q];
    float* out = which ? dbeta : dgamma;
    if (out) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t col = cg * 16 + q * 4 + e;
            if (col < d) out[col] = accumulate ? out[col] + s[e] : s[e];
        }
    }
}

// Sums `nparts` partial rows of 2·d floats into dgamma / dbeta.  A block owns
// 64 columns of one output (lane = column, so every load is a 256-byte
// coalesced run); its 16 waves take the partial rows round-robin, each with
// kReduceUnroll independent loads in flight, and combine in LDS in wave order,
// so the summation order is fixed.
__global__ __launch_bounds__(kReduceThreads) void col_reduce_kernel(const float* __restrict__ partial, int64_t nparts,
                                                                    int64_t d, float* __restrict__ dgamma,
                                                                    float* __restrict__ dbeta, int accumulate) {
    __shared__ float red[kReduceWaves][64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int which = blockIdx.y;
    const int64_t col = (int64_t)blockIdx.x * 64 + lane;
    float s = 0.f;
    if (col < d) {
        const float* src = partial + (int64_t)which * d + col;
        for (int64_t b = wid; b < nparts; b += kReduceUnroll * kReduceWaves) {
            // all kReduceUnroll loads in flight at once (indices past the end
            // re-read the last partial row and are not added)
            float t[kReduceUnroll];
#pragma unroll
            for (int u = 0; u < kReduceUnroll; ++u) {
                const int64_t i = b + u * kReduceWaves;
                t[u] = src[(i < nparts ? i : nparts - 1) * 2 * d];
            }
#pragma unroll
            for (int u = 0; u < kReduceUnroll; ++u) s += (b + u * kReduceWaves < nparts) ? t[u] : 0.f;
        }
    }
    red[wid][lane] = s;
    __syncthreads();
    if (wid == 0 && col < d) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < kReduceWaves; ++w) t += red[w][lane];
        float* out = which ? dbeta : dgamma;
        if (out) out[col] = accumulate ? out[col] + t : t;
    }
}

// Rows past 16384 columns: one block per row, three passes over the row.
template <typename T>
__global__ __launch_bounds__(kThreads) void ln_fwd_generic(const T* __restrict__ x, const T* __restrict__ gamma,
                                                           const T* __restrict__ beta, float eps, T* __restrict__ y,
                                                           float* __restrict__ mean, float* __restrict__ rstd,
                                                           int64_t d) {
    __shared__ float red[kWaves];
    const int64_t r = blockIdx.x;
    const T* xr = x + r * d;
    float s = 0.f;
    for (int64_t j = threadIdx.x; j < d; j += kThreads) s += Io<T>::ld(xr, j);
    const float mu = block_sum<kWaves>(s, red) / (float)d;
    float ss = 0.f;
    for (int64_t j = threadIdx.x; j < d; j += kThreads) {
        const float t = Io<T>::ld(xr, j) - mu;
        ss += t * t;
    }
    const float rs = 1.f / sqrtf(block_sum<kWaves>(ss, red) / (float)d + eps);
    for (int64_t j = threadIdx.x; j < d; j += kThreads)
        Io<T>::st(y + r * d, j, (Io<T>::ld(xr, j) - mu) * rs * Io<T>::ld(gamma, j) + Io<T>::ld(beta, j));
    if (threadIdx.x == 0) {
        mean[r] = mu;
        rstd[r] = rs;
    }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void ln_bwd_generic(const T* __restrict__ x, const T* __restrict__ dy,
                                                           const float* __restrict__ mean,
                                                           const float* __restrict__ rstd, const T* __restrict__ gamma,
                                                           T* __restrict__ dx, float* __restrict__ partial, int64_t d) {
    __shared__ float red[kWaves];
    const int64_t r = blockIdx.x;
    const float mu = mean[r], rs = rstd[r];
    float sg = 0.f, sgx = 0.f;
    for (int64_t j = threadIdx.x; j < d; j += kThreads) {
        const float xh = (Io<T>::ld(x, r * d + j) - mu) * rs;
        const float dyv = Io<T>::ld(dy, r * d + j);
        const float g = dyv * Io<T>::ld(gamma, j);
        sg += g;
        sgx += g * xh;
        partial[(r * 2 + 0) * d + j] = dyv * xh;
        partial[(r * 2 + 1) * d + j] = dyv;
    }
    sg = block_sum<kWaves>(sg, red) / (float)d;
    sgx = block_sum<kWaves>(sgx, red) / (float)d;
    for (int64_t j = threadIdx.x; j < d; j += kThreads) {
        const float xh = (Io<T>::ld(x, r * d + j) - mu) * rs;
        const float g = Io<T>::ld(dy, r * d + j) * Io<T>::ld(gamma, j);
        Io<T>::st(dx, r * d + j, rs * (g - sg - xh * sgx));
    }
}

constexpr int64_t kMaxRegCols = 1024 * 16;   // the widest row held in registers (16 waves)

// 16-byte accesses need 16-byte aligned rows of whole 16-byte groups.
template <typename T>
bool vec_ok(int64_t d, std::initializer_list<const void*> ptrs) {
    if (d % Pack16<T>::N != 0) return false;
    for (const void* p : ptrs)
        if ((uintptr_t)p % 16 != 0) return false;
    return true;
}

// The kernel shape of a row length, as f(DPL, G, WPR constants): the fewest
// waves per row that leave a lane at most 16 values.
template <typename T, int G, class F>
void for_shape_g(int64_t d, F f) {
    constexpr int kLeast = G > 4 ? G : 4;
    if (kLeast == 4 && d <= 64 * 4) f.template operator()<kLeast == 4 ? 4 : 8, G, 1>();
    else if (d <= 64 * 8) f.template operator()<8, G, 1>();
    else if (d <= 64 * 16) f.template operator()<16, G, 1>();
    else if (d <= 128 * 16) f.template operator()<16, G, 2>();
    else if (d <= 256 * 16) f.template operator()<16, G, 4>();
    else if (d <= 512 * 16) f.template operator()<16, G, 8>();
    else f.template operator()<16, G, 16>();
}
template <typename T, class F>
void for_shape(bool vec, int64_t d, F f) {
    if (vec) for_shape_g<T, Pack16<T>::N>(d, f);
    else for_shape_g<T, 1>(d, f);
}

template <typename T>
struct FwdArgs {
    nott_ctx ctx;
    const T *x, *gamma, *beta;
    float eps;
    T* y;
    float *mean, *rstd;
    int64_t rows, d;
    template <int DPL, int G, int WPR>
    void operator()() const {
        constexpr int GROUPS = WPR < kWaves ? kWaves / WPR : 1;
        const int64_t blocks = std::min<int64_t>(nott::ceil_div(rows, GROUPS), (int64_t)ctx->num_cu * 8);
        hipLaunchKernelGGL((ln_fwd_kernel<T, DPL, G, WPR, GROUPS>), dim3((unsigned)blocks), dim3(64 * WPR * GROUPS), 0,
                           ctx->stream, x, gamma, beta, eps, y, mean, rstd, rows, d);
    }
};

template <typename T>
int fwd(nott_ctx ctx, int64_t rows, int64_t d, const void* x, const void* gamma, const void* beta, float eps, void* y,
        float* mean, float* rstd) {
    const FwdArgs<T> a{ctx, static_cast<const T*>(x), static_cast<const T*>(gamma), static_cast<const T*>(beta), eps,
                       static_cast<T*>(y), mean, rstd, rows, d};
    if (d <= kMaxRegCols)
        for_shape<T>(vec_ok<T>(d, {x, gamma, beta, y}), d, a);
    else
        hipLaunchKernelGGL(ln_fwd_generic<T>, dim3((unsigned)rows), dim3(kThreads), 0, ctx->stream, a.x, a.gamma, a.beta,
                           eps, a.y, mean, rstd, d);
    return nott::launch_status(ctx, "layernorm_fwd");
}

// Scratch for the column partials of the allocation-free entry point
// (nott_layernorm_bwd_noalloc): one copy per GPU, alive until the process
// ends.  Host code never passes `scratch` itself to a kernel; it uses the
// device address hipGetSymbolAddress returns for the current device.
constexpr size_t kScratchBytes = size_t(16) << 20;
static __device__ __align__(256) float scratch[kScratchBytes / sizeof(float)];

// Rows a block of the backward takes at a time: 8 waves over the waves per row.
constexpr int bwd_groups(int wpr) { return wpr < 8 ? 8 / wpr : 1; }

template <typename T>
struct BwdArgs {
    nott_ctx ctx;
    const T *x, *dy;
    const float *mean, *rstd;
    const T* gamma;
    T* dx;
    float* partial;
    int64_t rows, d;
    int64_t* nparts;   // in: at most this many blocks (0: plan only); out: blocks
    template <int DPL, int G, int WPR>
    void operator()() const {
        constexpr int GROUPS = bwd_groups(WPR);
        const int64_t most = std::max<int64_t>(
            1, std::min<int64_t>(nott::ceil_div(rows, GROUPS), (int64_t)ctx->num_cu));
        if (!partial) {
            *nparts = most;
            return;
        }
        // at most 64 KB, beside the kernel's own few words
        const size_t lds = GROUPS > 1 ? sizeof(float) * GROUPS * 2 * (size_t)d : 0;
        static bool attr = false;
        if (GROUPS > 1 && !attr) {
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&ln_bwd_kernel<T, DPL, G, WPR, GROUPS>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)(64 << 10));
            attr = true;
        }
        hipLaunchKernelGGL((ln_bwd_kernel<T, DPL, G, WPR, GROUPS>), dim3((unsigned)*nparts), dim3(64 * WPR * GROUPS),
                           lds, ctx->stream, x, dy, mean, rstd, gamma, dx, partial, rows, d);
    }
};

// `fixed` (nullable) replaces the context workspace for the partials;
// `fixed_bytes` is its size.
template <typename T>
int bwd(nott_ctx ctx, int64_t rows, int64_t d, const void* x, const void* dy, const float* mean, const float* rstd,
        const void* gamma, void* dx, float* dgamma, float* dbeta, int accumulate, float* fixed = nullptr,
        size_t fixed_bytes = 0) {
    int64_t nparts = 0;
    BwdArgs<T> a{ctx, static_cast<const T*>(x), static_cast<const T*>(dy), mean, rstd, static_cast<const T*>(gamma),
                 static_cast<T*>(dx), nullptr, rows, d, &nparts};
    const bool vec = vec_ok<T>(d, {x, dy, gamma, dx}), reg = d <= kMaxRegCols;
    // Partials: 2 rows (dgamma, dbeta) of `pcols` columns per block.
    size_t pcols = (size_t)d;
    if (reg) {
        for_shape<T>(vec, d, a);   // the block count
        pcols = (size_t)nott::ceil_div(d, 16) * 16;
    } else {
        nparts = rows;
    }
    if (fixed) {
        // The entry point's bound is 8·d bytes a row outside aligned rows of up
        // to 2048 columns; inside it the blocks' partials fit (fewer blocks where
        // the columns' rounding to 16 would not).
        const size_t bound = vec && d <= 2048 ? 0 : sizeof(float) * 2 * (size_t)d * (size_t)rows;
        if (bound > fixed_bytes)
            return nott::fail(ctx, NOTT_ERR_UNSUPPORTED,
                              "nott_layernorm_bwd_noalloc: rows=" + std::to_string(rows) + ", d=" + std::to_string(d) +
                                  " needs " + std::to_string(bound) + " bytes of scratch; the static scratch holds " +
                                  std::to_string(fixed_bytes));
        if (reg) nparts = std::min<int64_t>(nparts, (int64_t)(fixed_bytes / (sizeof(float) * 2 * pcols)));
        a.partial = fixed;
    } else {
        a.partial = static_cast<float*>(nott::workspace(ctx, sizeof(float) * 2 * pcols * (size_t)nparts));
        if (!a.partial) return NOTT_ERR_ALLOC;
    }
    if (reg)
        for_shape<T>(vec, d, a);
    else
        hipLaunchKernelGGL(ln_bwd_generic<T>, dim3((unsigned)nparts), dim3(kThreads), 0, ctx->stream, a.x, a.dy, mean,
                           rstd, a.gamma, a.dx, a.partial, d);
    if ((dgamma || dbeta) && reg)
        hipLaunchKernelGGL(col_reduce_grouped_kernel, dim3((unsigned)(2 * nott::ceil_div(d, 16))), dim3(256), 0,
                           ctx->stream, a.partial, nparts, d, dgamma, dbeta, accumulate);
    else if (dgamma || dbeta)
        hipLaunchKernelGGL(col_reduce_kernel, dim3((unsigned)nott::ceil_div(d, 64), 2), dim3(kReduceThreads), 0,
                           ctx->stream, a.partial, nparts, d, dgamma, dbeta, accumulate);
    return nott::launch_status(ctx, "layernorm_bwd");
}

}  // namespace

namespace nott {

// Device address of `scratch` on each device, looked up once per device by
// nott_create (the context's device is current there).
int layernorm_scratch_setup(nott_ctx ctx) {
    static std::mutex mu;
    static void* addr[64] = {};
    std::lock_guard<std::mutex> g(mu);
    if (ctx->device < 0 || ctx->device >= 64) return fail(ctx, NOTT_ERR_INVALID_ARG, "device index out of range");
    if (!addr[ctx->device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return hip_fail(ctx, e, "hipGetSymbolAddress(layernorm scratch)");
        addr[ctx->device] = p;
    }
    ctx->ln_scratch = addr[ctx->device];
    return NOTT_OK;
}

}  // namespace nott

extern "C" int nott_layernorm_fwd(nott_ctx ctx, nott_dtype dtype, int64_t rows, int64_t d, const void* x,
                                  const void* gamma, const void* beta, double eps, void* y, float* mean, float* rstd) {
    NOTT_CHECK_CTX(ctx);
    NOTT_REQUIRE(ctx, nott::valid_dtype(dtype) && rows >= 0 && d > 0, "nott_layernorm_fwd: bad arguments");
    if (rows == 0) return NOTT_OK;
    NOTT_REQUIRE(ctx, x && gamma && beta && y && mean && rstd, "nott_layernorm_fwd: null buffer");
    nott::DeviceScope scope(ctx->device);
    return dtype == NOTT_F32 ? fwd<float>(ctx, rows, d, x, gamma, beta, (float)eps, y, mean, rstd)
                             : fwd<bf16_t>(ctx, rows, d, x, gamma, beta, (float)eps, y, mean, rstd);
}

extern "C" int nott_layernorm_bwd(nott_ctx ctx, nott_dtype dtype, int64_t rows, int64_t d, const void* x,
                                  const void* dy, const float* mean, const float* rstd, const void* gamma, void* dx,
                                  float* dgamma, float* dbeta, int accumulate) {
    NOTT_CHECK_CTX(ctx);
    NOTT_REQUIRE(ctx, nott::valid_dtype(dtype) && rows >= 0 && d > 0, "nott_layernorm_bwd: bad arguments");
    NOTT_REQUIRE(ctx, rows == 0 || (x && dy && mean && rstd && gamma && dx), "nott_layernorm_bwd: null buffer");
    nott::DeviceScope scope(ctx->device);
    if (rows == 0) {
        // Σ over no rows: the parameter gradients are zero (or unchanged).
        if (!accumulate) {
            if (dgamma && nott_zero(ctx, sizeof(float) * d, dgamma) != NOTT_OK) return NOTT_ERR_HIP;
            if (dbeta && nott_zero(ctx, sizeof(float) * d, dbeta) != NOTT_OK) return NOTT_ERR_HIP;
        }
        return NOTT_OK;
    }
    return dtype == NOTT_F32 ? bwd<float>(ctx, rows, d, x, dy, mean, rstd, gamma, dx, dgamma, dbeta, accumulate)
                             : bwd<bf16_t>(ctx, rows, d, x, dy, mean, rstd, gamma, dx, dgamma, dbeta, accumulate);
}

extern "C" int nott_layernorm_bwd_noalloc(nott_ctx ctx, nott_dtype dtype, int64_t rows, int64_t d, const void* x,
                                          const void* dy, const float* mean, const float* rstd, const void* gamma,
                                          void* dx, float* dgamma, float* dbeta, int accumulate) {
    NOTT_CHECK_CTX(ctx);
    NOTT_REQUIRE(ctx, nott::valid_dtype(dtype) && rows >= 0 && d > 0, "nott_layernorm_bwd_noalloc: bad arguments");
    NOTT_REQUIRE(ctx, rows == 0 || (x && dy && mean && rstd && gamma && dx), "nott_layernorm_bwd_noalloc: null buffer");
    NOTT_REQUIRE(ctx, ctx->ln_scratch != nullptr, "nott_layernorm_bwd_noalloc: scratch not set up");
    nott::DeviceScope scope(ctx->device);
    if (rows == 0) {
        if (!accumulate) {
            if (dgamma && nott_zero(ctx, sizeof(float) * d, dgamma) != NOTT_OK) return NOTT_ERR_HIP;
            if (dbeta && nott_zero(ctx, sizeof(float) * d, dbeta) != NOTT_OK) return NOTT_ERR_HIP;
        }
        return NOTT_OK;
    }
    float* sp = static_cast<float*>(ctx->ln_scratch);
    return dtype == NOTT_F32
               ? bwd<float>(ctx, rows, d, x, dy, mean, rstd, gamma, dx, dgamma, dbeta, accumulate, sp, kScratchBytes)
               : bwd<bf16_t>(ctx, rows, d, x, dy, mean, rstd, gamma, dx, dgamma, dbeta, accumulate, sp, kScratchBytes);
}
