// Fused softmax cross-entropy: loss and logit gradient in one read of the
// logits.
//
// Replaces F::cross_entropy as called by Nott::Loss::Details::compute
// (reference loss/details/ce.hpp:21-37; mean reduction, ignore_index -100,
// label smoothing ε), whose backward libtorch runs as two passes
// (nll_loss_backward, then _log_softmax_backward_data).  Per valid row i:
//   lse = max + log Σ exp(z − max)
//   dz  = grad_scale · (exp(z − lse) − (1−ε)·[j == y] − ε/c) / n_valid
//   loss_i = (1−ε)·(lse − z_y) + (ε/c)·(c·lse − Σ_j z_j)
// (a logit of −inf makes the smoothed loss infinite, as Σ_j z_j does.)
// Each row lives in registers of one workgroup: one HBM read, one write; what a
// row's stores follow is read before them, so dlogits may be logits itself.
#include "common.hpp"

#include <algorithm>

namespace {

constexpr int64_t kIgnoreIndex = -100;

// Counts valid labels and flags out-of-range ones.  One workgroup.
__global__ __launch_bounds__(1024) void xent_count_kernel(const int64_t* __restrict__ labels, int64_t n, int64_t c,
                                                          int* __restrict__ nvalid,
                                                          unsigned long long* __restrict__ err) {
    __shared__ float red[16];
    float cnt = 0.f;
    unsigned bad = 0;
    constexpr int kBatch = 16;   // labels per thread in flight
    for (int64_t base = threadIdx.x; base < n; base += 1024 * kBatch) {
        int64_t y[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int64_t i = base + (int64_t)u * 1024;
            y[u] = labels[i < n ? i : n - 1];
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            if (base + (int64_t)u * 1024 >= n || y[u] == kIgnoreIndex) continue;
            if (y[u] < 0 || y[u] >= c) ++bad;
            else cnt += 1.f;
        }
    }
    // counts up to 2^24 are exact in fp32; larger n is rejected on the host.
    const float total = block_sum<16>(cnt, red);
    if (bad) atomicAdd(err, (unsigned long long)bad);
    if (threadIdx.x == 0) *nvalid = (int)total;
}

template <int NWAVES>
__device__ __forceinline__ void block_sum2(float& a, float& b, float* red) {
    a = wave_sum(a);
    b = wave_sum(b);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) {
        red[wid] = a;
        red[NWAVES + wid] = b;
    }
    __syncthreads();
    float ta = 0.f, tb = 0.f;
#pragma unroll
    for (int i = 0; i < NWAVES; ++i) {
        ta += red[i];
        tb += red[NWAVES + i];
    }
    __syncthreads();
    a = ta;
    b = tb;
}

// Row body: v holds this thread's EPT elements of row `row` (element e of
// group g is column (g·NT + tid)·G + e; −inf past the end).  Writes the
// gradient row and the row's loss.  Every thread calls it (block reductions).
// One exponential per element: p = 2^(v·log2 e − max·log2 e) = e^(v − max)
// is kept in v, and the gradient is scale·(p/Σp − ε/C − (1 − ε)·[j = y])
// (the label's term applied once, by the thread that holds it); the row sum
// of the logits is formed only when label smoothing needs it.
template <typename T, int NT, int EPT>
__device__ __forceinline__ void xent_row_body(float (&v)[EPT], int64_t row, int64_t y, const T* z,
                                              int64_t c, float smoothing, float grad_scale, int nv, T* dz,
                                              float* __restrict__ row_loss, float* red) {
    constexpr int NWAVES = NT / 64;
    constexpr int G = Pack16<T>::N;
    constexpr int NG = EPT / G;
    constexpr float kLog2e = 1.4426950408889634f;
    const int ci = (int)c;
    if (!(y >= 0 && y < c)) {
        // Ignored (or out-of-range) row: zero gradient, no loss.
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int j0 = (g * NT + (int)threadIdx.x) * G;
            if (j0 >= ci) continue;
            float t[G];
#pragma unroll
            for (int e = 0; e < G; ++e) t[e] = 0.f;
            Pack16<T>::template st<true>(dz + j0, t);
        }
        if (threadIdx.x == 0 && row_loss) row_loss[row] = 0.f;
        return;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < EPT; ++e) mx = fmaxf(mx, v[e]);
    mx = block_max<NWAVES>(mx, red);
    const float mxl = mx * kLog2e;
    float se = 0.f, sz = 0.f;
    if (smoothing != 0.f) {
#pragma unroll
        for (int g = 0; g < NG; ++g)
            if ((g * NT + (int)threadIdx.x) * G < ci) {
#pragma unroll
                for (int e = 0; e < G; ++e) sz += v[g * G + e];
            }
    }
    const float zy = Io<T>::ld(z, y);   // before the stores: dlogits may be logits
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
        const float pe = __builtin_amdgcn_exp2f(fmaf(v[e], kLog2e, -mxl));
        se += pe;
        v[e] = pe;
    }
    block_sum2<NWAVES>(se, sz, red);
    const float lse = mx + __logf(se);
    const float scale = grad_scale / (float)nv;
    const float off = smoothing / (float)c;
    const float hit = 1.f - smoothing;
    const float ga = scale / se, gb = -scale * off;
    const int yi = (int)y;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        const int j0 = (g * NT + (int)threadIdx.x) * G;
        if (j0 >= ci) continue;
        float t[G];
#pragma unroll
        for (int e = 0; e < G; ++e) t[e] = fmaf(v[g * G + e], ga, gb);
        if ((unsigned)(yi - j0) < (unsigned)G) {
#pragma unroll
            for (int e = 0; e < G; ++e)
                if (j0 + e == yi) t[e] -= scale * hit;
        }
        Pack16<T>::template st<true>(dz + j0, t);
    }
    if (threadIdx.x == 0 && row_loss) row_loss[row] = hit * (lse - zy) + off * ((float)c * lse - sz);
}

// Vector path: 16-byte groups of G = 4 (fp32) or 8 (bf16) elements, strided
// by NT·G, loaded unconditionally (past-the-end groups re-read group 0 and
// count as −inf) so all of a thread's loads are in flight together.  The
// grid is persistent (rows blockIdx.x, + gridDim.x, ...) and the next row's
// loads are issued before the current row is reduced and written, so a CU's
// loads stay in flight through the block reductions and the stores.
template <typename T, int NT, int EPT>
__global__ __launch_bounds__(NT) void xent_rows_vec_kernel(const T* logits, const int64_t* __restrict__ labels,
                                                           int64_t n, int64_t c, float smoothing, float grad_scale,
                                                           const int* __restrict__ nvalid, T* dlogits,
                                                           float* __restrict__ row_loss) {
    constexpr int G = Pack16<T>::N;
    constexpr int NG = EPT / G;
    __shared__ float red[2 * (NT / 64)];
    typename Pack16<T>::Raw raw[NG];
    int64_t ny = 0;
    auto fetch = [&](int64_t row) {
        const T* z = logits + row * c;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int j0 = (g * NT + (int)threadIdx.x) * G;
            raw[g] = Pack16<T>::template raw<true>(z + (j0 < (int)c ? j0 : 0));
        }
        ny = labels[row];
    };
    const int nv = *nvalid;
    if ((int64_t)blockIdx.x < n) fetch(blockIdx.x);
    for (int64_t row = blockIdx.x; row < n; row += gridDim.x) {
        float v[EPT];
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int j0 = (g * NT + (int)threadIdx.x) * G;
            float t[G];
            Pack16<T>::unpack(raw[g], t);
#pragma unroll
            for (int e = 0; e < G; ++e) v[g * G + e] = j0 < (int)c ? t[e] : -INFINITY;
        }
        const int64_t y = ny;
        if (row + gridDim.x < n) fetch(row + gridDim.x);
        xent_row_body<T, NT, EPT>(v, row, y, logits + row * c, c, smoothing, grad_scale, nv,
                                        dlogits + row * c, row_loss, red);
    }
}

// Block-wide maximum / pair of sums with one LDS word per wave and a second
// wave reduction (the unrolled reads of block_max and block_sum2 would cost the
// wide rows their registers).  `red` is not reused by a later call.
template <int NWAVES>
__device__ __forceinline__ float row_max(float v, float* red) {
    v = wave_max(v);
    const int lane = threadIdx.x & 63;
    if (lane == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return wave_max(lane < NWAVES ? red[lane] : -INFINITY);
}
template <int NWAVES>
__device__ __forceinline__ void row_sum2(float& a, float& b, float* red) {
    a = wave_sum(a);
    b = wave_sum(b);
    const int lane = threadIdx.x & 63;
    if (lane == 0) {
        red[threadIdx.x >> 6] = a;
        red[NWAVES + (threadIdx.x >> 6)] = b;
    }
    __syncthreads();
    a = wave_sum(lane < NWAVES ? red[lane] : 0.f);
    b = wave_sum(lane < NWAVES ? red[NWAVES + lane] : 0.f);
}

// A group of −inf.
template <typename T>
__device__ __forceinline__ typename Pack16<T>::Raw minus_inf() {
    if constexpr (sizeof(T) == 2) return u32x4{0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u};
    else return f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
}

// Rows of any length at any alignment: c not a multiple of the 16-byte group,
// rows past the vector path's 32768, views that start off a 16-byte boundary.
// Each row is taken as its own 16-byte aligned groups, every one a single
// access, and the fewer than 2·G columns before the first and after the last
// whole group, one per thread (an element each, by itself).
//
// The first NT·NG groups are held in registers: one HBM read and one write, as
// in the vector path.  With REST the groups past them are streamed twice,
// before the held ones are loaded (a running maximum and sum per thread) and
// after they are stored, when their registers are free; the second read of a
// row of a few hundred KiB comes from the caches.  104 elements are what a
// thread holds at 4 waves per SIMD (128 VGPRs), which keeps two 512-thread rows
// (up to 53248 columns) or one 1024-thread row on a CU.  Bound by memory: it
// moves 4096 x 50257 fp32 at 5.1 TB/s (324 us), 8192 x 128256 bf16 at 5.4 TB/s
// (780 us) and 2048 x 151936 fp32 at 5.2 TB/s (482 us); three passes of single
// elements per row took 846, 3529 and 1247 us.  Short rows share the lines at their
// ends: up to 1024 columns loads, and fp32 stores, go through the caches (16000 x
// 1001 fp32 31.7 us, 33.8 past them).
template <typename T, int NT, int EPT, bool REST>
__global__ __launch_bounds__(NT, EPT > 64 ? 4 : 1) void xent_any_kernel(
    const T* logits, const int64_t* __restrict__ labels, int64_t c, float smoothing, float grad_scale,
    const int* __restrict__ nvalid, T* dlogits, float* __restrict__ row_loss) {
    constexpr int G = Pack16<T>::N;
    constexpr int NG = EPT / G;
    constexpr int NWAVES = NT / 64;
    constexpr int kUnroll = 4;       // streamed groups in flight per thread
    constexpr float kLog2e = 1.4426950408889634f;
    __shared__ float red[3 * NWAVES];
    const int tid = (int)threadIdx.x;
    const float off = smoothing / (float)c, hit = 1.f - smoothing;
    const int64_t row = blockIdx.x;
    const T* z = logits + row * c;
    T* dz = dlogits + row * c;
    const int64_t y = labels[row];
    // [0, s0) and [s0 + groups·G, c) are the single columns; thread i
    // holds the i-th of them (ej: its column, none for the other threads)
    const int s0 = (int)min((int64_t)((G - ((uintptr_t)z / sizeof(T)) % G) % G), c);
    const int64_t groups = (c - s0) / G, tail = s0 + groups * G;
    const int64_t ej = tid < s0 ? tid : tid - s0 < (int)(c - tail) ? tail + (tid - s0) : -1;
    const T* zb = z + s0;
    T* db = dz + s0;
    const bool vec_st = ((uintptr_t)db % 16) == 0;
    // group g·NT + tid is held iff g·NT < rem
    const int rem = (int)min(groups, (int64_t)NT * NG) - tid;
    if (!(y >= 0 && y < c)) {
        // Ignored (or out-of-range) row: zero gradient, no loss.
        for (int64_t j = tid; j < c; j += NT) Io<T>::st(dz, j, 0.f);
        if (tid == 0 && row_loss) row_loss[row] = 0.f;
        return;
    }
    float mx = ej >= 0 ? Io<T>::ld(z, ej) : -INFINITY;
    const float ez = mx;
    float se = 0.f, sz = 0.f;
    if constexpr (REST) {
        for (int64_t k = (int64_t)NT * NG + tid; k < groups; k += NT * kUnroll) {
            float t[kUnroll][G];
            float m = mx;
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                if (k + u * NT < groups) {
                    Pack16<T>::ld(zb + (k + u * NT) * G, t[u]);
                } else {
#pragma unroll
                    for (int e = 0; e < G; ++e) t[u][e] = -INFINITY;
                }
            }
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
#pragma unroll
                for (int e = 0; e < G; ++e) m = fmaxf(m, t[u][e]);
            // Nothing but −inf so far: no maximum to subtract (−inf − (−inf)
            // is no exponent); a NaN still reaches the sum.
            const bool none = m == -INFINITY;
            const float ml = none ? 0.f : m * kLog2e;
            se = none ? se : se * __builtin_amdgcn_exp2f((mx - m) * kLog2e);
            mx = m;
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
#pragma unroll
                for (int e = 0; e < G; ++e) {
                    se += __builtin_amdgcn_exp2f(fmaf(t[u][e], kLog2e, -ml));
                    if (k + u * NT < groups) sz += t[u][e];
                }
        }
    }
    // Every load is of a whole group of the row (past the last held one, that
    // one again); a row of fewer than 2·G columns may have none.
    typename Pack16<T>::Raw raw[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) raw[g] = minus_inf<T>();
    if (groups > 0) {
#pragma unroll
        for (int g = 0; g < NG; ++g)
            raw[g] = Pack16<T>::template raw<(EPT > 16)>(zb + (unsigned)(tid + min(g * NT, rem - 1)) * G);
    }
    float m = mx;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        raw[g] = g * NT < rem ? raw[g] : minus_inf<T>();
        float t[G];
        Pack16<T>::unpack(raw[g], t);
#pragma unroll
        for (int e = 0; e < G; ++e) m = fmaxf(m, t[e]);
        // unpacked again below: held packed until then, not as EPT floats more
        asm volatile("" : "+v"(raw[g]));
    }
    m = row_max<NWAVES>(m, red);
    const float ml = m * kLog2e;
    const float ep = __builtin_amdgcn_exp2f(fmaf(ez, kLog2e, -ml));
    const float zy = Io<T>::ld(z, y);   // (before the stores: dlogits may be logits)
    if constexpr (REST) se = mx == -INFINITY ? se : se * __builtin_amdgcn_exp2f((mx - m) * kLog2e);
    se += ej >= 0 ? ep : 0.f;
    if (smoothing != 0.f) {
        if (ej >= 0) sz += ez;
#pragma unroll
        for (int g = 0; g < NG; ++g)
            if (g * NT < rem) {
                float t[G];
                Pack16<T>::unpack(raw[g], t);
#pragma unroll
                for (int e = 0; e < G; ++e) sz += t[e];
                asm volatile("" : "+v"(raw[g]));
            }
    }
    float v[EPT];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        float t[G];
        Pack16<T>::unpack(raw[g], t);
#pragma unroll
        for (int e = 0; e < G; ++e) {
            v[g * G + e] = __builtin_amdgcn_exp2f(fmaf(t[e], kLog2e, -ml));
            se += v[g * G + e];
        }
    }
    row_sum2<NWAVES>(se, sz, red + NWAVES);
    const float lse = m + __logf(se);
    const float scale = grad_scale / (float)(*nvalid);
    const float ga = scale / se, gb = -scale * off;
    // The label's group, counted from this thread's first, and its element there.
    const int64_t yk = y >= s0 && y < tail ? (y - s0) / G - tid : -1;
    const int ye = yk >= 0 ? (int)((y - s0) % G) : 0;
    const int yh = yk < NT * NG ? (int)yk : -1;
    auto grad = [&](bool mine, float (&t)[G]) {
#pragma unroll
        for (int e = 0; e < G; ++e) t[e] = fmaf(t[e], ga, gb);
        if (mine) {
#pragma unroll
            for (int e = 0; e < G; ++e)
                if (e == ye) t[e] -= scale * hit;
        }
    };
    auto put = [&](T* p, const float (&t)[G]) {
        if (vec_st) {
            Pack16<T>::template st<(EPT > 16 || sizeof(T) == 2)>(p, t);
        } else {
#pragma unroll
            for (int e = 0; e < G; ++e) Io<T>::st(p, e, t[e]);
        }
    };
    if (ej >= 0) Io<T>::st(dz, ej, fmaf(ep, ga, gb) - (ej == y ? scale * hit : 0.f));
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        if (g * NT >= rem) continue;
        float t[G];
#pragma unroll
        for (int e = 0; e < G; ++e) t[e] = v[g * G + e];
        grad(g * NT == yh, t);
        put(db + g * NT * G + (unsigned)(tid * G), t);
    }
    if constexpr (REST) {
        for (int64_t k = (int64_t)NT * NG + tid; k < groups; k += NT * kUnroll) {
            float t[kUnroll][G];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
                if (k + u * NT < groups) Pack16<T>::ld(zb + (k + u * NT) * G, t[u]);
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                if (k + u * NT >= groups) break;
#pragma unroll
                for (int e = 0; e < G; ++e) t[u][e] = __builtin_amdgcn_exp2f(fmaf(t[u][e], kLog2e, -ml));
                grad(k + u * NT - tid == yk, t[u]);
                put(db + (k + u * NT) * G, t[u]);
            }
        }
    }
    if (tid == 0 && row_loss)
        row_loss[row] = hit * (lse - zy) + (smoothing != 0.f ? off * ((float)c * lse - sz) : 0.f);
}

__global__ __launch_bounds__(1024) void xent_loss_kernel(const float* __restrict__ row_loss, int64_t n,
                                                         const int* __restrict__ nvalid, float* __restrict__ loss) {
    __shared__ float red[16];
    float acc = 0.f;
    for (int64_t i = threadIdx.x; i < n; i += 1024) acc += row_loss[i];
    acc = block_sum<16>(acc, red);
    if (threadIdx.x == 0) *loss = (*nvalid > 0) ? acc / (float)(*nvalid) : __builtin_nanf("");
}

__global__ void xent_nan_kernel(float* __restrict__ loss) { *loss = __builtin_nanf(""); }

// One row of c <= 64·EPL columns per wave, lane j holding columns j, j + 64, ...:
// writes the gradient and returns the row's loss (0 for an ignored row).
template <typename T, int EPL>
__device__ __forceinline__ float xent_wave_row(const T* z, int64_t y, int64_t c, float smoothing, float grad_scale,
                                               int nv, T* dz) {
    constexpr float kLog2e = 1.4426950408889634f;
    const int lane = threadIdx.x & 63, ci = (int)c;
    float v[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) v[e] = e * 64 + lane < ci ? Io<T>::ld(z, e * 64 + lane) : -INFINITY;
    if (!(y >= 0 && y < c)) {
#pragma unroll
        for (int e = 0; e < EPL; ++e)
            if (e * 64 + lane < ci) Io<T>::st(dz, e * 64 + lane, 0.f);
        return 0.f;
    }
    const float zy = Io<T>::ld(z, y);
    float mx = v[0], sz = 0.f, se = 0.f;
#pragma unroll
    for (int e = 1; e < EPL; ++e) mx = fmaxf(mx, v[e]);
    mx = wave_max(mx);
    if (smoothing != 0.f) {
#pragma unroll
        for (int e = 0; e < EPL; ++e) sz += e * 64 + lane < ci ? v[e] : 0.f;
        sz = wave_sum(sz);
    }
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
        v[e] = __builtin_amdgcn_exp2f(fmaf(v[e], kLog2e, -mx * kLog2e));
        se += v[e];
    }
    se = wave_sum(se);
    const float lse = mx + __logf(se);
    const float scale = grad_scale / (float)nv;
    const float off = smoothing / (float)c;
    const float hit = 1.f - smoothing;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
        const int j = e * 64 + lane;
        if (j >= ci) continue;
        float g = fmaf(v[e], scale / se, -scale * off);
        if (j == (int)y) {
            // not contracted, whatever a caller's loop hoists: both kernels give the same bits
#pragma clang fp contract(off)
            g = g - scale * hit;
        }
        Io<T>::st(dz, j, g);
    }
    return hit * (lse - zy) + off * ((float)c * lse - sz);
}

// Rows of c <= 64·EPL columns that are not whole 16-byte groups (of up to 64
// columns when there are too many for the single-workgroup kernel below): one
// row per wave.
template <typename T, int EPL>
__global__ __launch_bounds__(256) void xent_wave_kernel(const T* logits, const int64_t* __restrict__ labels, int64_t n,
                                                        int64_t c, float smoothing, float grad_scale,
                                                        const int* __restrict__ nvalid, T* dlogits,
                                                        float* __restrict__ row_loss) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= n) return;
    const float l =
        xent_wave_row<T, EPL>(logits + row * c, labels[row], c, smoothing, grad_scale, *nvalid, dlogits + row * c);
    if ((threadIdx.x & 63) == 0 && row_loss) row_loss[row] = l;
}

// Small problems (c <= 64 classes, n <= kSmallRows rows; a classifier head at
// a small batch): the label count, every row and the mean loss in one
// 1024-thread workgroup, where the general path takes three launches and a
// workspace (without one, as under capture on a new context, up to
// kMostSmallRows rows go this way).  A wave
// owns rows wid, wid + 16, ...; the arithmetic and the summation orders are
// those of xent_count_kernel, xent_wave_kernel and xent_loss_kernel, so where
// the general path takes that kernel (c not a multiple of the 16-byte group)
// both give the same bits; its vector path sums each thread's group first.
// (One row per wave at a time costs 40 ns a row, 167 us at 4096 x 10 fp32
// against 17 us on the general path; the two meet near 250 rows.)
constexpr int64_t kSmallRows = 256, kMostSmallRows = 4096;
template <typename T>
__global__ __launch_bounds__(1024) void xent_small_kernel(const T* logits, const int64_t* __restrict__ labels, int64_t n,
                                                          int64_t c, float smoothing, float grad_scale, T* dlogits,
                                                          float* __restrict__ loss,
                                                          unsigned long long* __restrict__ err) {
    __shared__ float red[16];
    __shared__ float rl[kMostSmallRows];
    __shared__ int nvs;
    float cnt = 0.f;
    unsigned bad = 0;
    for (int64_t i = threadIdx.x; i < n; i += 1024) {
        const int64_t y = labels[i];
        if (y == kIgnoreIndex) continue;
        if (y < 0 || y >= c) ++bad;
        else cnt += 1.f;
    }
    const float total = block_sum<16>(cnt, red);
    if (bad) atomicAdd(err, (unsigned long long)bad);
    if (threadIdx.x == 0) nvs = (int)total;
    __syncthreads();
    const int nv = nvs;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int64_t row = wid; row < n; row += 16) {
        const float l =
            xent_wave_row<T, 1>(logits + row * c, labels[row], c, smoothing, grad_scale, nv, dlogits + row * c);
        if (lane == 0) rl[row] = l;
    }
    if (!loss) return;
    __syncthreads();
    float acc = 0.f;
    for (int64_t i = threadIdx.x; i < n; i += 1024) acc += rl[i];
    acc = block_sum<16>(acc, red);
    if (threadIdx.x == 0) *loss = nv > 0 ? acc / (float)nv : __builtin_nanf("");
}

// As many workgroups as are resident at once, at most one per row.
template <class K>
unsigned resident_grid(nott_ctx ctx, K kernel, int threads, int64_t n, int& per_cu) {
    if (per_cu == 0 &&
        (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0) != hipSuccess || per_cu < 1))
        per_cu = 1;
    return (unsigned)std::min<int64_t>(n, (int64_t)ctx->num_cu * per_cu);
}

template <typename T>
struct RowArgs {
    int64_t n, c;
    const T* logits;
    const int64_t* labels;
    float eps, scale;
    const int* nvalid;
    T* dl;
    float* row_loss;
};

template <typename T, int NT, int EPT>
void launch_vec(nott_ctx ctx, const RowArgs<T>& a) {
    static int per_cu = 0;
    const unsigned grid = resident_grid(ctx, xent_rows_vec_kernel<T, NT, EPT>, NT, a.n, per_cu);
    hipLaunchKernelGGL((xent_rows_vec_kernel<T, NT, EPT>), dim3(grid), dim3(NT), 0, ctx->stream, a.logits, a.labels,
                       a.n, a.c, a.eps, a.scale, a.nvalid, a.dl, a.row_loss);
}

template <typename T, int EPL>
void launch_wave(nott_ctx ctx, const RowArgs<T>& a) {
    hipLaunchKernelGGL((xent_wave_kernel<T, EPL>), dim3((unsigned)nott::ceil_div(a.n, 4)), dim3(256), 0, ctx->stream,
                       a.logits, a.labels, a.n, a.c, a.eps, a.scale, a.nvalid, a.dl, a.row_loss);
}

template <typename T, int NT, int EPT, bool REST>
void launch_any(nott_ctx ctx, const RowArgs<T>& a) {
    hipLaunchKernelGGL((xent_any_kernel<T, NT, EPT, REST>), dim3((unsigned)a.n), dim3(NT), 0, ctx->stream, a.logits,
                       a.labels, a.c, a.eps, a.scale, a.nvalid, a.dl, a.row_loss);
}

template <typename T>
void dispatch(nott_ctx ctx, const RowArgs<T>& a) {
    constexpr int G = Pack16<T>::N;
    // Whole aligned groups of up to 32768 columns: the persistent kernel, whose
    // next row is in flight during the reductions (5.7 TB/s at 16384 x 32000
    // fp32).  Everything else: up to 512 columns one wave a row, single elements
    // (16000 x 77 15.7 us, x 255 18.2 to 19.9, x 511 23.1 to 24.8; one 64-thread
    // workgroup of the kernel for any row 21.3, 22, 22.9 to 24.5 and 0.8 us more
    // at 100 rows); past that the kernel for any row, in the smallest shape that
    // holds it.
    const int64_t c = a.c;
    const bool vec = (c % G == 0) && ((uintptr_t)a.logits % 16 == 0) && ((uintptr_t)a.dl % 16 == 0);
    if (vec && c <= 64 * 16) return launch_vec<T, 64, 16>(ctx, a);
    if (vec && c <= 256 * 32) return launch_vec<T, 256, 32>(ctx, a);
    // bf16 rows of up to 32768: two 512-thread workgroups per CU, so that
    // two rows (plus the two prefetched ones) are in flight per CU.
    if (vec && sizeof(T) == 2 && c <= 512 * 64) return launch_vec<T, 512, 64>(ctx, a);
    if (vec && c <= 1024 * 32) return launch_vec<T, 1024, 32>(ctx, a);
    if (c <= 64) return launch_wave<T, 1>(ctx, a);
    if (c <= 128) return launch_wave<T, 2>(ctx, a);
    if (c <= 256) return launch_wave<T, 4>(ctx, a);
    if (c <= 512) return launch_wave<T, 8>(ctx, a);
    if (c <= 64 * 16) return launch_any<T, 64, 16, false>(ctx, a);
    if (c <= 256 * 32) return launch_any<T, 256, 32, false>(ctx, a);
    if (c <= 512 * 32) return launch_any<T, 512, 32, false>(ctx, a);
    if (c <= 512 * 64) return launch_any<T, 512, 64, false>(ctx, a);
    if (c <= 512 * 104) return launch_any<T, 512, 104, false>(ctx, a);
    if (c <= 1024 * 104) return launch_any<T, 1024, 104, false>(ctx, a);
    return launch_any<T, 1024, 104, true>(ctx, a);
}

}  // namespace

extern "C" int nott_softmax_xent_bwd(nott_ctx ctx, nott_dtype dtype, int64_t n, int64_t c, const void* logits,
                                     const int64_t* labels, double label_smoothing, double grad_scale, void* dlogits,
                                     float* loss) {
    NOTT_CHECK_CTX(ctx);
    NOTT_REQUIRE(ctx, nott::valid_dtype(dtype), "nott_softmax_xent_bwd: bad dtype");
    NOTT_REQUIRE(ctx, n >= 0 && c > 0, "nott_softmax_xent_bwd: need n >= 0 and c > 0");
    NOTT_REQUIRE(ctx, n < (int64_t(1) << 24) && n <= 0x7fffffff, "nott_softmax_xent_bwd: n too large");
    NOTT_REQUIRE(ctx, label_smoothing >= 0.0 && label_smoothing <= 1.0, "nott_softmax_xent_bwd: label_smoothing in [0,1]");
    NOTT_REQUIRE(ctx, n == 0 || (logits && labels && dlogits), "nott_softmax_xent_bwd: null buffer");
    nott::DeviceScope scope(ctx->device);
    if (n == 0) {
        if (loss) hipLaunchKernelGGL(xent_nan_kernel, dim3(1), dim3(1), 0, ctx->stream, loss);  // mean of nothing
        return nott::launch_status(ctx, "softmax_xent");
    }
    const float eps = (float)label_smoothing, scale = (float)grad_scale;
    // workspace: [nvalid int][pad to 256 B][row_loss n floats]
    const size_t need = 256 + sizeof(float) * (size_t)n;
    if (c <= 64 && (n <= kSmallRows || (n <= kMostSmallRows && !nott::optional_workspace(ctx, need)))) {
        if (dtype == NOTT_F32)
            hipLaunchKernelGGL(xent_small_kernel<float>, dim3(1), dim3(1024), 0, ctx->stream,
                               static_cast<const float*>(logits), labels, n, c, eps, scale,
                               static_cast<float*>(dlogits), loss, ctx->err_word);
        else
            hipLaunchKernelGGL(xent_small_kernel<bf16_t>, dim3(1), dim3(1024), 0, ctx->stream,
                               static_cast<const bf16_t*>(logits), labels, n, c, eps, scale,
                               static_cast<bf16_t*>(dlogits), loss, ctx->err_word);
        return nott::launch_status(ctx, "softmax_xent");
    }
    char* ws = static_cast<char*>(nott::workspace(ctx, need));
    if (!ws) return NOTT_ERR_ALLOC;
    int* nvalid = reinterpret_cast<int*>(ws);
    float* row_loss = loss ? reinterpret_cast<float*>(ws + 256) : nullptr;
    hipLaunchKernelGGL(xent_count_kernel, dim3(1), dim3(1024), 0, ctx->stream, labels, n, c, nvalid, ctx->err_word);
    if (dtype == NOTT_F32)
        dispatch<float>(ctx, {n, c, static_cast<const float*>(logits), labels, eps, scale, nvalid,
                              static_cast<float*>(dlogits), row_loss});
    else
        dispatch<bf16_t>(ctx, {n, c, static_cast<const bf16_t*>(logits), labels, eps, scale, nvalid,
                               static_cast<bf16_t*>(dlogits), row_loss});
    if (loss) hipLaunchKernelGGL(xent_loss_kernel, dim3(1), dim3(1024), 0, ctx->stream, row_loss, n, nvalid, loss);
    return nott::launch_status(ctx, "softmax_xent");
}
