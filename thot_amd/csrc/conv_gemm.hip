// bf16 NCHW convolutions as implicit GEMMs over a channels-last copy: every
// stride, dilation and tap count up to 25 with channels in whole 8s, where the
// 3×3 stride-1 kernels do not apply (strided, 1×1, 5×5 layers; conv.hpp:177 of
// the reference and its backward).
//
// A first launch writes the streamed tensor channels-last, zero-padded (so that
// no tap of any pixel needs a bounds check), and the weights as [row][tap][channel].
// The products then read 16-byte channel chunks straight into LDS, as the
// direct-to-LDS GEMM does (gemm_dma.hpp), with the row address of the gathered
// operand = pixel offset + tap offset:
//   forward : y[pixel, co] = Σ_{tap, ci} xp[pixel·stride + tap, ci] · w[co, tap, ci]
//   data    : dx[pixel of a stride parity class, ci] = Σ over the class's taps
//             and co of dyp[…, co] · w[ci, tap, co]: up to two row classes in one
//             launch, each with the one or two column phases side by side
//   weights : dw[co, (tap, ci)] = Σ_pixel dy[pixel, co] · xp[pixel·stride + tap, ci],
//             split over the pixels, partials summed in order
// 128×128 (or 128×64) tiles of 32×32×16 MFMAs, a 3-deep ring of 64-deep stages.
//
// With the copies, µs of forward / data / weight gradient, against the tap and im2col
// paths (which take other channel counts, and where the rules below say so):
//   [64, 128, 28, 28] → 256, 3×3 stride 2    29 / 38 / 38    was  56 / 60 / 54
//   [64, 64, 56, 56] → 128, 3×3 stride 2     38 / 41 / 50    was  53 / 59 / 69
//   [64, 512, 14, 14] → 512, 1×1             35 / 35 / 34    was  51 / 73 / 46
//   [64, 2048, 7, 7] → 512, 1×1              35 / 36 / 31    was  47 / 73 / 42
//   [16, 32, 32, 32] → 64, 5×5               14 / 21 / 23    was  38 / 52 / 38
// A strided product has few tiles (196 of 18 stages at the first shape, 370 TF), so
// it is bound by the latency of a stage; 10 µs of each pass is the copy.
#include "conv_fast.hpp"
#include "gemm_dma.hpp"

namespace nott {
namespace conv_fast {
namespace {

using gemm::dma::BK;
using gemm::dma::Frag;
using gemm::dma::FragAddr;
using gemm::dma::fill_block;
using gemm::dma::read_all;
using gemm::dma::zero_chunk;
using lds::barrier;
using lds::dma16;
using lds::lds_addr;
using lds::wait_vm_lgkm0;

constexpr int kMaxTaps = 25;
constexpr int NW = 4;           // waves per workgroup
constexpr int S = 3;            // ring depth
constexpr int BM = 128;

// ------------------------------------------------------------------- prep
// One tensor: xp[n][hp][wp][c] from x[n][c][h][w], position (i, j) holding pixel
// (i·sh − pt, j·sw − pl) or zeros.
template <typename T> struct PrepPart {
    const T* x;
    T* xp;
    int32_t c, h, w, pt, pl, sh, sw, cblocks, npos;
    FastDiv fij, fj, fcb;    // by hp·wp, wp and cblocks
};
template <typename T> struct PrepParams {
    PrepPart<T> part[2];        // the second may be empty (blocks[1] = blocks[0])
    int32_t blocks[2];       // first block after each part
    const T* wt;        // [k][cin][taps]
    T* wp2;
    int32_t k, cin, taps, by_cin;   // by_cin: rows are input channels (data gradient), columns output channels
    int32_t base[kMaxTaps], nt[kMaxTaps], t[kMaxTaps];   // by_cin, of a tap: its matrix, that matrix's taps, its place
};

// A block of a part: 64 positions × 64 channels, read along the positions,
// turned in LDS, written 16 bytes of channels at a time.  Positions are
// counted through all rows and images, so that narrow images fill the lanes
// too.  The blocks after the parts lay out the weights.  Bound by memory: the
// 128 MB of x and dy of [64, 64, 56, 56] → 256, 1×1, take 46 µs, 5.5 TB/s.
template <typename T> __global__ __launch_bounds__(256) void nhwc_prep_kernel(PrepParams<T> p) {
    constexpr int E = 16 / sizeof(T), CH = 64 / E;   // elements of a chunk, chunks of 64 channels
    __shared__ T tile[64][sizeof(T) == 2 ? 66 : 65];
    const int tid = threadIdx.x, b = (int)blockIdx.x;
    if (b >= p.blocks[1] && !p.by_cin) {
        // destination order: [row][tap][channel], a row's channels side by side
        const int64_t i = (int64_t)(b - p.blocks[1]) * 256 + tid;
        if (i >= (int64_t)p.taps * p.k * p.cin) return;
        const int32_t tap = (int32_t)(i / ((int64_t)p.k * p.cin));
        const int32_t j = (int32_t)(i - (int64_t)tap * p.k * p.cin), ko = j / p.cin, ci = j - ko * p.cin;
        p.wp2[((int64_t)ko * p.taps + tap) * p.cin + ci] = p.wt[(int64_t)j * p.taps + tap];
        return;
    }
    if (b >= p.blocks[1]) {
        // [k][cin·taps] turned: 64 output channels × 64 (input channel, tap)
        const int32_t kb = (p.k + 63) / 64, ct = p.cin * p.taps, wb = b - p.blocks[1];
        const int32_t k0 = wb % kb * 64, j0 = wb / kb * 64, nk = min(64, p.k - k0), nj = min(64, ct - j0);
        T v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int c = u * 4 + (tid >> 6);
            v[u] = (tid & 63) < nj && c < nk ? p.wt[(int64_t)(k0 + c) * ct + j0 + (tid & 63)] : T(0);
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) tile[u * 4 + (tid >> 6)][tid & 63] = v[u];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < CH / 4; ++u) {
            const int n = u * 256 + tid, ch = n % CH, at = n / CH;
            if (at >= nj || ch * E >= nk) continue;
            const int32_t ci = (j0 + at) / p.taps, tap = j0 + at - ci * p.taps;
            if (!p.nt[tap]) continue;   // a tap that only pixels past the edge would take
            T e[E];
#pragma unroll
            for (int z = 0; z < E; ++z) e[z] = tile[ch * E + z][at];
            *reinterpret_cast<u32x4*>(p.wp2 + p.base[tap] + (int64_t)(ci * p.nt[tap] + p.t[tap]) * p.k + k0 + ch * E) =
                gemm::Pack<T>::make(e);
        }
        return;
    }
    const int second = b >= p.blocks[0];
    const PrepPart<T>& q = p.part[second];
    uint32_t pb, cb, img, rest, i, j;
    q.fcb.divmod((uint32_t)(b - (second ? p.blocks[0] : 0)), pb, cb);
    const int32_t c0 = (int32_t)cb * 64, nc = min(64, q.c - c0), pos0 = (int32_t)pb * 64;
    const int32_t pos = min(pos0 + (tid & 63), q.npos - 1);
    q.fij.divmod((uint32_t)pos, img, rest);
    q.fj.divmod(rest, i, j);
    const int32_t hh = (int32_t)i * q.sh - q.pt, ww = (int32_t)j * q.sw - q.pl, hw = q.h * q.w;
    const bool in = hh >= 0 && hh < q.h && ww >= 0 && ww < q.w;
    const T* src = q.x + ((int64_t)img * q.c + c0) * hw + (in ? hh * q.w + ww : 0);
    T v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int c = u * 4 + (tid >> 6);
        v[u] = in && c < nc ? src[(int64_t)c * hw] : T(0);
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) tile[u * 4 + (tid >> 6)][tid & 63] = v[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < CH / 4; ++u) {
        const int n = u * 256 + tid, ch = n % CH, at = n / CH;
        if (pos0 + at >= q.npos || ch * E >= nc) continue;
        T e[E];
#pragma unroll
        for (int z = 0; z < E; ++z) e[z] = tile[ch * E + z][at];
        *reinterpret_cast<u32x4*>(q.xp + (int64_t)(pos0 + at) * q.c + c0 + ch * E) = gemm::Pack<T>::make(e);
    }
}

// ------------------------------------------------- forward and data gradient
// One product: rows are the pixels (image, i, j) of an ni × nj grid; of a data
// gradient with stride 2 along the width, P = 2 products over the same grid, whose
// results lie side by side.
struct RowClass {
    int32_t M, tile0;         // pixels; first tile of the launch
    int32_t K[2], woff[2];    // taps · channels, and the weights, of each product
    FastDiv fij, fj;          // by ni·nj and nj
    int32_t o0;               // first output element
    int32_t taps[2][kMaxTaps];   // element offsets into xp
};
struct RowParams {
    const bf16_t *xp, *w;
    bf16_t* out;
    const float* bias;
    int32_t relu, N, ncls, tiles;
    FastDiv fc;
    int32_t sn, si, sj;       // xp strides of image, i, j
    int32_t on, oc, oi;       // output strides of image, column, i
    int32_t wlim;             // output width
    int32_t vec;              // elements per store: 8, 4, 2 or 1
    int32_t ring;             // LDS bytes of the ring and, after it, of the staged results
    RowClass cls[2];
};

template <int BN, int P>
__global__ __launch_bounds__(64 * NW) void conv_rows_kernel(RowParams p) {
    constexpr int WM = BN == 128 ? 2 : 4, WN = BN == 128 ? 2 : 1;
    constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 32, FN = TN / 32;
    constexpr int A_BYTES = BM * 128, B_BYTES = BN * 128, STAGE = A_BYTES + B_BYTES;
    constexpr int LA = BM / 8 / NW, LB = BN / 8 / NW, LOADS = LA + LB;
    constexpr int PITCH = 2 * (P * BM + 8);   // bytes of a staged output column
    static_assert(BN * PITCH <= S * STAGE, "the results are staged in the ring");
    extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
    char NOTT_LDS* smem = (char NOTT_LDS*)smem_raw;
    int32_t NOTT_LDS* ltap = (int32_t NOTT_LDS*)(smem + p.ring);

    int id = (int)blockIdx.x;
    if ((p.tiles & 7) == 0) id = (id & 7) * (p.tiles >> 3) + (id >> 3);
    const RowClass& q = p.cls[p.ncls > 1 && id >= p.cls[1].tile0];
    const int tn = (p.N + BN - 1) / BN;
    id -= q.tile0;
    const int32_t m0 = id / tn * BM, n0 = id % tn * BN;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int wm = wid / WN, wn = wid % WN;
    if ((int)threadIdx.x < P * kMaxTaps) ltap[threadIdx.x] = (&q.taps[0][0])[threadIdx.x];
    __syncthreads();
    const int nk0 = (q.K[0] + BK - 1) / BK, nk = nk0 + (P == 2 ? (q.K[1] + BK - 1) / BK : 0);

    // This lane's rows of the A fills, and the chunk it takes of each (the
    // swizzle depends on the row through the wave's parity only).
    int32_t off[LA];
#pragma unroll
    for (int i = 0; i < LA; ++i) {
        const uint32_t m = (uint32_t)min(m0 + 8 * (i * NW + wid) + (lane >> 3), q.M - 1);
        uint32_t img, rest, y, x;
        q.fij.divmod(m, img, rest);
        q.fj.divmod(rest, y, x);
        off[i] = (int32_t)img * p.sn + (int32_t)y * p.si + (int32_t)x * p.sj;
    }
    const int chunk = (lane & 7) ^ ((4 * wid + (lane >> 4)) & 7);
    auto issue = [&](int t, int slot) {
        char NOTT_LDS* st = smem + slot * STAGE;
        const int ph = P == 2 && t >= nk0, k0 = (ph ? t - nk0 : t) * BK, K = q.K[ph];
        const bf16_t* w = p.w + q.woff[ph];
        const uint32_t k = (uint32_t)(k0 + 8 * chunk);
        const bool in = k < (uint32_t)K;
        uint32_t tap, c;
        p.fc.divmod(in ? k : 0u, tap, c);
        const int32_t toff = ltap[ph * kMaxTaps + tap] + (int32_t)c;
#pragma unroll
        for (int i = 0; i < LA; ++i)
            dma16(in ? p.xp + (off[i] + toff) : reinterpret_cast<const bf16_t*>(&zero_chunk),
                  lds_addr(st) + 1024 * (i * NW + wid));
        if (k0 + BK <= K) {
#pragma unroll
            for (int i = 0; i < LB; ++i)
                fill_block<false, BN, NW, false>(i, w, K, n0, p.N, k0, K, st + A_BYTES, wid, lane);
        } else {
#pragma unroll
            for (int i = 0; i < LB; ++i)
                fill_block<false, BN, NW, true>(i, w, K, n0, p.N, k0, K, st + A_BYTES, wid, lane);
        }
    };
    f32x16 acc[P][FM][FN];
#pragma unroll
    for (int h = 0; h < P; ++h)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[h][i][j][e] = 0.f;
    FragAddr<false, BM, FM> fa;
    FragAddr<false, BN, FN> fb;
    fa.init(wm * TM, lane);
    fb.init(wn * TN, lane);
    Frag<false> a[2][FM], b[2][FN];
#pragma unroll
    for (int s = 0; s < S - 1; ++s)
        if (s < nk) issue(s, s);
    if (nk > 0) {
        if (nk >= S - 1) wait_vm_lgkm0<(S - 2) * LOADS>();
        else wait_vm_lgkm0<0>();
        barrier();
        read_all<0>(a[0], fa, smem);
        read_all<0>(b[0], fb, smem + A_BYTES);
    }
    int slot = 0, free = S - 1;
    auto stages = [&](int t, int end, f32x16 (&c)[FM][FN]) {
        auto mma = [&](int s) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    c[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s][i].get(), b[s][j].get(), c[i][j], 0, 0, 0);
        };
        for (; t < end; ++t) {
            const char NOTT_LDS* sa = smem + slot * STAGE;
            const char NOTT_LDS* sb = sa + A_BYTES;
            const bool more = t + S - 1 < nk;
            read_all<1>(a[1], fa, sa);
            read_all<1>(b[1], fb, sb);
            if (more) issue(t + S - 1, free);
            mma(0);
            read_all<2>(a[0], fa, sa);
            read_all<2>(b[0], fb, sb);
            mma(1);
            read_all<3>(a[1], fa, sa);
            read_all<3>(b[1], fb, sb);
            mma(0);
            const int nslot = slot + 1 == S ? 0 : slot + 1;
            if (t + 1 < nk) {
                if (more) wait_vm_lgkm0<(S - 2) * LOADS>();
                else wait_vm_lgkm0<0>();
                barrier();
                const char NOTT_LDS* na = smem + nslot * STAGE;
                read_all<0>(a[0], fa, na);
                read_all<0>(b[0], fb, na + A_BYTES);
            }
            mma(1);
            free = slot;
            slot = nslot;
        }
    };
    stages(0, nk0, acc[0]);
    if constexpr (P == 2) stages(nk0, nk, acc[1]);

    // Lane l holds column l % 32 and, in register 4r + e, row 8r + 4·(l/32) + e.
    // The tile goes through LDS as [column][pixel], so that a wave stores runs
    // of one output channel: stored from the registers, 8 bytes per channel
    // plane, the strided data gradient of [64, 128, 28, 28] took 70 µs.
    __syncthreads();
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int col = wn * TN + 32 * j + (lane & 31);
        const float bias = p.bias ? p.bias[min(n0 + col, p.N - 1)] : 0.f;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v[P][4];
#pragma unroll
                for (int h = 0; h < P; ++h)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[h][e] = acc[h][i][j][4 * r + e];
                        if (p.bias) v[h][e] += bias;
                        if (p.relu) v[h][e] = relu_out(v[h][e]);
                    }
                char NOTT_LDS* at = smem + col * PITCH + 2 * P * (wm * TM + 32 * i + 8 * r + 4 * (lane >> 5));
                if constexpr (P == 2)
                    *reinterpret_cast<u32x4 NOTT_LDS*>(at) =
                        u32x4{pack_bf16x2(v[0][0], v[P - 1][0]), pack_bf16x2(v[0][1], v[P - 1][1]),
                              pack_bf16x2(v[0][2], v[P - 1][2]), pack_bf16x2(v[0][3], v[P - 1][3])};
                else
                    *reinterpret_cast<u32x2 NOTT_LDS*>(at) =
                        u32x2{pack_bf16x2(v[0][0], v[0][1]), pack_bf16x2(v[0][2], v[0][3])};
            }
    }
    __syncthreads();
    auto put = [&](auto tag) {
        typedef decltype(tag) V;
        constexpr int E = sizeof(V) / 2, RUNS = P * BM / E;
        const int e0 = (int)threadIdx.x % RUNS * E, m = m0 + e0 / P;
        if (m >= q.M) return;
        uint32_t img, rest, y, x;
        q.fij.divmod((uint32_t)m, img, rest);
        q.fj.divmod(rest, y, x);
        const int32_t px = (int32_t)x * P + e0 % P;
        if (E == 1 && px >= p.wlim) return;   // an odd width's last pair
        bf16_t* o = p.out + q.o0 + (int64_t)img * p.on + (int64_t)y * p.oi + px;
        for (int col = (int)threadIdx.x / RUNS; col < BN && n0 + col < p.N; col += 64 * NW / RUNS)
            *reinterpret_cast<V*>(o + (int64_t)(n0 + col) * p.oc) =
                *reinterpret_cast<const V NOTT_LDS*>(smem + col * PITCH + 2 * e0);
    };
    if (p.vec == 8) put(u32x4{});
    else if (p.vec == 4) put(u32x2{});
    else if (p.vec == 2) put(uint32_t{});
    else put(uint16_t{});
}

// ---------------------------------------------------------- weight gradient
template <typename T> struct WgradParams {
    const T *dyt, *xp;   // [pixel][k], [n][hp][wp][c]
    int32_t M, N, K, kps, splits;   // M = k, N = taps · C, K = pixels
    FastDiv fij, fj, fc;
    int32_t sn, si, sj;
    int32_t taps[kMaxTaps];
    float* ws;                // [split][M][N]
};
constexpr int kMaxPixels = 14336;   // of a split: their offsets sit in LDS beside the ring

// The operand slices of one wave: 16 k of the stage's 64 (bf16), 8 of its 32
// (fp32), for two 32-row fragments.
template <typename T> struct Slices;
template <> struct Slices<bf16_t> {
    static constexpr int kStageK = 64;
    FragAddr<true, 128, 2> at;
    Frag<true> f[2][2];
    __device__ __forceinline__ void init(int row0, int lane) { at.init(row0, lane); }
    template <int SL> __device__ __forceinline__ void read(const char NOTT_LDS* tile) { read_all<SL>(f[SL & 1], at, tile); }
};
// fp32 tiles are [k][128 rows]; odd k hold their rows with bit 5 flipped, so
// that the two halves of a wave (k and k + 1) read different banks.
template <> struct Slices<float> {
    static constexpr int kStageK = 32;
    int at[2];
    float f[2][2][4];
    __device__ __forceinline__ void init(int row0, int lane) {
        for (int i = 0; i < 2; ++i) at[i] = (lane >> 5) * 512 + 4 * ((row0 + 32 * i + (lane & 31)) ^ (lane & 32));
    }
    template <int SL> __device__ __forceinline__ void read(const char NOTT_LDS* tile) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                f[SL & 1][i][e] = *reinterpret_cast<const float NOTT_LDS*>(tile + at[i] + (SL * 4 + e) * 1024);
    }
};

template <typename T> __global__ __launch_bounds__(64 * NW) void conv_wgrad_rows_kernel(WgradParams<T> p) {
    constexpr int BN = 128, FM = 2, FN = 2, TILE = 128 * 128, STAGE = 2 * TILE, LOADS = 2 * 16 / NW;
    constexpr int BK = Slices<T>::kStageK, E = 16 / sizeof(T), KPB = 1024 / (128 * (int)sizeof(T));   // k of a 1 KB block
    extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
    char NOTT_LDS* smem = (char NOTT_LDS*)smem_raw;
    int32_t NOTT_LDS* lpix = (int32_t NOTT_LDS*)(smem + S * STAGE);
    int pm, pn, z;
    gemm::dma::tile_of((int)blockIdx.x, (p.M + BM - 1) / BM, (p.N + BN - 1) / BN, p.splits, 4, 0, pm, pn, z);
    const int32_t m0 = pm * BM, n0 = pn * BN, kb = z * p.kps, ke = min(p.K, kb + p.kps);
    const int nk = (ke - kb + BK - 1) / BK;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int wm = wid >> 1, wn = wid & 1;
    for (int i = threadIdx.x; i < nk * BK; i += 64 * NW) {
        uint32_t img, rest, y, x;
        p.fij.divmod((uint32_t)min(kb + i, p.K - 1), img, rest);
        p.fj.divmod(rest, y, x);
        lpix[i] = (int32_t)img * p.sn + (int32_t)y * p.si + (int32_t)x * p.sj;
    }
    // This lane's 16 bytes of columns of every fill (for B a tap and channels),
    // and its pixel in each 1 KB block.
    const int pix = lane / (128 / E);
    const int crow = E * ((lane % (128 / E)) ^ (E == 8 ? pix << 2 : pix << 3));   // its columns within the tile
    const uint32_t col = (uint32_t)min(n0 + crow, p.N - E);
    const int64_t arow = min(m0 + crow, p.M - E);
    uint32_t tap, c;
    p.fc.divmod(col, tap, c);
    int32_t toff = (int32_t)c;
#pragma unroll
    for (int i = 0; i < kMaxTaps; ++i) toff += (uint32_t)i == tap ? p.taps[i] : 0;
    __syncthreads();
    auto issue = [&](int t, int slot) {
        char NOTT_LDS* st = smem + slot * STAGE;
        const int32_t k0 = kb + t * BK;
#pragma unroll
        for (int i = 0; i < 16 / NW; ++i) {
            const int k = KPB * (i * NW + wid) + pix;
            const bool in = k0 + k < p.K;
            const T* zero = reinterpret_cast<const T*>(&zero_chunk);
            dma16(in ? p.dyt + ((int64_t)(k0 + k) * p.M + arow) : zero, lds_addr(st) + 1024 * (i * NW + wid));
            dma16(in ? p.xp + (lpix[t * BK + k] + toff) : zero, lds_addr(st + TILE) + 1024 * (i * NW + wid));
        }
    };
    // Even and odd slices have sums of their own, added at the end, so that an
    // fp32 sum runs over half of the split's pixels.  One sum for all was up to 1.38
    // times further from 64 bits than the generic path, which splits more ([64,
    // 128, 28, 28] → 256, 3×3 stride 2, fp32: 5.3e-7 against 3.8e-7; now 3.7e-7),
    // and 0.4 µs a launch faster.
    f32x16 acc[2][FM][FN];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[h][i][j][e] = 0.f;
    Slices<T> a, b;
    a.init(wm * 64, lane);
    b.init(wn * 64, lane);
    auto mma = [&](int s) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                if constexpr (sizeof(T) == 2) {
                    acc[s][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.f[s][i].get(), b.f[s][j].get(),
                                                                           acc[s][i][j], 0, 0, 0);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[s][i][j] =
                            __builtin_amdgcn_mfma_f32_32x32x2f32(a.f[s][i][e], b.f[s][j][e], acc[s][i][j], 0, 0, 0);
                }
            }
    };
#pragma unroll
    for (int s = 0; s < S - 1; ++s)
        if (s < nk) issue(s, s);
    if (nk > 0) {
        if (nk >= S - 1) wait_vm_lgkm0<(S - 2) * LOADS>();
        else wait_vm_lgkm0<0>();
        barrier();
        a.template read<0>(smem);
        b.template read<0>(smem + TILE);
    }
    int slot = 0, free = S - 1;
    for (int t = 0; t < nk; ++t) {
        const char NOTT_LDS* sa = smem + slot * STAGE;
        const char NOTT_LDS* sb = sa + TILE;
        const bool more = t + S - 1 < nk;
        a.template read<1>(sa);
        b.template read<1>(sb);
        if (more) issue(t + S - 1, free);
        mma(0);
        a.template read<2>(sa);
        b.template read<2>(sb);
        mma(1);
        a.template read<3>(sa);
        b.template read<3>(sb);
        mma(0);
        const int nslot = slot + 1 == S ? 0 : slot + 1;
        if (t + 1 < nk) {
            if (more) wait_vm_lgkm0<(S - 2) * LOADS>();
            else wait_vm_lgkm0<0>();
            barrier();
            const char NOTT_LDS* na = smem + nslot * STAGE;
            a.template read<0>(na);
            b.template read<0>(na + TILE);
        }
        mma(1);
        free = slot;
        slot = nslot;
    }
    float* ws = p.ws + (int64_t)z * p.M * p.N;
    const int col0 = lane & 31, rh = (lane >> 5) * 4;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int32_t m = m0 + wm * 64 + 32 * i + 8 * r + rh + e, n = n0 + wn * 64 + 32 * j + col0;
                    if (m < p.M && n < p.N) 
                        ws[(int64_t)m * p.N + n] = acc[0][i][j][4 * r + e] + acc[1][i][j][4 * r + e];
                }
}

// dw[k][c][tap] from column (tap, c).
struct TapMajorStore {
    float* dw;
    FastDiv fc;
    int32_t c, taps, accumulate;
    __device__ __forceinline__ void store(int64_t k, int64_t n, float v) const {
        uint32_t tap, ch;
        fc.divmod((uint32_t)n, tap, ch);
        float* o = dw + (k * c + ch) * taps + tap;
        *o = accumulate ? *o + v : v;
    }
};

int64_t align256(int64_t b) { return (b + 255) / 256 * 256; }

template <typename T>
PrepPart<T> part_of(const T* x, T* xp, int64_t n, int64_t c, int64_t h, int64_t w, int64_t hp, int64_t wp, int64_t pt,
                    int64_t pl, int64_t sh = 1, int64_t sw = 1) {
    PrepPart<T> p{};
    p.x = x; p.xp = xp;
    p.c = (int32_t)c; p.h = (int32_t)h; p.w = (int32_t)w;
    p.pt = (int32_t)pt; p.pl = (int32_t)pl; p.sh = (int32_t)sh; p.sw = (int32_t)sw;
    p.cblocks = (int32_t)ceil_div(c, 64);
    p.npos = (int32_t)(n * hp * wp);
    p.fij = FastDiv((uint32_t)(hp * wp)); p.fj = FastDiv((uint32_t)wp); p.fcb = FastDiv((uint32_t)p.cblocks);
    return p;
}

template <typename T> int launch_prep(nott_ctx ctx, PrepParams<T>& p) {
    int64_t blocks = 0;
    for (int i = 0; i < 2; ++i) {
        blocks += ceil_div(p.part[i].npos, 64) * p.part[i].cblocks;
        p.blocks[i] = (int32_t)blocks;
    }
    if (p.wt)
        blocks += p.by_cin ? ceil_div(p.k, 64) * ceil_div((int64_t)p.cin * p.taps, 64)
                           : ceil_div((int64_t)p.taps * p.k * p.cin, 256);
    hipLaunchKernelGGL(nhwc_prep_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, p);
    return launch_status(ctx, "conv channels-last prep");
}

template <int BN, int P> int launch_rows_as(nott_ctx ctx, RowParams& p) {
    int64_t tiles = 0;
    for (int i = 0; i < p.ncls; ++i) {
        p.cls[i].tile0 = (int32_t)tiles;
        tiles += ceil_div(p.cls[i].M, BM) * ceil_div(p.N, BN);
    }
    p.tiles = (int32_t)tiles;
    // A short product fills part of the ring only; the LDS it leaves holds more
    // workgroups per CU.
    int64_t nk = 0;
    for (int i = 0; i < p.ncls; ++i) nk = std::max(nk, ceil_div(p.cls[i].K[0], BK) + ceil_div(p.cls[i].K[1], BK));
    p.ring = (int32_t)std::max<int64_t>(std::min<int64_t>(S, nk) * (BM + BN) * 128, BN * 2 * (P * BM + 8));
    constexpr size_t kLds = (size_t)S * (BM + BN) * 128 + 8 * kMaxTaps;
    auto fn = conv_rows_kernel<BN, P>;
    static bool attr = false;
    if (!attr) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)kLds) != hipSuccess)
            return fail(ctx, NOTT_ERR_HIP, "conv_gemm: cannot reserve LDS");
        attr = true;
    }
    hipLaunchKernelGGL(fn, dim3((unsigned)tiles), dim3(64 * NW), (size_t)p.ring + 8 * kMaxTaps, ctx->stream, p);
    return launch_status(ctx, "conv_gemm");
}
bool narrow_tiles(nott_ctx ctx, int64_t wide, int64_t N);
int launch_rows(nott_ctx ctx, RowParams& p, int products) {
    int64_t wide = 0;
    for (int i = 0; i < p.ncls; ++i) wide += ceil_div(p.cls[i].M, BM) * ceil_div(p.N, 128);
    const bool n64 = narrow_tiles(ctx, wide, p.N);
    if (products == 2) return n64 ? launch_rows_as<64, 2>(ctx, p) : launch_rows_as<128, 2>(ctx, p);
    return n64 ? launch_rows_as<64, 1>(ctx, p) : launch_rows_as<128, 1>(ctx, p);
}

// Elements a store may take: runs of `run` consecutive output elements, all
// starting at multiples of the strides.
int32_t store_width(const void* out, int64_t run, int64_t a, int64_t b, int64_t c, int64_t d) {
    for (int32_t v = 8; v > 1; v /= 2)
        if (run % v == 0 && a % v == 0 && b % v == 0 && c % v == 0 && d % v == 0 && (uintptr_t)out % (2 * v) == 0)
            return v;
    return 1;
}

// The copy of x that the forward pass and the weight gradient read, and the
// step of the pixels in it.  A 1×1 kernel's copy holds only the pixels it takes.
struct Gather {
    int64_t hp, wp, sh, sw, ph, pw;   // copy's size, its stride over x, the pixels' stride over it
    explicit Gather(const nott_conv2d_desc* d, int64_t p, int64_t q) {
        const bool one = d->r == 1 && d->s == 1;
        hp = one ? p : d->h + 2 * d->pad_h;
        wp = one ? q : d->w + 2 * d->pad_w;
        sh = one ? d->stride_h : 1;
        sw = one ? d->stride_w : 1;
        ph = one ? 1 : d->stride_h;
        pw = one ? 1 : d->stride_w;
    }
};

// The padding of dy and the taps of the data gradient's parity classes:
// dx pixel (st_h·i + a, st_w·j + b) takes tap (r, s) from dy[i + dh, j + dw]
// where (a + pad − r·dil) = st·dh exactly.
// Taps (position and shift) of phase a along one axis.
int axis_taps(int64_t a, int64_t pad, int64_t taps, int64_t st, int64_t dil, int64_t* pos, int64_t* shift) {
    int n = 0;
    for (int64_t r = 0; r < taps; ++r) {
        const int64_t v = a + pad - r * dil;
        if (((v % st) + st) % st) continue;
        pos[n] = r;
        shift[n++] = v / st;
    }
    return n;
}
void axis_padding(int64_t size, int64_t out, int64_t pad, int64_t taps, int64_t st, int64_t dil, int64_t& lo,
                  int64_t& padded) {
    int64_t first = 0, last = out - 1;
    const int64_t rows = ceil_div(size, st);   // an odd size's last phase runs one past its end
    for (int64_t a = 0; a < st && a < size; ++a) {
        int64_t pos[kMaxTaps], sh[kMaxTaps];
        const int n = axis_taps(a, pad, taps, st, dil, pos, sh);
        for (int i = 0; i < n; ++i) {
            first = std::min(first, sh[i]);
            last = std::max(last, rows - 1 + sh[i]);
        }
    }
    lo = -first;
    padded = last - first + 1;
}

bool shape_ok(nott_ctx ctx, const nott_conv2d_desc* d, int64_t chunk = 8) {
    return ctx->conv_tap && d->layout == NOTT_NCHW && d->c % chunk == 0 && d->k % chunk == 0 && d->r * d->s <= kMaxTaps;
}
bool fits(int64_t elems) { return elems < (int64_t(1) << 31); }

// Tiles of M rows and N columns of a product over `classes` row classes of about M
// rows each: 128 × 64 ones also where the wide ones would not give every CU one ([64,
// 256, 14, 14] → 512, stride 2, 34 µs forward and 42 data gradient against 36 and 46).
bool narrow_tiles(nott_ctx ctx, int64_t wide, int64_t N) { return N <= 64 || wide < ctx->num_cu; }
int64_t row_tiles(nott_ctx ctx, int64_t M, int64_t N, int64_t classes) {
    const int64_t wide = ceil_div(M, BM) * ceil_div(N, 128);
    return narrow_tiles(ctx, wide * classes, N) ? ceil_div(M, BM) * ceil_div(N, 64) : wide;
}

}  // namespace

// A product of `stages` 64-deep stages on few tiles is one long chain, about 7 +
// 0.5·stages µs; the column path splits it, after an im2col of 17 µs and 1 µs a MB:
// [6, 512, 28, 32] → 32, 3×3 stride 2, 72 stages on 11 tiles, 45 µs against 30, [1,
// 256, 16, 16] → 64 24 against 19; but [8, 256, 28, 28] → 64, 5×5, 59 against 73.
// Up to 64 output channels the tap kernel (which reads x once where it lies) keeps
// three cases: many pixels in output planes of whole 1024s, whose channels' stores
// fall on the same memory channels ([64, 64, 64, 64] → 64, stride 2, 35 µs against
// 30, [64, 256, 64, 64] 97 against 70; half the images 23 against 26), and one
// channel chunk on 256 to 384 tiles ([64, 32, 48, 48] 21 against 17, [32, 32, 64, 64]
// 19 against 16; 10 against 15 at half, 32 against 35 at twice the images); and an
// input of up to 128 channels that with its copy outgrows the 256 MB of cache ([64,
// 96, 96, 96] 119 against 99; [64, 64, 112, 112] still 91 against 97).
bool rows_fwd_applies(nott_ctx ctx, const nott_conv2d_desc* d, int64_t p, int64_t q, bool col) {
    if (!shape_ok(ctx, d) || !fits(d->n * (d->h + 2 * d->pad_h) * (d->w + 2 * d->pad_w) * d->c)) return false;
    const int64_t M = d->n * p * q, K = d->r * d->s * d->c, stages = ceil_div(K, BK);
    if (col && row_tiles(ctx, M, d->k, 1) <= 64 && (double)stages > 20 + 4e-6 * (double)(K * M)) return false;
    const bool same_channels = p * q % 1024 == 0 && M >= 65536, one_chunk = d->c <= 32 && M >= 32768 && M < 49152;
    const bool past_cache = d->c <= 128 && d->n * d->h * d->w * d->c >= 55000000;
    return !(d->k <= 64 && (same_channels || one_chunk || past_cache) && tap_fwd_applies(ctx, d, 2));
}
// The other paths go through no copies and no partials, whose turn and sum cost
// about 10 µs a million weights: with few pixels a large gradient is better there.
// [2, 512, 8, 8] → 512, 3×3 stride 2 (32 pixels) 32 µs against 12 in bf16, 33 against
// 14 in fp32; with 32 pixels or fewer every one ([1, 32, 8, 8] → 32 12.0 against 7.6
// fp32, 10.2 against 8.7 bf16).  The lines are where they meet: the column path
// (whole 64s of pixels) 64 pixels, from 100 thousand weights 128 or the weights over
// 2300 ([8, 512, 16, 16], 512 pixels, 39 against 33); else 64 pixels from 500
// thousand weights ([1, 256, 16, 16] fp32 19.7 against 18.4) or the weights over 16000
// ([1, 512, 14, 14], 5×5, 196 pixels, bf16 74 against 46; 3×3 equal).
bool rows_wgrad_applies(nott_ctx ctx, const nott_conv2d_desc* d, int64_t p, int64_t q, size_t elem, bool col) {
    if (!shape_ok(ctx, d, 16 / (int64_t)elem) || !fits(d->n * (d->h + 2 * d->pad_h) * (d->w + 2 * d->pad_w) * d->c))
        return false;
    const int64_t K = d->n * p * q, MN = d->k * d->c * d->r * d->s;
    if (col) return K > (MN < 100000 ? 64 : std::max<int64_t>(128, std::min<int64_t>(512, MN / 2300)));
    return K > std::max<int64_t>(MN < 500000 ? 32 : 64, std::min<int64_t>(256, MN / 16000));
}
bool rows_dgrad_applies(nott_ctx ctx, const nott_conv2d_desc* d, int64_t p, int64_t q) {
    if (!shape_ok(ctx, d) || d->stride_h > 2 || d->stride_w > 2) return false;
    // A 1×1 kernel's gradient reads dy where it lies (conv_tap.hip): once, up to
    // 128 output columns, so the copy only costs.  64 images of 56×56: 64 → 64
    // channels 24 µs against 28 with the copy, k = 256 → c = 64 51 against 63; 28×28,
    // k = 512 → c = 128 40 against 42; but k = 64 → c = 256 at 56×56 66 against 41,
    // and planes that are not whole 16 bytes (512 → 512 at 14×14) 73 against 35.
    // k in odd 32s from 45000 pixels: up to 64 columns (16 images of 64×64, k = 96 →
    // c = 64 13 against 20; of 28×28 10 against 9), up to 128 where the planes are whole
    // 1024s of pixels, or k is at least 128 or, below 100000 pixels, 96 (16 images of
    // 56×56, k = 160 → c = 128 24 against 28; 64 images, k = 32 31 against 34).
    if (d->r == 1 && d->s == 1 && d->stride_h == 1 && d->stride_w == 1 && d->pad_h == 0 && d->pad_w == 0 &&
        d->c <= 128 && p * q % 8 == 0) {
        if (d->k % 64 == 0) return false;
        if (d->k % 32 == 0 && d->n * p * q >= 45000 &&
            (d->c <= 64 || p * q % 1024 == 0 || d->k >= 128 || (d->k >= 96 && d->n * p * q < 100000)) &&
            tap_dgrad_applies(ctx, d, 2))
            return false;
    }
    int64_t lo, hp, wp;
    axis_padding(d->h, p, d->pad_h, d->r, d->stride_h, d->dil_h, lo, hp);
    axis_padding(d->w, q, d->pad_w, d->s, d->stride_w, d->dil_w, lo, wp);
    if (!fits(d->n * hp * wp * d->k)) return false;
    // A long chain on few tiles, as in the forward: the tap kernel splits it ([4, 32,
    // 7, 7], k = 512, 3×3 stride 2, 48 stages on 2 tiles, 33 µs against 17; 24 stages on
    // 8 tiles 24 against 17, on 56 24 against 31), the other paths past 9 taps are
    // slower until about 100 stages (200 on 32 tiles 107 against 70, 100 on 15 equal).
    int64_t stages = 0, tiles = 0;
    for (int64_t a = 0; a < d->stride_h && a < d->h; ++a) {
        int64_t pos[kMaxTaps], sh[kMaxTaps], deep = 0;
        const int nr = axis_taps(a, d->pad_h, d->r, d->stride_h, d->dil_h, pos, sh);
        for (int64_t b = 0; b < d->stride_w && b < d->w; ++b)
            deep += ceil_div(nr * axis_taps(b, d->pad_w, d->s, d->stride_w, d->dil_w, pos, sh) * d->k, BK);
        stages = std::max(stages, deep);
        tiles += row_tiles(ctx, d->n * ceil_div(d->h - a, d->stride_h) * ceil_div(d->w, d->stride_w), d->c, d->stride_h);
    }
    if (d->r * d->s > 9) return stages <= 100 || tiles > 64;
    return stages < 12 || 20 * stages <= 120 + 11 * tiles || !tap_dgrad_applies(ctx, d, 2);
}

int rows_fwd(nott_ctx ctx, const nott_conv2d_desc* d, int64_t p, int64_t q, const bf16_t* x, const bf16_t* w,
             const float* b, bf16_t* y, int relu) {
    const Gather g(d, p, q);
    const int64_t taps = d->r * d->s;
    const int64_t xb = align256(2 * d->n * g.hp * g.wp * d->c);
    char* ws = static_cast<char*>(optional_workspace(ctx, (size_t)(xb + 2 * d->k * d->c * taps)));
    if (!ws) return NOTT_ERR_ALLOC;
    PrepParams<bf16_t> pp{};
    pp.part[0] = part_of(x, reinterpret_cast<bf16_t*>(ws), d->n, d->c, d->h, d->w, g.hp, g.wp, d->pad_h, d->pad_w,
                         g.sh, g.sw);
    pp.wt = w;
    pp.wp2 = reinterpret_cast<bf16_t*>(ws + xb);
    pp.k = (int32_t)d->k; pp.cin = (int32_t)d->c; pp.taps = (int32_t)taps;
    const int st = launch_prep(ctx, pp);
    if (st != NOTT_OK) return st;
    RowParams rp{};
    rp.xp = pp.part[0].xp; rp.w = pp.wp2; rp.out = y; rp.bias = b; rp.relu = relu;
    rp.N = (int32_t)d->k; rp.fc = FastDiv((uint32_t)d->c); rp.ncls = 1;
    rp.sn = (int32_t)(g.hp * g.wp * d->c); rp.si = (int32_t)(g.ph * g.wp * d->c); rp.sj = (int32_t)(g.pw * d->c);
    rp.on = (int32_t)(d->k * p * q); rp.oc = (int32_t)(p * q); rp.oi = (int32_t)q; rp.wlim = (int32_t)q;
    rp.vec = store_width(y, p * q, 0, 0, 0, 0);
    RowClass& c = rp.cls[0];
    c.M = (int32_t)(d->n * p * q); c.K[0] = (int32_t)(taps * d->c);
    c.fij = FastDiv((uint32_t)(p * q)); c.fj = FastDiv((uint32_t)q);
    for (int64_t i = 0; i < taps; ++i)
        c.taps[0][i] = (int32_t)(((i / d->s) * d->dil_h * g.wp + (i % d->s) * d->dil_w) * d->c);
    return launch_rows(ctx, rp, 1);
}

int rows_dgrad(nott_ctx ctx, const nott_conv2d_desc* d, int64_t p, int64_t q, const bf16_t* dy, const bf16_t* w,
               bf16_t* dx) {
    const int64_t taps = d->r * d->s;
    int64_t pt, pl, hp, wp;
    axis_padding(d->h, p, d->pad_h, d->r, d->stride_h, d->dil_h, pt, hp);
    axis_padding(d->w, q, d->pad_w, d->s, d->stride_w, d->dil_w, pl, wp);
    const int64_t xb = align256(2 * d->n * hp * wp * d->k);
    char* ws = static_cast<char*>(optional_workspace(ctx, (size_t)(xb + 2 * d->k * d->c * taps)));
    if (!ws) return NOTT_ERR_ALLOC;
    PrepParams<bf16_t> pp{};
    pp.part[0] = part_of(dy, reinterpret_cast<bf16_t*>(ws), d->n, d->k, p, q, hp, wp, pt, pl);
    pp.wt = w;
    pp.wp2 = reinterpret_cast<bf16_t*>(ws + xb);
    pp.k = (int32_t)d->k; pp.cin = (int32_t)d->c; pp.taps = (int32_t)taps; pp.by_cin = 1;
    RowParams rp{};
    rp.xp = pp.part[0].xp; rp.w = pp.wp2; rp.out = dx;
    rp.N = (int32_t)d->c; rp.fc = FastDiv((uint32_t)d->k);
    rp.sn = (int32_t)(hp * wp * d->k); rp.si = (int32_t)(wp * d->k); rp.sj = (int32_t)d->k;
    rp.on = (int32_t)(d->c * d->h * d->w); rp.oc = (int32_t)(d->h * d->w);
    rp.oi = (int32_t)(d->stride_h * d->w); rp.wlim = (int32_t)d->w;
    // one run per image and channel where all rows are taken, else one per row
    rp.vec = d->stride_h == 1 && d->w % d->stride_w == 0 ? store_width(dx, d->h * d->w, 0, 0, 0, 0)
                                                         : store_width(dx, d->w, 0, 0, 0, 0);
    const int products = (int)d->stride_w;
    const int64_t nj = ceil_div(d->w, d->stride_w);
    int64_t woff = 0;
    for (int64_t a = 0; a < d->stride_h && a < d->h; ++a) {
        RowClass& c = rp.cls[rp.ncls++];
        const int64_t ni = ceil_div(d->h - a, d->stride_h);
        c.M = (int32_t)(d->n * ni * nj);
        c.fij = FastDiv((uint32_t)(ni * nj)); c.fj = FastDiv((uint32_t)nj);
        c.o0 = (int32_t)(a * d->w);
        for (int64_t bb = 0; bb < d->stride_w && bb < d->w; ++bb) {
            int64_t pr[kMaxTaps], sr[kMaxTaps], ps[kMaxTaps], ss[kMaxTaps];
            const int nr = axis_taps(a, d->pad_h, d->r, d->stride_h, d->dil_h, pr, sr);
            const int ns = axis_taps(bb, d->pad_w, d->s, d->stride_w, d->dil_w, ps, ss);
            c.K[bb] = (int32_t)(nr * ns * d->k);
            c.woff[bb] = (int32_t)woff;
            for (int i = 0; i < nr; ++i)
                for (int j = 0; j < ns; ++j) {
                    const int t = i * ns + j, tap = (int)(pr[i] * d->s + ps[j]);
                    c.taps[bb][t] = (int32_t)(((sr[i] + pt) * wp + ss[j] + pl) * d->k);
                    pp.base[tap] = (int32_t)woff;
                    pp.nt[tap] = nr * ns;
                    pp.t[tap] = t;
                }
            woff += (int64_t)nr * ns * d->k * d->c;
        }
    }
    const int st = launch_prep(ctx, pp);
    if (st != NOTT_OK) return st;
    return launch_rows(ctx, rp, products);
}

template <typename T>
int rows_wgrad(nott_ctx ctx, const nott_conv2d_desc* d, int64_t p, int64_t q, const T* x, const T* dy, float* dw,
               int accumulate) {
    constexpr int BK = Slices<T>::kStageK;
    const Gather g(d, p, q);
    const int64_t taps = d->r * d->s;
    const int64_t M = d->k, N = taps * d->c, K = d->n * p * q;
    const int64_t tiles = ceil_div(M, BM) * ceil_div(N, 128), nkb = ceil_div(K, BK);
    // Splits: rounds of workgroups × (stages × a stage + 3.2 µs), the partials' write
    // and read, and 0.04 µs a split for the sum over a small result's partials ([16,
    // 96, 40, 40], 1×1, 96 outputs: 25 µs at 64 splits, 30 at 200); at most kMaxPixels
    // pixels each.  A stage is 0.6 to 1.2 µs in bf16 (loads), 2.1 in fp32: its MFMAs
    // alone are 128·128·32 multiply-adds at 128 a cycle, 1.7 µs at 2.4 GHz.
    int64_t stages = 0;
    float best = 0.f;
    for (int64_t s = 1; s <= std::max<int64_t>(ctx->num_cu, ceil_div(K, kMaxPixels)); ++s) {
        const int64_t per = ceil_div(nkb, s), n = ceil_div(nkb, per);
        if (per * BK > kMaxPixels) continue;
        const float fill = std::min(1.f, (float)(tiles * n) / (float)ctx->num_cu);
        const float us = (float)ceil_div(tiles * n, ctx->num_cu) * ((float)per * (sizeof(T) == 2 ? 0.63f + 0.53f * fill : 2.1f) + 3.2f) +
                         8.f * (float)(n * M * N) / 7.85e6f + 0.04f * (float)n;
        if (best == 0.f || us < best) {
            best = us;
            stages = per;
        }
    }
    const int64_t splits = ceil_div(nkb, stages);
    const int64_t xb = align256((int64_t)sizeof(T) * d->n * g.hp * g.wp * d->c), yb = align256((int64_t)sizeof(T) * K * M);
    char* ws = static_cast<char*>(optional_workspace(ctx, (size_t)(xb + yb + 4 * splits * M * N)));
    if (!ws) return NOTT_ERR_ALLOC;
    PrepParams<T> pp{};
    pp.part[0] = part_of(x, reinterpret_cast<T*>(ws), d->n, d->c, d->h, d->w, g.hp, g.wp, d->pad_h, d->pad_w,
                         g.sh, g.sw);
    pp.part[1] = part_of(dy, reinterpret_cast<T*>(ws + xb), d->n, d->k, p, q, p, q, 0, 0);
    const int st = launch_prep(ctx, pp);
    if (st != NOTT_OK) return st;
    WgradParams<T> wg{};
    wg.dyt = reinterpret_cast<const T*>(ws + xb);
    wg.xp = reinterpret_cast<const T*>(ws);
    wg.M = (int32_t)M; wg.N = (int32_t)N; wg.K = (int32_t)K;
    wg.kps = (int32_t)(stages * BK); wg.splits = (int32_t)splits;
    wg.fij = FastDiv((uint32_t)(p * q)); wg.fj = FastDiv((uint32_t)q); wg.fc = FastDiv((uint32_t)d->c);
    wg.sn = (int32_t)(g.hp * g.wp * d->c); wg.si = (int32_t)(g.ph * g.wp * d->c);
    wg.sj = (int32_t)(g.pw * d->c);
    for (int64_t i = 0; i < taps; ++i)
        wg.taps[i] = (int32_t)(((i / d->s) * d->dil_h * g.wp + (i % d->s) * d->dil_w) * d->c);
    wg.ws = reinterpret_cast<float*>(ws + xb + yb);
    constexpr size_t kLds = (size_t)S * 2 * 128 * 128 + 4 * kMaxPixels;
    const size_t lds = (size_t)S * 2 * 128 * 128 + 4 * (size_t)wg.kps;
    static bool attr = false;
    if (!attr) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_wgrad_rows_kernel<T>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds) != hipSuccess)
            return fail(ctx, NOTT_ERR_HIP, "conv_gemm: cannot reserve LDS");
        attr = true;
    }
    hipLaunchKernelGGL(conv_wgrad_rows_kernel<T>, dim3((unsigned)(tiles * splits)), dim3(64 * NW), lds, ctx->stream, wg);
    gemm::launch_splitk_reduce(ctx, wg.ws, splits, M, N,
                               TapMajorStore{dw, wg.fc, (int32_t)d->c, (int32_t)taps, accumulate});
    return launch_status(ctx, "conv_gemm wgrad");
}

template int rows_wgrad<float>(nott_ctx, const nott_conv2d_desc*, int64_t, int64_t, const float*, const float*, float*,
                               int);
template int rows_wgrad<bf16_t>(nott_ctx, const nott_conv2d_desc*, int64_t, int64_t, const bf16_t*, const bf16_t*,
                                float*, int);

}  // namespace conv_fast
}  // namespace nott
