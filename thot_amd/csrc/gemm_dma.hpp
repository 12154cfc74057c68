// bf16 MFMA GEMM with direct-to-LDS operand fills (gfx950).
//
//   C[M×N] = Σ_k A(m, k)·B(n, k),  fp32 accumulate, bf16 operands:
//   A(m, k) = A[m·lda + k]  (AT = false)   or   A[k·lda + m]  (AT = true)
//   B(n, k) = B[n·ldb + k]  (BT = false)   or   B[k·ldb + n]  (BT = true)
//
// Work decomposition.  A workgroup owns a BM×BN output tile and walks K in
// 64-deep stages; its WM×WN waves each own a (BM/WM)×(BN/WN) sub-tile made
// of 32×32 v_mfma_f32_32x32x16_bf16 blocks (one 32×32×16 product per issue).
//
// Fills.  Operands go from global memory straight into LDS with
// global_load_lds_dwordx4: one instruction moves 1 KB (16 bytes per lane,
// lane i to byte 16·i of a wave-uniform LDS base), so no VGPRs, no VALU
// repacking and no ds_write are spent on staging.  The lane→global mapping
// is chosen so that the 1 KB blocks land in a swizzled layout:
//   k-contiguous operand (AT/BT false), tile [row][k] (128 bytes per row):
//     16-byte chunk c (k = 8c..8c+7) of row r at r·128 + ((c ^ ((r>>1)&7))·16);
//     a 32×32×16 operand read (rows r0..r0+31, chunk 2s + lane/32) hits 16
//     distinct 16-byte slots in every quarter-wave.
//   row-contiguous operand (AT/BT true), tile [k][row] (2·R bytes per k):
//     chunk cr (rows 8cr..8cr+7) of k-row k at k·2R + ((cr ^ 4·(k&3))·16);
//     operands are read with ds_read_b64_tr_b16, which hands lane i of each
//     16-lane group the 4 k-consecutive values of row i from a [k][row]
//     block, i.e. the MFMA operand layout, so no transpose is ever stored.
// Stages form an S-deep ring: the loads of stage t+S-1 go into the slot of
// stage t-1 once every wave has passed the barrier that follows its last read
// of it, so S-1 stages are in flight while one is multiplied.  A 3-deep ring
// issues them in three parts between the slices of stage t (a burst of them
// after the barrier stalled the issuing waves: 8192x1024, K = 3072 60 -> 56 us);
// a 2-deep one at once, as they are needed a stage later.  Only s_waitcnt vmcnt
// (how many of this wave's loads may still be outstanding) and s_barrier order
// the ring; the compiler's workgroup fence (which would wait for every load) is
// not used, and the DMA is issued as inline assembly (see dma16).  Within a
// stage the four 16-deep slices are software-pipelined: the fragments of slice
// s+1 are read while slice s is multiplied.  The last stage of a K that is no
// multiple of 64 is filled up with zeros.
//
// Tile order.  Workgroups are dispatched round-robin over the 8 XCDs (each
// with its own L2); the linear tile index is remapped so that each XCD gets
// a contiguous band of tiles (grouped `gm` tile-rows at a time) and its L2
// holds the A rows and B columns that band shares.
#pragma once

#include "gemm.hpp"
#include "lds_dma.hpp"

namespace nott {
namespace gemm {
namespace dma {

constexpr int BK = 64;

using lds::barrier;
using lds::dma16;
using lds::lds_addr;
using lds::wait_vm_lgkm0;

// Issues block qq of this wave's share of one operand tile (R rows × 64 k, its
// NB = R/8 1 KB blocks dealt to the NW waves in turn) of stage k0.  Rows past
// `rows` are clamped to the last row (their results are never stored);
// row-contiguous operands need rows % 8 == 0 and rows >= 8.  TAIL: the stage
// may reach past K; its 16-byte chunks from K on (a k-contiguous operand's K is
// a multiple of 8) are filled with zeros.
static __device__ u32x4 zero_chunk;

template <bool TR, int R, int NW, bool TAIL>
__device__ __forceinline__ void fill_block(int qq, const bf16_t* __restrict__ p, int64_t ld, int64_t row0,
                                           int64_t rows, int64_t k0, int64_t K, char NOTT_LDS* dst, int wid,
                                           int lane) {
    constexpr int NB = R / 8;
    static_assert(NB % NW == 0, "tile blocks must split evenly over the waves");
    const int q = qq * NW + wid;
    const bf16_t* src;
    if constexpr (!TR) {
        const int r = 8 * q + (lane >> 3);
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        int64_t gr = row0 + r;
        gr = gr < rows ? gr : rows - 1;
        src = p + gr * ld + k0 + 8 * c;
        if (TAIL && k0 + 8 * c >= K) src = reinterpret_cast<const bf16_t*>(&zero_chunk);
    } else {
        static_assert(R >= 128, "row-contiguous tiles need at least 128 rows");
        constexpr int KPB = 1024 / (2 * R);   // k-rows per block
        const int b = 16 * lane;
        const int k = q * KPB + b / (2 * R);
        const int cr = ((b % (2 * R)) >> 4) ^ ((k & 3) << 2);
        int64_t gc = row0 + 8 * cr;
        gc = gc <= rows - 8 ? gc : rows - 8;
        src = p + (k0 + k) * ld + gc;
        if (TAIL && k0 + k >= K) src = reinterpret_cast<const bf16_t*>(&zero_chunk);
    }
    dma16(src, lds_addr(dst) + 1024 * q);
}

// A 32×16 MFMA operand (lane l: row l % 32, k = 8·(l/32) + 0..7): one
// 16-byte read from a [row][k] tile, or two transposing 8-byte reads from a
// [k][row] tile.
typedef short v4i16 __attribute__((ext_vector_type(4)));
template <bool TR> struct Frag;
template <> struct Frag<false> {
    u32x4 v;
    __device__ __forceinline__ bf16x8 get() const { return __builtin_bit_cast(bf16x8, v); }
    __device__ __forceinline__ void ld(const char NOTT_LDS* p) { v = *reinterpret_cast<const u32x4 NOTT_LDS*>(p); }
};
template <> struct Frag<true> {
    v4i16 lo, hi;
    __device__ __forceinline__ bf16x8 get() const {
        const v4i16 w[2] = {lo, hi};
        return __builtin_bit_cast(bf16x8, w);
    }
    __device__ __forceinline__ void ld(const char NOTT_LDS* p, int hi_off) {
        lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4i16 NOTT_LDS*)p);
        hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4i16 NOTT_LDS*)(p + hi_off));
    }
};

// Per-lane LDS byte offsets of one operand's fragments inside a stage tile
// (R rows; this wave's rows start at w0; F fragments of 32 rows).
//   [row][k] tile: fragment f, slice s at off[s] + 4096·f, where
//     off[s] = (w0 + l%32)·128 + ((2s + l/32) ^ ((l>>1)&7))·16
//     (w0 + 32f is a multiple of 16, so the swizzle depends on l only).
//   [k][row] tile: fragment f, slice s, half h at off[f] + (16s + 4h)·2R, where
//     off[f] = k·2R + (((r>>3) ^ 4·(k&3))·16) + (r&7)·2 with
//     r = w0 + 32f + 16·((l>>4)&1) + 4·(l&3), k = 8·(l/32) + ((l&15)>>2).
template <bool TR, int R, int F>
struct FragAddr {
    uint32_t off[TR ? F : 4];
    __device__ __forceinline__ void init(int w0, int lane) {
        if constexpr (!TR) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
                off[s] = (uint32_t)((w0 + (lane & 31)) * 128 + ((((2 * s) | (lane >> 5)) ^ ((lane >> 1) & 7)) << 4));
        } else {
            const int k = 8 * (lane >> 5) + ((lane & 15) >> 2);
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const int r = w0 + 32 * f + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
                off[f] = (uint32_t)(k * (2 * R) + (((r >> 3) ^ ((k & 3) << 2)) << 4) + (r & 7) * 2);
            }
        }
    }
    // Reads fragment FI of slice S of the tile at `base`.
    template <int S, int FI>
    __device__ __forceinline__ void read(Frag<TR>& d, const char NOTT_LDS* base) const {
        if constexpr (!TR) d.ld(base + off[S] + 4096 * FI);
        else d.ld(base + off[FI] + 16 * S * 2 * R, 4 * 2 * R);
    }
};

template <int S, bool TR, int R, int F, int I = 0>
__device__ __forceinline__ void read_all(Frag<TR> (&d)[F], const FragAddr<TR, R, F>& a, const char NOTT_LDS* base) {
    if constexpr (I < F) {
        a.template read<S, I>(d[I], base);
        read_all<S, TR, R, F, I + 1>(d, a, base);
    }
}

// Maps the linear workgroup index to its split and tile: the workgroups of an
// XCD (every eighth) take one contiguous run of the order split-major, then
// grouped `gm` tile-rows at a time, so that an XCD's L2 serves few k ranges and
// a compact block of tiles of each.  (With the splits outermost over all XCDs,
// every XCD read a part of every k range: 3072x1024, K = 8192 in 4 splits.)  Any
// count is shared out so: 252 workgroups in order, 18 tiles of 768x768, K = 32768 in
// 14 splits, took 81 us, 52 this way.
// Where the operands are small (by_tile) an XCD takes the same tiles of all splits:
// 2048x1024, K = 1024 in 4 splits 19.0 us against 20.1, 512x768, K = 3072 in 8 16
// against 18; with 61 MB of operands, 512x256, K = 40000 in 32, 33 against 24.
__device__ __forceinline__ void tile_of(int id, int tm, int tn, int splits, int gm, int by_tile, int& pm, int& pn,
                                        int& z) {
    const int nt = tm * tn, all = by_tile ? nt : nt * splits;
    if (by_tile) z = id / nt, id -= z * nt;
    id = (id & 7) * (all >> 3) + min(id & 7, all & 7) + (id >> 3);   // the first all % 8 XCDs have one more
    if (!by_tile) z = id / nt, id -= z * nt;
    const int per_group = gm * tn;
    const int g = id / per_group;
    const int first = g * gm;
    const int gsz = min(tm - first, gm);
    const int in = id - g * per_group;
    pm = first + in % gsz;
    pn = in / gsz;
}

// Split-K partials ws[split][m][n], and with row sums rows[split][m]; at() is
// the store of one split.
struct PartialRowStore {
    float* ws;
    float* rows;
    int64_t M, N;
    __device__ __forceinline__ PartialRowStore at(int z) const { return {ws + z * M * N, rows + z * M, M, N}; }
    __device__ __forceinline__ void store(int64_t m, int64_t n, float v) const {
        if (m < M && n < N) ws[m * N + n] = v;
    }
    __device__ __forceinline__ void rowsum(int64_t m, float v) const {
        if (m < M) rows[m] = v;
    }
};
template <class EP>
__device__ __forceinline__ const EP& at_split(const EP& ep, int) { return ep; }
__device__ __forceinline__ PartialRowStore at_split(const PartialRowStore& ep, int z) { return ep.at(z); }

// Sum of the 8 bf16 values of an operand fragment, in k order.
__device__ __forceinline__ void add_bf16x2(float& s, uint32_t w) {
    s += __builtin_bit_cast(float, w << 16);
    s += __builtin_bit_cast(float, w & 0xffff0000u);
}
__device__ __forceinline__ void add_frag(float& s, const Frag<false>& f) {
    add_bf16x2(s, f.v.x);
    add_bf16x2(s, f.v.y);
    add_bf16x2(s, f.v.z);
    add_bf16x2(s, f.v.w);
}
__device__ __forceinline__ void add_frag(float& s, const Frag<true>& f) {
    const u32x4 w = __builtin_bit_cast(u32x4, f.get());
    add_bf16x2(s, w.x);
    add_bf16x2(s, w.y);
    add_bf16x2(s, w.z);
    add_bf16x2(s, w.w);
}

template <class EP> struct IsBf16RowMajor { static constexpr bool value = false; };
template <> struct IsBf16RowMajor<RowMajorStore<bf16_t>> { static constexpr bool value = true; };

// Stores a wave's TM×64 block of a bf16 result.  acc holds transposed 32×32
// blocks (the MFMA operands exchanged): lane l has row l % 32 and, in
// register 4q + e, column 8q + 4·(l/32) + e, so four consecutive columns round
// to one 8-byte LDS write.  Staged as [row][64] with the 16-byte chunk at
// chunk ^ (row & 7) and its halves exchanged on rows with bit 3 set (16 lanes
// writing 16 rows hit every bank once), then written as whole 128-byte row
// pieces: 16 bytes per lane where C's rows allow it, else element by element
// with a row's 64 columns side by side.  Against 2-byte stores straight from
// the accumulators: 8192x1024->3072 with bias 115 -> 82 us (most of it the
// bias, see RowMajorStore), its data gradient 68 -> 66 us.
template <int TM, int FM, int FN, class EP>
__device__ __forceinline__ void store_tile(const EP& ep, const f32x16 (&acc)[FM][FN], char NOTT_LDS* buf, int64_t m0,
                                           int64_t n0, int lane) {
    const int r = lane & 31, h = lane >> 5;
    wait_vm_lgkm0<0>();   // this wave has read its last stage;
    barrier();            // every wave has: the ring is free
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        float cv[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) cv[e] = ep.column(n0 + 32 * j + 8 * (e >> 2) + 4 * h + (e & 3));
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int row = 32 * i + r;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = ep.finish(acc[i][j][4 * q + e], cv[4 * q + e]);
                const u32x2 w = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
                *reinterpret_cast<u32x2 NOTT_LDS*>(buf + row * 128 + (((4 * j + q) ^ (row & 7)) << 4) +
                                                   ((h ^ ((row >> 3) & 1)) << 3)) = w;
            }
        }
    }
    const bool vec = ep.ldc % 8 == 0 && ep.N % 8 == 0 && ((uintptr_t)ep.c % 16) == 0 &&
                     (!ep.mask || ((uintptr_t)ep.mask % 16) == 0);
    if (vec) {
        const int c = lane & 7;
        const int64_t n = n0 + 8 * c;
#pragma unroll
        for (int it = 0; it < TM / 8; ++it) {
            const int row = 8 * it + (lane >> 3);
            const int64_t m = m0 + row;
            u32x4 w = *reinterpret_cast<const u32x4 NOTT_LDS*>(buf + row * 128 + ((c ^ (row & 7)) << 4));
            if ((row >> 3) & 1) w = u32x4{w.z, w.w, w.x, w.y};
            if (m >= ep.M || n >= ep.N) continue;
            if (ep.mask) {
                const u32x4 k = *reinterpret_cast<const u32x4*>(ep.mask + m * ep.ldc + n);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (__builtin_bit_cast(float, k[e] << 16) <= 0.f) w[e] &= 0xffff0000u;
                    if (__builtin_bit_cast(float, k[e] & 0xffff0000u) <= 0.f) w[e] &= 0xffffu;
                }
            }
            *reinterpret_cast<u32x4*>(ep.c + m * ep.ldc + n) = w;
        }
    } else {
        const int64_t n = n0 + lane;
        for (int row = 0; row < TM; ++row) {
            const int64_t m = m0 + row;
            if (m >= ep.M || n >= ep.N) continue;
            const int b = row * 128 + (((lane >> 3) ^ (row & 7)) << 4) + ((((lane >> 2) & 1) ^ ((row >> 3) & 1)) << 3) +
                          (lane & 3) * 2;
            bf16_t v = *reinterpret_cast<const bf16_t NOTT_LDS*>(buf + b);
            if (ep.mask && bf16_to_f32(ep.mask[m * ep.ldc + n]) <= 0.f) v = 0;
            ep.c[m * ep.ldc + n] = v;
        }
    }
}

// grid: tiles (tm·tn) times k splits of kps (a multiple of BK) each.  TAIL: K is
// not a multiple of 64 (a test at every fill, and the other fill's addresses, cost 2
// to 5%: 1080x1000, K = 2368 21.3 us against 20.3 without).
// ROWSUM: also Σ_k A(m, k) for every row m of the tile (the bias gradient
// when A is the output gradient of a Linear), summed in fp32 from the A
// fragments already in registers: only the tiles of tile column 0 sum, and
// there fragment f's sum is kept by wave column f % WN, so each row is
// summed once; the two k-halves of a row are held by lanes l and l+32 and
// combined at the end; the epilogue receives it via ep.rowsum(m, v).
template <bool AT, bool BT, int BM, int BN, int WM, int WN, int S, bool ROWSUM, bool TAIL, class EP>
__global__ __launch_bounds__(64 * WM * WN) void gemm_kernel(const bf16_t* __restrict__ A, int64_t lda,
                                                             const bf16_t* __restrict__ B, int64_t ldb, EP ep0,
                                                             int64_t M, int64_t N, int64_t K, int64_t kps, int splits,
                                                             int gm, int by_tile) {
    constexpr int NW = WM * WN;
    constexpr int TM = BM / WM, TN = BN / WN;
    constexpr int FM = TM / 32, FN = TN / 32;
    constexpr int A_BYTES = BM * 128, B_BYTES = BN * 128, STAGE = A_BYTES + B_BYTES;
    constexpr int LOADS = (BM / 8 + BN / 8) / NW;   // global_load_lds per wave per stage
    static_assert(TM % 32 == 0 && TN % 32 == 0, "wave tiles are whole 32x32 blocks");
    static_assert(S >= 2 && (S - 2) * LOADS < 64, "ring depth");
    // bf16 results: transposed accumulators, stored through LDS (store_tile)
    constexpr bool SWAP = IsBf16RowMajor<EP>::value && !ROWSUM;
    static_assert(!SWAP || (TN == 64 && NW * TM * 128 <= S * STAGE), "the staged output tile fits the ring");
    extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
    char NOTT_LDS* smem = (char NOTT_LDS*)smem_raw;

    const int tm = (int)((M + BM - 1) / BM), tn = (int)((N + BN - 1) / BN);
    int pm, pn, z;
    tile_of((int)blockIdx.x, tm, tn, splits, gm, by_tile, pm, pn, z);
    const EP ep = at_split(ep0, z);
    const int64_t m0 = (int64_t)pm * BM, n0 = (int64_t)pn * BN;
    const int64_t kb = (int64_t)z * kps;
    const int64_t ke = kb + kps < K ? kb + kps : K;
    const int nk = ke > kb ? (int)((ke - kb + BK - 1) / BK) : 0;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int wm = wid / WN, wn = wid % WN;

    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    // Issues loads [from, to) of this wave's LOADS for stage t.
    constexpr int LA = BM / 8 / NW;
    auto issue = [&](int t, int slot, int from, int to) {
        char NOTT_LDS* st = smem + slot * STAGE;
        const int64_t k0 = kb + (int64_t)t * BK;
        if (!TAIL || k0 + BK <= K) {
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                if (i < from || i >= to) continue;
                if (i < LA) fill_block<AT, BM, NW, false>(i, A, lda, m0, M, k0, K, st, wid, lane);
                else fill_block<BT, BN, NW, false>(i - LA, B, ldb, n0, N, k0, K, st + A_BYTES, wid, lane);
            }
        } else {
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                if (i < from || i >= to) continue;
                if (i < LA) fill_block<AT, BM, NW, true>(i, A, lda, m0, M, k0, K, st, wid, lane);
                else fill_block<BT, BN, NW, true>(i - LA, B, ldb, n0, N, k0, K, st + A_BYTES, wid, lane);
            }
        }
    };
    FragAddr<AT, BM, FM> fa;
    FragAddr<BT, BN, FN> fb;
    fa.init(wm * TM, lane);
    fb.init(wn * TN, lane);

    Frag<AT> a[2][FM];
    Frag<BT> b[2][FN];
    float rs[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) rs[i] = 0.f;
    auto mma = [&](int p) {
        if constexpr (ROWSUM) {
            if (pn == 0) {
#pragma unroll
                for (int i = 0; i < FM; ++i)
                    if (i % WN == wn) add_frag(rs[i], a[p][i]);
            }
        }
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                acc[i][j] = SWAP ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[p][j].get(), a[p][i].get(), acc[i][j], 0, 0, 0)
                                 : __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[p][i].get(), b[p][j].get(), acc[i][j], 0, 0, 0);
    };

    // Stages 0..S-2 are in flight before the loop.  The loads of stage t+S
    // go into slot t % S once every wave has passed the barrier that follows
    // its last read of stage t.
#pragma unroll
    for (int s = 0; s < S - 1; ++s)
        if (s < nk) issue(s, s, 0, LOADS);
    if (nk > 0) {
        if (nk >= S - 1) wait_vm_lgkm0<(S - 2) * LOADS>();
        else wait_vm_lgkm0<0>();
        barrier();
        read_all<0>(a[0], fa, smem);
        read_all<0>(b[0], fb, smem + A_BYTES);
    }
    // The refill of a freed slot (stage t+S-1 while stage t is multiplied) is
    // issued in three parts between the slices.
    constexpr int P1 = S == 2 ? LOADS : (LOADS + 2) / 3, P2 = S == 2 ? LOADS : (2 * LOADS + 2) / 3;
    int slot = 0, free = S - 1;   // ring slots of stage t and of the refill
    for (int t = 0; t < nk; ++t) {
        const char NOTT_LDS* sa = smem + slot * STAGE;
        const char NOTT_LDS* sb = sa + A_BYTES;
        const bool more = t + S - 1 < nk;
        read_all<1>(a[1], fa, sa);
        read_all<1>(b[1], fb, sb);
        if (more) issue(t + S - 1, free, 0, P1);
        mma(0);
        read_all<2>(a[0], fa, sa);
        read_all<2>(b[0], fb, sb);
        if (more) issue(t + S - 1, free, P1, P2);
        mma(1);
        read_all<3>(a[1], fa, sa);
        read_all<3>(b[1], fb, sb);
        if (more) issue(t + S - 1, free, P2, LOADS);
        mma(0);
        const int nslot = slot + 1 == S ? 0 : slot + 1;
        if (t + 1 < nk) {
            // Stage t+1 must have landed; stages t+2 .. t+S-1 may be in flight.
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
    if constexpr (ROWSUM) {
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            if (pn != 0 || i % WN != wn) continue;
            const float v = rs[i] + __shfl_xor(rs[i], 32);
            if (lane < 32) ep.rowsum(m0 + wm * TM + 32 * i + lane, v);
        }
    }
    if constexpr (SWAP) {
        store_tile<TM, FM, FN>(ep, acc, smem + wid * (TM * 128), m0 + wm * TM, n0 + wn * TN, lane);
        return;
    }
    // Accumulator layout of a 32×32 block: lane l holds column l % 32 and,
    // in register 4q + e, row 8q + 4·(l/32) + e.
    const int col = lane & 31, rh = (lane >> 5) * 4;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    ColumnOf<EP>::store(ep, m0 + wm * TM + 32 * i + 8 * q + rh + e, n0 + wn * TN + 32 * j + col,
                                        acc[i][j][4 * q + e], 0);
}

template <bool AT, bool BT, int BM, int BN, int WM, int WN, int S>
struct Config {
    static constexpr bool kAT = AT, kBT = BT;
    static constexpr int kBM = BM, kBN = BN, kWM = WM, kWN = WN, kS = S;
    static constexpr int kThreads = 64 * WM * WN;
    static constexpr size_t kLds = (size_t)S * (BM + BN) * 128;
};

// Tile shapes the dispatcher picks from: 256×256 with 8 waves of 128×64 and a
// 2-deep ring (128 KB of LDS), 256×128 with 8 waves of 64×64 and a 3-deep ring
// (144 KB), 128×128 with 4 waves and a 3-deep ring (96 KB, one workgroup per
// CU) or a 2-deep one (64 KB, two per CU).
enum class Shape { T256x256, T256x128, T128x128, T128x128x2 };

struct Plan {
    Shape shape;
    int64_t splits, kps;
};

// Picks the tile shape and the split-K count with the least estimated time:
//   rounds of workgroups × (64-deep stages × stage + tile),
//   stage: idle + load · (how much of the chip's slots is filled), the load
//   another where both operands are row-contiguous (both_tr, weight gradients),
//   and more with the row sums (rowsum);
//   tile: the first fill and the output; for a split also the second launch
//   with a chain over the partials, the partials' write and read, and uneven
//   splits, of which the 8 XCDs share some (tile_of).
// The constants (us) are a fit to each shape and split forced on 118 products of
// 128..65536 rows, 128..8192 columns and K = 64..65536, forward and both gradients,
// with inputs changing from call to call; the pick is 0.7% off the best of them in
// the mean (at most 12%).  A pick of at most 16 splits with constants from fewer
// products was 2.9% off (34%): weight gradients of 16384 tokens, 256 → 256, 20 us
// against 16, 128 → 1024 23 against 18, of 65536 tokens, 128 → 128, 56 against 20.
inline Plan plan(nott_ctx ctx, int64_t M, int64_t N, int64_t K, bool both_tr, bool rowsum, int64_t splits) {
    struct Cost {
        Shape shape;
        int bm, bn, per_cu;
        float idle, load, load_tr, rows, tile;
    };
    static constexpr Cost kCosts[] = {
        {Shape::T256x256, 256, 256, 1, 1.31f, 0.08f, 0.015f, 0.14f, 6.6f},
        {Shape::T256x128, 256, 128, 1, 0.73f, 0.06f, 0.005f, 0.15f, 4.8f},
        {Shape::T128x128, 128, 128, 1, 0.50f, 0.14f, 0.03f, 0.51f, 3.0f},
        {Shape::T128x128x2, 128, 128, 2, 0.70f, 0.50f, 0.27f, 0.00f, 3.0f},
    };
    constexpr float kSplitUs = 1.8f, kUnevenUs = 1.4f, kPartialUs = 0.04f, kPartialRowsUs = 0.21f;
    constexpr float kPartialBytesPerUs = 5.9e6f;
    const int64_t nkb = ceil_div(K, BK);
    Plan best{Shape::T128x128, 1, K};
    float best_us = 0.f;
    for (const Cost& c : kCosts) {
        const int64_t tiles = ceil_div(M, c.bm) * ceil_div(N, c.bn), slots = (int64_t)ctx->num_cu * c.per_cu;
        const float idle = c.idle + (rowsum ? c.rows : 0.f), load = both_tr ? c.load_tr : c.load;
        // past 16 in steps of a quarter of the power of two below: the best lie in a flat valley
        for (int64_t s = 1, step = 1; s <= 256; s += step) {
            if (s >= 16 && (s & (s - 1)) == 0) step = s / 4;
            const int64_t want = splits > 0 ? std::min(splits, std::min<int64_t>(nkb, 65535)) : s;
            if (want > 1 && splits <= 0 && nkb / want < 4) break;
            const int64_t stages = ceil_div(nkb, want), n = ceil_div(nkb, stages);
            const float fill = std::min(1.f, (float)(tiles * n) / (float)slots);
            float us = (float)ceil_div(tiles * n, slots) * ((float)stages * (idle + load * fill) + c.tile);
            if (n > 1)
                us += kSplitUs + (n % 8 && n != 2 && n != 4 ? kUnevenUs : 0.f) + (float)n * (rowsum ? kPartialRowsUs : kPartialUs) +
                      8.f * (float)(n * M * N) / kPartialBytesPerUs;
            if (best_us == 0.f || us < best_us) {
                best_us = us;
                best = Plan{c.shape, n, n > 1 ? stages * BK : K};
            }
            if (splits > 0) break;
        }
    }
    return best;
}

// Whether the operands qualify: 16-byte aligned bases and leading dimensions,
// k-contiguous operands in whole 8-k chunks and row-contiguous ones in whole
// 8-row groups, and at least 128 rows and columns (narrower products waste
// most of a tile).
template <bool AT, bool BT>
inline bool applies(const bf16_t* A, int64_t lda, const bf16_t* B, int64_t ldb, int64_t M, int64_t N, int64_t K) {
    auto ok16 = [](const void* p, int64_t ld) { return ((uintptr_t)p % 16) == 0 && (ld % 8) == 0; };
    if (K <= 0 || ((!AT || !BT) && K % 8 != 0) || !ok16(A, lda) || !ok16(B, ldb)) return false;
    if (M < 128 || N < 128) return false;
    if ((AT && M % 8 != 0) || (BT && N % 8 != 0)) return false;
    return ceil_div(M, 128) * ceil_div(N, 128) < (int64_t)1 << 26;   // tiles times splits in an int
}

template <class Cfg, bool ROWSUM, bool TAIL, class EP>
int launch_as(nott_ctx ctx, const bf16_t* A, int64_t lda, const bf16_t* B, int64_t ldb, const EP& ep, int64_t M,
           int64_t N, int64_t K, int64_t splits, int64_t kps) {
    auto fn = gemm_kernel<Cfg::kAT, Cfg::kBT, Cfg::kBM, Cfg::kBN, Cfg::kWM, Cfg::kWN, Cfg::kS, ROWSUM, TAIL, EP>;
    static bool attr = false;   // one setting per kernel instantiation
    if (!attr) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)Cfg::kLds) != hipSuccess)
            return fail(ctx, NOTT_ERR_HIP, "gemm_dma: cannot reserve LDS");
        attr = true;
    }
    const int64_t tiles = ceil_div(M, Cfg::kBM) * ceil_div(N, Cfg::kBN);
    const int64_t bytes = 2 * (M + N) * K;
    const int by_tile = splits > 1 && tiles % 8 == 0 && bytes >= 5000000 && bytes < 22000000;
    hipLaunchKernelGGL(fn, dim3((unsigned)(tiles * splits)), dim3(Cfg::kThreads), Cfg::kLds, ctx->stream, A, lda, B,
                       ldb, ep, M, N, K, kps, (int)splits, 4, by_tile);
    return launch_status(ctx, "gemm_dma");
}

template <class Cfg, bool ROWSUM, class EP>
int launch(nott_ctx ctx, const bf16_t* A, int64_t lda, const bf16_t* B, int64_t ldb, const EP& ep, int64_t M,
           int64_t N, int64_t K, int64_t splits, int64_t kps) {
    return K % BK ? launch_as<Cfg, ROWSUM, true>(ctx, A, lda, B, ldb, ep, M, N, K, splits, kps)
                  : launch_as<Cfg, ROWSUM, false>(ctx, A, lda, B, ldb, ep, M, N, K, splits, kps);
}

template <bool AT, bool BT, bool ROWSUM, class EP>
int launch_shape(nott_ctx ctx, Shape sh, const bf16_t* A, int64_t lda, const bf16_t* B, int64_t ldb, const EP& ep,
                 int64_t M, int64_t N, int64_t K, int64_t splits, int64_t kps) {
    switch (sh) {
        case Shape::T256x128:
            return launch<Config<AT, BT, 256, 128, 4, 2, 3>, ROWSUM>(ctx, A, lda, B, ldb, ep, M, N, K, splits, kps);
        case Shape::T256x256:
            return launch<Config<AT, BT, 256, 256, 2, 4, 2>, ROWSUM>(ctx, A, lda, B, ldb, ep, M, N, K, splits, kps);
        case Shape::T128x128x2:
            return launch<Config<AT, BT, 128, 128, 2, 2, 2>, ROWSUM>(ctx, A, lda, B, ldb, ep, M, N, K, splits, kps);
        default:
            return launch<Config<AT, BT, 128, 128, 2, 2, 3>, ROWSUM>(ctx, A, lda, B, ldb, ep, M, N, K, splits, kps);
    }
}

// C = A·B, or NOTT_ERR_UNSUPPORTED when the operands do not qualify (the
// caller then uses another engine).  Split-K partials go to the workspace and
// are summed in split order by the reduce kernel, which applies the epilogue.
// ROWSUM also hands ep.rowsum(m, Σ_k A(m, k)) for every row (see gemm_kernel).
template <bool AT, bool BT, bool ROWSUM = false, class EP>
int run(nott_ctx ctx, const bf16_t* A, int64_t lda, const bf16_t* B, int64_t ldb, const EP& ep, int64_t M, int64_t N,
        int64_t K, int64_t splits = 0) {
    if (M <= 0 || N <= 0) return NOTT_OK;
    if (!applies<AT, BT>(A, lda, B, ldb, M, N, K)) return NOTT_ERR_UNSUPPORTED;
    // The split reduce that also sums rows works on 4-column groups.
    if (ROWSUM && N % 4 != 0) splits = 1;
    Plan p = plan(ctx, M, N, K, AT && BT, ROWSUM, splits);
    const size_t body = (size_t)(p.splits * M * N), rows = ROWSUM ? (size_t)(p.splits * M) : 0;
    float* ws = p.splits > 1 ? static_cast<float*>(optional_workspace(ctx, sizeof(float) * (body + rows))) : nullptr;
    if (p.splits > 1 && !ws) p = plan(ctx, M, N, K, AT && BT, ROWSUM, 1);   // no room for the partials
    if (p.splits == 1) return launch_shape<AT, BT, ROWSUM>(ctx, p.shape, A, lda, B, ldb, ep, M, N, K, 1, p.kps);
    const int st = launch_shape<AT, BT, ROWSUM>(ctx, p.shape, A, lda, B, ldb, PartialRowStore{ws, ws + body, M, N}, M,
                                                N, K, p.splits, p.kps);
    if (st != NOTT_OK) return st;
    if constexpr (ROWSUM) launch_splitk_reduce(ctx, ws, p.splits, M, N, ep, ws + body);
    else launch_splitk_reduce(ctx, ws, p.splits, M, N, ep);
    return launch_status(ctx, "gemm_dma_splitk");
}

}  // namespace dma
}  // namespace gemm
}  // namespace nott
