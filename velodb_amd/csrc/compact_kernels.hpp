// compact_kernels.hpp -- device bodies and __global__ wrappers of the
// oblivious order-preserving compaction (ORCompact routing network), the
// Q6-style filter + exact int128 SUM and OP_SCATTER, used by compact.hip in
// launch mode and by the resident queue kernel.
//
// Reference method: oblivious_compact_elem / _inner_elem / _2power_inner_elem
// (obliviator/join/enclave/oblivious_compact.c:59-153, 327-338).  For a
// power-of-two n the recursion unrolls into log2(n) levels: at level q
// (block size s = 2^(q+1), half = 2^q) every aligned block [b, b+s) with
// offset o = C[b] mod s (C = exclusive prefix count of the selected rows)
// conditionally swaps rows b+i and b+half+i for all i < half, with
//   s == 2 : swap = (!sel[b] & sel[b+1]) ^ o
//   s  > 2 : m1 = C[b+half] - C[b], om = o mod half, om1 = (o+m1) mod half,
//            swap = ((om + m1 >= half) ^ (o >= half)) ^ (i >= om1)
// (the offset form of :88-105; the chain of :121-153 reduces to o = C[b]
// mod s for the blocks it creates).  With D = C[b+half] = C[b] + m1 the second
// form is one bit: om1 is D mod half, the first exclusive-or is bit q of D
// (C[b]'s bit q plus the carry of om + m1), and adding half-1-i to D carries
// into bit q exactly when i < om1, so
//   s  > 2 : swap = !bit q of (D + half - 1 - i).
// Every row is read and written at every level; the swap decision is a select,
// so addresses depend on n_pad only.
//
// Passes: count (selected rows per tile) -> tile scan -> local levels
// q < T_LOG inside each tile (LDS) -> fused global levels, S per HBM pass,
// rows at stride 2^q_lo as in the sort's global passes.
//
// Each body takes its block index explicitly (vb) and its larger LDS arrays
// from the caller, so the resident kernel can run it over its own blocks.
#pragma once

#include "sort_core.hpp"

#include <type_traits>

namespace vo {
namespace compact_k {
namespace {

constexpr int CT_LOG = 12; // tile: 4096 rows
constexpr int CT = 1 << CT_LOG;
constexpr int CBLOCK = 256;

// A word the network moves: up to kParts columns (pointer and element width 1,
// 2, 4 or 8 bytes; width 0 ends the list) side by side in 64 bits, so that
// narrow columns share a run of the network instead of taking a register pair
// and LDS traffic each.
constexpr int kParts = 4;
struct Word {
    void *p[kParts];
    uint32_t w[kParts];
};

template <int NW>
struct Cols {
    Word c[NW];
};

// Row loads and stores of the network passes.  NT: non-temporal, for rows
// beyond the 256 MB MALL, which every pass streams through once (below it
// the next pass re-reads them from the MALL).
template <bool NT, typename T>
__device__ __forceinline__ T ld_row(const T *p)
{
    if constexpr (NT)
        return __builtin_nontemporal_load(p);
    else
        return *p;
}

template <bool NT, typename T>
__device__ __forceinline__ void st_row(T *p, T v)
{
    if constexpr (NT)
        __builtin_nontemporal_store(v, p);
    else
        *p = v;
}

// Rows idx(m), m < RR, of every word.  W8: every word is one 8-byte column;
// otherwise the widths are uniform over the launch, and each part's loads (or
// stores) are issued together.
template <bool W8, bool NT, int RR, int NW, class I>
__device__ __forceinline__ void ld_rows(uint64_t (&r)[RR][NW], const Cols<NW> &c, I idx)
{
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        uint32_t sh = 0;
#pragma unroll
        for (int k = 0; k < (W8 ? 1 : kParts); ++k) {
            const uint32_t wd = W8 ? 8 : c.c[w].w[k];
            if (wd == 0) break;
            uint32_t z = 0; // a row index of its own per part (register pressure)
            if (!W8) asm volatile("" : "+v"(z));
            auto part = [&](auto *p) {
#pragma unroll
                for (int m = 0; m < RR; ++m) {
                    const uint64_t v = ld_row<NT>(p + (idx(m) + z));
                    r[m][w] = k == 0 ? v : r[m][w] | (v << sh);
                }
            };
            if (wd == 8)
                part((const uint64_t *)c.c[w].p[k]);
            else if (wd == 4)
                part((const uint32_t *)c.c[w].p[k]);
            else if (wd == 2)
                part((const uint16_t *)c.c[w].p[k]);
            else
                part((const uint8_t *)c.c[w].p[k]);
            sh += 8 * wd;
        }
    }
}

template <bool W8, bool NT, int RR, int NW, class I>
__device__ __forceinline__ void st_rows(const uint64_t (&r)[RR][NW], const Cols<NW> &c, I idx)
{
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        uint32_t sh = 0;
#pragma unroll
        for (int k = 0; k < (W8 ? 1 : kParts); ++k) {
            const uint32_t wd = W8 ? 8 : c.c[w].w[k];
            if (wd == 0) break;
            uint32_t z = 0;
            if (!W8) asm volatile("" : "+v"(z));
            auto part = [&](auto *p) {
                using E = std::remove_reference_t<decltype(*p)>;
#pragma unroll
                for (int m = 0; m < RR; ++m) st_row<NT>(p + (idx(m) + z), (E)(k == 0 ? r[m][w] : r[m][w] >> sh));
            };
            if (wd == 8)
                part((uint64_t *)c.c[w].p[k]);
            else if (wd == 4)
                part((uint32_t *)c.c[w].p[k]);
            else if (wd == 2)
                part((uint16_t *)c.c[w].p[k]);
            else
                part((uint8_t *)c.c[w].p[k]);
            sh += 8 * wd;
        }
    }
}

// Lanes whose pair swaps at level q > 0: d = low word of the prefix count at
// the block's middle plus half - 1 - i (see the top; only the low q + 1 bits
// matter, and q <= 31).
__device__ __forceinline__ uint64_t swap_lanes(uint32_t d, int q)
{
    return __builtin_amdgcn_ballot_w64((d & (1u << q)) == 0);
}

template <int NW>
__device__ __forceinline__ void swap_rows(uint64_t m, uint64_t (&x)[NW], uint64_t (&y)[NW])
{
    uint32_t a[2 * NW], b[2 * NW];
#pragma unroll
    for (int w = 0; w < 2 * NW; ++w) {
        a[w] = (uint32_t)(x[w / 2] >> (32 * (w & 1)));
        b[w] = (uint32_t)(y[w / 2] >> (32 * (w & 1)));
    }
    dev::swap_words<dev::Join::kCopy, 2 * NW>({m, 0}, a, b);
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        x[w] = (uint64_t)a[2 * w] | ((uint64_t)a[2 * w + 1] << 32);
        y[w] = (uint64_t)b[2 * w] | ((uint64_t)b[2 * w + 1] << 32);
    }
}

// Instances of one size class 2^c of a batch: virtual row v of the class is
// row v mod 2^c of instance v >> c, stored at physical row
// off[v >> c] + (v mod 2^c), whose live rows are n[v >> c].  off == nullptr:
// a single compaction, virtual rows are physical rows and the caller's n
// applies.  Every caller passes a v whose instance is the same for the whole
// wavefront, so the table reads are scalar.
struct Inst {
    const uint64_t *off;
    const uint64_t *n;
    int c;
};

__device__ __forceinline__ uint64_t uni64(uint64_t v)
{
    return ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32)) << 32) |
           __builtin_amdgcn_readfirstlane((uint32_t)v);
}

__device__ __forceinline__ uint32_t inst_of(const Inst &in, uint64_t v)
{
    return __builtin_amdgcn_readfirstlane((uint32_t)(v >> in.c));
}

// physical row of virtual row v
__device__ __forceinline__ uint64_t inst_row(const Inst &in, uint64_t v)
{
    if (in.off == nullptr) return v;
    return uni64(in.off[inst_of(in, v)]) + (v & ((1ull << in.c) - 1));
}

// row of v inside its instance, and that instance's live rows
__device__ __forceinline__ uint64_t inst_local(const Inst &in, uint64_t v)
{
    return in.off == nullptr ? v : (v & ((1ull << in.c) - 1));
}

__device__ __forceinline__ uint64_t inst_live(const Inst &in, uint64_t v, uint64_t n)
{
    return in.off == nullptr ? n : uni64(in.n[inst_of(in, v)]);
}

// ---------------------------------------------------------------- counting

// Selected rows per tile: sel[i] = mask[i] != 0 && i < n.
__device__ __forceinline__ void b_count_mask(const uint8_t *__restrict__ mask, uint64_t n,
                                             uint32_t *__restrict__ tile_cnt, Inst in, TraceSlot *slot, uint32_t vb)
{
    __shared__ uint32_t red[CBLOCK / 64];
    dev::Atr tr(slot);
    const uint64_t tv = (uint64_t)vb * CT;
    const uint64_t t0 = inst_row(in, tv), l0 = inst_local(in, tv), nn = inst_live(in, tv, n);
    uint32_t c = 0;
#pragma unroll 4
    for (int k = 0; k < CT / CBLOCK; ++k) {
        const uint32_t i = k * CBLOCK + threadIdx.x;
        c += (mask[t0 + i] != 0) & (l0 + i < nn);
        tr.at(1, t0 + i);
    }
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t s = 0;
        for (int w = 0; w < CBLOCK / 64; ++w) s += red[w];
        tile_cnt[vb] = s;
        tr.at(2, vb);
    }
    tr.done(dev::gtid());
}

__global__ __launch_bounds__(CBLOCK) void k_count_mask(const uint8_t *__restrict__ mask, uint64_t n,
                                                       uint32_t *__restrict__ tile_cnt, Inst in, TraceSlot *slot)
{
    b_count_mask(mask, n, tile_cnt, in, slot, blockIdx.x);
}

// Q6-style predicate: writes mask[i] and per-tile counts in one pass.
struct Pred {
    int32_t day_lo, day_hi;
    int64_t disc_lo, disc_hi, qty_lt;
};

template <bool NT = false>
__device__ __forceinline__ void b_filter_count(const int32_t *__restrict__ day, const int64_t *__restrict__ qty,
                                               const int64_t *__restrict__ disc, uint64_t n, Pred pr,
                                               uint8_t *__restrict__ mask, uint32_t *__restrict__ tile_cnt,
                                               TraceSlot *slot, uint32_t vb)
{
    __shared__ uint32_t red[CBLOCK / 64];
    dev::Atr tr(slot);
    const uint64_t t0 = (uint64_t)vb * CT;
    uint32_t c = 0;
#pragma unroll 4
    for (int k = 0; k < CT / CBLOCK; ++k) {
        const uint64_t i = t0 + k * CBLOCK + threadIdx.x;
        const int32_t d = ld_row<NT>(day + i);
        const int64_t q = ld_row<NT>(qty + i), ds = ld_row<NT>(disc + i);
        const uint32_t m = (d >= pr.day_lo) & (d < pr.day_hi) & (ds >= pr.disc_lo) & (ds <= pr.disc_hi) &
                           (q < pr.qty_lt) & (i < n);
        st_row<NT>(mask + i, (uint8_t)m);
        c += m;
        tr.at(3, i); // day, qty, disc read and mask written at row i
    }
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t s = 0;
        for (int w = 0; w < CBLOCK / 64; ++w) s += red[w];
        tile_cnt[vb] = s;
        tr.at(2, vb);
    }
    tr.done(dev::gtid());
}

template <bool NT = false>
__global__ __launch_bounds__(CBLOCK) void k_filter_count(const int32_t *__restrict__ day,
                                                         const int64_t *__restrict__ qty,
                                                         const int64_t *__restrict__ disc, uint64_t n, Pred pr,
                                                         uint8_t *__restrict__ mask, uint32_t *__restrict__ tile_cnt,
                                                         TraceSlot *slot)
{
    b_filter_count<NT>(day, qty, disc, n, pr, mask, tile_cnt, slot, blockIdx.x);
}

// Exclusive scan of the tile counts by one block of NT threads:
// pre[0..nt], pre[nt] = total; part holds NT words of LDS.
template <uint32_t NT, bool TOTAL = true>
__device__ __forceinline__ void b_scan_tiles(const uint32_t *__restrict__ cnt, uint32_t nt, uint64_t *__restrict__ pre,
                                             uint64_t *__restrict__ out_count, TraceSlot *slot, uint64_t *part)
{
    dev::Atr tr(slot);
    const uint32_t per = (nt + NT - 1) / NT;
    const uint32_t lo = threadIdx.x * per;
    // a thread's chunk in groups of 16 counts, loaded before any is used: one
    // memory round trip per group rather than per count
    constexpr int G = 16;
    uint64_t s = 0;
    for (uint32_t k0 = 0; k0 < per; k0 += G) {
        uint32_t v[G];
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const uint32_t k = k0 + j, i = lo + k;
            v[j] = (k < per && i < nt) ? cnt[i] : 0u;
        }
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const uint32_t k = k0 + j, i = lo + k;
            if (k < per && i < nt) tr.at(4, i);
            s += v[j];
        }
    }
    part[threadIdx.x] = s;
    __syncthreads();
    for (uint32_t off = 1; off < NT; off <<= 1) {
        const uint64_t v = threadIdx.x >= (uint32_t)off ? part[threadIdx.x - off] : 0;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    uint64_t run = part[threadIdx.x] - s; // exclusive prefix of this thread's chunk
    for (uint32_t k0 = 0; k0 < per; k0 += G) {
        uint32_t v[G];
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const uint32_t k = k0 + j, i = lo + k;
            v[j] = (k < per && i < nt) ? cnt[i] : 0u;
        }
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const uint32_t k = k0 + j, i = lo + k;
            if (k < per && i < nt) {
                pre[i] = run;
                run += v[j];
                tr.at(5, i);
            }
        }
    }
    if (threadIdx.x == NT - 1) {
        if (TOTAL) pre[nt] = part[NT - 1];
        if (out_count) *out_count = part[NT - 1];
        tr.at(6, nt);
    }
    tr.done(dev::gtid());
}

__global__ __launch_bounds__(1024) void k_scan_tiles(const uint32_t *__restrict__ cnt, uint32_t nt,
                                                     uint64_t *__restrict__ pre, uint64_t *__restrict__ out_count,
                                                     TraceSlot *slot)
{
    __shared__ uint64_t part[1024];
    b_scan_tiles<1024>(cnt, nt, pre, out_count, slot, part);
}

// Tile scans of many tiles (launch mode): segments of kScanSeg counts, one
// 1024-thread block each, kScanPer contiguous counts per thread.
// k_scan_part writes each segment's sum (<= 2^25, so 32 bits), k_scan_tiles
// scans those sums into segment bases, and k_scan_fin writes every tile's
// exclusive prefix from its segment's base.  The sums and the prefixes are
// those of the one-block scan: integer addition in any grouping.
constexpr uint32_t kScanPer = 8;
constexpr uint32_t kScanSeg = 1024 * kScanPer;

// Exclusive prefix of v over a 1024-thread block and the block's total;
// sh: 16 words of LDS.
__device__ __forceinline__ uint64_t block_scan1024(uint64_t v, uint64_t *sh, uint64_t &total)
{
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint64_t inc = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint64_t u = __shfl_up(inc, off, 64);
        inc += lane >= (uint32_t)off ? u : 0;
    }
    if (lane == 63) sh[w] = inc;
    __syncthreads();
    uint64_t before = 0, tot = 0;
#pragma unroll
    for (uint32_t k = 0; k < 16; ++k) {
        const uint64_t x = sh[k];
        before += k < w ? x : 0;
        tot += x;
    }
    total = tot;
    return before + inc - v;
}

__global__ __launch_bounds__(1024) void k_scan_part(const uint32_t *__restrict__ cnt, uint32_t nt,
                                                    uint32_t *__restrict__ seg_sum, TraceSlot *slot)
{
    __shared__ uint64_t sh[16];
    dev::Atr tr(slot);
    const uint64_t lo = (uint64_t)blockIdx.x * kScanSeg + (uint64_t)threadIdx.x * kScanPer;
    uint32_t v[kScanPer];
#pragma unroll
    for (uint32_t j = 0; j < kScanPer; ++j) v[j] = lo + j < nt ? cnt[lo + j] : 0u;
    uint64_t s = 0;
#pragma unroll
    for (uint32_t j = 0; j < kScanPer; ++j) {
        s += v[j];
        if (lo + j < nt) tr.at(4, lo + j);
    }
    uint64_t total;
    (void)block_scan1024(s, sh, total);
    if (threadIdx.x == 0) {
        seg_sum[blockIdx.x] = (uint32_t)total;
        tr.at(7, blockIdx.x);
    }
    tr.done(dev::gtid());
}

__global__ __launch_bounds__(1024) void k_scan_fin(const uint32_t *__restrict__ cnt, uint32_t nt,
                                                   const uint64_t *__restrict__ seg_base, uint64_t *__restrict__ pre,
                                                   TraceSlot *slot)
{
    __shared__ uint64_t sh[16];
    dev::Atr tr(slot);
    const uint64_t lo = (uint64_t)blockIdx.x * kScanSeg + (uint64_t)threadIdx.x * kScanPer;
    uint32_t v[kScanPer];
#pragma unroll
    for (uint32_t j = 0; j < kScanPer; ++j) v[j] = lo + j < nt ? cnt[lo + j] : 0u;
    uint64_t s = 0;
#pragma unroll
    for (uint32_t j = 0; j < kScanPer; ++j) s += v[j];
    uint64_t total;
    uint64_t run = seg_base[blockIdx.x] + block_scan1024(s, sh, total);
    tr.at(7, blockIdx.x);
#pragma unroll
    for (uint32_t j = 0; j < kScanPer; ++j) {
        if (lo + j < nt) {
            pre[lo + j] = run;
            tr.at(4, lo + j);
            tr.at(5, lo + j);
        }
        run += v[j];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        pre[nt] = seg_base[gridDim.x]; // the total
        tr.at(6, nt);
    }
    tr.done(dev::gtid());
}

// The tile scans of every instance of a batch class, instance vb by block vb:
// its nts tiles' exclusive prefix counts go to pre[vb * nts ..] (each
// instance restarts at zero, so each compacts to its own front) and its
// selected count to out[idx[vb]] when out is given.
__device__ __forceinline__ void b_scan_seg(const uint32_t *__restrict__ cnt, uint32_t nts, uint64_t *__restrict__ pre,
                                           uint64_t *__restrict__ out, const uint64_t *__restrict__ idx,
                                           TraceSlot *slot, uint64_t *part, uint32_t vb)
{
    const uint64_t o = (uint64_t)vb * nts;
    uint64_t *oc = out ? out + uni64(idx[vb]) : nullptr;
    b_scan_tiles<CBLOCK, false>(cnt + o, nts, pre + o, oc, slot, part);
}

__global__ __launch_bounds__(CBLOCK) void k_scan_seg(const uint32_t *__restrict__ cnt, uint32_t nts,
                                                     uint64_t *__restrict__ pre, uint64_t *__restrict__ out,
                                                     const uint64_t *__restrict__ idx, TraceSlot *slot)
{
    __shared__ uint64_t part[CBLOCK];
    b_scan_seg(cnt, nts, pre, out, idx, slot, part, blockIdx.x);
}

// ---------------------------------------------------------- local levels

// Levels q = 0 .. T-1 inside each 2^T-row tile (T = 12, or 13 where that
// saves a later pass).  A thread holds 16 rows of each column in registers
// under layout a: rows lay_base(tau, a) | m << a (sort_core.hpp); levels
// a .. a+3 pair rows inside a thread.  Layout 0 (levels 0-3) is 16 consecutive
// rows, the ones whose mask bytes the thread reads for the scan, so its prefix
// counts come from registers; levels from 4 up need counts at multiples of 16
// only, one word of LDS per thread.  Of the relayouts 6 -> 0 -> 4 (-> 5) -> T-4
// only the last leaves the wavefront; rows are loaded in layout 6 and stored in
// layout T-4, both 64 lanes on consecutive rows.  Rows are read from `src` and
// written to `dst` (which may be the same columns).  (With two counts in LDS
// per pair and the offset form's arithmetic the pass was issue-bound: two
// 8-byte columns of 2^23 rows 61.9 -> 51.2 us, 12 bytes of 2^24 144 -> 122 us.)
template <int T>
using CTileOf = dev::TileCT<dev::Rec<1, uint64_t, true>, T, 4, false>;

// relayout buffer: one 8-byte column
template <int T>
constexpr size_t cbuf_bytes() { return (size_t)CTileOf<T>::TPAD * 8; }

template <int NW, int T, int A_FROM, int A_TO>
__device__ __forceinline__ void crelayout(uint64_t (&r)[16][NW], dev::TileBuf &buf, uint32_t tau)
{
    using TL = CTileOf<T>;
    constexpr bool IN = TL::in_wave(A_FROM, A_TO);
    uint64_t h = 0;
    uint32_t n = 0;
    if (buf.shared || A_FROM > 6)
        __syncthreads();
    else
        TL::wave_fence();
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        uint64_t v[16];
#pragma unroll
        for (int m = 0; m < 16; ++m) v[m] = r[m][w];
        TL::template move_col<A_FROM, A_TO>(v, reinterpret_cast<uint64_t *>(buf.p), tau, h, n);
        if (w + 1 < NW) {
            if constexpr (IN)
                TL::wave_fence();
            else
                __syncthreads();
        }
#pragma unroll
        for (int m = 0; m < 16; ++m) r[m][w] = v[m];
    }
    buf.shared = !IN;
}

// Levels 0-3 in layout 0: selm = the select bits of the thread's rows, c0 =
// low word of the prefix count at its first row.
template <int NW>
__device__ __forceinline__ void clevels0(uint64_t (&r)[16][NW], uint32_t selm, uint32_t c0)
{
    auto cnt = [&](int e) { return c0 + __popc(selm & ((1u << e) - 1)); };
#pragma unroll
    for (int m = 0; m < 16; m += 2) {
        const uint32_t s0 = selm >> m, s1 = selm >> (m + 1);
        const uint64_t sw = __builtin_amdgcn_ballot_w64((((~s0 & s1) ^ cnt(m)) & 1u) != 0);
        swap_rows<NW>(sw, r[m], r[m | 1]);
    }
#pragma unroll
    for (int q = 1; q < 4; ++q) {
        const int half = 1 << q;
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            if (m & half) continue;
            const uint32_t d = cnt((m & ~(2 * half - 1)) + half) + (uint32_t)(half - 1 - (m & (half - 1)));
            swap_rows<NW>(swap_lanes(d, q), r[m], r[m | half]);
        }
    }
}

// Levels Q0 .. Q1 in layout A >= 4; c16 = the tile's prefix counts at rows
// 16 j, tbase = the low word of the tile's first.
template <int NW, int A, int Q0, int Q1>
__device__ __forceinline__ void clevels(uint64_t (&r)[16][NW], const uint32_t *c16, uint32_t tbase, uint32_t tau)
{
    const uint32_t base = dev::lay_base<4>(tau, A);
    const uint32_t top = (base >> (A + 4)) << A; // 16-row index of the thread's rows, register bits clear
    const uint32_t rest = tbase + ((1u << A) - 1) - (base & ((1u << A) - 1));
#pragma unroll
    for (int q = Q0; q <= Q1; ++q) {
        const int k = q - A;
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            if (m & (1 << k)) continue;
            const uint32_t mid = (uint32_t)((m & ~((2 << k) - 1)) | (1 << k)) << (A - 4);
            const uint32_t over = (uint32_t)(((1 << k) - 1) - (m & ((1 << k) - 1))) << A;
            swap_rows<NW>(swap_lanes(c16[top + mid] + rest + over, q), r[m], r[m | (1 << k)]);
        }
    }
}

// Exact sum of a[i] * b[i] over the thread's selected rows (layout 0), added
// over the block into partial[vb].  Summing selected rows here, where the tile
// has them in registers with their mask bits, is the sum over the compacted
// prefix without the pass that re-read both columns (1.46 of 13.2 ms at 2^29).
template <int NTHR>
__device__ __forceinline__ void csum(const uint64_t (&r)[16][2], uint32_t selm, __int128 *__restrict__ partial,
                                     uint32_t vb, uint32_t tid)
{
    __shared__ __int128 red[NTHR / 64];
    unsigned __int128 acc = 0;
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        const __int128 prod = (__int128)(int64_t)r[m][0] * (__int128)(int64_t)r[m][1];
        const uint64_t on = 0 - (uint64_t)((selm >> m) & 1u);
        acc += ((unsigned __int128)((uint64_t)((unsigned __int128)prod >> 64) & on) << 64) | ((uint64_t)prod & on);
        // one product at a time: all sixteen in flight pass the 128 VGPRs that
        // let two 2^13-row blocks share a CU
        uint64_t lo = (uint64_t)acc, hi = (uint64_t)(acc >> 64);
        asm volatile("" : "+v"(lo), "+v"(hi));
        acc = ((unsigned __int128)hi << 64) | lo;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const uint64_t lo = __shfl_xor((uint64_t)acc, off), hi = __shfl_xor((uint64_t)(acc >> 64), off);
        acc += ((unsigned __int128)hi << 64) | lo;
    }
    if ((tid & 63) == 0) red[tid >> 6] = (__int128)acc;
    __syncthreads();
    if (tid == 0) {
        unsigned __int128 t = 0;
        for (int w = 0; w < NTHR / 64; ++w) t += (unsigned __int128)red[w];
        partial[vb] = (__int128)t;
    }
}

// W8: every column is 8 bytes wide (no per-load width dispatch).  partial (two
// 8-byte columns only): the tile's sum of products of its selected rows.
template <int NW, bool W8, bool TRACE, bool NT = false, int T = CT_LOG>
__device__ __forceinline__ void b_compact_local(Cols<NW> src, Cols<NW> dst, const uint8_t *__restrict__ mask,
                                                uint64_t n, const uint64_t *__restrict__ tile_pre, Inst in,
                                                __int128 *__restrict__ partial, TraceSlot *slot, char *lds_raw,
                                                uint32_t vb)
{
    constexpr int NTHR = 1 << (T - 4), AS = T - 4;
    dev::TileBuf buf{lds_raw};
    uint32_t *c16 = reinterpret_cast<uint32_t *>(lds_raw + cbuf_bytes<T>());
    __shared__ uint32_t wsum[NTHR / 64];
    const uint32_t tid = threadIdx.x;
    const uint64_t tv = (uint64_t)vb << T;
    const uint64_t t0 = inst_row(in, tv), l0 = inst_local(in, tv), nn = inst_live(in, tv, n);
    const uint32_t tbase = (uint32_t)tile_pre[tv >> CT_LOG];
    dev::AtrT<TRACE> tr(slot);
    tr.at(7, tv >> CT_LOG);

    // rows, coalesced; issued before the scan
    const uint32_t lb = dev::lay_base<4>(tid, 6);
    uint64_t r[16][NW];
    auto at_in = [&](int m) { return t0 + lb + 64u * m; };
    ld_rows<W8, NT>(r, src, at_in);
#pragma unroll
    for (int m = 0; m < 16; ++m)
#pragma unroll
        for (int w = 0; w < NW; ++w) tr.at(8 + w, at_in(m));

    // select bits and exclusive prefix: thread tid owns rows [16 tid, 16 tid + 16)
    uint32_t selm = 0;
    const uint8_t *mp = mask + t0 + tid * 16;
    if (((uintptr_t)(mask + t0) & 15) == 0) { // tiles of a 16-byte aligned mask
        const uint4 v = *reinterpret_cast<const uint4 *>(mp);
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int k = 0; k < 16; ++k) selm |= (((x[k >> 2] >> (8 * (k & 3))) & 0xFFu) != 0 ? 1u : 0u) << k;
    } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) selm |= (mp[k] != 0 ? 1u : 0u) << k;
    }
    const uint64_t row0 = l0 + tid * 16;
    const uint32_t live = row0 + 16 <= nn ? 16u : row0 < nn ? (uint32_t)(nn - row0) : 0u;
    selm &= (1u << live) - 1;
#pragma unroll
    for (int k = 0; k < 16; ++k) tr.at(1, t0 + tid * 16 + k);
    const uint32_t run = __popc(selm);
    uint32_t incl = run;
    const uint32_t lane = tid & 63;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_up(incl, off);
        incl += lane >= (uint32_t)off ? v : 0;
    }
    if (lane == 63) wsum[tid >> 6] = incl;
    __syncthreads();
    uint32_t wpre = 0;
    for (uint32_t w = 0; w < (tid >> 6); ++w) wpre += wsum[w];
    const uint32_t c0 = wpre + incl - run;
    // read inside the wavefront up to layout 6, beyond it after the relayout's barriers
    c16[tid] = c0;
    crelayout<NW, T, 6, 0>(r, buf, tid);
    if constexpr (NW == 2 && W8) {
        if (partial) {
            csum<NTHR>(r, selm, partial, vb, tid);
            tr.at(16, vb);
        }
    }
    clevels0<NW>(r, selm, tbase + c0);
    crelayout<NW, T, 0, 4>(r, buf, tid);
    clevels<NW, 4, 4, 7>(r, c16, tbase, tid);
    if constexpr (T == 13) {
        crelayout<NW, T, 4, 5>(r, buf, tid);
        clevels<NW, 5, 8, 8>(r, c16, tbase, tid);
        crelayout<NW, T, 5, AS>(r, buf, tid);
        clevels<NW, AS, 9, 12>(r, c16, tbase, tid);
    } else {
        static_assert(T == 12, "tiles of 2^12 or 2^13 rows");
        crelayout<NW, T, 4, AS>(r, buf, tid);
        clevels<NW, AS, 8, 11>(r, c16, tbase, tid);
    }
    uint32_t tid_s = tid; // store addresses recomputed here (register pressure)
    asm volatile("" : "+v"(tid_s));
    auto at_out = [&](int m) { return t0 + tid_s + ((uint32_t)m << AS); };
    st_rows<W8, NT>(r, dst, at_out);
#pragma unroll
    for (int m = 0; m < 16; ++m)
#pragma unroll
        for (int w = 0; w < NW; ++w) tr.at(16 + w, at_out(m));
    tr.done((uint64_t)vb * NTHR + tid);
}

// dynamic LDS of the local pass: the relayout buffer and a count per thread
template <int T>
constexpr size_t clocal_lds() { return cbuf_bytes<T>() + ((size_t)4 << (T - 4)); }

// XC: contiguous block ranges per XCD (dev::xcd_block)
template <int NW, bool W8, bool TRACE, bool NT = false, int T = CT_LOG, bool XC = true>
__global__ __launch_bounds__(1 << (T - 4), W8 ? 4 : 1) void k_compact_local(Cols<NW> src, Cols<NW> dst,
                                                                const uint8_t *__restrict__ mask, uint64_t n,
                                                                const uint64_t *__restrict__ tile_pre, Inst in,
                                                                __int128 *__restrict__ partial, TraceSlot *slot)
{
    extern __shared__ __align__(16) char lds_raw[];
    b_compact_local<NW, W8, TRACE, NT, T>(src, dst, mask, n, tile_pre, in, partial, slot, lds_raw,
                                          dev::xcd_block<XC>());
}

// ---------------------------------------------------------- global levels

// Levels q_lo .. q_lo+S-1 (ascending, q_lo >= CT_LOG): thread g owns the 2^S
// rows base + m * 2^q_lo.  The block start of any pair has every bit below
// q_lo + 1 clear, so its prefix counts are the same for all lanes of a
// wavefront and come from the tile prefix array.
template <int NW, int S, bool TRACE, bool NT = false>
__device__ __forceinline__ void b_compact_global(Cols<NW> cols, const uint64_t *__restrict__ tile_pre, int q_lo,
                                                 Inst in, TraceSlot *slot, uint32_t vb)
{
    dev::AtrT<TRACE> tr(slot);
    const uint64_t g = (uint64_t)vb * 256 + threadIdx.x;
    const uint64_t base = (g & ((1ull << q_lo) - 1)) | ((g >> q_lo) << (q_lo + S));
    // the 2^S rows lie in one instance (q_lo + S <= its size class)
    const uint64_t pb = inst_row(in, base);
    uint64_t r[1 << S][NW];
    auto at = [&](int m) { return pb + ((uint64_t)m << q_lo); };
    ld_rows<false, NT>(r, cols, at);
#pragma unroll
    for (int m = 0; m < (1 << S); ++m)
#pragma unroll
        for (int w = 0; w < NW; ++w) tr.at(8 + w, at(m));
    // uniform part of base (bits >= 8 are shared by the wavefront)
    const uint64_t ubase = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(base >> 32)) << 32) |
                           __builtin_amdgcn_readfirstlane((uint32_t)base & ~0xFFu);
    const uint32_t rest = (uint32_t)((1ull << q_lo) - 1) - ((uint32_t)base & (uint32_t)((1ull << q_lo) - 1));
#pragma unroll
    for (int k = 0; k < S; ++k) {
#pragma unroll
        for (int m = 0; m < (1 << S); ++m) {
            if (m & (1 << k)) continue;
            const uint64_t ue = ubase + ((uint64_t)m << q_lo);
            const uint64_t mid = (ue & ~((2ull << (q_lo + k)) - 1)) + (1ull << (q_lo + k));
            const uint32_t d = (uint32_t)tile_pre[mid >> CT_LOG] + rest +
                               ((uint32_t)(((1 << k) - 1) - (m & ((1 << k) - 1))) << q_lo);
            tr.at(7, mid >> CT_LOG);
            swap_rows<NW>(swap_lanes(d, q_lo + k), r[m], r[m | (1 << k)]);
        }
    }
    st_rows<false, NT>(r, cols, at);
#pragma unroll
    for (int m = 0; m < (1 << S); ++m)
#pragma unroll
        for (int w = 0; w < NW; ++w) tr.at(16 + w, at(m));
    tr.done(dev::gtid());
}

template <int NW, int S, bool TRACE, bool NT = false>
__global__ __launch_bounds__(256) void k_compact_global(Cols<NW> cols, const uint64_t *__restrict__ tile_pre, int q_lo,
                                                        Inst in, TraceSlot *slot)
{
    b_compact_global<NW, S, TRACE, NT>(cols, tile_pre, q_lo, in, slot, dev::xcd_block<!NT>());
}

// ------------------------------------------------- LDS-staged global levels

// S = 5 .. T-4 levels q_lo .. q_lo+S-1 (q_lo >= T) in one pass.  A block takes
// the 2^T rows hibase + g * 2^q_lo + j0 + c (g < 2^S, c < 2^C, C = T - S):
// local row l = g << C | c, so level q_lo+k pairs local bit C+k.  Loaded in
// layout C, where the first levels run, stored in layout T-4, where the last
// four do; the prefix counts the levels need, tile_pre at hibase + g * 2^q_lo,
// go to LDS.
template <int NW, int T, int A, int S, int B0, int B1>
__device__ __forceinline__ void hlevels(uint64_t (&r)[16][NW], const uint32_t *P, uint32_t tau, int q_lo, uint32_t j0)
{
    constexpr int C = T - S;
    const uint32_t base = dev::lay_base<4>(tau, A);
    const uint32_t g0 = base >> C; // the thread's g, register bits clear
    const uint32_t rest = ((1u << q_lo) - 1) - j0 - (base & ((1u << C) - 1));
#pragma unroll
    for (int bit = B0; bit <= B1; ++bit) {
        const int k = bit - C; // level q_lo + k
        const uint32_t low = (1u << k) - 1;
        const uint32_t restk = rest + ((low & ~g0) << q_lo);
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            if (m & (1 << (bit - A))) continue;
            const uint32_t gm = (uint32_t)m << (A - C);
            const uint32_t mid = ((g0 & ~(low * 2 + 1)) | (gm & ~(low * 2 + 1))) + (1u << k);
            const uint32_t d = P[mid] + restk - ((gm & low) << q_lo);
            swap_rows<NW>(swap_lanes(d, q_lo + k), r[m], r[m | (1 << (bit - A))]);
        }
    }
}

template <int NW, int S, bool W8, bool TRACE, bool NT = false, int T = CT_LOG>
__device__ __forceinline__ void b_compact_hybrid(Cols<NW> cols, const uint64_t *__restrict__ tile_pre, int q_lo,
                                                 Inst in, TraceSlot *slot, char *lds_raw, uint32_t vb)
{
    dev::AtrT<TRACE> tr(slot);
    constexpr int C = T - S, NTHR = 1 << (T - 4), AS = T - 4;
    static_assert(S >= 5 && C >= 4, "hybrid widths 5..T-4");
    dev::TileBuf buf{lds_raw};
    uint32_t *P = reinterpret_cast<uint32_t *>(lds_raw + cbuf_bytes<T>()); // low words of 2^S prefix counts
    const uint32_t tid = threadIdx.x;
    // row indices fit 32 bits (n_pad <= 2^32)
    const uint32_t runs = (1u << q_lo) >> C; // blocks per group of 2^(q_lo+S) rows
    const uint32_t hibase = (vb / runs) << (q_lo + S);
    const uint32_t j0 = (vb % runs) << C;
    // the group's 2^(q_lo+S) rows lie in one instance: physical row of its first
    const uint64_t ph = inst_row(in, hibase);
    auto grow = [&](uint32_t l) { return ((l >> C) << q_lo) + (l & ((1u << C) - 1)); }; // additive over bit fields
    uint64_t r[16][NW];
    {
        const uint32_t gl = j0 + grow(dev::lay_base<4>(tid, C));
        auto at = [&](int m) { return ph + gl + grow((uint32_t)m << C); };
        ld_rows<W8, NT>(r, cols, at);
#pragma unroll
        for (int m = 0; m < 16; ++m)
#pragma unroll
            for (int w = 0; w < NW; ++w) tr.at(8 + w, at(m));
    }
    __syncthreads(); // (resident blocks: the last step's reads of P)
    for (uint32_t k = tid; k < (1u << S); k += NTHR) {
        P[k] = (uint32_t)tile_pre[((uint64_t)hibase + ((uint64_t)k << q_lo)) >> CT_LOG];
        tr.at(7, ((uint64_t)hibase + ((uint64_t)k << q_lo)) >> CT_LOG);
    }
    __syncthreads();
    if constexpr (S == 9) { // five bits below the last four: layouts C and C + 1
        hlevels<NW, T, C, S, C, C + 3>(r, P, tid, q_lo, j0);
        crelayout<NW, T, C, C + 1>(r, buf, tid);
        hlevels<NW, T, C + 1, S, C + 4, C + 4>(r, P, tid, q_lo, j0);
        crelayout<NW, T, C + 1, AS>(r, buf, tid);
    } else {
        hlevels<NW, T, C, S, C, T - 5>(r, P, tid, q_lo, j0);
        crelayout<NW, T, C, AS>(r, buf, tid);
    }
    hlevels<NW, T, AS, S, T - 4, T - 1>(r, P, tid, q_lo, j0);
    // recompute the store addresses here rather than keep the load addresses
    // live across the levels (register pressure)
    uint32_t tid_s = tid;
    asm volatile("" : "+v"(tid_s));
    const uint32_t gs = j0 + grow(dev::lay_base<4>(tid_s, AS));
    auto at_out = [&](int m) { return ph + gs + grow((uint32_t)m << AS); };
    st_rows<W8, NT>(r, cols, at_out);
#pragma unroll
    for (int m = 0; m < 16; ++m)
#pragma unroll
        for (int w = 0; w < NW; ++w) tr.at(16 + w, at_out(m));
    tr.done((uint64_t)vb * NTHR + tid);
}

template <int S, int T>
constexpr size_t chybrid_lds() { return cbuf_bytes<T>() + ((size_t)4 << S); }

template <int NW, int S, bool W8, bool TRACE, bool NT = false, int T = CT_LOG, bool XC = true>
__global__ __launch_bounds__(1 << (T - 4), W8 ? 4 : 1) void k_compact_hybrid(Cols<NW> cols, const uint64_t *__restrict__ tile_pre,
                                                                 int q_lo, Inst in, TraceSlot *slot)
{
    extern __shared__ __align__(16) char lds_raw[];
    b_compact_hybrid<NW, S, W8, TRACE, NT, T>(cols, tile_pre, q_lo, in, slot, lds_raw, dev::xcd_block<XC>());
}

// --------------------------------------------------------- int128 SUM

// One 256-thread block: strided partial sums, then a tree in LDS (exact:
// int128 addition is associative).
__device__ __forceinline__ void b_sum_final(const __int128 *__restrict__ partial, uint32_t np,
                                            const uint64_t *__restrict__ count, uint64_t *__restrict__ out,
                                            TraceSlot *slot, __int128 *red)
{
    dev::Atr tr(slot);
    // groups of 8 loads in flight (one per tile: 2^16 partials at 2^29 rows)
    constexpr uint32_t G = 8;
    __int128 s = 0;
    for (uint32_t i0 = threadIdx.x; i0 < np; i0 += 256 * G) {
        __int128 v[G];
#pragma unroll
        for (uint32_t j = 0; j < G; ++j) v[j] = i0 + 256 * j < np ? partial[i0 + 256 * j] : 0;
#pragma unroll
        for (uint32_t j = 0; j < G; ++j) {
            s += v[j];
            if (i0 + 256 * j < np) tr.at(8, i0 + 256 * j);
        }
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < (uint32_t)off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const __int128 t = red[0];
        out[0] = *count;
        out[1] = 0;
        out[2] = (uint64_t)t;
        out[3] = (uint64_t)(t >> 64);
        tr.at(16, 0);
    }
    tr.done(dev::gtid());
}

__global__ __launch_bounds__(256) void k_sum_final(const __int128 *__restrict__ partial, uint32_t np,
                                                   const uint64_t *__restrict__ count, uint64_t *__restrict__ out,
                                                   TraceSlot *slot)
{
    __shared__ __int128 red[256];
    b_sum_final(partial, np, count, out, slot, red);
}

// ------------------------------------------------------------ OP_SCATTER

__device__ __forceinline__ void b_scatter_positions(const uint8_t *__restrict__ mask, uint64_t n,
                                                    const uint64_t *__restrict__ tile_pre, int32_t *__restrict__ out,
                                                    TraceSlot *slot, uint32_t vb)
{
    __shared__ uint32_t wsum[CBLOCK / 64];
    dev::Atr tr(slot);
    const uint32_t tid = threadIdx.x;
    const uint64_t t0 = (uint64_t)vb * CT;
    constexpr int PER = CT / CBLOCK;
    uint32_t sel[PER], run = 0;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const uint64_t i = t0 + tid * PER + k;
        if (i < n) {
            sel[k] = mask[i] != 0;
            tr.at(1, i);
        } else {
            sel[k] = 0;
        }
        run += sel[k];
    }
    uint32_t incl = run;
    const uint32_t lane = tid & 63;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_up(incl, off);
        incl += lane >= (uint32_t)off ? v : 0;
    }
    if (lane == 63) wsum[tid >> 6] = incl;
    __syncthreads();
    uint32_t wpre = 0;
    for (uint32_t w = 0; w < (tid >> 6); ++w) wpre += wsum[w];
    uint64_t c = tile_pre[vb] + wpre + incl - run;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const uint64_t i = t0 + tid * PER + k;
        if (sel[k]) { // reference semantics: only selected rows are written (not oblivious)
            out[i] = (int32_t)c;
            tr.at(16, i);
        }
        c += sel[k];
    }
    tr.done(dev::gtid());
}

__global__ __launch_bounds__(CBLOCK) void k_scatter_positions(const uint8_t *__restrict__ mask, uint64_t n,
                                                              const uint64_t *__restrict__ tile_pre,
                                                              int32_t *__restrict__ out, TraceSlot *slot)
{
    b_scatter_positions(mask, n, tile_pre, out, slot, blockIdx.x);
}

} // namespace
} // namespace compact_k
} // namespace vo
