// sort_kernels.hpp -- oblivious bitonic sort kernels and their pass schedule.
//
// Reference: executeBitonicSort (include/cuda/sort.cuh:70-118) runs one
// grid-wide pass per (k, j) stage, S = log2N(log2N+1)/2 passes.  Here the
// same compare-exchange network is grouped into far fewer HBM passes:
//   pass 0       k_sort_local_ct : every tile of 2^T_LOG records fully
//                                  sorted (levels p <= T_LOG), registers+LDS;
// then either the wrapped schedule (the default, plan_wrapped), on tiles of
// 2^T_LOG or 2^W_LOG records:
//                k_sort_global   : up to S_MAX strided stages in registers;
//                k_sort_hybrid   : 4 and more strided stages through LDS;
//                k_sort_merge    : a level's stages inside contiguous tiles;
//                k_sort_wrap     : a level's last stages and the next one's
//                                  first ones in one pass;
// or level by level (plan_passes; tuning words and recorded programs): for
// each p > T_LOG the stages q >= T_LOG by global and hybrid passes, then a
// merge.  Either is a function of the sizes, the record kind and the tuning.
//
// Addressing: a block's records sit at one uniform (scalar) base; every column
// has a buffer resource there, the register's element offset goes to the
// scalar offset field and the thread's to the vector offset.  In strided tiles
// and global passes both reach across the array: below 2^29 elements
// (kMaxSortRows) and of disjoint bits, so that their sum is below 2^32 bytes
// for 8-byte columns too.  Batched sorts map a block's uniform virtual base
// through a per-instance offset table (instances are never smaller than a tile
// on these kernels).
#pragma once

#include "sort_core.hpp"

#include <algorithm>

namespace vo {
namespace dev {

// Uniform virtual index -> physical index (identity without a table).  The
// table entry is made wave-uniform explicitly: where the compiler cannot
// prove the table unwritten (the resident queue kernel's bodies) it would
// load it into vector registers, and every buffer access based on it would
// become a loop over lanes.
__device__ __forceinline__ uint64_t map_uniform(const IMap &m, uint64_t v)
{
    if (m.offsets == nullptr) return v;
    const uint64_t o = m.offsets[v >> m.c];
    const uint64_t ou = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(o >> 32)) << 32) |
                        __builtin_amdgcn_readfirstlane((uint32_t)o);
    return ou + (v & ((1ull << m.c) - 1));
}

// Cache policy of the passes' buffer loads and stores (the instructions'
// aux field): 0 for arrays that fit the 256 MB MALL, where the next pass
// re-reads them from it; kCpStream (non-temporal) for larger ones, which
// every pass streams through once.
constexpr int kCpStream = 2;

// Raw buffer access: the uniform base goes into a buffer resource (scalar
// registers), the per-thread part is a 32-bit byte offset.  Dword 3 of the
// resource selects the 32-bit data format (0x00020000) used for untyped
// loads on gfx9-family parts.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *ubase)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(ubase), (short)0, (int)0xFFFFFFFFu, 0x00020000);
}

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Tile form: one buffer resource per column for the tile's uniform base u,
// the per-register offset so (elements, uniform) in the scalar offset field and
// the per-thread offset vi in the vector offset; so + vi < 2^29 (see the top).
template <typename T, int CP = 0>
__device__ __forceinline__ T ld_t(__amdgpu_buffer_rsrc_t r, uint32_t vi, uint32_t so)
{
    if constexpr (sizeof(T) == 8)
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, vi * 8u, so * 8u, CP));
    else
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, vi * 4u, so * 4u, CP));
}

template <typename T, int CP = 0>
__device__ __forceinline__ void st_t(__amdgpu_buffer_rsrc_t r, uint32_t vi, uint32_t so, T v)
{
    if constexpr (sizeof(T) == 8)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, vi * 8u, so * 8u, CP);
    else
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, vi * 4u, so * 4u, CP);
}

template <class R, bool TRACE, int CP = 0>
__device__ __forceinline__ void gload_t(R &r, const Bufs<R> &b, uint64_t u, uint32_t so, uint32_t vi, uint64_t &h,
                                        uint32_t &n)
{
#pragma unroll
    for (int w = 0; w < R::KW; ++w) r.k[w] = ld_t<uint64_t, CP>(buf_rsrc(b.k[w] + u), vi, so);
    r.p = ld_t<typename R::P, CP>(buf_rsrc(b.p + u), vi, so);
    if constexpr (TRACE) {
        h = tfold(h, 1, u + so + vi);
        ++n;
    }
}

template <class R, bool TRACE, int CP = 0>
__device__ __forceinline__ void gstore_t(const R &r, const Bufs<R> &b, uint64_t u, uint32_t so, uint32_t vi,
                                         uint64_t &h, uint32_t &n)
{
#pragma unroll
    for (int w = 0; w < R::KW; ++w) st_t<uint64_t, CP>(buf_rsrc(b.k[w] + u), vi, so, r.k[w]);
    st_t<typename R::P, CP>(buf_rsrc(b.p + u), vi, so, r.p);
    if constexpr (TRACE) {
        h = tfold(h, 2, u + so + vi);
        ++n;
    }
}

// ----------------------------------------------------------- tiny arrays

// n_pad <= 8: one thread runs the network directly.
// Each kernel is a device body taking its block index explicitly plus a thin
// __global__ wrapper; the resident queue kernel (queue.hip) runs the same
// bodies over its own block loop.

template <class R, bool TRACE>
__device__ __forceinline__ void body_tiny(Bufs<R> b, int n_log, uint64_t n_valid, int fill, TraceSlot *slot,
                                          uint32_t blk)
{
    if (threadIdx.x != 0 || blk != 0) return;
    uint64_t h = 0;
    uint32_t nops = 0;
    const uint32_t N = 1u << n_log;
    R r[8];
    for (uint32_t i = 0; i < 8; ++i) {
        if (i < N) {
            gload<R, TRACE>(r[i], b, i, h, nops);
            if (fill) pad_select(r[i], i, n_valid);
        }
    }
    for (int p = 1; p <= n_log; ++p)
        for (int q = p - 1; q >= 0; --q)
            for (uint32_t i = 0; i < N; ++i) {
                const uint32_t ixj = i ^ (1u << q);
                if (i < ixj) cmpx_scalar(r[i], r[ixj], dir_asc(i, p, n_log));
            }
    for (uint32_t i = 0; i < 8; ++i)
        if (i < N) gstore<R, TRACE>(r[i], b, i, h, nops);
    if constexpr (TRACE) tcommit(slot, 0, h, nops);
}

template <class R, bool TRACE>
__global__ void k_sort_tiny(Bufs<R> b, int n_log, uint64_t n_valid, int fill, TraceSlot *slot)
{
    body_tiny<R, TRACE>(b, n_log, n_valid, fill, slot, blockIdx.x);
}

// ---------------------------------------------------------- tile kernels

// Tiles of 2^t records for t < T_LOG (small arrays): levels 1 .. p_max with
// runtime layouts.  Loads and stores use the coalesced layout a = t - R_LOG.
template <class R, int T_LOG, int R_LOG, int BLOCK, bool TRACE>
__device__ __forceinline__ void body_local(Bufs<R> b, IMap map, int t, int p_max, int p_top, uint64_t n_valid,
                                           int fill, TraceSlot *slot, char *lds_raw, uint32_t blk)
{
    const uint32_t T = 1u << t;
    const Lds<R> s = lds_view<R>(lds_raw, T + (T >> 4));
    const uint32_t tau = threadIdx.x;
    const bool act = tau < (T >> R_LOG);
    const uint64_t vbase = (uint64_t)blk << t;
    uint64_t h = 0;
    uint32_t nops = 0;
    R r[1 << R_LOG];
    int a = t - R_LOG;
    if (act) {
        const uint32_t base = lay_base<R_LOG>(tau, a);
#pragma unroll
        for (int m = 0; m < (1 << R_LOG); ++m) {
            const uint64_t v = vbase + (base | ((uint32_t)m << a));
            gload<R, TRACE>(r[m], b, phys(map, v), h, nops);
            if (fill) pad_select(r[m], local_row(map, v), live_rows(map, v, n_valid));
        }
    }
    for (int p = 1; p <= p_max; ++p) tile_level<R, R_LOG, TRACE>(r, s, tau, act, a, p, p - 1, p_top, vbase, h, nops);
    const int a_out = t - R_LOG;
    if (a != a_out) {
        relayout<R, R_LOG, TRACE>(r, s, tau, act, a, a_out, h, nops);
        a = a_out;
    }
    if (act) {
        const uint32_t base = lay_base<R_LOG>(tau, a);
#pragma unroll
        for (int m = 0; m < (1 << R_LOG); ++m)
            gstore<R, TRACE>(r[m], b, phys(map, vbase + (base | ((uint32_t)m << a))), h, nops);
    }
    if constexpr (TRACE) tcommit(slot, (uint64_t)blk * BLOCK + tau, h, nops);
}

template <class R, int T_LOG, int R_LOG, int BLOCK, bool TRACE>
__global__ __launch_bounds__(BLOCK) void k_sort_local(Bufs<R> b, IMap map, int t, int p_max, int p_top, uint64_t n_valid,
                                                      int fill, TraceSlot *slot)
{
    extern __shared__ __align__(16) char lds_raw[];
    body_local<R, T_LOG, R_LOG, BLOCK, TRACE>(b, map, t, p_max, p_top, n_valid, fill, slot, lds_raw, blockIdx.x);
}

// Full 2^T_LOG tiles: all levels p = 1 .. T_LOG with a compile-time schedule.
template <class R, int T_LOG, int R_LOG, int BLOCK, bool TRACE, int CP = 0>
__device__ __forceinline__ void body_local_ct(Bufs<R> b, IMap map, int p_top, uint64_t n_valid, int fill,
                                              TraceSlot *slot, char *lds, uint32_t blk)
{
    using TL = TileCT<R, T_LOG, R_LOG, TRACE>;
    constexpr int A0 = TL::A_IO;
    TileBuf buf{lds};
    const uint32_t tau = threadIdx.x;
    const uint64_t vbase = (uint64_t)blk << T_LOG;
    const uint64_t pbase = map_uniform(map, vbase);
    uint64_t h = 0;
    uint32_t nops = 0;
    R r[1 << R_LOG];
    const uint32_t base = lay_base<R_LOG>(tau, A0);
#pragma unroll
    for (int m = 0; m < (1 << R_LOG); ++m) {
        gload_t<R, TRACE, CP>(r[m], b, pbase, (uint32_t)m << A0, base, h, nops);
        if (fill) {
            const uint64_t v = vbase + (base | ((uint32_t)m << A0));
            pad_select(r[m], local_row(map, v), live_rows(map, vbase, n_valid));
        }
    }
    const bool asc_hi = dir_asc(vbase, T_LOG, p_top);
    TL::template levels<1, A0>(r, buf, tau, asc_hi, p_top, h, nops);
    TL::template relayout<TL::end_all(1, A0), A0>(r, buf, tau, h, nops);
#pragma unroll
    for (int m = 0; m < (1 << R_LOG); ++m) gstore_t<R, TRACE, CP>(r[m], b, pbase, (uint32_t)m << A0, base, h, nops);
    if constexpr (TRACE) tcommit(slot, (uint64_t)blk * BLOCK + tau, h, nops);
}

// 1024-thread blocks: two per CU, 8 waves per SIMD (at most 64 VGPRs; the
// second bound is the minimum waves per execution unit)
template <class R, int T_LOG, int R_LOG, int BLOCK, bool TRACE, int CP = 0, bool XC = true>
__global__ __launch_bounds__(BLOCK, BLOCK >= 1024 ? 8 : 1) void k_sort_local_ct(Bufs<R> b, IMap map, int p_top,
                                                                                uint64_t n_valid, int fill,
                                                                                TraceSlot *slot)
{
    extern __shared__ __align__(16) char lds[];
    body_local_ct<R, T_LOG, R_LOG, BLOCK, TRACE, CP>(b, map, p_top, n_valid, fill, slot, lds, xcd_block<XC>());
}

// Stages (p, T_LOG-1 .. 0) of one level p > T_LOG on tiles of 2^T_LOG.
template <class R, int T_LOG, int R_LOG, int BLOCK, bool TRACE, int CP = 0>
__device__ __forceinline__ void body_merge(Bufs<R> b, IMap map, int p, int p_top, TraceSlot *slot, char *lds,
                                           uint32_t blk)
{
    using TL = TileCT<R, T_LOG, R_LOG, TRACE>;
    constexpr int A0 = T_LOG - R_LOG, AS = TL::A_IO;
    TileBuf buf{lds};
    const uint32_t tau = threadIdx.x;
    const uint64_t vbase = (uint64_t)blk << T_LOG;
    const uint64_t pbase = map_uniform(map, vbase);
    uint64_t h = 0;
    uint32_t nops = 0;
    R r[1 << R_LOG];
    const uint32_t base = lay_base<R_LOG>(tau, A0);
#pragma unroll
    for (int m = 0; m < (1 << R_LOG); ++m) gload_t<R, TRACE, CP>(r[m], b, pbase, (uint32_t)m << A0, base, h, nops);
    const bool asc = dir_asc(vbase, p, p_top);
    TL::template level<-1, T_LOG - 1, A0>(r, buf, tau, asc, p_top, h, nops);
    TL::template relayout<TL::end_layout(T_LOG - 1, A0), AS>(r, buf, tau, h, nops);
#pragma unroll
    for (int m = 0; m < (1 << R_LOG); ++m)
        gstore_t<R, TRACE, CP>(r[m], b, pbase, (uint32_t)m << AS, lay_base<R_LOG>(tau, AS), h, nops);
    if constexpr (TRACE) tcommit(slot, (uint64_t)blk * BLOCK + tau, h, nops);
}

template <class R, int T_LOG, int R_LOG, int BLOCK, bool TRACE, int CP = 0, bool XC = true>
__global__ __launch_bounds__(BLOCK, BLOCK >= 1024 ? 8 : 1) void k_sort_merge(Bufs<R> b, IMap map, int p, int p_top, TraceSlot *slot)
{
    extern __shared__ __align__(16) char lds[];
    body_merge<R, T_LOG, R_LOG, BLOCK, TRACE, CP>(b, map, p, p_top, slot, lds, xcd_block<XC>());
}

// The same merge with resident blocks: each block walks tiles
// blockIdx.x, blockIdx.x + gridDim.x, ... and issues the HBM loads of its
// next tile before working on the current one, so the loads overlap the LDS
// and compare-exchange phase of the tile in hand.
template <class R, int T_LOG, int R_LOG, int BLOCK, bool TRACE>
__global__ __launch_bounds__(BLOCK) void k_sort_merge_pipe(Bufs<R> b, IMap map, int p, int p_top, uint32_t n_tiles,
                                                           TraceSlot *slot)
{
    using TL = TileCT<R, T_LOG, R_LOG, TRACE>;
    constexpr int A0 = T_LOG - R_LOG;
    constexpr int RR = 1 << R_LOG;
    extern __shared__ __align__(16) char lds[];
    TileBuf buf{lds};
    const uint32_t tau = threadIdx.x;
    const uint32_t base = lay_base<R_LOG>(tau, A0);
    uint64_t h = 0;
    uint32_t nops = 0;
    R cur[RR], nxt[RR];
    uint32_t t = blockIdx.x;
    if (t < n_tiles) {
        const uint64_t pb = map_uniform(map, (uint64_t)t << T_LOG);
#pragma unroll
        for (int m = 0; m < RR; ++m) gload_t<R, TRACE>(cur[m], b, pb, (uint32_t)m << A0, base, h, nops);
    }
    for (; t < n_tiles; t += gridDim.x) {
        const uint32_t tn = t + gridDim.x;
        if (tn < n_tiles) {
            const uint64_t pn = map_uniform(map, (uint64_t)tn << T_LOG);
#pragma unroll
            for (int m = 0; m < RR; ++m) gload_t<R, TRACE>(nxt[m], b, pn, (uint32_t)m << A0, base, h, nops);
        }
        const uint64_t vbase = (uint64_t)t << T_LOG;
        const uint64_t pbase = map_uniform(map, vbase);
        const bool asc = dir_asc(vbase, p, p_top);
        TL::template level<-1, T_LOG - 1, A0>(cur, buf, tau, asc, p_top, h, nops);
        TL::template relayout<TL::end_layout(T_LOG - 1, A0), A0>(cur, buf, tau, h, nops);
#pragma unroll
        for (int m = 0; m < RR; ++m) gstore_t<R, TRACE>(cur[m], b, pbase, (uint32_t)m << A0, base, h, nops);
#pragma unroll
        for (int m = 0; m < RR; ++m) cur[m] = nxt[m];
    }
    if constexpr (TRACE) tcommit(slot, (uint64_t)blockIdx.x * BLOCK + tau, h, nops);
}

// ------------------------------------------------------ LDS-staged passes

// A strided tile of 2^T_LOG records: 2^(T_LOG - C) runs of 2^C contiguous
// records, run r starting at element ubase + r * 2^q_lo.  Tile-local index l
// maps to element (l mod 2^C) + (l >> C) * 2^q_lo (plus the block's uniform
// bits), so tile bits [0, C) are the array's low bits and tile bits
// [C, T_LOG) its bits [q_lo, q_lo + T_LOG - C).  Two passes run on it:
//   * hybrid (TAIL = false): the S = T_LOG - C stages (p, q_lo+S-1 .. q_lo);
//   * wrap (TAIL = true, q_lo + S == p): the end of level p - 1, its stages
//     C-1 .. 0, and then the start of level p, its stages p-1 .. q_lo.  A
//     level's end and the next one's start need the array's lowest and
//     highest bits, which a tile of contiguous records and a hybrid tile
//     hold only one half of each; a wrap tile holds both, so one trip to
//     memory does the work of two.
// A tile is loaded and stored in whatever layout its first and last stages
// run in (at least 16 consecutive lanes on consecutive records), which saves
// the relayouts from and to the layout of 64.
template <int T_LOG, int R_LOG>
constexpr int strided_load_layout(int c, bool tail)
{
    int a = T_LOG - R_LOG;
    if (tail)
        while (a > c - 1 && a - R_LOG >= 4) a -= R_LOG;
    return a;
}

template <class R, int T_LOG, int R_LOG, int BLOCK, int C, bool TAIL, bool TRACE, int CP = 0>
__device__ __forceinline__ void body_strided(Bufs<R> b, IMap map, int p, int q_lo, int p_top, TraceSlot *slot,
                                             char *lds, uint32_t blk32)
{
    using TL = TileCT<R, T_LOG, R_LOG, TRACE>;
    constexpr int S = T_LOG - C;
    TileBuf buf{lds};
    constexpr int AL = strided_load_layout<T_LOG, R_LOG>(C, TAIL);
    constexpr int AT = TAIL ? TL::end_layout(C - 1, AL) : AL;
    constexpr int AS = TL::end_layout(T_LOG - 1, AT, C);
    static_assert(C >= 5 && AL >= 4 && AS >= 4, "runs of at least 32 records, 16 lanes on each");
    const uint32_t tau = threadIdx.x;
    const uint64_t blk = blk32;
    const uint64_t b_lo = blk & ((1ull << (q_lo - C)) - 1);
    const uint64_t b_hi = blk >> (q_lo - C);
    const uint64_t ublk = (b_lo << C) | (b_hi << (q_lo + S));
    const uint64_t pb = map_uniform(map, ublk);
    // element offset of tile-local index l (a bit permutation, additive over
    // disjoint bit fields; below 2^29, so a byte offset fits 32 bits)
    auto eoff = [&](uint32_t l) { return (l & ((1u << C) - 1)) | ((l >> C) << q_lo); };
    uint64_t h = 0;
    uint32_t nops = 0;
    R r[1 << R_LOG];
    {
        const uint32_t vl = eoff(lay_base<R_LOG>(tau, AL));
#pragma unroll
        for (int m = 0; m < (1 << R_LOG); ++m)
            gload_t<R, TRACE, CP>(r[m], b, pb, eoff((uint32_t)m << AL), vl, h, nops);
    }
    // tile bit T_LOG - 1 is array bit p - 1, the direction bit of level p - 1
    // (which is below the top level)
    if constexpr (TAIL) TL::template level<T_LOG - 1, C - 1, AL>(r, buf, tau, false, 64, h, nops);
    const bool asc = dir_asc(ublk, p, p_top);
    TL::template level<-1, T_LOG - 1, AT, C>(r, buf, tau, asc, p_top, h, nops);
    {
        const uint32_t vs = eoff(lay_base<R_LOG>(tau, AS));
#pragma unroll
        for (int m = 0; m < (1 << R_LOG); ++m)
            gstore_t<R, TRACE, CP>(r[m], b, pb, eoff((uint32_t)m << AS), vs, h, nops);
    }
    if constexpr (TRACE) tcommit(slot, blk * BLOCK + tau, h, nops);
}

template <class R, int T_LOG, int R_LOG, int BLOCK, int S, bool TRACE, int CP = 0, bool XC = true>
__global__ __launch_bounds__(BLOCK, BLOCK >= 1024 ? 8 : 1) void k_sort_hybrid(Bufs<R> b, IMap map, int p, int q_lo, int p_top,
                                                       TraceSlot *slot)
{
    extern __shared__ __align__(16) char lds[];
    body_strided<R, T_LOG, R_LOG, BLOCK, T_LOG - S, false, TRACE, CP>(b, map, p, q_lo, p_top, slot, lds,
                                                                      xcd_block<XC>());
}

template <class R, int T_LOG, int R_LOG, int BLOCK, int S, bool TRACE, int CP = 0, bool XC = true>
__global__ __launch_bounds__(BLOCK, BLOCK >= 1024 ? 8 : 1) void k_sort_wrap(Bufs<R> b, IMap map, int p, int q_lo, int p_top, TraceSlot *slot)
{
    extern __shared__ __align__(16) char lds[];
    body_strided<R, T_LOG, R_LOG, BLOCK, T_LOG - S, true, TRACE, CP>(b, map, p, q_lo, p_top, slot, lds,
                                                                     xcd_block<XC>());
}

// ------------------------------------------------------------ global pass

// S fused stages (p, q_lo+S-1 .. q_lo): thread g owns the 2^S records
// base(g) + m * 2^q_lo, base(g) = (g mod 2^q_lo) + (g / 2^q_lo) * 2^(q_lo+S).
// With q_lo >= 8 a block's 256 threads share every bit of base(g) above bit 7,
// so base(g) = ubase + tid and consecutive lanes touch consecutive records:
// each wavefront load or store is one contiguous 512-byte (keys) or 256-byte
// (payload) run.
template <class R, int S, bool TRACE, int CP = 0>
__device__ __forceinline__ void body_global(Bufs<R> b, IMap map, int p, int q_lo, int p_top, TraceSlot *slot,
                                            uint32_t blk, uint32_t tid)
{
    const uint64_t g0 = (uint64_t)blk * 256;
    const uint64_t ubase = (g0 & ((1ull << q_lo) - 1)) | ((g0 >> q_lo) << (q_lo + S));
    const uint64_t pbase = map_uniform(map, ubase);
    uint64_t h = 0;
    uint32_t nops = 0;
    R r[1 << S];
#pragma unroll
    for (int m = 0; m < (1 << S); ++m) gload_t<R, TRACE, CP>(r[m], b, pbase, (uint32_t)m << q_lo, tid, h, nops);
    const bool asc = dir_asc(ubase, p, p_top);
#pragma unroll
    for (int qq = S - 1; qq >= 0; --qq) cmpx_stage(r, qq, [&](int) { return asc; });
#pragma unroll
    for (int m = 0; m < (1 << S); ++m) gstore_t<R, TRACE, CP>(r[m], b, pbase, (uint32_t)m << q_lo, tid, h, nops);
    if constexpr (TRACE) tcommit(slot, g0 + tid, h, nops);
}

template <class R, int S, bool TRACE, int CP = 0, bool XC = true>
__global__ __launch_bounds__(256) void k_sort_global(Bufs<R> b, IMap map, int p, int q_lo, int p_top,
                                                     TraceSlot *slot)
{
    body_global<R, S, TRACE, CP>(b, map, p, q_lo, p_top, slot, xcd_block<XC>(), threadIdx.x);
}

} // namespace dev

// ================================================================== host

namespace sortimpl {

using dev::Bufs;
using dev::IMap;

// Largest padded row count: 8-byte columns of 2^29 rows keep every byte
// offset of the buffer-resource addressing below 2^32.
constexpr uint64_t kMaxSortRows = 1ull << 29;

struct Pass {
    // 0 tiny, 1 local, 2 global, and on tiles of the local pass's size 3 merge,
    // 4 hybrid; on tiles of 2^w records 5 wrap, 6 merge, 7 hybrid
    int kind;
    int p, q_lo, s;
    int w = 0;
};

// Pass schedule for n_log = log2(n_pad) with tiles of 2^t_log and at most
// s_max fused global stages.  Depends on public sizes only.
// With h_max > s_max, groups larger than s_max run as LDS-staged hybrid
// passes (kind 4) of up to h_max stages; a level's stages above the tile are
// split into the fewest passes, as evenly as possible.
// Width of group gi when `count` stages are split into `groups` passes.
__host__ __device__ constexpr int plan_width(int count, int groups, int gi)
{
    return count / groups + (gi < count % groups ? 1 : 0);
}

// Fewest groups of one level's `count` stages such that every group is a
// register pass (width <= s_max) or a hybrid pass (h_min <= width <= h_max):
// a caller passes the widths it has built.
__host__ __device__ inline int plan_groups(int count, int s_max, int h_max, int h_min)
{
    const int g_max = s_max > h_max ? s_max : h_max;
    for (int groups = (count + g_max - 1) / g_max;; ++groups) {
        bool ok = true;
        for (int gi = 0; gi < groups; ++gi) {
            const int s = plan_width(count, groups, gi);
            if (!(s <= s_max || (s >= h_min && s <= h_max))) ok = false;
        }
        if (ok) return groups;
    }
}

inline std::vector<Pass> plan_passes(int n_log, int t_log, int s_max, int r_log, int h_max = 0)
{
    std::vector<Pass> v;
    if (n_log < r_log) {
        v.push_back({0, n_log, 0, 0});
        return v;
    }
    const int t = std::min(n_log, t_log);
    v.push_back({1, t, 0, t});
    for (int p = t_log + 1; p <= n_log; ++p) {
        const int count = p - t_log;
        const int groups = plan_groups(count, s_max, h_max, 4); // launch path: hybrid widths 4..8
        int q = p - 1;
        for (int gi = 0; gi < groups; ++gi) {
            const int s = plan_width(count, groups, gi);
            v.push_back({s <= s_max ? 2 : 4, p, q - s + 1, s});
            q -= s;
        }
        v.push_back({3, p, 0, 0});
    }
    return v;
}

// The default schedule: the cheapest sequence of passes over the stages above
// the tile, in network order, where a pass may also end one level and start the
// next (wrap).  Found by dynamic programming from the end over (level p, next
// stage q); the costs are one pass's time at 2^28 records relative to a copy of
// the array.  (Inside the MALL they differ: at 2^23 records the nine-stage hybrid,
// here the dearest one, is the cheapest pass, 31 us against 37 for the merge and
// 40-44 for wraps; the plan found with those times is the same 16 passes.)  A
// level-by-level schedule needs ceil((p - t_log) / h_max) + 1 passes for level
// p; this one, on tiles of 2^w_log records above the local pass's 2^t_log, comes
// close to (p - 5) / (w_log - 5) on average: at 2^28 31 passes instead of 38 on
// 2^13-record tiles and 28 on 2^14-record ones.
inline std::vector<Pass> plan_wrapped(int n_log, int t_log, int w_log, int s_max, int r_log)
{
    std::vector<Pass> v;
    if (n_log <= t_log) return plan_passes(n_log, t_log, s_max, r_log);
    v.push_back({1, t_log, 0, t_log});
    struct Best {
        float cost;
        Pass pass;
        int p, q; // state after the pass
    };
    std::vector<std::vector<Best>> best(n_log + 2, std::vector<Best>(n_log + 1, Best{0.f, {}, 0, 0}));
    for (int p = n_log; p > t_log; --p)
        for (int q = 0; q < p; ++q) {
            Best &b = best[p][q];
            b.cost = 1e30f;
            // the pass ends at (p2, q2); stage -1 of a level is the start of the next
            auto consider = [&](float cost, Pass ps, int p2, int q2) {
                if (q2 < 0) {
                    ++p2;
                    q2 = p2 - 1;
                }
                const float c = cost + (p2 > n_log ? 0.f : best[p2][q2].cost);
                if (c < b.cost) b = Best{c, ps, p2, q2};
            };
            for (int s = 1; s <= s_max && q - s + 1 >= 8; ++s)
                consider(s <= 3 ? 1.f : 1.08f, {2, p, q - s + 1, s}, p, q - s);
            for (int s = 4; s <= w_log - 5; ++s) // runs of 2^(w_log - s) records, at least 32
                if (q - s + 1 >= w_log - s) consider(s <= w_log - 6 ? 1.1f : 1.14f, {7, p, q - s + 1, s, w_log}, p, q - s);
            if (q < w_log) consider(1.12f, {6, p, 0, 0, w_log}, p, -1);
            // stages q .. 0 and the next level's first s (a run of 32 records
            // may repeat a stage above q, which changes nothing)
            const int c = std::max(5, q + 1), s = w_log - c;
            if (s >= 1 && p < n_log) consider(c <= 5 ? 1.17f : 1.13f, {5, p + 1, p + 1 - s, s, w_log}, p + 1, p - s);
        }
    for (int p = t_log + 1, q = t_log; p <= n_log;) {
        const Best &b = best[p][q];
        v.push_back(b.pass);
        p = b.p;
        q = b.q;
    }
    return v;
}

// S_LARGE / LARGE_LOG: from n_pad = 2^LARGE_LOG up, register passes take at
// most S_LARGE stages (wider groups go to the hybrid pass); below, S_MAX.
// Hybrid passes of at most HW_MAX stages run with twice the threads per block
// and half the records per thread (the same tiles, so the same records per
// block): more waves per SIMD where that pass is faster.
// WRAP = false builds the level-by-level schedule alone, LEVELS = false the
// wrapped one alone (its callers ask wrapped() first), BATCH = true the
// passes over many small instances whose arrays together exceed the MALL.
template <class R, int T_LOG, int R_LOG, int BLOCK, int S_MAX, int H_MAX = 0, int S_LARGE = S_MAX, int LARGE_LOG = 64,
          int HW_MAX = 0, int W_LOG = T_LOG, bool WRAP = true, bool BATCH = false, bool LEVELS = true>
struct SortImpl {
    static_assert(T_LOG >= 8, "global passes need q_lo >= 8 (256-thread blocks)");
    static_assert(H_MAX == 0 || (T_LOG - H_MAX >= 5 && BLOCK << R_LOG == 1 << T_LOG), "hybrid tile shape");
    static_assert(S_LARGE >= 1 && S_LARGE <= S_MAX, "register cap for large sorts");
    static_assert(W_LOG >= T_LOG && W_LOG - R_LOG <= 10, "wide tiles");

    static int smax(vo_ctx *ctx, int n_log)
    {
        const int cap = n_log >= LARGE_LOG ? S_LARGE : S_MAX;
        return std::max(1, std::min(cap, ctx->tuning.max_fused_stages));
    }
    static int hmax(vo_ctx *ctx) { return std::min(H_MAX, ctx->tuning.max_hybrid_stages); }

    // The default tuning runs the wrapped schedule; a tuning word that picks
    // pass widths or block shapes, and recorded programs (whose bodies they
    // are), run level by level.
    static bool wrapped(vo_ctx *ctx)
    {
        const SortTuning &t = ctx->tuning, d;
        return WRAP && !ctx->rec && t.max_fused_stages == d.max_fused_stages &&
               t.max_hybrid_stages == d.max_hybrid_stages && !t.pipe_merge && !t.wide_block && !t.flip_hybrid_block;
    }

    // Wide tiles take one more stage bit per pass (28 passes instead of 31 for
    // 2^28 12-byte records, 32 instead of 37 for 16-byte ones) with twice the
    // threads behind each barrier.  They are used from 512 tiles, two a CU:
    // 12-byte records at 2^22 (256 tiles) 366 -> 420 us, 2^23 748 -> 728, 2^24
    // 1553 -> 1507, 2^26 8.39 -> 7.89 ms, 2^28 39.5 -> 37.1; 16-byte ones at 2^22
    // 549 -> 546 us, 2^24 2.40 -> 2.30 ms, 2^26 12.9 -> 12.0; two key words at
    // 2^22 758 -> 749 us, 2^24 3.90 -> 3.59 ms, 2^26 18.1 -> 16.0.
    static std::vector<Pass> plan(vo_ctx *ctx, int n_log, uint64_t n_virtual)
    {
        if (!wrapped(ctx)) return plan_passes(n_log, T_LOG, smax(ctx, n_log), R_LOG, hmax(ctx));
        static const auto make = [](int w) {
            std::vector<std::vector<Pass>> v;
            for (int l = 0; (1ull << l) <= kMaxSortRows; ++l)
                v.push_back(plan_wrapped(l, T_LOG, w, l >= LARGE_LOG ? S_LARGE : S_MAX, R_LOG));
            return v;
        };
        static const std::vector<std::vector<Pass>> plans = make(T_LOG), wide = make(W_LOG);
        return (n_log >= W_LOG && (n_virtual >> W_LOG) >= 512 ? wide : plans)[n_log];
    }

    template <bool TRACE, int S, int RL, int BL, int CP, bool XC>
    static void hybrid_shape(vo_ctx *ctx, Bufs<R> b, IMap map, int p, int q_lo, int p_top, uint64_t n_virtual)
    {
        using TL = dev::TileCT<R, T_LOG, RL, TRACE>;
        const size_t lds = TL::lds_bytes();
        static const char *const names[] = {"sort_hybrid_s4", "sort_hybrid_s5", "sort_hybrid_s6", "sort_hybrid_s7",
                                            "sort_hybrid_s8"};
        LaunchInfo li{names[S - 4], dim3((uint32_t)(n_virtual >> T_LOG)), dim3(BL), (uint32_t)lds,
                      hash_mix(hash_mix(p, q_lo), hash_mix(S + 100, p_top))};
        auto k = dev::k_sort_hybrid<R, T_LOG, RL, BL, S, TRACE, CP, XC>;
        VO_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        launch(ctx, li, k, b, map, p, q_lo, p_top, trace_slot(ctx));
    }

    template <bool TRACE, int S, int CP, bool XC>
    static void launch_hybrid(vo_ctx *ctx, Bufs<R> b, IMap map, int p, int q_lo, int p_top, uint64_t n_virtual)
    {
        if constexpr (S <= H_MAX && T_LOG - S >= 5) {
            static_assert(S >= 4 && S <= 8, "hybrid pass widths 4..8");
            // tuning may flip the shape (both are built when the wide one is)
            const bool wide = (S <= HW_MAX) != (HW_MAX > 0 && ctx->tuning.flip_hybrid_block);
            if (wide) {
                // the 6-stage pass on 1024-thread blocks measured faster with
                // the default policy even at 2^28 (5.53 vs 5.13 TB/s)
                constexpr int CPS = S == 6 ? 0 : CP;
                if constexpr (HW_MAX > 0)
                    hybrid_shape<TRACE, S, R_LOG - 1, 2 * BLOCK, CPS, XC>(ctx, b, map, p, q_lo, p_top, n_virtual);
            } else {
                hybrid_shape<TRACE, S, R_LOG, BLOCK, CP, XC>(ctx, b, map, p, q_lo, p_top, n_virtual);
            }
        } else {
            throw Error{VO_ERR_INVALID, "hybrid pass width not built"};
        }
    }

    // Arrays of one tile smaller than 2^T_LOG (t = 8 .. T_LOG - 1), of at most
    // two key words: the compile-time tile sort at their own size, on at least
    // one whole wavefront.  (The run-time form below keeps its LDS addresses in
    // registers and a barrier around every relayout: one array of 4096 12-byte
    // records, call and wait included, 61 -> 40 us.)  Batch classes of these
    // sizes run the same form, however many their instances (64 of 2^10 records
    // 81 -> 51 us, 1024 of 2^12 423 -> 354, call and item table included).
    template <bool TRACE, int T = 8>
    static bool launch_small(vo_ctx *ctx, Bufs<R> b, IMap map, int t, int p_top, uint64_t n_valid, int fill,
                             uint64_t n_virtual)
    {
        if constexpr (WRAP && T < T_LOG && R::KW <= 2) {
            if (t != T) return launch_small<TRACE, T + 1>(ctx, b, map, t, p_top, n_valid, fill, n_virtual);
            // few records a thread: a lone tile's time is its waves' latency
            // (2^12 records on 256, 512 and 1024 threads: 29.0, 23.4, 28.3 us;
            // 2^10 on 64, 128 and 256: 18.3, 11.4, 9.6)
            constexpr int RL = std::min(R_LOG, T >= 12 ? 3 : 2);
            const size_t lds = dev::TileCT<R, T, RL, TRACE>::lds_bytes();
            LaunchInfo li{"sort_local", dim3((uint32_t)(n_virtual >> T)), dim3(1u << (T - RL)), (uint32_t)lds,
                          hash_mix(hash_mix(T, p_top), fill)};
            launch(ctx, li, dev::k_sort_local_ct<R, T, RL, 1 << (T - RL), TRACE, 0, true>, b, map, p_top, n_valid,
                   fill, trace_slot(ctx));
            return true;
        }
        return false;
    }

    // A kernel over tiles of 2^WL records.
    template <bool TRACE, int WL, class K, class... A>
    static void launch_tiles(vo_ctx *ctx, const char *family, uint64_t n_virtual, uint64_t hash, K k, A... args)
    {
        const size_t lds = dev::TileCT<R, WL, R_LOG, TRACE>::lds_bytes();
        LaunchInfo li{family, dim3((uint32_t)(n_virtual >> WL)), dim3(1u << (WL - R_LOG)), (uint32_t)lds, hash};
        VO_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        launch(ctx, li, k, args..., trace_slot(ctx));
    }

    // Wrap passes of S = 1 .. WL - 5 stages of the upper level, hybrid passes of
    // S = 4 .. WL - 5 stages, and the merge, on tiles of 2^WL records.
    template <bool TRACE, int CP, bool XC, int WL, int S = 1>
    static void tile_pass(vo_ctx *ctx, Bufs<R> b, IMap map, const Pass &ps, int p_top, uint64_t n_virtual, bool txc)
    {
        constexpr int BW = 1 << (WL - R_LOG);
        if constexpr (!WRAP || S > WL - 5) {
            throw Error{VO_ERR_INVALID, "tile pass not built"};
        } else {
            static const char *const wraps[] = {"sort_wrap_s1", "sort_wrap_s2", "sort_wrap_s3",
                                                "sort_wrap_s4", "sort_wrap_s5", "sort_wrap_s6",
                                                "sort_wrap_s7", "sort_wrap_s8", "sort_wrap_s9"};
            static const char *const hybrids[] = {"sort_hybrid_s4", "sort_hybrid_s5", "sort_hybrid_s6",
                                                  "sort_hybrid_s7", "sort_hybrid_s8", "sort_hybrid_s9"};
            if (ps.kind == 6) {
                auto k = dev::k_sort_merge<R, WL, R_LOG, BW, TRACE, CP, XC>;
                if (!XC && txc) k = dev::k_sort_merge<R, WL, R_LOG, BW, TRACE, CP, true>;
                launch_tiles<TRACE, WL>(ctx, "sort_merge", n_virtual, hash_mix(ps.p, p_top), k, b, map, ps.p, p_top);
                return;
            }
            if (ps.s != S) return tile_pass<TRACE, CP, XC, WL, S + 1>(ctx, b, map, ps, p_top, n_virtual, txc);
            const uint64_t h = hash_mix(ps.p, ps.q_lo);
            if (ps.kind == 5)
                launch_tiles<TRACE, WL>(ctx, wraps[S - 1], n_virtual, hash_mix(h, hash_mix(S + 200, p_top)),
                                        dev::k_sort_wrap<R, WL, R_LOG, BW, S, TRACE, CP, XC>, b, map, ps.p, ps.q_lo,
                                        p_top);
            if constexpr (S >= 4)
                if (ps.kind == 7)
                    launch_tiles<TRACE, WL>(ctx, hybrids[S - 4], n_virtual, hash_mix(h, hash_mix(S + 100, p_top)),
                                            dev::k_sort_hybrid<R, WL, R_LOG, BW, S, TRACE, CP, XC>, b, map, ps.p,
                                            ps.q_lo, p_top);
        }
    }

    template <bool TRACE, int S, int CP, bool XC>
    static void launch_global(vo_ctx *ctx, const LaunchInfo &li, Bufs<R> b, IMap map, int p, int q_lo, int p_top)
    {
        if constexpr (S <= S_MAX)
            launch(ctx, li, dev::k_sort_global<R, S, TRACE, CP, XC>, b, map, p, q_lo, p_top, trace_slot(ctx));
    }

    template <bool TRACE, int CP, bool XC>
    static void global_pass(vo_ctx *ctx, Bufs<R> b, IMap map, int p, int q_lo, int s, int p_top, uint64_t n_virtual)
    {
        const uint64_t threads = n_virtual >> s;
        VO_CHECK(threads >= 256 && q_lo >= 8, VO_ERR_INVALID, "global pass below one block");
        static const char *const names[] = {"sort_global_s0", "sort_global_s1", "sort_global_s2", "sort_global_s3",
                                            "sort_global_s4", "sort_global_s5"};
        VO_CHECK(s >= 1 && s <= 5, VO_ERR_INVALID, "bad fused stage count");
        LaunchInfo li{names[s], dim3((uint32_t)(threads / 256)), dim3(256), 0,
                      hash_mix(hash_mix(p, q_lo), hash_mix(s, p_top))};
        switch (s) {
        case 1: launch_global<TRACE, 1, CP, XC>(ctx, li, b, map, p, q_lo, p_top); break;
        case 2: launch_global<TRACE, 2, CP, XC>(ctx, li, b, map, p, q_lo, p_top); break;
        case 3: launch_global<TRACE, 3, CP, XC>(ctx, li, b, map, p, q_lo, p_top); break;
        case 4: launch_global<TRACE, 4, CP, XC>(ctx, li, b, map, p, q_lo, p_top); break;
        case 5: launch_global<TRACE, 5, CP, XC>(ctx, li, b, map, p, q_lo, p_top); break;
        default: throw Error{VO_ERR_INVALID, "bad fused stage count"};
        }
    }

    // The level-by-level schedule's passes above the local one: merge (kind 3)
    // and hybrid (kind 4) on tiles of the local pass's size.
    template <bool TRACE, int CP, bool XC>
    static void level_pass(vo_ctx *ctx, Bufs<R> b, IMap map, const Pass &ps, int n_log, int p_top, uint64_t n_virtual)
    {
        if (ps.kind == 4) {
            switch (ps.s) {
            case 4: launch_hybrid<TRACE, 4, CP, XC>(ctx, b, map, ps.p, ps.q_lo, p_top, n_virtual); break;
            case 5: launch_hybrid<TRACE, 5, CP, XC>(ctx, b, map, ps.p, ps.q_lo, p_top, n_virtual); break;
            case 6: launch_hybrid<TRACE, 6, CP, XC>(ctx, b, map, ps.p, ps.q_lo, p_top, n_virtual); break;
            case 7: launch_hybrid<TRACE, 7, CP, XC>(ctx, b, map, ps.p, ps.q_lo, p_top, n_virtual); break;
            case 8: launch_hybrid<TRACE, 8, CP, XC>(ctx, b, map, ps.p, ps.q_lo, p_top, n_virtual); break;
            default: throw Error{VO_ERR_INVALID, "bad hybrid stage count"};
            }
            return;
        }
        const size_t lds = dev::TileCT<R, T_LOG, R_LOG, TRACE>::lds_bytes();
        const uint32_t n_tiles = (uint32_t)(n_virtual >> T_LOG);
        if (ctx->tuning.pipe_merge && !ctx->rec) { // resident: plain merge blocks
            auto k = dev::k_sort_merge_pipe<R, T_LOG, R_LOG, BLOCK, TRACE>;
            VO_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            int per_cu = 0;
            VO_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k, BLOCK, lds));
            const uint32_t grid = std::min<uint32_t>(n_tiles, (uint32_t)std::max(1, per_cu) * ctx->num_cus);
            LaunchInfo li{"sort_merge", dim3(grid), dim3(BLOCK), (uint32_t)lds, hash_mix(ps.p, p_top)};
            launch(ctx, li, k, b, map, ps.p, p_top, n_tiles, trace_slot(ctx));
        } else {
            LaunchInfo li{"sort_merge", dim3(n_tiles), dim3(BLOCK), (uint32_t)lds, hash_mix(ps.p, p_top)};
            auto k = dev::k_sort_merge<R, T_LOG, R_LOG, BLOCK, TRACE, CP, XC>;
            if (!XC && tiles_xc(n_log)) k = dev::k_sort_merge<R, T_LOG, R_LOG, BLOCK, TRACE, CP, true>;
            VO_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            launch(ctx, li, k, b, map, ps.p, p_top, trace_slot(ctx));
        }
    }

    template <bool TRACE, int CP, bool XC>
    static void run_t(vo_ctx *ctx, Bufs<R> b, int n_log, uint64_t n_valid, int fill, IMap map, int p_top,
                      uint64_t n_virtual)
    {
        for (const Pass &ps : plan(ctx, n_log, n_virtual)) {
            switch (ps.kind) {
            case 0: {
                LaunchInfo li{"sort_tiny", dim3(1), dim3(64), 0, hash_mix(n_log, fill)};
                launch(ctx, li, dev::k_sort_tiny<R, TRACE>, b, n_log, n_valid, fill, trace_slot(ctx));
                break;
            }
            case 1: {
                const int t = ps.p;
                const bool ct = (t == T_LOG && p_top >= T_LOG);
                if (!ct && !ctx->rec && launch_small<TRACE>(ctx, b, map, t, p_top, n_valid, fill, n_virtual)) break;
                const size_t lds = ct ? dev::TileCT<R, T_LOG, R_LOG, TRACE>::lds_bytes() : dev::lds_bytes<R>(t);
                LaunchInfo li{"sort_local", dim3((uint32_t)(n_virtual >> t)), dim3(BLOCK), (uint32_t)lds,
                              hash_mix(hash_mix(t, p_top), fill)};
                if (ct) {
                    auto k = dev::k_sort_local_ct<R, T_LOG, R_LOG, BLOCK, TRACE, CP, XC>;
                    if (!XC && tiles_xc(n_log)) k = dev::k_sort_local_ct<R, T_LOG, R_LOG, BLOCK, TRACE, CP, true>;
                    VO_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
                    launch(ctx, li, k, b, map, p_top, n_valid, fill, trace_slot(ctx));
                } else {
                    auto k = dev::k_sort_local<R, T_LOG, R_LOG, BLOCK, TRACE>;
                    VO_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
                    launch(ctx, li, k, b, map, t, std::min(t, p_top), p_top, n_valid, fill, trace_slot(ctx));
                }
                break;
            }
            case 2: global_pass<TRACE, CP, XC>(ctx, b, map, ps.p, ps.q_lo, ps.s, p_top, n_virtual); break;
            case 5:
            case 6:
            case 7:
                if (ps.w == T_LOG)
                    tile_pass<TRACE, CP, XC, T_LOG>(ctx, b, map, ps, p_top, n_virtual, tiles_xc(n_log));
                else
                    tile_pass<TRACE, CP, XC, W_LOG>(ctx, b, map, ps, p_top, n_virtual, tiles_xc(n_log));
                break;
            case 3:
            case 4:
                if constexpr (LEVELS)
                    level_pass<TRACE, CP, XC>(ctx, b, map, ps, n_log, p_top, n_virtual);
                else
                    throw Error{VO_ERR_INVALID, "level-by-level pass not built"};
                break;
            }
        }
    }

    // Streaming loads and stores (dev::kCpStream) when the arrays a launch
    // covers exceed the 256 MB MALL, so that no pass re-reads them from it.
    // Measured on the 12-byte sort: +4% at 2^26 and +2.7% at 2^28, but -8% at
    // 2^24, which the MALL holds.  Resident programs keep the default (their
    // bodies are built with it); tuning bit 0x800 flips the choice.
    static constexpr uint64_t kMallBytes = 256ull << 20;
    static uint64_t bytes(uint64_t rows) { return rows * (8 * R::KW + sizeof(typename R::P)); }
    static bool streaming(vo_ctx *ctx, uint64_t n_virtual)
    {
        const bool big = bytes(n_virtual) > kMallBytes;
        return !ctx->rec && (big != (ctx->tuning.flip_streaming != 0));
    }

    // Block order of the contiguous tile passes (dev::xcd_block) of an instance
    // above the MALL.
    static bool tiles_xc(int n_log) { return bytes(1ull << n_log) >= 3 * kMallBytes; }

    static void dispatch(vo_ctx *ctx, Bufs<R> b, int n_log, uint64_t n_valid, int fill, IMap map, int p_top,
                         uint64_t n_virtual)
    {
        if (ctx->tracing)
            run_t<true, 0, true>(ctx, b, n_log, n_valid, fill, map, p_top, n_virtual);
        else if (!streaming(ctx, n_virtual))
            run_t<false, 0, true>(ctx, b, n_log, n_valid, fill, map, p_top, n_virtual);
        else if (BATCH && bytes(1ull << n_log) <= kMallBytes)
            run_t<false, dev::kCpStream, BATCH>(ctx, b, n_log, n_valid, fill, map, p_top, n_virtual);
        else
            run_t<false, dev::kCpStream, false>(ctx, b, n_log, n_valid, fill, map, p_top, n_virtual);
    }

    static void run(vo_ctx *ctx, Bufs<R> b, int n_log, uint64_t n_valid, int fill)
    {
        VO_CHECK((1ull << n_log) <= kMaxSortRows, VO_ERR_INVALID,
                 "n_pad above 2^29 (32-bit buffer offsets of 8-byte columns)");
        dispatch(ctx, b, n_log, n_valid, fill, IMap{nullptr, 0, nullptr}, n_log, 1ull << n_log);
    }

    // `count` independent instances of 2^c rows, instance i at element
    // offsets[i] with ns[i] live rows (both device arrays): one schedule for
    // all of them, every launch covering every instance.
    static void run_mapped(vo_ctx *ctx, Bufs<R> b, int c, uint64_t count, const uint64_t *offsets, const uint64_t *ns)
    {
        VO_CHECK(c >= R_LOG && (1ull << c) <= kMaxSortRows, VO_ERR_INVALID, "batched instance size out of range");
        dispatch(ctx, b, c, 0, 1, IMap{offsets, c, ns}, c, count << c);
    }

    static int passes(vo_ctx *ctx, int n_log) { return (int)plan(ctx, n_log, 1ull << n_log).size(); }
};

// Record kinds and their tile shapes (LDS = 2^T_LOG * 17/16 * record bytes).
using RecKP = dev::Rec<1, uint32_t, true>; // 12 B: u64 key + u32 payload
using RecKV = dev::Rec<1, uint64_t, true>; // 16 B: u64 key + u64 value
// multi-column: packed key words + the u32 row index (the unpack pass widens
// it into the caller's int64 index column)
using RecM1 = dev::Rec<1, uint32_t, false>;
using RecM2 = dev::Rec<2, uint32_t, false>;
using RecM4 = dev::Rec<4, uint32_t, false>;
using RecM8 = dev::Rec<8, uint32_t, false>;

} // namespace sortimpl
} // namespace vo
