// sort_core.hpp -- device building blocks of the oblivious bitonic network.
//
// The network is the reference's: for k = 2, 4, ..., N and j = k/2, ..., 1,
// element i is compare-exchanged with i ^ j, ascending when (i & k) == 0
// (include/cuda/sort.cuh:104-117).  Stage (k = 2^p, j = 2^q) is written
// (p, q).  The schedule here executes exactly those compare-exchanges in the
// same per-element order, but groups stages so that one HBM pass applies many
// of them:
//   * tile kernels hold a 2^t-element tile per block; each thread keeps
//     2^R_LOG elements in registers whose indices differ in R_LOG adjacent
//     bits [a, a + R_LOG) ("layout a"); stages on those bits run in
//     registers, and a change of layout goes through LDS;
//   * global kernels apply S consecutive stages (p, q_lo + S - 1 .. q_lo) to
//     groups of 2^S elements at stride 2^q_lo, one group per thread.
// Every compare-exchange reads and writes both slots and selects with
// v_cndmask, so the address stream depends only on the public sizes.
#pragma once

#include "vo_internal.hpp"

namespace vo {
namespace dev {

// ---------------------------------------------------------------- records

// A record: KW 64-bit key words compared lexicographically, then (when TIE)
// the payload.  Stored as KW + 1 separate arrays (structure of arrays).
template <int KW_, typename P_, bool TIE_>
struct Rec {
    static constexpr int KW = KW_;
    using P = P_;
    static constexpr bool TIE = TIE_;
    uint64_t k[KW];
    P p;
};

template <class R>
struct Bufs {
    uint64_t *k[R::KW];
    typename R::P *p;
};

template <class R>
__device__ __forceinline__ bool rec_gt(const R &a, const R &b)
{
    bool gt = false, eq = true;
#pragma unroll
    for (int w = 0; w < R::KW; ++w) {
        gt = gt | (eq & (a.k[w] > b.k[w]));
        eq = eq & (a.k[w] == b.k[w]);
    }
    if constexpr (R::TIE) gt = gt | (eq & (a.p > b.p));
    return gt;
}

// Compare-exchange: afterwards a <= b when asc, a >= b otherwise.  Ties
// (equal over every compared field) are left in place, as needSwap does
// (sort.cuh:31-40).
// The comparison runs on wavefront lane masks and the swap is v_cndmask on the
// resulting mask (2 per 32-bit word).  `ascm` holds the lanes whose pair sorts
// ascending.
//
// Wait states.  On gfx950 a VALU instruction that reads a mask or a carry (an
// SGPR pair or vcc) stands at least two wait states behind the VALU instruction
// that wrote it: hipcc puts s_nop 1 between v_sub_co and v_subb_co, and fills
// the distance from a v_cmp to its v_cndmask.  It does not look into asm blocks,
// so they keep the distance themselves: borrow chains run interleaved (or on
// s_nop), and a block of selects makes its mask with a scalar instruction of its
// own, whose operands and result the hardware waits for (outside the block a
// mask may come from a v_cmp, or from the v_readlane of a spilled register).

// lt[i] = lanes where pair i has a < b as one unsigned integer of WORDS 32-bit
// words: the borrow out of a subtract-with-borrow chain, a VALU instruction a
// word and no scalar logic.  Four chains side by side keep the two wait states
// for nothing; two need one s_nop 0 a word.
#define VO_SUB(M, A, B) "v_sub_co_u32_e64 %[t], %[" M "], %[" A "], %[" B "]\n\t"
#define VO_SUBB(M, A, B) "v_subb_co_u32_e64 %[t], %[" M "], %[" A "], %[" B "], %[" M "]\n\t"
#define VO_WORD4(OP, W) OP("m0", "a0" W, "b0" W) OP("m1", "a1" W, "b1" W) OP("m2", "a2" W, "b2" W) OP("m3", "a3" W, "b3" W)
#define VO_WORD2(OP, W) OP("m0", "a0" W, "b0" W) OP("m1", "a1" W, "b1" W)
#define VO_WORD1(OP, W) OP("m0", "a0" W, "b0" W)
#define VO_IN(I, W) [a##I##W] "v"(a[I][W]), [b##I##W] "v"(b[I][W])
#define VO_IN3(I) VO_IN(I, 0), VO_IN(I, 1), VO_IN(I, 2)
#define VO_IN4(I) VO_IN3(I), VO_IN(I, 3)
#define VO_OUT(I) [m##I] "=&s"(lt[I])

template <int N, int WORDS>
__device__ __forceinline__ void lt_masks(uint64_t (&lt)[N], const uint32_t (&a)[N][WORDS],
                                         const uint32_t (&b)[N][WORDS])
{
    static_assert((N == 1 || N == 2 || N == 4) && (WORDS == 3 || WORDS == 4), "chains built");
    uint32_t t;
    if constexpr (N == 4 && WORDS == 3)
        asm(VO_WORD4(VO_SUB, "0") VO_WORD4(VO_SUBB, "1") VO_WORD4(VO_SUBB, "2")
            : [t] "=&v"(t), VO_OUT(0), VO_OUT(1), VO_OUT(2), VO_OUT(3)
            : VO_IN3(0), VO_IN3(1), VO_IN3(2), VO_IN3(3));
    else if constexpr (N == 4)
        asm(VO_WORD4(VO_SUB, "0") VO_WORD4(VO_SUBB, "1") VO_WORD4(VO_SUBB, "2") VO_WORD4(VO_SUBB, "3")
            : [t] "=&v"(t), VO_OUT(0), VO_OUT(1), VO_OUT(2), VO_OUT(3)
            : VO_IN4(0), VO_IN4(1), VO_IN4(2), VO_IN4(3));
    else if constexpr (N == 2 && WORDS == 3)
        asm(VO_WORD2(VO_SUB, "0") "s_nop 0\n\t" VO_WORD2(VO_SUBB, "1") "s_nop 0\n\t" VO_WORD2(VO_SUBB, "2")
            : [t] "=&v"(t), VO_OUT(0), VO_OUT(1)
            : VO_IN3(0), VO_IN3(1));
    else if constexpr (N == 2)
        asm(VO_WORD2(VO_SUB, "0") "s_nop 0\n\t" VO_WORD2(VO_SUBB, "1") "s_nop 0\n\t" VO_WORD2(VO_SUBB, "2")
            "s_nop 0\n\t" VO_WORD2(VO_SUBB, "3")
            : [t] "=&v"(t), VO_OUT(0), VO_OUT(1)
            : VO_IN4(0), VO_IN4(1));
    else if constexpr (WORDS == 3)
        asm(VO_WORD1(VO_SUB, "0") "s_nop 1\n\t" VO_WORD1(VO_SUBB, "1") "s_nop 1\n\t" VO_WORD1(VO_SUBB, "2")
            : [t] "=&v"(t), VO_OUT(0)
            : VO_IN3(0));
    else
        asm(VO_WORD1(VO_SUB, "0") "s_nop 1\n\t" VO_WORD1(VO_SUBB, "1") "s_nop 1\n\t" VO_WORD1(VO_SUBB, "2")
            "s_nop 1\n\t" VO_WORD1(VO_SUBB, "3")
            : [t] "=&v"(t), VO_OUT(0)
            : VO_IN4(0));
}

#undef VO_SUB
#undef VO_SUBB
#undef VO_WORD4
#undef VO_WORD2
#undef VO_WORD1
#undef VO_IN
#undef VO_IN3
#undef VO_IN4
#undef VO_OUT

// The lanes that swap, as two masks and the scalar instruction that joins them.
enum class Join { kXor, kOr, kCopy };
struct SwapMask {
    uint64_t a, b; // kCopy: a alone
};

// Exchanges x[0 .. W-1] and y[0 .. W-1] in the lanes of m.  Selects run as the
// VOP3 form of v_cndmask on a mask in scalar registers: the compiler shrinks a
// select whose mask it has put in vcc to the VOP2 form, and that form issues in
// 23 cycles a wavefront on this chip where the VOP3 one takes 4.5 (a compare,
// its wait states and three selects: 14.2 against 4.2 cycles an instruction).
// OWN: the new y stays in y's registers.  It saves W registers, which the
// 12-byte sort's 64-VGPR passes need (nine-stage pass: no spill instead of 7
// VGPRs), but costs moves where 8-byte columns must stand in register pairs
// (two key words, local pass: 10477 VALU instructions instead of 9035).
#define VO_SEL(I, D)                                                                                                   \
    "v_cndmask_b32_e64 %[o" I "], %[x" I "], %[y" I "], %[s]\n\t"                                                     \
    "v_cndmask_b32_e64 %[" D I "], %[y" I "], %[x" I "], %[s]\n\t"
#define VO_NEW(I) [o##I] "=&v"(o[I]), [n##I] "=&v"(n[I])
#define VO_OWN(I) [o##I] "=&v"(o[I]), [y##I] "+v"(y[I])
#define VO_IN(I) [x##I] "v"(x[I]), [y##I] "v"(y[I])
#define VO_SWAP(OP, ...)                                                                                               \
    if constexpr (OWN)                                                                                                 \
        asm(OP VO_SEL("0", "y") VO_SEL("1", "y") VO_SEL("2", "y")                                                      \
            : [s] "=&s"(s), VO_OWN(0), VO_OWN(1), VO_OWN(2)                                                            \
            : [x0] "v"(x[0]), [x1] "v"(x[1]), [x2] "v"(x[2]), __VA_ARGS__                                              \
            : "scc");                                                                                                  \
    else if constexpr (W == 2)                                                                                         \
        asm(OP VO_SEL("0", "n") VO_SEL("1", "n")                                                                       \
            : [s] "=&s"(s), VO_NEW(0), VO_NEW(1)                                                                       \
            : VO_IN(0), VO_IN(1), __VA_ARGS__                                                                          \
            : "scc");                                                                                                  \
    else if constexpr (W == 3)                                                                                         \
        asm(OP VO_SEL("0", "n") VO_SEL("1", "n") VO_SEL("2", "n")                                                      \
            : [s] "=&s"(s), VO_NEW(0), VO_NEW(1), VO_NEW(2)                                                            \
            : VO_IN(0), VO_IN(1), VO_IN(2), __VA_ARGS__                                                                \
            : "scc");                                                                                                  \
    else if constexpr (W == 4)                                                                                         \
        asm(OP VO_SEL("0", "n") VO_SEL("1", "n") VO_SEL("2", "n") VO_SEL("3", "n")                                     \
            : [s] "=&s"(s), VO_NEW(0), VO_NEW(1), VO_NEW(2), VO_NEW(3)                                                 \
            : VO_IN(0), VO_IN(1), VO_IN(2), VO_IN(3), __VA_ARGS__                                                      \
            : "scc");                                                                                                  \
    else                                                                                                               \
        asm(OP VO_SEL("0", "n") VO_SEL("1", "n") VO_SEL("2", "n") VO_SEL("3", "n") VO_SEL("4", "n")                    \
            : [s] "=&s"(s), VO_NEW(0), VO_NEW(1), VO_NEW(2), VO_NEW(3), VO_NEW(4)                                      \
            : VO_IN(0), VO_IN(1), VO_IN(2), VO_IN(3), VO_IN(4), __VA_ARGS__                                            \
            : "scc")

template <Join J, int W>
__device__ __forceinline__ void swap_block(SwapMask m, uint32_t *x, uint32_t *y)
{
    static_assert(W >= 2 && W <= 5, "words of one block");
    constexpr bool OWN = J == Join::kXor && W == 3;
    uint64_t s;
    uint32_t o[W], n[W];
    if constexpr (J == Join::kXor) {
        VO_SWAP("s_xor_b64 %[s], %[a], %[b]\n\t", [a] "s"(m.a), [b] "s"(m.b));
    } else if constexpr (J == Join::kOr) {
        VO_SWAP("s_or_b64 %[s], %[a], %[b]\n\t", [a] "s"(m.a), [b] "s"(m.b));
    } else {
        VO_SWAP("s_mov_b64 %[s], %[a]\n\t", [a] "s"(m.a));
    }
#pragma unroll
    for (int w = 0; w < W; ++w) {
        x[w] = o[w];
        if constexpr (!OWN) y[w] = n[w];
    }
}

#undef VO_SEL
#undef VO_NEW
#undef VO_OWN
#undef VO_IN
#undef VO_SWAP

template <Join J, int W>
__device__ __forceinline__ void swap_words(SwapMask m, uint32_t *x, uint32_t *y)
{
    if constexpr (W > 5) {
        constexpr int F = W == 6 ? 4 : 5; // at least two words stay
        swap_block<J, F>(m, x, y);
        swap_words<J, W - F>(m, x + F, y + F);
    } else {
        swap_block<J, W>(m, x, y);
    }
}

// A record as 32-bit words, payload lowest.
template <class R>
constexpr int rec_words() { return 2 * R::KW + (int)sizeof(typename R::P) / 4; }

template <class R>
__device__ __forceinline__ void rec_to_words(uint32_t (&v)[rec_words<R>()], const R &r)
{
    constexpr int PW = (int)sizeof(typename R::P) / 4;
#pragma unroll
    for (int w = 0; w < PW; ++w) v[w] = (uint32_t)((uint64_t)r.p >> (32 * w));
#pragma unroll
    for (int w = 0; w < 2 * R::KW; ++w) v[PW + w] = (uint32_t)(r.k[w / 2] >> (32 * (w & 1)));
}

template <class R>
__device__ __forceinline__ void rec_from_words(R &r, const uint32_t (&v)[rec_words<R>()])
{
    constexpr int PW = (int)sizeof(typename R::P) / 4;
    if constexpr (PW == 2)
        r.p = (typename R::P)((uint64_t)v[0] | ((uint64_t)v[1] << 32));
    else
        r.p = (typename R::P)v[0];
#pragma unroll
    for (int w = 0; w < R::KW; ++w) r.k[w] = (uint64_t)v[PW + 2 * w] | ((uint64_t)v[PW + 2 * w + 1] << 32);
}

// Compare-exchanges of one stage on a thread's registers: register m with
// m | 1 << bit, ascending where asc(m).  Four pairs at a time, whose compares
// are interleaved.
template <class R, int RR, class D>
__device__ __forceinline__ void cmpx_stage(R (&r)[RR], int bit, D asc)
{
    constexpr int N = RR / 2 < 4 ? RR / 2 : 4, W = rec_words<R>();
#pragma unroll
    for (int g = 0; g < RR / 2; g += N) {
        auto lower = [&](int i) { return (((g + i) >> bit) << (bit + 1)) | ((g + i) & ((1 << bit) - 1)); };
        uint32_t x[N][W], y[N][W];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            rec_to_words(x[i], r[lower(i)]);
            rec_to_words(y[i], r[lower(i) | (1 << bit)]);
        }
        if constexpr (R::TIE && R::KW == 1) {
            // (key, payload) records compare as one integer, key high.  Records
            // equal in every field are identical, so exchanging them on a tie
            // changes nothing and the swap is simply lt(x, y) xor ascending.
            uint64_t lt[N];
            lt_masks<N, W>(lt, x, y);
#pragma unroll
            for (int i = 0; i < N; ++i)
                swap_words<Join::kXor, W>({lt[i], __builtin_amdgcn_ballot_w64(asc(lower(i)))}, x[i], y[i]);
        } else {
            static_assert(!R::TIE, "other records leave ties in place");
            // each key word costs one v_cmp for > and one for <; the lexicographic
            // combination and the direction are scalar mask operations
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const R &a = r[lower(i)], &b = r[lower(i) | (1 << bit)];
                const uint64_t ascm = __builtin_amdgcn_ballot_w64(asc(lower(i)));
                uint64_t gt = 0, lt = 0, eq = ~0ull;
#pragma unroll
                for (int w = 0; w < R::KW; ++w) {
                    const uint64_t g = __builtin_amdgcn_ballot_w64(a.k[w] > b.k[w]);
                    const uint64_t l = __builtin_amdgcn_ballot_w64(a.k[w] < b.k[w]);
                    gt |= eq & g;
                    lt |= eq & l;
                    eq &= ~(g | l);
                }
                swap_words<Join::kOr, W>({ascm & gt, ~ascm & lt}, x[i], y[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < N; ++i) {
            rec_from_words(r[lower(i)], x[i]);
            rec_from_words(r[lower(i) | (1 << bit)], y[i]);
        }
    }
}

// Scalar reference form of the same exchange (used by the one-thread kernel,
// where lane masks would not describe the per-iteration pairs).
template <class R>
__device__ __forceinline__ void cmpx_scalar(R &a, R &b, bool asc)
{
    const bool sw = asc ? rec_gt(a, b) : rec_gt(b, a);
#pragma unroll
    for (int w = 0; w < R::KW; ++w) {
        const uint64_t x = a.k[w], y = b.k[w];
        a.k[w] = sw ? y : x;
        b.k[w] = sw ? x : y;
    }
    const typename R::P x = a.p, y = b.p;
    a.p = sw ? y : x;
    b.p = sw ? x : y;
}

// Direction of stage level p for (virtual) element index g: ascending when
// bit p of g is clear, and always at the top level p_top of an instance.
__device__ __forceinline__ bool dir_asc(uint64_t g, int p, int p_top)
{
    return (p >= p_top) | (((g >> p) & 1) == 0);
}

// Virtual-to-physical index map.  Plain sorts use the identity; batched
// sorts place instance v >> c at offsets[v >> c].
struct IMap {
    const uint64_t *offsets; // nullptr -> identity
    int c;                   // log2 instance size when offsets != nullptr
    const uint64_t *ns;      // live rows per instance (pad fill), or nullptr
};

__device__ __forceinline__ uint64_t phys(const IMap &m, uint64_t v)
{
    if (m.offsets == nullptr) return v;
    return m.offsets[v >> m.c] + (v & ((1ull << m.c) - 1));
}

// Pad fill for virtual row v: its row index inside its instance and the
// instance's live row count.
__device__ __forceinline__ uint64_t local_row(const IMap &m, uint64_t v)
{
    return m.offsets == nullptr ? v : (v & ((1ull << m.c) - 1));
}

__device__ __forceinline__ uint64_t live_rows(const IMap &m, uint64_t v, uint64_t n_valid)
{
    return m.ns == nullptr ? n_valid : m.ns[v >> m.c];
}

template <class R, bool TRACE>
__device__ __forceinline__ void gload(R &r, const Bufs<R> &b, uint64_t i, uint64_t &h, uint32_t &n)
{
#pragma unroll
    for (int w = 0; w < R::KW; ++w) r.k[w] = b.k[w][i];
    r.p = b.p[i];
    if constexpr (TRACE) {
        h = tfold(h, 1, i);
        ++n;
    }
}

template <class R, bool TRACE>
__device__ __forceinline__ void gstore(const R &r, const Bufs<R> &b, uint64_t i, uint64_t &h, uint32_t &n)
{
#pragma unroll
    for (int w = 0; w < R::KW; ++w) b.k[w][i] = r.k[w];
    b.p[i] = r.p;
    if constexpr (TRACE) {
        h = tfold(h, 2, i);
        ++n;
    }
}

// Pad record for sorts that fill [n, n_pad): all key bits set, payload = index.
template <class R>
__device__ __forceinline__ void pad_select(R &r, uint64_t g, uint64_t n_valid)
{
    const bool pad = g >= n_valid;
#pragma unroll
    for (int w = 0; w < R::KW; ++w) r.k[w] = pad ? ~0ull : r.k[w];
    r.p = pad ? (typename R::P)g : r.p;
}

// Blocks go to the 8 XCDs in turn; this order gives every XCD one contiguous
// range of the launch's blocks (the first grid mod 8 ranges are one longer),
// so a pass finds in its XCD's L2 what the pass before left there.  While an
// instance fits the MALL every pass gains (12-byte sort, one-stage pass: 8.8
// -> 5.8 us at 2^20 records, 29.5 -> 28.9 at 2^23; batched sorts 59.2 -> 57.8
// ms).  Above it strided passes lose (1009 -> 1060 us at 2^28: every run they
// read is another DRAM page) and keep the plain order; contiguous tiles gain
// from 3 times the MALL up (merge pass 1219 -> 1123 us at 2^28; whole sorts at
// 2^26, 2^27 and 2^28: 10.18 -> 10.03, 22.4 -> 21.9 and 48.8 -> 47.3 ms) but
// lose between (16-byte sort at 2^25: 6.72 -> 6.88 ms; two key words at 2^24:
// 4.37 -> 4.45 ms), where part of a pass is still found in the MALL.
template <bool XC = true>
__device__ __forceinline__ uint32_t xcd_block()
{
    if constexpr (!XC) return blockIdx.x;
    const uint32_t q = gridDim.x >> 3, rem = gridDim.x & 7, x = blockIdx.x & 7;
    return x * q + (x < rem ? x : rem) + (blockIdx.x >> 3);
}

// ------------------------------------------------------------ tile layout

// LDS position of tile element l: one pad slot per 16 elements keeps the
// strided layouts free of bank conflicts for 4- and 8-byte columns.
__device__ __forceinline__ uint32_t lpos(uint32_t l) { return l + (l >> 4); }

// Element held in register m by thread tau under layout a.
template <int R_LOG>
__device__ __forceinline__ uint32_t lay_base(uint32_t tau, int a)
{
    return (tau & ((1u << a) - 1)) | ((tau >> a) << (a + R_LOG));
}

template <class R>
struct Lds {
    uint64_t *k; // KW arrays of tpad words
    typename R::P *p;
    uint32_t tpad;
};

template <class R>
__device__ __forceinline__ Lds<R> lds_view(char *base, uint32_t tpad)
{
    Lds<R> s;
    s.k = reinterpret_cast<uint64_t *>(base);
    s.p = reinterpret_cast<typename R::P *>(base + sizeof(uint64_t) * R::KW * tpad);
    s.tpad = tpad;
    return s;
}

template <class R>
constexpr size_t lds_bytes(int t)
{
    return (size_t)((1u << t) + ((1u << t) >> 4)) * (sizeof(uint64_t) * R::KW + sizeof(typename R::P));
}

template <class R, int R_LOG, bool TRACE>
__device__ __forceinline__ void lds_put(const R (&r)[1 << R_LOG], const Lds<R> &s, uint32_t tau, int a,
                                        uint64_t &h, uint32_t &n)
{
    const uint32_t base = lay_base<R_LOG>(tau, a);
#pragma unroll
    for (int m = 0; m < (1 << R_LOG); ++m) {
        const uint32_t l = lpos(base | ((uint32_t)m << a));
#pragma unroll
        for (int w = 0; w < R::KW; ++w) s.k[w * s.tpad + l] = r[m].k[w];
        s.p[l] = r[m].p;
        if constexpr (TRACE) {
            h = tfold(h, 3, l);
            ++n;
        }
    }
}

template <class R, int R_LOG, bool TRACE>
__device__ __forceinline__ void lds_get(R (&r)[1 << R_LOG], const Lds<R> &s, uint32_t tau, int a, uint64_t &h,
                                        uint32_t &n)
{
    const uint32_t base = lay_base<R_LOG>(tau, a);
#pragma unroll
    for (int m = 0; m < (1 << R_LOG); ++m) {
        const uint32_t l = lpos(base | ((uint32_t)m << a));
#pragma unroll
        for (int w = 0; w < R::KW; ++w) r[m].k[w] = s.k[w * s.tpad + l];
        r[m].p = s.p[l];
        if constexpr (TRACE) {
            h = tfold(h, 4, l);
            ++n;
        }
    }
}

// Stages (p, q) for q = q_hi down to q_lo, all inside the register bits of
// layout a (a <= q_lo <= q_hi < a + R_LOG).  `vbase` is the virtual index of
// tile element 0.
template <class R, int R_LOG>
__device__ __forceinline__ void reg_stages(R (&r)[1 << R_LOG], uint32_t tau, int a, int q_hi, int q_lo, int p,
                                           int p_top, uint64_t vbase)
{
    const uint32_t base = lay_base<R_LOG>(tau, a);
#pragma unroll
    for (int qq = R_LOG - 1; qq >= 0; --qq) {
        const int q = a + qq;
        if (q > q_hi || q < q_lo) continue;
        cmpx_stage(r, qq, [&](int m) { return dir_asc(vbase + (base | ((uint32_t)m << a)), p, p_top); });
    }
}

// Moves the tile from layout a_old to layout a_new through LDS.
template <class R, int R_LOG, bool TRACE>
__device__ __forceinline__ void relayout(R (&r)[1 << R_LOG], const Lds<R> &s, uint32_t tau, bool act, int a_old,
                                         int a_new, uint64_t &h, uint32_t &n)
{
    __syncthreads();
    if (act) lds_put<R, R_LOG, TRACE>(r, s, tau, a_old, h, n);
    __syncthreads();
    if (act) lds_get<R, R_LOG, TRACE>(r, s, tau, a_new, h, n);
}

// Runs stages (p, q_start .. 0) of one level on the tile in registers,
// changing layout whenever the next stage bit is not a register bit.
template <class R, int R_LOG, bool TRACE>
__device__ __forceinline__ void tile_level(R (&r)[1 << R_LOG], const Lds<R> &s, uint32_t tau, bool act, int &a,
                                           int p, int q_start, int p_top, uint64_t vbase, uint64_t &h, uint32_t &n)
{
    int q = q_start;
    while (q >= 0) {
        if (!(a <= q && q < a + R_LOG)) {
            const int a_new = q - R_LOG + 1 > 0 ? q - R_LOG + 1 : 0;
            relayout<R, R_LOG, TRACE>(r, s, tau, act, a, a_new, h, n);
            a = a_new;
        }
        if (act) reg_stages<R, R_LOG>(r, tau, a, q, a, p, p_top, vbase);
        q = a - 1;
    }
}

// ------------------------------------------------- compile-time tile schedule

// Same schedule as tile_level, with the tile size, every layout and every
// level fixed at compile time, so that all LDS offsets are immediates and the
// stage loops fully unroll.  Used for full 2^T_LOG tiles.
// A block's relayout buffer.  shared: other waves may still read what they (or
// the block's last tile) moved through it.
struct TileBuf {
    char *p;
    bool shared = true;
};

template <class R, int T_LOG, int R_LOG, bool TRACE>
struct TileCT {
    static constexpr int RR = 1 << R_LOG;
    static constexpr uint32_t T = 1u << T_LOG;
    static constexpr uint32_t TPAD = T + (T >> 4);
    using P = typename R::P;

    // Layout in which contiguous tiles meet memory when their stages leave the
    // choice: 64 lanes on consecutive records, a wavefront on its own ones.
    static constexpr int A_IO = T_LOG - R_LOG < 6 ? T_LOG - R_LOG : 6;

    // Layout for stage q: as many of the stages below it as the registers hold,
    // but none below the last one wanted.
    static constexpr int layout_for(int q, int qlo)
    {
        const int a = q - R_LOG + 1 > qlo ? q - R_LOG + 1 : qlo;
        return a < T_LOG - R_LOG ? a : T_LOG - R_LOG;
    }
    // Stages on bits below layouts 1 and 2 run between lanes (LANES) and keep
    // the layout.
    static constexpr bool lane_stage(int q, int a) { return LANES && a <= 2 && q < a; }

    // layout reached after stages (q_start .. qlo) starting from layout a
    static constexpr int end_layout(int q, int a, int qlo = 0)
    {
        while (q >= qlo) {
            if (lane_stage(q, a)) break;
            if (!(a <= q && q < a + R_LOG)) a = layout_for(q, qlo);
            q = (a > qlo ? a : qlo) - 1;
        }
        return a;
    }

    // Stage Q (0 or 1) of level P in layouts 1 and 2: record index bit Q is
    // thread index bit Q, so the pair of register m is register m of two lanes
    // of a quad.  Issue-bound, so it is kept to six VALU instructions a record:
    // the borrow chain of lt_masks reads the partner's words through a DPP quad
    // permutation, and the words move by DPP moves under the execution mask of
    // the swapping pairs.  (Written with selects it compiled to 64-bit compares
    // per record and took 10 us of a 2^23-record pass, as long as the other
    // twelve stages and the three relayouts together.)
    // Built for the 12-byte record, the only one whose layouts need it.
    static constexpr bool LANES = R::TIE && R::KW == 1 && sizeof(P) == 4;

    // Exchanges the records of the lane pairs that are out of order: ascending
    // pairs where the upper lane's record is the smaller one, descending pairs
    // (both lanes set in descm) where it is not (equal records are identical).
    template <int Q>
    static __device__ __forceinline__ void lane_cmpx(R &r, uint64_t descm)
    {
        uint32_t w0 = (uint32_t)r.p, w1 = (uint32_t)r.k[0], w2 = (uint32_t)(r.k[0] >> 32), t;
        uint64_t sw, ex;
        // s_nop: two wait states before a DPP read of a register that a VALU
        // instruction wrote, and before each read of the borrow (see
        // lt_masks); %6 holds the lower lane of every pair
#define VO_LANE_CMPX(PERM, SHIFT, LOWER)                                                                               \
    asm("s_nop 1\n\t"                                                                                                  \
        "v_sub_co_u32_dpp %3, vcc, %0, %0 quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"                            \
        "s_nop 1\n\t"                                                                                                 \
        "v_subb_co_u32_dpp %3, vcc, %1, %1, vcc quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"                      \
        "s_nop 1\n\t"                                                                                                 \
        "v_subb_co_u32_dpp %3, vcc, %2, %2, vcc quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"                      \
        "s_and_b64 %4, vcc, %6\n\t"                                                                                    \
        "s_lshl_b64 vcc, %4, " SHIFT "\n\t"                                                                            \
        "s_or_b64 %4, %4, vcc\n\t"                                                                                     \
        "s_xor_b64 %4, %4, %7\n\t"                                                                                     \
        "s_and_saveexec_b64 %5, %4\n\t"                                                                                \
        "v_mov_b32_dpp %0, %0 quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"                                        \
        "v_mov_b32_dpp %1, %1 quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"                                        \
        "v_mov_b32_dpp %2, %2 quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"                                        \
        "s_mov_b64 exec, %5"                                                                                           \
        : "+v"(w0), "+v"(w1), "+v"(w2), "=&v"(t), "=&s"(sw), "=&s"(ex)                                                 \
        : "s"(LOWER), "s"(descm)                                                                                       \
        : "vcc", "scc")
        if constexpr (Q == 0)
            VO_LANE_CMPX("[1,0,3,2]", "1", 0x5555555555555555ull);
        else
            VO_LANE_CMPX("[2,3,0,1]", "2", 0x3333333333333333ull);
#undef VO_LANE_CMPX
        r.p = (P)w0;
        r.k[0] = (uint64_t)w1 | ((uint64_t)w2 << 32);
    }

    template <int P, int A, int Q>
    static __device__ __forceinline__ void lane_stages(R (&r)[RR], uint32_t tau, bool asc_hi, int p_top)
    {
        const uint32_t base = lay_base<R_LOG>(tau, A);
#pragma unroll
        for (int m = 0; m < RR; ++m) {
            bool asc;
            if constexpr (P < 0) {
                asc = asc_hi;
            } else {
                const uint32_t l = base | ((uint32_t)m << A);
                asc = (P >= p_top) | (P >= T_LOG ? asc_hi : (((l >> P) & 1u) == 0));
            }
            lane_cmpx<Q>(r[m], __builtin_amdgcn_ballot_w64(!asc));
        }
        if constexpr (Q > 0) lane_stages<P, A, Q - 1>(r, tau, asc_hi, p_top);
    }

    // LDS of one block: a single buffer that every column passes through in
    // turn.  On 2^14-record tiles the 12-byte records pass in 32-bit words: half
    // the buffer, and 64 VGPRs instead of 72-75, so two 1024-thread blocks share
    // a CU.  On 2^13-record tiles the same gives four blocks a CU instead of two
    // and is faster at 2^23 records (748 -> 699 us) but slower below (one tile a
    // CU at 2^20: 176 -> 184 us, barriers) and above (39.5 -> 40.6 ms at 2^28).
    // Other records keep 8-byte columns (halves cost them registers and moves:
    // two key words 108 -> 133 VGPRs).
    static constexpr bool NARROW = R::TIE && R::KW == 1 && sizeof(P) == 4 && T_LOG >= 14;
    static constexpr size_t lds_bytes() { return (size_t)TPAD * (NARROW ? 4 : 8); }

    template <int A, typename C>
    static __device__ __forceinline__ void put_col(const C (&v)[RR], C *buf, uint32_t tau, uint64_t &h, uint32_t &n)
    {
        const uint32_t lb = lpos(lay_base<R_LOG>(tau, A));
#pragma unroll
        for (int m = 0; m < RR; ++m) {
            const uint32_t l = lb + lpos((uint32_t)m << A);
            buf[l] = v[m];
            if constexpr (TRACE) {
                h = tfold(h, 3, l);
                ++n;
            }
        }
    }

    template <int A, typename C>
    static __device__ __forceinline__ void get_col(C (&v)[RR], const C *buf, uint32_t tau, uint64_t &h, uint32_t &n)
    {
        const uint32_t lb = lpos(lay_base<R_LOG>(tau, A));
#pragma unroll
        for (int m = 0; m < RR; ++m) {
            const uint32_t l = lb + lpos((uint32_t)m << A);
            v[m] = buf[l];
            if constexpr (TRACE) {
                h = tfold(h, 4, l);
                ++n;
            }
        }
    }

    // Layouts up to 6 hold the 64 << R_LOG records of a wavefront in tile order
    // (the thread bits above the lane's are the tile's top bits), so a relayout
    // between two of them stays inside one wavefront: it runs in the
    // wavefront's own part of the buffer without a barrier, and the waves of a
    // block drift apart, one's LDS phase over another's compare-exchanges.
    // (With barriers in all 23 relayouts of the local pass its VALU and LDS
    // times added up.)
    static constexpr bool in_wave(int a_old, int a_new) { return a_old <= 6 && a_new <= 6; }

    // Keeps the LDS accesses before and after in order for the compiler; a
    // wavefront's own are in order in hardware.
    static __device__ __forceinline__ void wave_fence()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    template <int A_OLD, int A_NEW, typename C>
    static __device__ __forceinline__ void move_col(C (&v)[RR], C *buf, uint32_t tau, uint64_t &h, uint32_t &n)
    {
        put_col<A_OLD>(v, buf, tau, h, n);
        if constexpr (in_wave(A_OLD, A_NEW))
            wave_fence();
        else
            __syncthreads();
        get_col<A_NEW>(v, buf, tau, h, n);
    }

    // Before a column enters the buffer: every wave is done with what it read
    // there.  Between relayouts inside the wavefronts each wave only uses its
    // own part, of one column slot a record.
    template <int A_OLD, int A_NEW>
    static __device__ __forceinline__ void relayout(R (&r)[RR], TileBuf &lds, uint32_t tau, uint64_t &h, uint32_t &n)
    {
        if constexpr (A_OLD != A_NEW) {
            constexpr bool IN = in_wave(A_OLD, A_NEW);
            if (lds.shared || A_OLD > 6)
                __syncthreads();
            else
                wave_fence();
            if constexpr (NARROW)
                move_words<A_OLD, A_NEW>(r, lds, tau, h, n);
            else
                move_cols<A_OLD, A_NEW>(r, lds, tau, h, n);
            lds.shared = !IN;
        }
    }

    // between two columns of one relayout
    template <bool IN>
    static __device__ __forceinline__ void next_col()
    {
        if constexpr (IN)
            wave_fence();
        else
            __syncthreads();
    }

    template <int A_OLD, int A_NEW>
    static __device__ __forceinline__ void move_words(R (&r)[RR], TileBuf &lds, uint32_t tau, uint64_t &h, uint32_t &n)
    {
        constexpr bool IN = in_wave(A_OLD, A_NEW);
        constexpr int WORDS = 2 + (int)sizeof(P) / 4;
        uint32_t *buf = reinterpret_cast<uint32_t *>(lds.p);
#pragma unroll
        for (int w = 0; w < WORDS; ++w) {
            uint32_t v[RR];
#pragma unroll
            for (int m = 0; m < RR; ++m) {
                const uint64_t x = w < 2 ? r[m].k[0] : (uint64_t)r[m].p;
                v[m] = (w & 1) ? (uint32_t)(x >> 32) : (uint32_t)x;
            }
            move_col<A_OLD, A_NEW>(v, buf, tau, h, n);
            if (w + 1 < WORDS) next_col<IN>();
#pragma unroll
            for (int m = 0; m < RR; ++m) {
                const uint64_t x = w < 2 ? r[m].k[0] : (uint64_t)r[m].p;
                const uint64_t y = (w & 1) ? (x & 0xFFFFFFFFull) | ((uint64_t)v[m] << 32)
                                           : (x & ~0xFFFFFFFFull) | v[m];
                if (w < 2)
                    r[m].k[0] = y;
                else
                    r[m].p = (P)y;
            }
        }
    }

    template <int A_OLD, int A_NEW>
    static __device__ __forceinline__ void move_cols(R (&r)[RR], TileBuf &lds, uint32_t tau, uint64_t &h, uint32_t &n)
    {
        constexpr bool IN = in_wave(A_OLD, A_NEW);
#pragma unroll
        for (int w = 0; w < R::KW; ++w) {
            uint64_t v[RR];
#pragma unroll
            for (int m = 0; m < RR; ++m) v[m] = r[m].k[w];
            move_col<A_OLD, A_NEW>(v, reinterpret_cast<uint64_t *>(lds.p), tau, h, n);
            next_col<IN>();
#pragma unroll
            for (int m = 0; m < RR; ++m) r[m].k[w] = v[m];
        }
        P v[RR];
#pragma unroll
        for (int m = 0; m < RR; ++m) v[m] = r[m].p;
        P *buf = reinterpret_cast<P *>(lds.p);
        // a narrower column starts where the wavefront's 8-byte part does
        if constexpr (IN && sizeof(P) < 8)
            buf += lpos(__builtin_amdgcn_readfirstlane(tau >> 6) << (6 + R_LOG)) * (8 / sizeof(P) - 1);
        move_col<A_OLD, A_NEW>(v, buf, tau, h, n);
#pragma unroll
        for (int m = 0; m < RR; ++m) r[m].p = v[m];
    }

    // Stages q = QHI .. QLO of level P (P >= 0 compile-time; P < 0 means a
    // level above the tile whose direction `asc_hi` is uniform per block).
    template <int P, int A, int QHI, int QLO>
    static __device__ __forceinline__ void stages(R (&r)[RR], uint32_t tau, bool asc_hi, int p_top)
    {
        const uint32_t base = lay_base<R_LOG>(tau, A);
#pragma unroll
        for (int q = QHI; q >= QLO; --q) {
            cmpx_stage(r, q - A, [&](int m) -> bool {
                if constexpr (P < 0) {
                    return asc_hi;
                } else {
                    const uint32_t l = base | ((uint32_t)m << A);
                    return (P >= p_top) | (P >= T_LOG ? asc_hi : (((l >> P) & 1u) == 0));
                }
            });
        }
    }

    // Stages (P, Q .. QLO) from layout A, changing layout as needed.
    template <int P, int Q, int A, int QLO = 0>
    static __device__ __forceinline__ void level(R (&r)[RR], TileBuf &lds, uint32_t tau, bool asc_hi, int p_top,
                                                 uint64_t &h, uint32_t &n)
    {
        if constexpr (Q >= QLO && lane_stage(Q, A)) {
            lane_stages<P, A, Q>(r, tau, asc_hi, p_top);
        } else if constexpr (Q >= QLO) {
            constexpr bool covered = (A <= Q && Q < A + R_LOG);
            constexpr int AN = covered ? A : layout_for(Q, QLO);
            constexpr int LO = AN > QLO ? AN : QLO;
            relayout<A, AN>(r, lds, tau, h, n);
            stages<P, AN, Q, LO>(r, tau, asc_hi, p_top);
            level<P, LO - 1, AN, QLO>(r, lds, tau, asc_hi, p_top, h, n);
        }
    }

    // Levels P .. T_LOG of a full local sort from layout A; returns through
    // the template chain and leaves the tile in layout end_all(P, A).
    static constexpr int end_all(int p, int a)
    {
        for (; p <= T_LOG; ++p) a = end_layout(p - 1, a);
        return a;
    }

    template <int P, int A>
    static __device__ __forceinline__ void levels(R (&r)[RR], TileBuf &lds, uint32_t tau, bool asc_hi, int p_top,
                                                  uint64_t &h, uint32_t &n)
    {
        if constexpr (P <= T_LOG) {
            level<P, P - 1, A>(r, lds, tau, asc_hi, p_top, h, n);
            levels<P + 1, end_layout(P - 1, A)>(r, lds, tau, asc_hi, p_top, h, n);
        }
    }
};

// A column of a 2^12-row tile on 256 threads between layout 6 (64 lanes on
// consecutive rows: what memory likes) and layout 0 (16 consecutive rows a
// thread: what a scan over rows likes), inside the wavefronts.  lds:
// kRowsLds bytes; a barrier stands between its last use by other waves and the
// first call.
using Rows12 = TileCT<Rec<1, uint64_t, true>, 12, 4, false>;
constexpr uint32_t kRowsLds = Rows12::TPAD * 8;

template <int A_FROM, int A_TO>
__device__ __forceinline__ void wave_rows(uint64_t (&v)[16], char *lds, uint32_t tau)
{
    static_assert(Rows12::in_wave(A_FROM, A_TO), "layouts inside the wavefront");
    uint64_t h = 0;
    uint32_t n = 0;
    Rows12::wave_fence();
    Rows12::move_col<A_FROM, A_TO>(v, reinterpret_cast<uint64_t *>(lds), tau, h, n);
}

} // namespace dev
} // namespace vo
