// sort_kv.hip -- the (u64 key, u64 value) oblivious sort used by the join, the
// shuffle with permutation output and the oblivious gather.
#include "resident_tables.hpp"
#include "sort_kernels.hpp"

namespace vo {

using namespace sortimpl;

namespace {

const std::pair<const void *, BodyInfo> kBodies[] = {VO_SORT_KV_BODIES(VO_BODY_ENTRY)};
const bool kRegistered = (register_bodies(kBodies, sizeof kBodies / sizeof kBodies[0]), true);

// As the 12-byte sort's, its passes change at 2^27 records: at 2^28 its 4-5 stage register passes ran at
// 4.80-4.99 TB/s against 5.11-5.36 for its LDS-staged passes
// (512-thread hybrid passes measured no faster for it: 78.04-78.05 vs 78.06-78.14 ms per
// 2^28-row shuffle with permutation output)
using SortKV = SortImpl<RecKV, 12, 4, 256, 5, 7, 3, 27, 0, 13>;
// Up to 2^20 records, one tile or fewer a CU: 512 threads of 8 records each (as
// in sort_kp.hip); a shuffle of 2^20 rows with its permutation 222 -> 203 us.
using SortKV_S = SortImpl<RecKV, 12, 3, 512, 5, 0, 3, 27, 0, 12, true, false, false>;

} // namespace

void sort_kv(vo_ctx *ctx, uint64_t *keys, uint64_t *vals, uint64_t n_pad)
{
    Bufs<RecKV> b;
    b.k[0] = keys;
    b.p = vals;
    const int n_log = ilog2(n_pad);
    if (n_log <= 20 && SortKV_S::wrapped(ctx))
        SortKV_S::run(ctx, b, n_log, n_pad, 0);
    else
        SortKV::run(ctx, b, n_log, n_pad, 0);
}

} // namespace vo
