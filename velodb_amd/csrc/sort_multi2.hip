// sort_multi2.hip -- the sort of two packed key words used by the multi-column
// OP_SORT (sort_multi.hip).
#include "resident_tables.hpp"
#include "sort_kernels.hpp"

namespace vo {

using namespace sortimpl;

namespace {

const std::pair<const void *, BodyInfo> kBodies[] = {VO_SORT_M2_BODIES(VO_BODY_ENTRY)};
const bool kRegistered = (register_bodies(kBodies, sizeof kBodies / sizeof kBodies[0]), true);

// register passes and tiles as for one key word (sort_multi.hip)
using SortM2 = SortImpl<RecM2, 12, 4, 256, 3, 7, 3, 64, 0, 13>;
// (as there; two key words, 2^20 rows: 289 -> 247 us)
using SortM2_S = SortImpl<RecM2, 12, 3, 512, 3, 0, 3, 64, 0, 12, true, false, false>;

} // namespace

void sort_words2(vo_ctx *ctx, uint64_t *const *words, uint32_t *payload, int n_log)
{
    Bufs<RecM2> b;
    for (int w = 0; w < 2; ++w) b.k[w] = words[w];
    b.p = payload;
    if (n_log <= 20 && SortM2_S::wrapped(ctx))
        SortM2_S::run(ctx, b, n_log, 1ull << n_log, 0);
    else
        SortM2::run(ctx, b, n_log, 1ull << n_log, 0);
}

} // namespace vo
