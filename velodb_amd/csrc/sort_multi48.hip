// sort_multi48.hip -- the sorts of four and eight packed key words used by the
// multi-column OP_SORT (sort_multi.hip).
#include "resident_tables.hpp"
#include "sort_kernels.hpp"

namespace vo {

using namespace sortimpl;

namespace {

const std::pair<const void *, BodyInfo> kBodies[] = {VO_SORT_M48_BODIES(VO_BODY_ENTRY)};
const bool kRegistered = (register_bodies(kBodies, sizeof kBodies / sizeof kBodies[0]), true);

using SortM4 = SortImpl<RecM4, 11, 3, 256, 3, 6>;
using SortM8 = SortImpl<RecM8, 10, 2, 256, 2>;

template <class S, class R>
void sort_words(vo_ctx *ctx, uint64_t *const *words, uint32_t *payload, int n_log)
{
    Bufs<R> b;
    for (int w = 0; w < R::KW; ++w) b.k[w] = words[w];
    b.p = payload;
    S::run(ctx, b, n_log, 1ull << n_log, 0);
}

} // namespace

void sort_words4(vo_ctx *ctx, uint64_t *const *words, uint32_t *payload, int n_log)
{
    sort_words<SortM4, RecM4>(ctx, words, payload, n_log);
}

void sort_words8(vo_ctx *ctx, uint64_t *const *words, uint32_t *payload, int n_log)
{
    sort_words<SortM8, RecM8>(ctx, words, payload, n_log);
}

} // namespace vo
