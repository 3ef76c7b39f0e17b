// C++ operator-level tests of the oblivious path through include/velodb_amd/operators.hpp
// (needs a GPU; tests/test_gpu_cpp_operators.py builds nothing and runs the binary that
// __graft_entry__.build() compiled).
//
// The ORDER BY cases follow the reference's tests/query/test_order_by.cpp (employees table
// :22-45, assertions :97-440); VARCHAR columns are dictionary ordinals in alphabetical order,
// as the device sort sees them.  The expected rows are written out as in the reference test;
// every case is also checked against a host stable sort of the same rows.
#include "velodb_amd/operators.hpp"

#include <dlfcn.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <new>
#include <numeric>
#include <random>
#include <set>
#include <string>
#include <tuple>
#include <vector>

using namespace velodb_amd;

// The CPU oracle (oracle/oracle.h), linked from oracle/_build/liboracle.so:
// the reference's multi-column bitonic sort, ORCompact and the oblivious
// equi-join restated on the host.
extern "C" {
int orc_bitonic_sort_multi(void *const *cols, const uint32_t *types, const uint8_t *asc, size_t ncols,
                           int64_t *indices, size_t n, size_t npad);
void orc_compact(void *buf, size_t elem_size, const uint8_t *selected, size_t n);
size_t orc_join_pairs(const uint64_t *lkey, size_t n_left, const uint64_t *rkey, size_t n_right, int64_t *out_left,
                      int64_t *out_right, size_t cap, int *status);
}

static int g_fail = 0;
#define CHECK(cond)                                                                                                    \
    do {                                                                                                               \
        if (!(cond)) {                                                                                                 \
            std::printf("  CHECK failed: %s (%s:%d)\n", #cond, __FILE__, __LINE__);                                   \
            ++g_fail;                                                                                                  \
        }                                                                                                              \
    } while (0)

// TaskManager::start with the library's message on failure.
#define CHECK_START(tm)                                                                                                \
    do {                                                                                                               \
        if (!(tm).start()) {                                                                                           \
            std::printf("  CHECK failed: start (%s:%d): %s\n", __FILE__, __LINE__, vo_last_error((tm).native()));      \
            ++g_fail;                                                                                                  \
        }                                                                                                              \
    } while (0)

// Host allocations made by the library itself while g_count_allocs is set (the
// library's operator new resolves to the program's).
static bool g_count_allocs = false;
static size_t g_lib_allocs = 0;

__attribute__((noinline)) void *operator new(std::size_t n)
{
    Dl_info at;
    if (g_count_allocs && dladdr(__builtin_return_address(0), &at) && at.dli_fname &&
        std::strstr(at.dli_fname, "libvelodb_amd"))
        ++g_lib_allocs;
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
__attribute__((noinline)) void operator delete(void *p) noexcept { std::free(p); }
__attribute__((noinline)) void operator delete(void *p, std::size_t) noexcept { std::free(p); }

// employees (test_order_by.cpp:35-42)
static const std::vector<int32_t> kId = {3, 1, 5, 2, 4, 6, 7, 8};
static const std::vector<const char *> kName = {"Charlie", "Alice", "Eve", "Bob", "David", "Frank", "Grace", "Helen"};
static const std::vector<double> kSalary = {75000, 50000, 90000, 60000, 75000, 45000, 80000, 55000};
static const std::vector<const char *> kDept = {"Engineering", "Marketing", "Engineering", "Sales",
                                                "Marketing",   "Sales",     "Engineering", "Marketing"};
static const std::vector<int32_t> kAge = {28, 30, 35, 25, 32, 28, 29, 26};
static const std::vector<uint8_t> kActive = {1, 1, 0, 1, 1, 0, 1, 1};

enum { C_ID, C_NAME, C_SALARY, C_DEPT, C_AGE, C_ACTIVE };

// alphabetical dictionary ordinal of a string column
static std::vector<uint64_t> ordinals(const std::vector<const char *> &v)
{
    std::vector<std::string> d(v.begin(), v.end());
    std::sort(d.begin(), d.end());
    d.erase(std::unique(d.begin(), d.end()), d.end());
    std::vector<uint64_t> o;
    for (const char *s : v) o.push_back(std::lower_bound(d.begin(), d.end(), std::string(s)) - d.begin());
    return o;
}

static RowBatch employees(const std::vector<size_t> &rows)
{
    const auto name_o = ordinals(kName), dept_o = ordinals(kDept);
    std::vector<int32_t> id, age;
    std::vector<uint64_t> name, dept;
    std::vector<double> sal;
    std::vector<uint8_t> act;
    for (size_t r : rows) {
        id.push_back(kId[r]);
        name.push_back(name_o[r]);
        sal.push_back(kSalary[r]);
        dept.push_back(dept_o[r]);
        age.push_back(kAge[r]);
        act.push_back(kActive[r]);
    }
    std::vector<Column> c;
    const size_t n = rows.size();
    c.push_back(Column::fromHost(VO_T_INTEGER, id.data(), n));
    c.push_back(Column::fromHost(VO_T_VARCHAR, name.data(), n));
    c.push_back(Column::fromHost(VO_T_DOUBLE, sal.data(), n));
    c.push_back(Column::fromHost(VO_T_VARCHAR, dept.data(), n));
    c.push_back(Column::fromHost(VO_T_INTEGER, age.data(), n));
    c.push_back(Column::fromHost(VO_T_BOOLEAN, act.data(), n));
    return RowBatch(std::move(c), n);
}

static std::vector<size_t> all_rows()
{
    std::vector<size_t> r(kId.size());
    std::iota(r.begin(), r.end(), 0);
    return r;
}

// Runs ORDER BY over the given employee rows; returns the sorted batch.
static RowBatch order_by(ExecutionContext &ctx, const std::vector<size_t> &rows, std::vector<size_t> keys,
                         std::vector<bool> asc)
{
    auto src = std::make_unique<BatchSourceOperator>(ctx, employees(rows));
    SortOperator sort(ctx, std::move(src), std::move(keys), std::move(asc));
    auto res = sort.next();
    if (!res) {
        std::printf("  sort failed: %s\n", res.error().c_str());
        ++g_fail;
        return RowBatch();
    }
    auto end = sort.next(); // the stream ends after the sorted batch
    CHECK(static_cast<bool>(end) && end.value().getRowCount() == 0);
    return std::move(res).value();
}

// host stable sort of the same rows (ties keep input order, as the device
// sort breaks ties by original row index)
static std::vector<int32_t> host_order_ids(const std::vector<size_t> &rows, const std::vector<size_t> &keys,
                                           const std::vector<bool> &asc)
{
    const auto name_o = ordinals(kName), dept_o = ordinals(kDept);
    auto key = [&](size_t r, size_t c) -> double {
        switch (c) {
        case C_ID: return kId[r];
        case C_NAME: return (double)name_o[r];
        case C_SALARY: return kSalary[r];
        case C_DEPT: return (double)dept_o[r];
        case C_AGE: return kAge[r];
        default: return kActive[r];
        }
    };
    std::vector<size_t> o = rows;
    std::stable_sort(o.begin(), o.end(), [&](size_t a, size_t b) {
        for (size_t i = 0; i < keys.size(); ++i) {
            const double x = key(a, keys[i]), y = key(b, keys[i]);
            if (x != y) return asc[i] ? x < y : x > y;
        }
        return false;
    });
    std::vector<int32_t> ids;
    for (size_t r : o) ids.push_back(kId[r]);
    return ids;
}

static void check_against_host(const RowBatch &b, const std::vector<size_t> &rows, const std::vector<size_t> &keys,
                               const std::vector<bool> &asc)
{
    const auto got = b.getColumn(C_ID).toHost<int32_t>(b.getRowCount());
    CHECK(got == host_order_ids(rows, keys, asc));
}

static void test_order_by_integer(ExecutionContext &ctx)
{
    // ORDER BY id / ORDER BY id ASC (test_order_by.cpp:97-134)
    auto b = order_by(ctx, all_rows(), {C_ID}, {true});
    CHECK(b.getRowCount() == 8);
    CHECK((b.getColumn(C_ID).toHost<int32_t>(8) == std::vector<int32_t>{1, 2, 3, 4, 5, 6, 7, 8}));
    // the non-key columns travel with their rows: Alice, Bob, Charlie first
    const auto names = b.getColumn(C_NAME).toHost<uint64_t>(3);
    CHECK((names == std::vector<uint64_t>{0, 1, 2}));
    check_against_host(b, all_rows(), {C_ID}, {true});
}

static void test_order_by_desc(ExecutionContext &ctx)
{
    // ORDER BY id DESC (:136-154)
    auto b = order_by(ctx, all_rows(), {C_ID}, {false});
    CHECK((b.getColumn(C_ID).toHost<int32_t>(8) == std::vector<int32_t>{8, 7, 6, 5, 4, 3, 2, 1}));
    check_against_host(b, all_rows(), {C_ID}, {false});
}

static void test_order_by_string(ExecutionContext &ctx)
{
    // ORDER BY name (:156-174): Alice, Bob, Charlie, David, ...
    auto b = order_by(ctx, all_rows(), {C_NAME}, {true});
    CHECK((b.getColumn(C_ID).toHost<int32_t>(4) == std::vector<int32_t>{1, 2, 3, 4}));
    check_against_host(b, all_rows(), {C_NAME}, {true});
}

static void test_order_by_double(ExecutionContext &ctx)
{
    // ORDER BY salary (:176-194): Frank 45000, Alice 50000, Helen 55000, Bob 60000
    auto b = order_by(ctx, all_rows(), {C_SALARY}, {true});
    CHECK((b.getColumn(C_SALARY).toHost<double>(4) == std::vector<double>{45000, 50000, 55000, 60000}));
    check_against_host(b, all_rows(), {C_SALARY}, {true});
}

static void test_order_by_multiple(ExecutionContext &ctx)
{
    // ORDER BY department, salary (:196-223)
    auto b = order_by(ctx, all_rows(), {C_DEPT, C_SALARY}, {true, true});
    CHECK((b.getColumn(C_DEPT).toHost<uint64_t>(3) == std::vector<uint64_t>{0, 0, 0}));
    CHECK((b.getColumn(C_SALARY).toHost<double>(3) == std::vector<double>{75000, 80000, 90000}));
    check_against_host(b, all_rows(), {C_DEPT, C_SALARY}, {true, true});
}

static void test_order_by_mixed(ExecutionContext &ctx)
{
    // ORDER BY department ASC, salary DESC (:225-250)
    auto b = order_by(ctx, all_rows(), {C_DEPT, C_SALARY}, {true, false});
    CHECK((b.getColumn(C_SALARY).toHost<double>(3) == std::vector<double>{90000, 80000, 75000}));
    check_against_host(b, all_rows(), {C_DEPT, C_SALARY}, {true, false});
}

static void test_order_by_boolean(ExecutionContext &ctx)
{
    // ORDER BY active, name (:252-273): the two inactive rows (Eve, Frank) first
    auto b = order_by(ctx, all_rows(), {C_ACTIVE, C_NAME}, {true, true});
    CHECK((b.getColumn(C_ACTIVE).toHost<uint8_t>(3) == std::vector<uint8_t>{0, 0, 1}));
    CHECK((b.getColumn(C_ID).toHost<int32_t>(2) == std::vector<int32_t>{5, 6}));
    check_against_host(b, all_rows(), {C_ACTIVE, C_NAME}, {true, true});
}

// WHERE <mask> then ORDER BY: the mask column is appended to the batch (the
// scan's "$_mask"), FilterCompactionOperator compacts every column.
static RowBatch where_order_by(ExecutionContext &ctx, const std::function<bool(size_t)> &pred,
                               std::vector<size_t> keys, std::vector<bool> asc)
{
    RowBatch b = employees(all_rows());
    std::vector<uint8_t> mask;
    for (size_t r = 0; r < kId.size(); ++r) mask.push_back(pred(r) ? 1 : 0);
    std::vector<Column> cols;
    for (size_t i = 0; i < b.getColumnCount(); ++i) cols.push_back(std::move(b.getColumn(i)));
    cols.push_back(Column::fromHost(VO_T_BOOLEAN, mask.data(), mask.size()));
    const size_t mask_index = cols.size() - 1;
    auto src = std::make_unique<BatchSourceOperator>(ctx, RowBatch(std::move(cols), kId.size()));
    auto filt = std::make_unique<FilterCompactionOperator>(ctx, std::move(src), mask_index);
    SortOperator sort(ctx, std::move(filt), std::move(keys), std::move(asc));
    auto res = sort.next();
    if (!res) {
        std::printf("  where+sort failed: %s\n", res.error().c_str());
        ++g_fail;
        return RowBatch();
    }
    return std::move(res).value();
}

static void test_where_order_by(ExecutionContext &ctx)
{
    // WHERE department = 'Engineering' ORDER BY salary DESC (:330-347): Eve, Grace, Charlie
    const auto dept_o = ordinals(kDept);
    auto b = where_order_by(ctx, [&](size_t r) { return dept_o[r] == 0; }, {C_SALARY}, {false});
    CHECK(b.getRowCount() == 3);
    CHECK((b.getColumn(C_SALARY).toHost<double>(3) == std::vector<double>{90000, 80000, 75000}));
    CHECK((b.getColumn(C_ID).toHost<int32_t>(3) == std::vector<int32_t>{5, 7, 3}));
    // WHERE salary = 75000.0 ORDER BY name (:387-403): Charlie, David
    auto d = where_order_by(ctx, [&](size_t r) { return kSalary[r] == 75000.0; }, {C_NAME}, {true});
    CHECK(d.getRowCount() == 2);
    CHECK((d.getColumn(C_ID).toHost<int32_t>(2) == std::vector<int32_t>{3, 4}));
    // WHERE salary > 100000.0 (:425-435): no rows
    auto e = where_order_by(ctx, [&](size_t r) { return kSalary[r] > 100000.0; }, {C_SALARY}, {true});
    CHECK(e.getRowCount() == 0);
    // WHERE name = 'Alice' (:437-...): one row
    auto s = where_order_by(ctx, [&](size_t r) { return std::string(kName[r]) == "Alice"; }, {C_SALARY}, {true});
    CHECK(s.getRowCount() == 1);
    CHECK((s.getColumn(C_SALARY).toHost<double>(1) == std::vector<double>{50000}));
}

static void test_nullable_bitmaps_travel(ExecutionContext &ctx)
{
    // a nullable non-key column: its bitmap is permuted with its rows
    const size_t n = 1000;
    std::mt19937_64 rng(7);
    std::vector<int64_t> key(n), val(n);
    std::vector<uint8_t> valid(n);
    for (size_t i = 0; i < n; ++i) {
        key[i] = (int64_t)(rng() % 100000) - 50000;
        val[i] = (int64_t)i;
        valid[i] = (uint8_t)(rng() & 1);
    }
    std::vector<Column> c;
    c.push_back(Column::fromHost(VO_T_BIGINT, key.data(), n));
    c.push_back(Column::fromHost(VO_T_BIGINT, val.data(), n, valid.data()));
    auto src = std::make_unique<BatchSourceOperator>(ctx, RowBatch(std::move(c), n));
    SortOperator sort(ctx, std::move(src), {0}, {true});
    auto res = sort.next();
    CHECK(static_cast<bool>(res));
    if (!res) return;
    RowBatch b = std::move(res).value();
    // keys ascending; each output row carries the value and bitmap byte of
    // one input row with that key (tied keys may come in any order: the
    // multi-column sort, like the reference's, is not stable), and every
    // input row appears once
    std::vector<int64_t> want = key;
    std::sort(want.begin(), want.end());
    const auto gk = b.getColumn(0).toHost<int64_t>(n), gv = b.getColumn(1).toHost<int64_t>(n);
    const auto gb = b.getColumn(1).bitmapToHost(n);
    CHECK(gk == want);
    std::vector<int> seen(n, 0);
    bool ok = true;
    for (size_t i = 0; i < n; ++i) {
        const int64_t j = gv[i];
        ok = ok && j >= 0 && (size_t)j < n && key[j] == gk[i] && valid[j] == gb[i] && ++seen[j] == 1;
    }
    CHECK(ok);
}

static void test_join_groupsum(ExecutionContext &ctx, bool dense)
{
    // dimension (key, group) and fact (fk, value); unmatched fact keys 4, 9, 11
    const std::vector<int32_t> dk = {1, 2, 3, 10}, dg = {0, 1, 0, 7}, fk = {1, 4, 3, 3, 9, 2, 11, 11};
    const std::vector<int64_t> fv = {10, 1000, 5, 7, 1000, 3, 99, 99};
    std::vector<Column> d, f;
    d.push_back(Column::fromHost(VO_T_INTEGER, dk.data(), dk.size()));
    d.push_back(Column::fromHost(VO_T_INTEGER, dg.data(), dg.size()));
    f.push_back(Column::fromHost(VO_T_INTEGER, fk.data(), fk.size()));
    f.push_back(Column::fromHost(VO_T_BIGINT, fv.data(), fv.size()));
    PKFKJoinGroupSumOperator op(ctx, std::make_unique<BatchSourceOperator>(ctx, RowBatch(std::move(d), dk.size())),
                                std::make_unique<BatchSourceOperator>(ctx, RowBatch(std::move(f), fk.size())), 0, 1,
                                0, 1, 8, dense);
    auto res = op.next();
    CHECK(static_cast<bool>(res));
    if (!res) return;
    RowBatch b = std::move(res).value();
    CHECK(b.getRowCount() == 2);
    CHECK((b.getColumn(0).toHost<int32_t>(2) == std::vector<int32_t>{0, 1}));
    CHECK((b.getColumn(1).toHost<int64_t>(2) == std::vector<int64_t>{22, 3}));

    // 50k dimension rows, 200k fact rows, 25 groups against a host group-by
    const size_t nd = 50000, nf = 200000;
    std::mt19937_64 rng(11);
    std::vector<int32_t> k2(nd), g2(nd), f2(nf);
    std::vector<int64_t> v2(nf);
    std::iota(k2.begin(), k2.end(), 1);
    std::shuffle(k2.begin(), k2.end(), rng);
    for (auto &g : g2) g = (int32_t)(rng() % 25);
    std::vector<int64_t> want(25, 0);
    std::vector<int32_t> group_of(nd + 1);
    for (size_t i = 0; i < nd; ++i) group_of[k2[i]] = g2[i];
    for (size_t i = 0; i < nf; ++i) {
        f2[i] = k2[rng() % nd];
        v2[i] = 100 + (int64_t)(rng() % 10000000);
        want[group_of[f2[i]]] += v2[i];
    }
    std::vector<Column> d2, fc2;
    d2.push_back(Column::fromHost(VO_T_INTEGER, k2.data(), nd));
    d2.push_back(Column::fromHost(VO_T_INTEGER, g2.data(), nd));
    fc2.push_back(Column::fromHost(VO_T_INTEGER, f2.data(), nf));
    fc2.push_back(Column::fromHost(VO_T_BIGINT, v2.data(), nf));
    PKFKJoinGroupSumOperator op2(ctx, std::make_unique<BatchSourceOperator>(ctx, RowBatch(std::move(d2), nd)),
                                 std::make_unique<BatchSourceOperator>(ctx, RowBatch(std::move(fc2), nf)), 0, 1, 0, 1,
                                 25, dense);
    auto r2 = op2.next();
    CHECK(static_cast<bool>(r2));
    if (!r2) return;
    RowBatch b2 = std::move(r2).value();
    CHECK(b2.getRowCount() == 25);
    std::vector<int32_t> wg(25);
    std::iota(wg.begin(), wg.end(), 0);
    CHECK(b2.getColumn(0).toHost<int32_t>(25) == wg);
    CHECK(b2.getColumn(1).toHost<int64_t>(25) == want);
}

// two-column INTEGER batch (id, value)
static RowBatch id_value(const std::vector<int32_t> &id, const std::vector<int32_t> &v)
{
    std::vector<Column> c;
    c.push_back(Column::fromHost(VO_T_INTEGER, id.data(), id.size()));
    c.push_back(Column::fromHost(VO_T_INTEGER, v.data(), v.size()));
    return RowBatch(std::move(c), id.size());
}

static void test_sort_merge_join(ExecutionContext &ctx)
{
    // tests/query/test_join_execution.cpp:12-66: A(id 0..4, x = 10 id) JOIN
    // B(id 0..4, y = 100 + id) ON A.id = B.id -> 5 rows, 4 columns
    std::vector<int32_t> id = {0, 1, 2, 3, 4}, x = {0, 10, 20, 30, 40}, y = {100, 101, 102, 103, 104};
    SortMergeJoinOperator j(ctx, std::make_unique<BatchSourceOperator>(ctx, id_value(id, x)),
                            std::make_unique<BatchSourceOperator>(ctx, id_value(id, y)), {0, 0});
    auto r = j.next();
    CHECK(static_cast<bool>(r));
    if (!r) return;
    RowBatch b = std::move(r).value();
    CHECK(b.getRowCount() == 5);
    CHECK(b.getColumnCount() == 4);
    CHECK(b.getColumn(0).toHost<int32_t>(5) == id);
    CHECK(b.getColumn(1).toHost<int32_t>(5) == x);
    CHECK(b.getColumn(2).toHost<int32_t>(5) == id);
    CHECK(b.getColumn(3).toHost<int32_t>(5) == y);
    auto end = j.next();
    CHECK(static_cast<bool>(end) && end.value().getRowCount() == 0);

    // tests/query/test_multi_join.cpp:14-86: A(1,2,3) JOIN B(1,2,4) JOIN C(1,3,5) -> 1 row (id 1)
    auto ab = std::make_unique<SortMergeJoinOperator>(
        ctx, std::make_unique<BatchSourceOperator>(ctx, id_value({1, 2, 3}, {10, 20, 30})),
        std::make_unique<BatchSourceOperator>(ctx, id_value({1, 2, 4}, {100, 200, 400})), std::make_pair(0, 0));
    SortMergeJoinOperator abc(ctx, std::move(ab),
                              std::make_unique<BatchSourceOperator>(ctx, id_value({1, 3, 5}, {1000, 3000, 5000})),
                              {2, 0});
    auto r3 = abc.next();
    CHECK(static_cast<bool>(r3));
    if (!r3) return;
    RowBatch b3 = std::move(r3).value();
    CHECK(b3.getRowCount() == 1);
    CHECK(b3.getColumnCount() == 6);
    std::vector<int32_t> row;
    for (size_t c = 0; c < 6; ++c) row.push_back(b3.getColumn(c).toHost<int32_t>(1)[0]);
    CHECK((row == std::vector<int32_t>{1, 10, 1, 100, 1, 1000}));
    auto e3 = abc.next();
    CHECK(static_cast<bool>(e3) && e3.value().getRowCount() == 0);

    // many-to-many with a nullable payload against host nested loops
    const size_t nl = 3000, nr = 2000;
    std::mt19937_64 rng(5);
    std::vector<int64_t> lk(nl), rk(nr), lv(nl), rv(nr);
    std::vector<uint8_t> lvalid(nl);
    for (size_t i = 0; i < nl; ++i) {
        lk[i] = (int64_t)(rng() % 300) - 150;
        lv[i] = (int64_t)i * 7;
        lvalid[i] = (uint8_t)(rng() & 1);
    }
    for (size_t i = 0; i < nr; ++i) {
        rk[i] = (int64_t)(rng() % 300) - 150;
        rv[i] = -(int64_t)i;
    }
    std::vector<std::tuple<int64_t, size_t, size_t>> want;
    for (size_t i = 0; i < nl; ++i)
        for (size_t k = 0; k < nr; ++k)
            if (lk[i] == rk[k]) want.emplace_back(lk[i], i, k);
    std::sort(want.begin(), want.end());
    std::vector<Column> lc, rc;
    lc.push_back(Column::fromHost(VO_T_BIGINT, lk.data(), nl));
    lc.push_back(Column::fromHost(VO_T_BIGINT, lv.data(), nl, lvalid.data()));
    rc.push_back(Column::fromHost(VO_T_BIGINT, rv.data(), nr));
    rc.push_back(Column::fromHost(VO_T_BIGINT, rk.data(), nr));
    SortMergeJoinOperator mm(ctx, std::make_unique<BatchSourceOperator>(ctx, RowBatch(std::move(lc), nl)),
                             std::make_unique<BatchSourceOperator>(ctx, RowBatch(std::move(rc), nr)), {0, 1});
    auto rm = mm.next();
    CHECK(static_cast<bool>(rm));
    if (!rm) return;
    RowBatch bm = std::move(rm).value();
    const size_t n = want.size();
    CHECK(bm.getRowCount() == n);
    if (bm.getRowCount() != n) return;
    const auto gk = bm.getColumn(0).toHost<int64_t>(n), gv = bm.getColumn(1).toHost<int64_t>(n);
    const auto gb = bm.getColumn(1).bitmapToHost(n);
    const auto grv = bm.getColumn(2).toHost<int64_t>(n), grk = bm.getColumn(3).toHost<int64_t>(n);
    bool ok = true;
    for (size_t i = 0; i < n; ++i) {
        const auto &[k, li, ri] = want[i];
        ok = ok && gk[i] == k && gv[i] == lv[li] && gb[i] == lvalid[li] && grv[i] == rv[ri] && grk[i] == k;
    }
    CHECK(ok);
    // a key index out of bounds is a failure Result, as in the reference
    SortMergeJoinOperator bad(ctx, std::make_unique<BatchSourceOperator>(ctx, id_value({1}, {1})),
                              std::make_unique<BatchSourceOperator>(ctx, id_value({1}, {1})), {5, 0});
    auto rb = bad.next();
    CHECK(!rb);
    if (!rb) CHECK(rb.error() == "Left join key index out of bounds");
}

// ---- children that yield several batches (collectBatches, slicing, prefetch)

struct KV {
    std::vector<int32_t> key;
    std::vector<int64_t> val;
    std::vector<uint8_t> valid;
};

static KV random_kv(size_t n, uint64_t seed, int32_t key_range)
{
    std::mt19937_64 rng(seed);
    KV kv;
    for (size_t i = 0; i < n; ++i) {
        kv.key.push_back((int32_t)(rng() % (uint64_t)key_range) - key_range / 2);
        kv.val.push_back((int64_t)(rng() >> 8) - (int64_t)(1ull << 54));
        kv.valid.push_back((uint8_t)(rng() % 5 != 0));
    }
    return kv;
}

// rows [a, b) of kv as a batch (key INTEGER, value BIGINT nullable)
static RowBatch kv_batch(const KV &kv, size_t a, size_t b)
{
    std::vector<Column> c;
    c.push_back(Column::fromHost(VO_T_INTEGER, kv.key.data() + a, b - a));
    c.push_back(Column::fromHost(VO_T_BIGINT, kv.val.data() + a, b - a, kv.valid.data() + a));
    return RowBatch(std::move(c), b - a);
}

static std::vector<RowBatch> kv_batches(const KV &kv, const std::vector<size_t> &cuts)
{
    std::vector<RowBatch> out;
    for (size_t i = 0; i + 1 < cuts.size(); ++i) out.push_back(kv_batch(kv, cuts[i], cuts[i + 1]));
    return out;
}

static void test_multi_batch_sort(ExecutionContext &ctx)
{
    // three child batches, 9100 rows; output in slices of at most 4000 rows
    const KV kv = random_kv(9100, 21, 600);
    Schema schema({ColumnInfo("k", VO_T_INTEGER), ColumnInfo("v", VO_T_BIGINT)});
    SortOperator op(ctx, schema.clone(), std::make_unique<BatchSourceOperator>(ctx, kv_batches(kv, {0, 3000, 7500, 9100})),
                    {0}, {false});
    op.setMaxBatchSize(4000);
    std::vector<int32_t> gk;
    std::vector<int64_t> gv;
    std::vector<uint8_t> gb;
    std::vector<size_t> sizes;
    for (;;) {
        auto r = op.next();
        CHECK(static_cast<bool>(r));
        if (!r) return;
        RowBatch b = std::move(r).value();
        if (b.getRowCount() == 0) break;
        const size_t n = b.getRowCount();
        sizes.push_back(n);
        const auto k = b.getColumn(0).toHost<int32_t>(n);
        const auto v = b.getColumn(1).toHost<int64_t>(n);
        const auto bits = b.getColumn(1).bitmapToHost(n);
        gk.insert(gk.end(), k.begin(), k.end());
        gv.insert(gv.end(), v.begin(), v.end());
        gb.insert(gb.end(), bits.begin(), bits.end());
    }
    CHECK((sizes == std::vector<size_t>{4000, 4000, 1100}));
    CHECK(op.getOutputSchema().getColumnIndex("v") == 1);
    // the oracle: the reference's network over the gathered rows (padded to 2^14), then permute
    const size_t n = 9100, npad = 16384;
    std::vector<int32_t> key(npad, 0);
    std::copy(kv.key.begin(), kv.key.end(), key.begin());
    std::vector<int64_t> idx(npad);
    void *cols[1] = {key.data()};
    const uint32_t types[1] = {VO_T_INTEGER};
    const uint8_t asc[1] = {0};
    CHECK(orc_bitonic_sort_multi(cols, types, asc, 1, idx.data(), n, npad) == 0);
    bool ok = gk.size() == n;
    for (size_t i = 0; ok && i < n; ++i)
        ok = gk[i] == key[i] && idx[i] < (int64_t)n && gv[i] == kv.val[idx[i]] && gb[i] == kv.valid[idx[i]];
    CHECK(ok);
}

static void test_multi_batch_filter(ExecutionContext &ctx)
{
    // three batches with a "$_mask" column; each compacted on its own while
    // the next is prefetched; the selected rows match ORCompact's prefix
    const std::vector<size_t> cuts = {0, 5000, 5001, 12000};
    const KV kv = random_kv(12000, 22, 1000);
    std::vector<uint8_t> mask(12000);
    std::mt19937_64 rng(23);
    for (auto &m : mask) m = (uint8_t)(rng() % 3 == 0);
    std::vector<RowBatch> batches;
    for (size_t i = 0; i + 1 < cuts.size(); ++i) {
        RowBatch b = kv_batch(kv, cuts[i], cuts[i + 1]);
        std::vector<Column> c;
        c.push_back(std::move(b.getColumn(0)));
        c.push_back(std::move(b.getColumn(1)));
        c.push_back(Column::fromHost(VO_T_BOOLEAN, mask.data() + cuts[i], cuts[i + 1] - cuts[i]));
        batches.emplace_back(std::move(c), cuts[i + 1] - cuts[i]);
    }
    Schema schema({ColumnInfo("t.k", VO_T_INTEGER), ColumnInfo("t.v", VO_T_BIGINT), ColumnInfo("t.$_mask", VO_T_BOOLEAN)});
    FilterCompactionOperator op(ctx, std::move(schema), std::make_unique<BatchSourceOperator>(ctx, std::move(batches)));
    for (size_t i = 0; i + 1 < cuts.size(); ++i) {
        auto r = op.next();
        CHECK(static_cast<bool>(r));
        if (!r) return;
        RowBatch b = std::move(r).value();
        const size_t a = cuts[i], n = cuts[i + 1] - a;
        // the oracle: ORCompact of (key, value, valid) rows of this batch
        struct Row {
            int32_t k;
            uint8_t valid, pad[3];
            int64_t v;
        };
        std::vector<Row> rows(n);
        for (size_t j = 0; j < n; ++j) rows[j] = Row{kv.key[a + j], kv.valid[a + j], {0, 0, 0}, kv.val[a + j]};
        orc_compact(rows.data(), sizeof(Row), mask.data() + a, n);
        size_t m = 0;
        for (size_t j = 0; j < n; ++j) m += mask[a + j] != 0;
        CHECK(b.getRowCount() == m);
        if (b.getRowCount() != m) return;
        const auto k = b.getColumn(0).toHost<int32_t>(m);
        const auto v = b.getColumn(1).toHost<int64_t>(m);
        const auto bits = b.getColumn(1).bitmapToHost(m);
        bool ok = true;
        for (size_t j = 0; j < m; ++j) ok = ok && k[j] == rows[j].k && v[j] == rows[j].v && bits[j] == rows[j].valid;
        CHECK(ok);
    }
    auto end = op.next();
    CHECK(static_cast<bool>(end) && end.value().getRowCount() == 0);
    // the reference's form needs a "$_mask" column in the schema
    bool threw = false;
    try {
        FilterCompactionOperator bad(ctx, Schema({ColumnInfo("k", VO_T_INTEGER)}),
                                     std::make_unique<BatchSourceOperator>(ctx, RowBatch()));
    } catch (const ExecutionError &) {
        threw = true;
    }
    CHECK(threw);
}

static void test_multi_batch_sort_merge_join(ExecutionContext &ctx)
{
    // left in two batches, right in three; the pairs match the oracle's join
    const KV l = random_kv(3000, 24, 400), r = random_kv(4000, 25, 400);
    Schema schema({ColumnInfo("l.k", VO_T_INTEGER), ColumnInfo("l.v", VO_T_BIGINT), ColumnInfo("r.k", VO_T_INTEGER),
                   ColumnInfo("r.v", VO_T_BIGINT)});
    SortMergeJoinOperator op(ctx, std::move(schema),
                             std::make_unique<BatchSourceOperator>(ctx, kv_batches(l, {0, 1700, 3000})),
                             std::make_unique<BatchSourceOperator>(ctx, kv_batches(r, {0, 100, 2600, 4000})), {0, 0},
                             {}, {}, JoinType::INNER);
    auto res = op.next();
    CHECK(static_cast<bool>(res));
    if (!res) return;
    RowBatch b = std::move(res).value();
    // oracle key codes: INTEGER keys sign-extended, sign bit flipped
    auto code = [](int32_t k) { return (uint64_t)(int64_t)k ^ (1ull << 63); };
    std::vector<uint64_t> lc, rc;
    for (int32_t k : l.key) lc.push_back(code(k));
    for (int32_t k : r.key) rc.push_back(code(k));
    int status = 0;
    std::vector<int64_t> ol(1), orr(1);
    const size_t n_out = orc_join_pairs(lc.data(), lc.size(), rc.data(), rc.size(), ol.data(), orr.data(), 0, &status);
    ol.resize(n_out);
    orr.resize(n_out);
    CHECK(orc_join_pairs(lc.data(), lc.size(), rc.data(), rc.size(), ol.data(), orr.data(), n_out, &status) == n_out);
    CHECK(status == 0);
    CHECK(b.getRowCount() == n_out);
    if (b.getRowCount() != n_out) return;
    const auto glk = b.getColumn(0).toHost<int32_t>(n_out), grk = b.getColumn(2).toHost<int32_t>(n_out);
    const auto glv = b.getColumn(1).toHost<int64_t>(n_out), grv = b.getColumn(3).toHost<int64_t>(n_out);
    const auto glb = b.getColumn(1).bitmapToHost(n_out), grb = b.getColumn(3).bitmapToHost(n_out);
    bool ok = true;
    for (size_t i = 0; ok && i < n_out; ++i)
        ok = glk[i] == l.key[ol[i]] && glv[i] == l.val[ol[i]] && glb[i] == l.valid[ol[i]] && grk[i] == r.key[orr[i]] &&
             grv[i] == r.val[orr[i]] && grb[i] == r.valid[orr[i]];
    CHECK(ok);
    auto end = op.next();
    CHECK(static_cast<bool>(end) && end.value().getRowCount() == 0);
}

// Plan nodes build the same operators as the direct calls above: the
// single-table WHERE + ORDER BY wiring, the planner's sort-merge join (sort
// each side on its key, then join), a materialization and a PK/FK GROUP BY
// plan; a plan runs again from a second createOperator; a node with the wrong
// number of children throws, as the reference's assertion does.
static std::vector<std::vector<int64_t>> rows_of(const RowBatch &b)
{
    std::vector<std::vector<int64_t>> out(b.getRowCount());
    for (size_t c = 0; c < b.getColumnCount(); ++c) {
        const Column &col = b.getColumn(c);
        std::vector<int64_t> v(b.getRowCount());
        if (col.getTypeId() == VO_T_BIGINT) {
            v = col.toHost<int64_t>(b.getRowCount());
        } else {
            const auto w = col.toHost<int32_t>(b.getRowCount());
            std::copy(w.begin(), w.end(), v.begin());
        }
        for (size_t r = 0; r < v.size(); ++r) out[r].push_back(v[r]);
    }
    return out;
}

static RowBatch run_plan(ExecutionContext &ctx, const AbstractPlanNode &plan)
{
    auto op = plan.createOperator(ctx);
    auto r = op->next();
    if (!r) {
        std::printf("  plan failed: %s\n", r.error().c_str());
        ++g_fail;
        return RowBatch();
    }
    return std::move(r).value();
}

static void test_plan_nodes(ExecutionContext &ctx)
{
    static_assert(static_cast<uint16_t>(PlanType::SORT_MERGE_JOIN) == 0x38 &&
                      static_cast<uint16_t>(PlanType::SORT) == 0x80 &&
                      static_cast<uint16_t>(PlanType::COMPACTION) == 0x02,
                  "reference PlanType values");
    // WHERE department = 'Engineering' ORDER BY salary DESC, as a plan
    const auto dept_o = ordinals(kDept);
    auto scan = std::make_unique<ScanPlanNode>(
        [&] {
            RowBatch b = employees(all_rows());
            std::vector<uint8_t> mask;
            for (size_t r = 0; r < kId.size(); ++r) mask.push_back(dept_o[r] == 0 ? 1 : 0);
            std::vector<Column> cols;
            for (size_t i = 0; i < b.getColumnCount(); ++i) cols.push_back(std::move(b.getColumn(i)));
            cols.push_back(Column::fromHost(VO_T_BOOLEAN, mask.data(), mask.size()));
            return RowBatch(std::move(cols), kId.size());
        },
        "employees");
    auto q = planFilterOrderBy(std::move(scan), 6, {C_SALARY}, {false});
    CHECK(q->getPlanType() == PlanType::SORT);
    CHECK(q->toString() == "Sort(#2 DESC)");
    CHECK(q->getChildren().size() == 1 && q->getChildren()[0]->toString() == "FilterCompaction(mask #6)");
    for (int run = 0; run < 2; ++run) { // the same plan twice
        RowBatch b = run_plan(ctx, *q);
        CHECK(b.getRowCount() == 3);
        if (b.getRowCount() == 3) CHECK((b.getColumn(C_ID).toHost<int32_t>(3) == std::vector<int32_t>{5, 7, 3}));
    }

    // the same WHERE as a predicate evaluated on the device (no mask column):
    // department = 'Engineering' AND salary >= 76000.0 -> Eve, Grace
    auto pf = std::make_unique<FilterCompactionPlanNode>(
        std::vector<PredicateTerm>{PredicateTerm::make<uint64_t>(C_DEPT, ComparisonType::EQUAL, 0),
                                   PredicateTerm::make<double>(C_SALARY, ComparisonType::GREATER_THAN_OR_EQUAL,
                                                               76000.0)});
    CHECK(pf->toString() == "FilterCompaction(#3 = c AND #2 >= c)");
    pf->addChild(std::make_unique<ScanPlanNode>([] { return employees(all_rows()); }));
    auto ps = std::make_unique<SortPlanNode>(std::vector<size_t>{C_SALARY}, std::vector<bool>{false});
    ps->addChild(std::move(pf));
    RowBatch pb = run_plan(ctx, *ps);
    CHECK(pb.getRowCount() == 2);
    if (pb.getRowCount() == 2) CHECK((pb.getColumn(C_ID).toHost<int32_t>(2) == std::vector<int32_t>{5, 7}));
    // OR of two terms over a nullable column: a NULL row is never selected
    {
        std::vector<int32_t> v = {5, 50, 7, 70}, w = {1, 1, 0, 0};
        std::vector<uint8_t> vvalid = {1, 0, 1, 1};
        std::vector<Column> c;
        c.push_back(Column::fromHost(VO_T_INTEGER, v.data(), 4, vvalid.data()));
        c.push_back(Column::fromHost(VO_T_INTEGER, w.data(), 4));
        FilterCompactionOperator f(ctx, std::make_unique<BatchSourceOperator>(ctx, RowBatch(std::move(c), 4)),
                                   std::vector<PredicateTerm>{PredicateTerm::make<int32_t>(0, ComparisonType::GREATER_THAN, 60),
                                                              PredicateTerm::make<int32_t>(1, ComparisonType::EQUAL, 1)},
                                   ConnectiveType::OR);
        auto r = f.next();
        CHECK(static_cast<bool>(r));
        if (r) {
            RowBatch b = std::move(r).value();
            // row 0 (5 > 60 OR 1 = 1), row 1 NULL, row 2 neither, row 3 (70 > 60)
            CHECK(b.getRowCount() == 2);
            if (b.getRowCount() == 2) CHECK((b.getColumn(0).toHost<int32_t>(2) == std::vector<int32_t>{5, 70}));
        }
    }

    // sort-merge join of unsorted inputs through the planner's wiring
    // (tests/query/test_join_execution.cpp:12-66 data, rows shuffled)
    const std::vector<int32_t> lid = {3, 0, 4, 1, 2}, rid = {2, 4, 0, 3, 1};
    std::vector<int32_t> lx, ry;
    for (int32_t i : lid) lx.push_back(10 * i);
    for (int32_t i : rid) ry.push_back(100 + i);
    for (bool obl : {false, true}) {
        auto j = planSortMergeJoin(std::make_unique<ScanPlanNode>([&] { return id_value(lid, lx); }, "A"),
                                   std::make_unique<ScanPlanNode>([&] { return id_value(rid, ry); }, "B"), {0, 0},
                                   obl);
        CHECK(j->getPlanType() == PlanType::SORT_MERGE_JOIN && j->toString() == "SortMergeJoin(#0 = #0)");
        CHECK(j->getChildren().size() == 2 && j->getChildren()[0]->toString() == "Sort(#0 ASC)");
        RowBatch b = run_plan(ctx, *j);
        std::vector<std::vector<int64_t>> want;
        for (int64_t i = 0; i < 5; ++i) want.push_back({i, 10 * i, i, 100 + i});
        CHECK(b.getRowCount() == 5 && rows_of(b) == want);
    }

    // materialization of row ids through a plan
    std::vector<int64_t> val = {7, 8, 9, 10};
    std::vector<Column> sc;
    sc.push_back(Column::fromHost(VO_T_BIGINT, val.data(), val.size()));
    RowBatch source(std::move(sc), val.size());
    std::vector<int64_t> ids = {3, 0, 0, 2};
    MaterializationPlanNode mp({{0, &source, 0}});
    mp.addChild(std::make_unique<ScanPlanNode>([&] {
        std::vector<Column> c;
        c.push_back(Column::fromHost(VO_T_BIGINT, ids.data(), ids.size()));
        return RowBatch(std::move(c), ids.size());
    }));
    RowBatch mb = run_plan(ctx, mp);
    CHECK(mb.getRowCount() == 4 && (mb.getColumn(0).toHost<int64_t>(4) == std::vector<int64_t>{10, 7, 7, 9}));

    // PK/FK join + GROUP BY as a plan (same data as test_join_groupsum)
    const std::vector<int32_t> dk = {1, 2, 3, 10}, dg = {0, 1, 0, 7}, fk = {1, 4, 3, 3, 9, 2, 11, 11};
    const std::vector<int64_t> fv = {10, 1000, 5, 7, 1000, 3, 99, 99};
    PKFKJoinGroupSumPlanNode gp(0, 1, 0, 1, 8, true);
    gp.addChild(std::make_unique<ScanPlanNode>([&] {
        std::vector<Column> d;
        d.push_back(Column::fromHost(VO_T_INTEGER, dk.data(), dk.size()));
        d.push_back(Column::fromHost(VO_T_INTEGER, dg.data(), dg.size()));
        return RowBatch(std::move(d), dk.size());
    }));
    gp.addChild(std::make_unique<ScanPlanNode>([&] {
        std::vector<Column> f;
        f.push_back(Column::fromHost(VO_T_INTEGER, fk.data(), fk.size()));
        f.push_back(Column::fromHost(VO_T_BIGINT, fv.data(), fv.size()));
        return RowBatch(std::move(f), fk.size());
    }));
    RowBatch gb = run_plan(ctx, gp);
    CHECK(gb.getRowCount() == 2 && (rows_of(gb) == std::vector<std::vector<int64_t>>{{0, 22}, {1, 3}}));

    // a join node with one child
    SortMergeJoinPlanNode lone({0, 0});
    lone.addChild(std::make_unique<ScanPlanNode>([&] { return id_value({1}, {1}); }));
    bool threw = false;
    try {
        (void)lone.createOperator(ctx);
    } catch (const ExecutionError &e) {
        threw = std::string(e.what()) == "SortMergeJoinPlanNode must have exactly 2 children";
    }
    CHECK(threw);
}

// tests/data/test_oblivious_table.cpp: a 1000-row table (id INTEGER, value BIGINT)
static RowBatch thousand_rows()
{
    std::vector<int32_t> id(1000);
    std::vector<int64_t> v(1000);
    for (int i = 0; i < 1000; ++i) {
        id[i] = i;
        v[i] = (int64_t)i * 100;
    }
    std::vector<Column> c;
    c.push_back(Column::fromHost(VO_T_INTEGER, id.data(), 1000));
    c.push_back(Column::fromHost(VO_T_BIGINT, v.data(), 1000));
    return RowBatch(std::move(c), 1000);
}

static bool is_permutation_of_rows(const ObliviousTable &t)
{
    std::set<uint32_t> pos;
    for (size_t i = 0; i < t.getRowCount(); ++i) {
        const uint32_t p = t.getPosition((uint32_t)i);
        if (p >= t.getRowCount()) return false;
        pos.insert(p);
    }
    return pos.size() == t.getRowCount();
}

static void test_oblivious_table(TaskManager &tm)
{
    RowBatch src = thousand_rows();
    // BasicCreation (:32-51)
    ObliviousTable ot("test_table", &src, tm, 1);
    CHECK(ot.getName() == "test_table");
    CHECK(ot.getRowCount() == 1000);
    CHECK(ot.getSourceTable() == &src);
    CHECK(is_permutation_of_rows(ot));
    // the initial shuffle moved most records
    size_t moved0 = 0;
    for (uint32_t i = 0; i < 1000; ++i) moved0 += ot.getPosition(i) != i;
    CHECK(moved0 > 900);
    // ShuffleChangesPositionMap (:54-84)
    std::vector<uint32_t> before(1000);
    for (uint32_t i = 0; i < 1000; ++i) before[i] = ot.getPosition(i);
    ot.startAsyncShuffle();
    CHECK(ot.isShuffling());
    CHECK(ot.getPosition(0) == before[0]); // the active map is unchanged until the wait
    ot.waitForShuffle();
    CHECK(!ot.isShuffling());
    size_t changed = 0;
    for (uint32_t i = 0; i < 1000; ++i) changed += ot.getPosition(i) != before[i];
    CHECK(changed > 900);
    CHECK(is_permutation_of_rows(ot));
    // MultipleShuffles (:150-170)
    ObliviousTable ot2("t2", &src, tm, 2);
    for (int round = 0; round < 5; ++round) {
        ot2.startAsyncShuffle();
        ot2.waitForShuffle();
        CHECK(is_permutation_of_rows(ot2));
    }
    CHECK(ot2.getShuffleCount() == 5);
    // a row count that is not a power of two keeps its positions in range
    // (checked above); a one-row table stays put
    std::vector<int32_t> one = {7};
    std::vector<Column> oc;
    oc.push_back(Column::fromHost(VO_T_INTEGER, one.data(), 1));
    RowBatch ob(std::move(oc), 1);
    ObliviousTable ot1("one", &ob, tm, 3);
    ot1.startAsyncShuffle();
    ot1.waitForShuffle();
    CHECK(ot1.getPosition(0) == 0);
}

static void test_oblivious_table_manager(TaskManager &tm)
{
    RowBatch src = thousand_rows();
    ObliviousTableManager mgr(tm);
    mgr.registerTable("test_table", &src, 4);
    // ManagerBasicUsage (:87-98)
    CHECK(mgr.hasTable("test_table"));
    CHECK(!mgr.hasTable("other"));
    CHECK(mgr.getStats().tables_registered == 1);
    // QueryLifecycle (:100-126)
    const uint32_t p0 = mgr.getTable("test_table").getPosition(0);
    mgr.beginQuery({"test_table"});
    mgr.markAccessed("test_table");
    mgr.endQuery(); // starts the shuffle
    CHECK(mgr.getTable("test_table").isShuffling());
    mgr.beginQuery({"test_table"}); // waits for it
    CHECK(!mgr.getTable("test_table").isShuffling());
    CHECK(is_permutation_of_rows(mgr.getTable("test_table")));
    (void)p0;
    mgr.endQuery();
    CHECK(mgr.getStats().total_shuffles >= 1);
    // ProfilesControlledShuffleForAccessedTables (:128-148)
    mgr.beginQuery({"test_table"});
    mgr.markAccessed("test_table");
    mgr.endQuery();
    const size_t count = mgr.getTable("test_table").getShuffleCount();
    mgr.profileAccessedTableShuffles();
    CHECK(mgr.getTable("test_table").getShuffleCount() == count + 1);
    CHECK(mgr.controlledShuffleMicros("test_table") > 0);
    // PositionEnrichment (:172-214)
    mgr.beginQuery({"test_table"});
    const size_t n = 100;
    std::vector<uint32_t> ids(n);
    std::iota(ids.begin(), ids.end(), 0u);
    uint32_t *d_ids = nullptr, *d_pos = nullptr;
    hip_check(hipMalloc(reinterpret_cast<void **>(&d_ids), n * 4), "hipMalloc");
    hip_check(hipMalloc(reinterpret_cast<void **>(&d_pos), n * 4), "hipMalloc");
    hip_check(hipMemcpy(d_ids, ids.data(), n * 4, hipMemcpyHostToDevice), "hipMemcpy");
    mgr.enrichPositions("test_table", d_ids, d_pos, n);
    std::vector<uint32_t> pos(n);
    hip_check(hipMemcpy(pos.data(), d_pos, n * 4, hipMemcpyDeviceToHost), "hipMemcpy");
    bool ok = true;
    for (size_t i = 0; i < n; ++i) ok = ok && pos[i] == mgr.getTable("test_table").getPosition((uint32_t)i);
    CHECK(ok);
    (void)hipFree(d_ids);
    (void)hipFree(d_pos);
    mgr.endQuery();
    bool threw = false;
    try {
        mgr.getTable("missing");
    } catch (const std::runtime_error &) {
        threw = true;
    }
    CHECK(threw);
}

// The operators submit every command to the TaskManager, as the reference's
// do; with the resident queue the launch-only ones (OP_SORT, the join, the
// shuffle) run in order between the queue's commands.
static void test_operators_over_resident_queue()
{
    TaskManager tm(64, true);
    CHECK_START(tm);
    ExecutionContext ctx(tm);
    std::vector<int32_t> id = {0, 1, 2, 3, 4}, x = {0, 10, 20, 30, 40}, y = {100, 101, 102, 103, 104};
    SortMergeJoinOperator j(ctx, std::make_unique<BatchSourceOperator>(ctx, id_value(id, x)),
                            std::make_unique<BatchSourceOperator>(ctx, id_value(id, y)), {0, 0});
    auto r = j.next();
    CHECK(static_cast<bool>(r));
    if (r) {
        RowBatch b = std::move(r).value();
        CHECK(b.getRowCount() == 5 && b.getColumnCount() == 4);
        CHECK(b.getColumn(3).toHost<int32_t>(5) == y);
    }
    auto sorted = order_by(ctx, all_rows(), {C_AGE, C_ID}, {false, true});
    CHECK(sorted.getRowCount() == 8);
    CHECK((sorted.getColumn(C_ID).toHost<int32_t>(8) == std::vector<int32_t>{5, 4, 1, 7, 3, 6, 8, 2}));
    test_oblivious_table_manager(tm);
    CHECK(tm.stop());
}

static void test_padded_transfers(TaskManager &tm)
{
    // columns through the padded staged transfer: the values round-trip, the
    // pad rows arrive as zeros, and the sort sees the same data
    const size_t n = 100000;
    std::vector<int64_t> v(n);
    std::mt19937_64 rng(9);
    for (auto &x : v) x = (int64_t)(rng() >> 1) - (1ll << 61);
    Column c = Column::fromHost(tm, VO_T_BIGINT, v.data(), n);
    CHECK(c.capacity() == 131072);
    CHECK(c.toHost<int64_t>(tm, n) == v);
    const auto all = c.toHost<int64_t>(tm, c.capacity());
    bool zeros = true;
    for (size_t i = n; i < all.size(); ++i) zeros = zeros && all[i] == 0;
    CHECK(zeros);
}

static void test_materialization(ExecutionContext &ctx)
{
    // MaterializationOperator: a source table (value BIGINT nullable, tag
    // INTEGER) and row ids with repeats and one id outside the table
    const size_t nt = 5000, n = 20000;
    std::mt19937_64 rng(21);
    std::vector<int64_t> val(nt);
    std::vector<int32_t> tag(nt);
    std::vector<uint8_t> valid(nt);
    for (size_t i = 0; i < nt; ++i) {
        val[i] = (int64_t)(rng() >> 2);
        tag[i] = (int32_t)(rng() % 1000);
        valid[i] = (uint8_t)(rng() % 4 != 0);
    }
    std::vector<Column> sc;
    sc.push_back(Column::fromHost(VO_T_BIGINT, val.data(), nt, valid.data()));
    sc.push_back(Column::fromHost(VO_T_INTEGER, tag.data(), nt));
    RowBatch source(std::move(sc), nt);
    std::vector<int64_t> ids(n);
    for (auto &x : ids) x = (int64_t)(rng() % nt);
    for (size_t i = 0; i < 3000; ++i) ids[i] = 42;
    ids[n - 1] = (int64_t)nt + 9; // outside the table
    std::vector<Column> ic;
    ic.push_back(Column::fromHost(VO_T_BIGINT, ids.data(), n));
    MaterializationOperator m(ctx, std::make_unique<BatchSourceOperator>(ctx, RowBatch(std::move(ic), n)),
                              {{0, &source, 1}, {0, &source, 0}});
    auto r = m.next();
    CHECK(static_cast<bool>(r));
    if (!r) return;
    RowBatch b = std::move(r).value();
    CHECK(b.getRowCount() == n && b.getColumnCount() == 2);
    const auto gt = b.getColumn(0).toHost<int32_t>(n);
    const auto gv = b.getColumn(1).toHost<int64_t>(n);
    const auto gb = b.getColumn(1).bitmapToHost(n);
    bool ok = true;
    for (size_t i = 0; i + 1 < n; ++i)
        ok = ok && gt[i] == tag[ids[i]] && gv[i] == val[ids[i]] && (gb[i] != 0) == (valid[ids[i]] != 0);
    CHECK(ok);
    CHECK(gt[n - 1] == 0 && gv[n - 1] == 0 && gb[n - 1] == 0);

    // the join with oblivious materialization equals the permute form
    std::vector<int32_t> lk(3000), rk(2000), lv(3000), rv(2000);
    for (size_t i = 0; i < 3000; ++i) {
        lk[i] = (int32_t)(rng() % 500);
        lv[i] = (int32_t)i;
    }
    for (size_t i = 0; i < 2000; ++i) {
        rk[i] = (int32_t)(rng() % 500);
        rv[i] = -(int32_t)i;
    }
    auto join = [&](bool obl) {
        SortMergeJoinOperator j(ctx, std::make_unique<BatchSourceOperator>(ctx, id_value(lk, lv)),
                                std::make_unique<BatchSourceOperator>(ctx, id_value(rk, rv)), {0, 0},
                                JoinType::INNER, obl);
        auto res = j.next();
        CHECK(static_cast<bool>(res));
        std::vector<std::vector<int32_t>> cols;
        if (!res) return cols;
        RowBatch jb = std::move(res).value();
        for (size_t c = 0; c < 4; ++c) cols.push_back(jb.getColumn(c).toHost<int32_t>(jb.getRowCount()));
        return cols;
    };
    const auto a = join(false), o = join(true);
    CHECK(!a.empty() && a == o);
}

static void test_errors_are_results(ExecutionContext &ctx)
{
    // a failure of the library comes back as Result::failure with its message
    std::vector<int32_t> k = {1, 2, 3};
    std::vector<int64_t> v = {1, 2, 3};
    std::vector<Column> d, f;
    d.push_back(Column::fromHost(VO_T_INTEGER, k.data(), 3));
    d.push_back(Column::fromHost(VO_T_INTEGER, k.data(), 3));
    f.push_back(Column::fromHost(VO_T_INTEGER, k.data(), 3));
    f.push_back(Column::fromHost(VO_T_BIGINT, v.data(), 3));
    PKFKJoinGroupSumOperator op(ctx, std::make_unique<BatchSourceOperator>(ctx, RowBatch(std::move(d), 3)),
                                std::make_unique<BatchSourceOperator>(ctx, RowBatch(std::move(f), 3)), 0, 1, 0, 1,
                                100, true); // dense GROUP BY takes at most 64 groups
    auto r = op.next();
    CHECK(!r);
    if (!r) CHECK(r.error().find("max_groups") != std::string::npos);
}

static void test_task_manager_queue(ExecutionContext &)
{
    // TaskManager::start / submitCommand / waitCommand / stop with the resident kernel
    TaskManager tm(64, true);
    CHECK_START(tm);
    CHECK(tm.isRunning());
    const size_t n = 5000, n_pad = 8192;
    std::vector<uint64_t> keys(n);
    std::vector<uint32_t> pay(n);
    std::mt19937_64 rng(3);
    for (size_t i = 0; i < n; ++i) {
        keys[i] = rng();
        pay[i] = (uint32_t)i;
    }
    Column ck = Column::fromHost(VO_T_UBIGINT, keys.data(), n), cp = Column::fromHost(VO_T_INTEGER, pay.data(), n);
    vo_command c{};
    c.opcode = VO_OP_SORT_KP;
    c.args.sort_kp = {static_cast<uint64_t *>(ck.rawData()), static_cast<uint32_t *>(cp.rawData()), n, n_pad};
    tm.waitCommand(tm.submitCommand(c));
    const auto gk = ck.toHost<uint64_t>(n);
    std::vector<uint64_t> want = keys;
    std::sort(want.begin(), want.end());
    CHECK(gk == want);
    CHECK(tm.stop());
    CHECK(!tm.isRunning());
}

// --persistent: the shared TaskManager runs every operator's commands in the
// resident queue kernel (TaskManager::start with persistent = true), as a
// reference caller with a persistent TaskManager would.
// vo_compact_noalloc allocates nothing, on the host either, and compacts every
// column in order of its rows (launch mode: a resident queue would be parked first).
static void test_compact_noalloc_allocates_nothing(TaskManager &tm)
{
    constexpr uint64_t N = 4096;
    const uint32_t widths[VO_MAX_SORT_COLUMNS] = {8, 4, 1, 2, 8, 1, 4, 2};
    char *dev = nullptr;
    CHECK(hipMalloc((void **)&dev, N * 8 * (VO_MAX_SORT_COLUMNS + 1)) == hipSuccess);
    std::vector<uint8_t> mask(N);
    std::vector<uint64_t> want;
    for (uint64_t i = 0; i < N; ++i) {
        mask[i] = i % 3 == 1;
        if (mask[i]) want.push_back(i);
    }
    vo_compact_args a{};
    a.mask = (const uint8_t *)dev;
    a.n = a.n_pad = N;
    a.n_cols = VO_MAX_SORT_COLUMNS;
    CHECK(hipMemcpy(dev, mask.data(), N, hipMemcpyHostToDevice) == hipSuccess);
    for (uint32_t c = 0; c < a.n_cols; ++c) {
        std::vector<char> host(N * 8);
        for (uint64_t i = 0; i < N; ++i) std::memcpy(&host[i * widths[c]], &i, widths[c]);
        a.cols[c] = dev + N * 8 * (c + 1);
        a.col_bytes[c] = widths[c];
        CHECK(hipMemcpy(a.cols[c], host.data(), N * widths[c], hipMemcpyHostToDevice) == hipSuccess);
    }
    g_lib_allocs = 0;
    g_count_allocs = true;
    const int st = vo_compact_noalloc(tm.native(), &a);
    g_count_allocs = false;
    CHECK(st == VO_OK);
    CHECK(vo_sync(tm.native()) == VO_OK);
    CHECK(g_lib_allocs == 0);
    for (uint32_t c = 0; c < a.n_cols; ++c) {
        std::vector<char> host(want.size() * widths[c]);
        CHECK(hipMemcpy(host.data(), a.cols[c], host.size(), hipMemcpyDeviceToHost) == hipSuccess);
        bool same = true;
        for (size_t k = 0; k < want.size(); ++k) same &= !std::memcmp(&host[k * widths[c]], &want[k], widths[c]);
        CHECK(same);
    }
    CHECK(hipFree(dev) == hipSuccess);
}

int main(int argc, char **argv)
{
    const bool persistent = argc > 1 && std::string(argv[1]) == "--persistent";
    TaskManager tm(1024, persistent);
    if (persistent && !tm.start()) {
        std::printf("FAILED: the resident queue did not start: %s\n", vo_last_error(tm.native()));
        return 1;
    }
    std::printf("mode: %s\n", persistent ? "persistent (resident queue)" : "launch");
    ExecutionContext ctx(tm);
    const std::vector<std::pair<const char *, std::function<void()>>> tests = {
        {"order_by_integer", [&] { test_order_by_integer(ctx); }},
        {"order_by_desc", [&] { test_order_by_desc(ctx); }},
        {"order_by_string", [&] { test_order_by_string(ctx); }},
        {"order_by_double", [&] { test_order_by_double(ctx); }},
        {"order_by_multiple", [&] { test_order_by_multiple(ctx); }},
        {"order_by_mixed", [&] { test_order_by_mixed(ctx); }},
        {"order_by_boolean", [&] { test_order_by_boolean(ctx); }},
        {"where_order_by", [&] { test_where_order_by(ctx); }},
        {"nullable_bitmaps_travel", [&] { test_nullable_bitmaps_travel(ctx); }},
        {"join_groupsum_sorted", [&] { test_join_groupsum(ctx, false); }},
        {"sort_merge_join", [&] { test_sort_merge_join(ctx); }},
        {"oblivious_table", [&] { test_oblivious_table(tm); }},
        {"padded_transfers", [&] { test_padded_transfers(tm); }},
        {"materialization", [&] { test_materialization(ctx); }},
        {"oblivious_table_manager", [&] { test_oblivious_table_manager(tm); }},
        {"operators_over_resident_queue", [&] { test_operators_over_resident_queue(); }},
        {"join_groupsum_dense", [&] { test_join_groupsum(ctx, true); }},
        {"errors_are_results", [&] { test_errors_are_results(ctx); }},
        {"task_manager_queue", [&] { test_task_manager_queue(ctx); }},
        {"plan_nodes", [&] { test_plan_nodes(ctx); }},
        {"compact_noalloc_allocates_nothing",
         [&] {
             if (!persistent) test_compact_noalloc_allocates_nothing(tm);
         }},
        {"multi_batch_sort", [&] { test_multi_batch_sort(ctx); }},
        {"multi_batch_filter", [&] { test_multi_batch_filter(ctx); }},
        {"multi_batch_sort_merge_join", [&] { test_multi_batch_sort_merge_join(ctx); }},
    };
    for (const auto &t : tests) {
        const int before = g_fail;
        std::printf("RUN  %s\n", t.first);
        std::fflush(stdout);
        // these two start a resident queue of their own: the shared one is
        // stopped around them, so one resident kernel holds the GPU at a time
        const bool own_queue = std::string(t.first) == "operators_over_resident_queue" ||
                               std::string(t.first) == "task_manager_queue";
        try {
            if (persistent && own_queue) CHECK(tm.stop());
            t.second();
            if (persistent && own_queue) CHECK_START(tm);
        } catch (const std::exception &e) {
            std::printf("  exception: %s\n", e.what());
            ++g_fail;
        }
        std::printf("%s %s\n", g_fail == before ? "PASS" : "FAIL", t.first);
        std::fflush(stdout);
    }
    if (persistent && !tm.stop()) {
        std::printf("  the resident queue did not stop\n");
        ++g_fail;
    }
    std::printf("%s: %d failed checks\n", g_fail ? "FAILED" : "OK", g_fail);
    return g_fail ? 1 : 0;
}
