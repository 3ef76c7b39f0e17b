"""Measured cases of the oblivious operators, through the package's public calls.

Each listed case is one operator call (or the short chain of calls that one
query operator makes) on columns resident in HBM, at a size a user runs:
point-query sorts, ordinary analytics tables and the largest tables.  Sizes
are the workloads of bench.py and of the tests, most of them ragged (rows
padded to a power of two).  `draw` gives further sizes, types and
selectivities of the same ranges.
"""
import math

import torch

import velodb_amd
from velodb_amd import _abi

_M63 = -(1 << 63)
_ctx = None


def _context():
    """The process's one library context, on torch's current stream."""
    global _ctx
    if _ctx is None:
        _ctx = velodb_amd.Context(stream=torch.cuda.current_stream().cuda_stream)
    return _ctx


def _pow2(n, least=1):
    p = least
    while p < n:
        p *= 2
    return p


def listed():
    return [
        # a point query's result sorted before it is returned: launch latency
        {"name": "sort_3k", "op": "sort", "n": 3000, "wait": True},
        # the plain sort of an ordinary table
        {"name": "sort_1m", "op": "sort", "n": 1 << 20, "wait": True},
        # the headline: the largest table
        {"name": "sort_2p28", "op": "sort", "n": 1 << 28, "wait": False},
        # ORDER BY of two keys with two payload columns (SortOperator)
        {"name": "order_by_12m", "op": "order_by", "n": 12_000_000, "second": "double"},
        # WHERE of three terms, then compaction of columns of mixed widths (FilterCompactionOperator)
        {"name": "where_10m", "op": "where", "n": 10_000_000, "keep": 0.25},
        # Q6-style filter + SUM over a scale-factor-1 fact table
        {"name": "filter_6m", "op": "filter", "n": 6_000_000},
        # the same over a scale-factor-50 fact table
        {"name": "filter_300m", "op": "filter", "n": 300_000_000},
        # PK/FK join + GROUP BY over 25 known group ids
        {"name": "join_dense_7m", "op": "join", "n_dim": 1_500_000, "n_fact": 6_000_000, "groups": 25, "dense": True},
        # the same with the sort-based GROUP BY on smaller tables
        {"name": "join_sorted_1m", "op": "join", "n_dim": 150_000, "n_fact": 800_000, "groups": 50, "dense": False},
        # equi-join into row pairs, COUNT then WRITE (SortMergeJoinOperator)
        {"name": "join_pairs_7m", "op": "pairs", "n_left": 1_500_000, "n_right": 6_000_000, "distinct": 1_500_000,
         "wide": False},
        # oblivious materialization of one BIGINT column
        {"name": "gather_8m", "op": "gather", "n_table": 1 << 22, "n": 1 << 23, "bytes": 8},
        # thousands of uneven sorts in one call
        {"name": "batch_4096", "op": "batch", "items": 4096, "lo": 10, "hi": 20, "sizes_seed": 0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["sort", "sort", "order_by", "where", "filter", "join", "pairs", "gather", "batch"])
    if op == "sort":
        n = _log(rng, 20, 100_000_000)
        return {"op": op, "n": n, "wait": rng.random() < 0.5}
    if op == "order_by":
        return {"op": op, "n": _log(rng, 200, 12_000_000), "second": rng.choice(["double", "bigint"])}
    if op == "where":
        return {"op": op, "n": _log(rng, 200, 30_000_000), "keep": round(rng.uniform(0.01, 0.9), 3)}
    if op == "filter":
        return {"op": op, "n": _log(rng, 500, 100_000_000)}
    if op == "join":
        nd = _log(rng, 100, 1_500_000)
        dense = rng.random() < 0.5
        return {"op": op, "n_dim": nd, "n_fact": int(nd * rng.uniform(1, 5)), "groups": rng.randint(2, 60),
                "dense": dense}
    if op == "pairs":
        nl = _log(rng, 100, 1_500_000)
        return {"op": op, "n_left": nl, "n_right": int(nl * rng.uniform(0.5, 4)),
                "distinct": max(1, int(nl * rng.uniform(0.5, 1.5))), "wide": rng.random() < 0.5}
    if op == "gather":
        n = _log(rng, 500, 1 << 23)
        return {"op": op, "n_table": max(1, int(n * rng.uniform(0.1, 1.0))), "n": n, "bytes": rng.choice([4, 8])}
    lo = rng.randint(6, 12)
    return {"op": "batch", "items": _log(rng, 8, 1024), "lo": lo, "hi": lo + rng.randint(2, 6),
            "sizes_seed": rng.randint(1, 1 << 20)}


# ------------------------------------------------------------------ inputs


def _gen(seed):
    return torch.Generator(device="cuda:0").manual_seed(int(seed) * 1_000_003 + 17)


def _ints(g, n, lo, hi, dtype=torch.int64, size=None):
    """n values of [lo, hi), in a buffer of `size` elements (the rest 0)."""
    v = torch.randint(lo, hi, (n,), device="cuda:0", generator=g, dtype=dtype)
    if size is None or size == n:
        return v
    b = torch.zeros(size, device="cuda:0", dtype=dtype)
    b[:n] = v
    return b


def _batch_items(case):
    """[(offset, rows, padded rows)]: sizes log-uniform in [2^lo, 2^hi], each at a multiple of its padded size."""
    g = torch.Generator().manual_seed(case["sizes_seed"])
    u = torch.rand(case["items"], generator=g, dtype=torch.float64).tolist()
    items, off = [], 0
    for x in u:
        n = max(1, int(2.0 ** (case["lo"] + x * (case["hi"] - case["lo"]))))
        p = _pow2(n)
        off = (off + p - 1) // p * p
        items.append((off, n, p))
        off += p
    return items, off


def _sort_columns(g, n, size):
    return _ints(g, n, _M63, (1 << 63) - 1, size=size), torch.arange(size, device="cuda:0", dtype=torch.int32)


def _inputs(case, seed):
    """The input columns alone, from the seed."""
    g, op = _gen(seed), case["op"]
    s = {}
    if op == "sort":
        s["n"], s["n_pad"] = case["n"], _pow2(case["n"])
        s["keys"], s["payload"] = _sort_columns(g, s["n"], s["n_pad"])
    elif op == "order_by":
        n, p = case["n"], _pow2(case["n"])
        s["n"], s["n_pad"] = n, p
        s["a0"] = _ints(g, n, -1000, 1000, torch.int32, p)
        if case["second"] == "double":
            s["b0"] = torch.zeros(p, device="cuda:0", dtype=torch.float64)
            s["b0"][:n] = torch.randn(n, device="cuda:0", generator=g, dtype=torch.float64)
        else:
            s["b0"] = _ints(g, n, -(1 << 62), 1 << 62, size=p)
        s["p1"] = torch.arange(p, device="cuda:0", dtype=torch.int64)
        s["p2"] = _ints(g, p, 0, 1 << 40)
    elif op == "where":
        n, p = case["n"], _pow2(case["n"])
        s["n"], s["n_pad"] = n, p
        s["x"] = _ints(g, n, 0, 1_000_000, torch.int32, p)
        s["y"] = _ints(g, n, 0, 100, torch.int64, p)
        s["c8"] = _ints(g, n, 0, 1 << 50, torch.int64, p)
        s["c4"] = _ints(g, n, 0, 1 << 30, torch.int32, p)
        s["c1"] = _ints(g, n, 0, 2, torch.uint8, p)
        s["hi"] = int(1_000_000 * case["keep"])
    elif op == "filter":
        n, p = case["n"], _pow2(case["n"], 2)
        s["n"], s["n_pad"] = n, p
        s["day"] = _ints(g, n, 8036, 10562, torch.int32, p)
        s["qty"] = _ints(g, n, 1, 51, size=p)
        s["price"] = _ints(g, n, 90_000, 10_495_001, size=p)
        s["disc"] = _ints(g, n, 0, 11, size=p)
    elif op == "join":
        nd, nf = case["n_dim"], case["n_fact"]
        s["n_pad"] = _pow2(nd + nf, 4096)
        s["dk"] = (torch.randperm(nd, device="cuda:0", generator=g) + 1).to(torch.int32)
        s["dg"] = _ints(g, nd, 0, case["groups"], torch.int32)
        s["fk"] = s["dk"][_ints(g, nf, 0, nd)]
        s["fv"] = _ints(g, nf, 100, 10_000_001)
    elif op == "pairs":
        nl, nr, d = case["n_left"], case["n_right"], case["distinct"]
        dt = torch.int64 if case["wide"] else torch.int32
        spread = 1_000_003 if case["wide"] else 1
        if d == nl:
            left = torch.randperm(nl, device="cuda:0", generator=g) + 1
        else:
            left = _ints(g, nl, 1, d + 1)
        s["left"] = (left * spread).to(dt)
        s["right"] = (_ints(g, nr, 1, d + 1) * spread).to(dt)
    elif op == "gather":
        dt = torch.int64 if case["bytes"] == 8 else torch.int32
        top = 1 << (8 * case["bytes"] - 2)
        s["table"] = _ints(g, case["n_table"], -top, top, dt)
        s["ids"] = _ints(g, case["n"], 0, case["n_table"])
        s["ids"][: case["n"] // 8] = case["n_table"] // 3  # a hot record
    else:
        s["items"], total = _batch_items(case)
        s["keys"] = _ints(g, total, _M63, (1 << 63) - 1)
        s["payload"] = torch.arange(total, device="cuda:0", dtype=torch.int32)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["op"], s["case"], s["ctx"] = case["op"], case, _context()
    dev = "cuda:0"
    if s["op"] == "order_by":
        s["a"], s["b"] = torch.empty_like(s["a0"]), torch.empty_like(s["b0"])
        s["idx"] = torch.zeros(s["n_pad"], dtype=torch.int64, device=dev)
        s["o1"], s["o2"] = torch.zeros_like(s["p1"]), torch.zeros_like(s["p2"])
    elif s["op"] == "where":
        s["mask"] = torch.zeros(s["n_pad"], dtype=torch.uint8, device=dev)
        s["o8"], s["o4"], s["o1"] = (torch.empty_like(s[k]) for k in ("c8", "c4", "c1"))
        s["count"] = torch.zeros(1, dtype=torch.int64, device=dev)
        s["terms"] = [(s["x"], _abi.T_INTEGER, _abi.CMP_GE, 0), (s["x"], _abi.T_INTEGER, _abi.CMP_LT, s["hi"]),
                      (s["y"], _abi.T_BIGINT, _abi.CMP_LT, 90)]
    elif s["op"] == "filter":
        s["op_"], s["od"] = torch.zeros_like(s["price"]), torch.zeros_like(s["disc"])
        s["out"] = torch.zeros(4, dtype=torch.int64, device=dev)
    elif s["op"] == "join":
        s["og"] = torch.zeros(64, dtype=torch.int32, device=dev)
        s["osum"] = torch.zeros(64, dtype=torch.int64, device=dev)
        s["on"] = torch.zeros(1, dtype=torch.int64, device=dev)
    elif s["op"] == "gather":
        s["out"] = torch.zeros(case["n"], dtype=s["table"].dtype, device=dev)
        s["found"] = torch.zeros(case["n"], dtype=torch.uint8, device=dev)
    return s


def run(s):
    ctx, op, case = s["ctx"], s["op"], s["case"]
    if op == "sort":
        if case["wait"]:
            ctx.sort_kp(s["keys"], s["payload"], s["n"], s["n_pad"])
        else:
            ctx.sort_kp_async(s["keys"], s["payload"], s["n"], s["n_pad"])
        return s["keys"], s["payload"]
    if op == "order_by":
        # the operator sorts copies of the key columns in place
        s["a"].copy_(s["a0"])
        s["b"].copy_(s["b0"])
        second = _abi.T_DOUBLE if case["second"] == "double" else _abi.T_BIGINT
        ctx.sort([s["a"], s["b"]], [_abi.T_INTEGER, second], [True, False], s["idx"], s["n"], s["n_pad"])
        ctx.permute(s["o1"], s["p1"], s["idx"], s["n"], _abi.T_BIGINT)
        ctx.permute(s["o2"], s["p2"], s["idx"], s["n"], _abi.T_BIGINT)
        return s["idx"], s["a"], s["b"], s["o1"], s["o2"]
    if op == "where":
        # the operator compacts copies of its input's columns in place
        for o, c in (("o8", "c8"), ("o4", "c4"), ("o1", "c1")):
            s[o].copy_(s[c])
        ctx.predicate_mask(s["terms"], s["mask"], s["n"], s["n_pad"])
        ctx.compact(s["mask"], [s["o8"], s["o4"], s["o1"]], [8, 4, 1], s["n"], s["n_pad"], out_count=s["count"])
        return s["mask"], s["count"], s["o8"], s["o4"], s["o1"]
    if op == "filter":
        ctx.filter_sum(s["day"], s["qty"], s["price"], s["disc"], s["n"], s["n_pad"], s["out"], out_price=s["op_"],
                       out_disc=s["od"])
        return s["out"], s["op_"], s["od"]
    if op == "join":
        ctx.join_groupsum(s["dk"], s["dg"], case["n_dim"], s["fk"], s["fv"], case["n_fact"], s["n_pad"], s["og"],
                          s["osum"], s["on"], case["groups"], dense_groups=case["dense"])
        return s["og"], s["osum"], s["on"]
    if op == "pairs":
        return ctx.join_pairs(s["left"], s["right"], _abi.T_BIGINT if case["wide"] else _abi.T_INTEGER)
    if op == "gather":
        ctx.gather_oblivious(s["table"], case["n_table"], s["ids"], case["n"], s["out"], case["bytes"],
                             out_found=s["found"])
        return s["out"], s["found"]
    ctx.sort_batch(s["keys"], s["payload"], s["items"])
    return s["keys"], s["payload"]


def work(case):
    """Each input read once and each output written once (padded columns are outputs too)."""
    op = case["op"]
    if op == "sort":
        b = 12 * case["n"] + 12 * _pow2(case["n"])
    elif op == "order_by":
        n, p = case["n"], _pow2(case["n"])
        b = 12 * n + (12 + 8) * p + 2 * 16 * n
    elif op == "where":
        n, p = case["n"], _pow2(case["n"])
        b = 12 * n + p + 13 * n + 13 * p
    elif op == "filter":
        b = 28 * case["n"] + 16 * _pow2(case["n"], 2)
    elif op == "join":
        b = 8 * case["n_dim"] + 12 * case["n_fact"] + 12 * case["groups"]
    elif op == "pairs":
        w = 8 if case["wide"] else 4
        out = case["n_left"] * case["n_right"] // case["distinct"]
        b = w * (case["n_left"] + case["n_right"]) + 16 * _pow2(out)
    elif op == "gather":
        b = case["bytes"] * case["n_table"] + (8 + case["bytes"] + 1) * case["n"]
    else:
        b = sum(12 * n + 12 * p for _, n, p in _batch_items(case)[0])
    return {"bytes": b, "flops": 0}


def tolerance(case):
    # integers, row ids and bytes moved whole
    return "exact"


# -------------------------------------------------------- plain torch results


def _sorted_kp(keys, payload, n, n_pad):
    """Unsigned 64-bit order by key, ties by payload (ascending here, so a stable sort), then the pads."""
    _, order = torch.sort(keys[:n] ^ _M63, stable=True)
    k = torch.full((n_pad,), -1, dtype=torch.int64, device=keys.device)
    k[:n] = keys[:n][order]
    p = torch.arange(n_pad, dtype=torch.int32, device=keys.device)
    p[:n] = payload[:n][order]
    return k, p


def exact(case, seed):
    s, op = _inputs(case, seed), case["op"]
    if op == "sort":
        return _sorted_kp(s["keys"], s["payload"], s["n"], s["n_pad"])
    if op == "order_by":
        n, p = s["n"], s["n_pad"]
        a, b = s["a0"][:n], s["b0"][:n]
        o = torch.sort(b, descending=True, stable=True).indices
        o = o[torch.sort(a[o], stable=True).indices]
        ea = torch.full((p,), (1 << 31) - 1, dtype=torch.int32, device=a.device)
        low = torch.finfo(torch.float64).min if b.dtype == torch.float64 else torch.iinfo(torch.int64).min
        eb = torch.full((p,), low, dtype=b.dtype, device=a.device)
        ea[:n], eb[:n] = a[o], b[o]
        o1, o2 = torch.zeros_like(s["p1"]), torch.zeros_like(s["p2"])
        o1[:n], o2[:n] = s["p1"][o], s["p2"][o]
        return None, ea, eb, o1, o2  # the pad rows' order is the network's own
    if op == "where":
        live = torch.arange(s["n_pad"], device="cuda:0") < s["n"]
        m = live & (s["x"] >= 0) & (s["x"] < s["hi"]) & (s["y"] < 90)
        # rows behind the selected ones are the network's own order
        return m.to(torch.uint8), m.sum().reshape(1), None, None, None
    if op == "filter":
        n = s["n"]
        m = ((s["day"][:n] >= 8766) & (s["day"][:n] < 9131) & (s["disc"][:n] >= 5) & (s["disc"][:n] <= 7)
             & (s["qty"][:n] < 24))
        total = int((s["price"][:n][m] * s["disc"][:n][m]).sum())  # below 2^63 at every size here
        return torch.tensor([int(m.sum()), 0, total, 0], dtype=torch.int64), None, None
    if op == "join":
        grp = torch.zeros(case["n_dim"] + 1, dtype=torch.int64, device="cuda:0")
        grp[s["dk"].long()] = s["dg"].long()
        g = grp[s["fk"].long()]
        sums = torch.zeros(64, dtype=torch.int64, device="cuda:0").index_add_(0, g, s["fv"])
        ids = torch.nonzero(torch.bincount(g, minlength=64)).reshape(-1)
        og, osum = torch.zeros(64, dtype=torch.int32), torch.zeros(64, dtype=torch.int64)
        og[: len(ids)], osum[: len(ids)] = ids.to(torch.int32).cpu(), sums[ids].cpu()
        # rows behind the last group are not results
        same = len(ids) == case["groups"]
        return (og if same else None), (osum if same else None), torch.tensor([len(ids)])
    if op == "pairs":
        lk, lo = torch.sort(s["left"], stable=True)
        rk, ro = torch.sort(s["right"], stable=True)
        first = torch.searchsorted(rk, lk)
        cnt = torch.searchsorted(rk, lk, right=True) - first
        n = int(cnt.sum())
        el, er = (torch.full((_pow2(n),), -1, dtype=torch.int64, device="cuda:0") for _ in range(2))
        start = torch.cumsum(cnt, 0) - cnt
        row = torch.repeat_interleave(torch.arange(len(lk), device="cuda:0"), cnt)
        el[:n] = lo[row]
        er[:n] = ro[first[row] + torch.arange(n, device="cuda:0") - start[row]]
        return n, el, er
    if op == "gather":
        return s["table"][s["ids"]], torch.ones(case["n"], dtype=torch.uint8)
    k, p = s["keys"].clone(), s["payload"].clone()
    for off, n, pad in s["items"]:
        k[off:off + pad], p[off:off + pad] = _batch_sorted(s, off, n, pad)
    return k, p


def _batch_sorted(s, off, n, pad):
    k, p = _sorted_kp(s["keys"][off:off + pad], s["payload"][off:off + pad], n, pad)
    return k, p
