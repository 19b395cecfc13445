"""Timed cases of the group-by library, through its public Python entry points.

Every case is one call a program makes on device-resident columns: a grouped
aggregation through the dispatcher (from thousands to 2^28 rows, a handful to
millions of groups, uniform and skewed keys, one or two value columns, one or
two key columns), one in key order, a planned batch of uneven queries, and the
sort, partition and dictionary sub-operators on their own.

Group-by results come in no particular order.  The keys of these cases stand
for dictionary codes (or ids made of one), as in a star schema, and each pass
ends as such a program does: it puts every aggregate at its code's place in a
dense column.  Passes whose result is ordered return the result itself.
"""
import math

import torch

from eiger_amd import gamax as G

T, A = G.type_id, G.aggregation_id
DEV = "cuda"
INT64_KEY_SHIFT = 12  # int64 keys: ids handed out in blocks, code << 12 | 7

TYPES = {
    "i32": (T.INT32, torch.int32, "<i4", 4),
    "i64": (T.INT64, torch.int64, "<i8", 8),
    "f32": (T.FLOAT32, torch.float32, "<f4", 4),
    "f64": (T.FLOAT64, torch.float64, "<f8", 8),
}
OF_ID = {t[0]: t for t in TYPES.values()}
AGGS = {"sum": A.SUM, "min": A.MIN, "max": A.MAX, "avg": A.AVG}

SUM_COUNT = "sum0,count"                     # the batched and partition-heavy workloads' requests
FIVE = "count,sum0,min0,max0,sum1"           # the strategy sweep's requests
BATCH_REQS = [(0, A.SUM), (-1, A.COUNT_ALL)]


def listed():
    return [
        # a dashboard tile over a small table: all latency
        dict(name="tiny", op="groupby", rows=3001, groups=120, key="i32", vals="i64", aggs=SUM_COUNT, s=0.0, bound=False),
        # the plain small workload: 2^20 rows, keys in [0, 1024), int32 values
        dict(name="small_1m", op="groupby", rows=1 << 20, groups=1024, key="i32", vals="i32", aggs="count,sum0", s=0.0, bound=False),
        # an ordinary query of the uneven mix: a few million rows, skewed, many groups
        dict(name="mid_3m_zipf", op="groupby", rows=3_000_017, groups=400_003, key="i32", vals="i64", aggs=SUM_COUNT, s=0.8, bound=False),
        # the strategy sweep: few groups (skewed), some, many; five aggregates over two columns
        dict(name="sweep_2e10_zipf", op="groupby", rows=1 << 28, groups=1 << 10, key="i32", vals="i64,f32", aggs=FIVE, s=1.0, bound=True),
        dict(name="sweep_2e16", op="groupby", rows=1 << 28, groups=1 << 16, key="i32", vals="i64,f32", aggs=FIVE, s=0.0, bound=True),
        dict(name="sweep_2e22", op="groupby", rows=1 << 28, groups=1 << 22, key="i32", vals="i64,f32", aggs=FIVE, s=0.0, bound=True),
        # partition-heavy: int64 ids, four rows a group, no hint (an odd row count)
        dict(name="heavy_i64", op="groupby", rows=(1 << 26) + 12_345, groups=1 << 24, key="i64", vals="i64", aggs=SUM_COUNT, s=0.0, bound=False),
        # a report in key order: the sort strategy, double values, AVG
        dict(name="ordered_f64", op="ordered", rows=40_000_003, groups=1 << 20, key="i64", vals="f64", aggs="avg0,min0,max0,count", s=0.5, bound=False),
        # two key columns (region, day) fused into one
        dict(name="two_keys", op="two_keys", rows=25_000_001, groups=700_000, key="i32", vals="f32", aggs="sum0,count", s=0.0, bound=False),
        # a planned batch of uneven queries, replayed
        dict(name="batch_512", op="batch", queries=512, max_rows=4_000_000),
        # ordering two columns by a full-width key
        dict(name="sort_pair", op="sort_pair", rows=(1 << 26) + 1001, key="i32", vals="i64"),
        # rows to codes against a dictionary of sparse ids
        dict(name="encode_sparse", op="encode", rows=100_000_007, groups=300_000, key="i32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["groupby"] * 7 + ["ordered", "two_keys", "batch", "sort_pair", "encode"])
    s = 0.0 if rng.random() < 0.5 else round(rng.uniform(0.5, 1.5), 2)
    if op == "batch":
        return dict(op=op, queries=_log(rng, 64, 512), max_rows=_log(rng, 200_000, 4_000_000))
    if op == "sort_pair":
        return dict(op=op, rows=_log(rng, 10_000, 1 << 26), key=rng.choice(["i32", "i64"]), vals=rng.choice(["i32", "i64"]))
    if op == "encode":
        return dict(op=op, rows=_log(rng, 100_000, 100_000_000), groups=_log(rng, 1000, 500_000), key=rng.choice(["i32", "i64"]))
    if op == "ordered":
        rows = _log(rng, 100_000, 40_000_000)
        return dict(op=op, rows=rows, groups=_log(rng, 16, rows // 4), key=rng.choice(["i32", "i64"]), vals=rng.choice(["f64", "f32", "i64"]),
                    aggs=rng.choice(["avg0,min0,max0,count", SUM_COUNT]), s=s, bound=False)
    if op == "two_keys":
        rows = _log(rng, 100_000, 25_000_000)
        return dict(op=op, rows=rows, groups=_log(rng, 100, min(1_000_000, rows // 4)), key="i32", vals=rng.choice(["f32", "i64"]), aggs=SUM_COUNT, s=s,
                    bound=False)
    if rng.random() < 0.4:  # the sweep's shape
        rows = _log(rng, 1 << 22, 1 << 28)
        return dict(op=op, rows=rows, groups=_log(rng, 16, min(1 << 22, rows // 4)), key="i32", vals="i64,f32", aggs=FIVE, s=s, bound=True)
    key = rng.choice(["i32", "i32", "i64"])
    rows = _log(rng, 1000, (1 << 26) if key == "i64" else (1 << 27))
    return dict(op=op, rows=rows, groups=_log(rng, 1, min(1 << 24, max(2, rows // 4))), key=key, vals=rng.choice(["i64", "i32", "f32", "f64"]),
                aggs=rng.choice([SUM_COUNT, SUM_COUNT, "sum0,min0,max0", "avg0,count"]), s=s, bound=rng.random() < 0.3)


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _codes(gen, rows, groups, s):
    """Codes in [0, groups): every code equally often in random order (s = 0),
    or Zipf-like with code r drawn about as often as 1/(r+1)^s."""
    if s == 0.0:
        out = torch.randint(0, groups, (rows,), device=DEV, generator=gen)
        m = min(rows, groups)
        # each code at least once where the rows allow it
        out[torch.randperm(rows, device=DEV, generator=gen)[:m] if rows <= (1 << 20) else torch.arange(m, device=DEV) * (rows // m)] = \
            torch.arange(m, device=DEV)
        return out
    u = torch.rand(rows, device=DEV, generator=gen, dtype=torch.float64)
    return _zipf(u, float(groups), s)


def _zipf(u, d, s):
    """The bounded Pareto law on [1, d+1) at u, floored: a continuous Zipf."""
    top = torch.as_tensor(d + 1.0, device=DEV, dtype=torch.float64)
    s = torch.as_tensor(s, device=DEV, dtype=torch.float64)
    e = 1.0 - s
    near = e.abs() < 1e-6
    e = torch.where(near, torch.ones_like(e), e)
    x = torch.where(near, torch.pow(top, u), torch.pow(u * (torch.pow(top, e) - 1.0) + 1.0, 1.0 / e))
    r = x.floor().long() - 1
    return torch.minimum(r.clamp_(min=0), top.long() - 2)


def _values(gen, rows, kind):
    if kind == "i64":
        return torch.randint(-(1 << 31), 1 << 31, (rows,), device=DEV, generator=gen)
    if kind == "i32":
        return torch.randint(0, 1000, (rows,), device=DEV, generator=gen, dtype=torch.int32)
    if kind == "f32":
        return torch.rand(rows, device=DEV, generator=gen)
    return torch.randn(rows, device=DEV, generator=gen, dtype=torch.float64)


def _keys(codes, key):
    return codes.to(torch.int32) if key == "i32" else (codes << INT64_KEY_SHIFT) + 7


def _view(t):
    for tid, dt, _, _ in TYPES.values():
        if t.dtype == dt:
            return G.column_view(t.data_ptr(), t.numel(), tid)
    raise TypeError(str(t.dtype))


def _requests(aggs):
    out = []
    for a in aggs.split(","):
        out.append((-1, A.COUNT_ALL) if a == "count" else (int(a[3:]), AGGS[a[:3]]))
    return out


def _second(groups):
    """Distinct values of the second of two key columns."""
    return max(1, int(math.sqrt(groups)))


def _table(case, seed):
    """(codes, value columns) of a group-by case."""
    gen = _gen(seed)
    codes = _codes(gen, case["rows"], case["groups"], case["s"])
    return codes, [_values(gen, case["rows"], v) for v in case["vals"].split(",")]


def _batch_table(case, seed):
    """The uneven mix: rows log-uniform in [1e3, max_rows], distinct codes
    log-uniform in [1, rows / 2], half the queries uniform, half Zipf with s
    in [0.5, 1.5].  Sizes come from the case, data from the seed."""
    nq = case["queries"]
    shape = torch.Generator().manual_seed(nq * 7919 + case["max_rows"])
    r = torch.rand(4, nq, generator=shape, dtype=torch.float64)
    rows = torch.exp(math.log(1e3) + r[0] * (math.log(case["max_rows"]) - math.log(1e3))).long()
    groups = torch.exp(r[1] * torch.log(rows.double() / 2)).long().clamp_(min=1)
    s = torch.where(r[2] < 0.5, torch.zeros(nq, dtype=torch.float64), 0.5 + r[3])
    padded = (rows + 63) // 64 * 64  # each query's columns start on their own line
    start = torch.cumsum(padded, 0) - padded
    total = int(padded.sum())
    gen = _gen(seed)
    u = torch.rand(total, device=DEV, generator=gen, dtype=torch.float64)
    q = torch.repeat_interleave(torch.arange(nq, device=DEV), padded.to(DEV), output_size=total)
    d = groups.to(DEV).double()[q]
    keys = _zipf(u, d, s.to(DEV)[q]).to(torch.int32)
    del u, d, q
    return rows.tolist(), groups.tolist(), start.tolist(), keys, _values(gen, total, "i64")


# ---------------------------------------------------------------- prepare
class _State:
    pass


def _ready():
    """What a serving program does once at its start."""
    if not G.mlp_loaded():
        G.load_dispatch_model()


def prepare(case, seed):
    _ready()
    st = _State()
    st.op = case["op"]
    if st.op == "batch":
        return _prepare_batch(st, case, seed)
    n = case["rows"]
    if st.op == "sort_pair":
        gen = _gen(seed)
        lo, hi, dt = (-(1 << 31), 1 << 31, torch.int32) if case["key"] == "i32" else (-(1 << 62), 1 << 62, torch.int64)
        st.data = [torch.randint(lo, hi, (n,), device=DEV, generator=gen, dtype=dt), _values(gen, n, case["vals"])]
        st.views = [_view(t) for t in st.data]
        return st
    if st.op == "encode":
        gen = _gen(seed)
        d = case["groups"]
        dt = TYPES[case["key"]][1]
        # sparse ids: the dictionary's keys spread over the type's positive range
        gap = ((1 << 31) - 1) // d if case["key"] == "i32" else 1 << 30
        ids = torch.arange(d, device=DEV) * gap + torch.randint(0, gap, (d,), device=DEV, generator=gen)
        ids = ids[torch.randperm(d, device=DEV, generator=gen)].to(dt)
        st.data = [ids[torch.randint(0, d, (n,), device=DEV, generator=gen)], ids]
        st.views = [_view(t) for t in st.data]
        return st
    codes, vals = _table(case, seed)
    st.reqs = _requests(case["aggs"])
    st.groups = case["groups"]
    st.bound = case["groups"] if case["bound"] else G.MAXIMUM_SIZE
    st.key = case["key"]
    if st.op == "two_keys":
        st.d1 = _second(st.groups)
        st.data = [torch.div(codes, st.d1, rounding_mode="floor").to(torch.int32), (codes % st.d1).to(torch.int32)] + vals
        st.nkeys, key_type = 2, T.UINT64
    else:
        st.data = [_keys(codes, st.key)] + vals
        st.nkeys, key_type = 1, TYPES[st.key][0]
    st.views = [_view(t) for t in st.data]
    # the program's requests are known before its data: their kernels are ready
    G.jit_prefetch(key_type, [v.type for v in st.views[st.nkeys:]], st.reqs)
    G.jit_wait()
    if st.op != "ordered":
        st.dense = []
        for c, kind in st.reqs:
            t = G.agg_output_data_type(kind, st.views[st.nkeys + c].type if c >= 0 else T.INT32)
            st.dense.append(torch.zeros(st.groups, device=DEV, dtype=OF_ID[t][1]))
    return st


def _prepare_batch(st, case, seed):
    rows, groups, start, keys, vals = _batch_table(case, seed)
    cap = [min(r, g) for r, g in zip(rows, groups)]
    total = sum(cap)
    st.data = [keys, vals]
    # one sentinel code per query (its group count): rows never written go there
    out_keys = torch.repeat_interleave(torch.tensor(groups, device=DEV, dtype=torch.int32), torch.tensor(cap, device=DEV), output_size=total)
    st.outs = [out_keys, torch.zeros(total, device=DEV, dtype=torch.int64), torch.zeros(total, device=DEV, dtype=torch.int64)]
    width = torch.tensor([g + 1 for g in groups])
    base = (torch.cumsum(width, 0) - width).to(DEV)
    st.base = torch.repeat_interleave(base, torch.tensor(cap, device=DEV), output_size=total)
    st.dense = [torch.zeros(int(width.sum()), device=DEV, dtype=torch.int64) for _ in range(2)]
    queries, at = [], 0
    for q in range(len(rows)):
        col = [G.column_view(t.data_ptr() + start[q] * t.element_size(), rows[q], tid) for t, tid in ((keys, T.INT32), (vals, T.INT64))]
        out = [G.column_view(t.data_ptr() + at * t.element_size(), cap[q], tid) for t, tid in zip(st.outs, (T.INT32, T.INT64, T.INT64))]
        queries.append(G.batch_query(col[0], col[1], groups[q], out[0], out[1:]))
        at += cap[q]
    st.plan = G.batch_plan(queries, T.INT32, T.INT64, BATCH_REQS, G.batch_tuning(tile_rows_log2=17, lds_slots_log2=11, lds_max_bound_log2=12,
                                                                                 blocks_per_cu=2, radix_bits=10))
    return st


# ---------------------------------------------------------------- run
class _Device:
    """A library column as torch sees device memory; keeps the column alive."""

    def __init__(self, col):
        self.col = col
        self.__cuda_array_interface__ = {"shape": (col.size,), "typestr": OF_ID[col.type][2], "data": (col.data, False), "version": 2}


def _torch(col):
    return torch.as_tensor(_Device(col), device=DEV)


def run(st):
    if st.op == "sort_pair":
        return [_torch(c) for c in G.sort_column_pair(st.views[0], st.views[1])]
    if st.op == "encode":
        return _torch(G.dictionary_encode_with_dict(st.views[0], st.views[1]))
    if st.op == "batch":
        st.plan.graph_launch()
        ngroups, status = st.plan.results()
        idx = st.outs[0].long() + st.base
        for d, o in zip(st.dense, st.outs[1:]):
            d.index_copy_(0, idx, o)
        return st.dense + [ngroups, status]
    hint = G.groupby_hint(groups_upper_bound=st.bound)
    if st.op == "ordered":
        hint.groupby_algo = G.groupby_algo.SORT
    cols = G.groupby(st.views[:st.nkeys], st.views[st.nkeys:], st.reqs, hint).columns()
    out = [_torch(c) for c in cols]
    if st.op == "ordered":
        return out
    if st.nkeys == 2:
        idx = out[0].long() * st.d1 + out[1]
    else:
        idx = out[0].long() if st.key == "i32" else out[0] >> INT64_KEY_SHIFT
    for d, o in zip(st.dense, out[st.nkeys:]):
        d.index_copy_(0, idx, o)
    return st.dense


# ---------------------------------------------------------------- work and exact results
def work(case):
    op = case["op"]
    if op == "batch":
        nq = case["queries"]
        span = math.log(case["max_rows"]) - math.log(1e3)
        rows = nq * (case["max_rows"] - 1e3) / span  # mean of a log-uniform draw
        return {"bytes": 12.0 * rows + 20.0 * rows / 24, "flops": 0.0}
    n, kb = case["rows"], TYPES[case["key"]][3]
    if op == "sort_pair":
        return {"bytes": 2.0 * n * (kb + TYPES[case["vals"]][3]), "flops": 0.0}
    if op == "encode":
        return {"bytes": float(n * (kb + 4) + case["groups"] * kb), "flops": 0.0}
    kb *= 2 if op == "two_keys" else 1
    vb = [TYPES[v][3] for v in case["vals"].split(",")]
    groups = min(n, case["groups"])
    out = kb + sum(4 if (a.startswith("sum") and case["vals"].split(",")[int(a[3:])] == "f32") or
                   (a[:3] in ("min", "max") and vb[int(a[3:])] == 4) else 8 for a in case["aggs"].split(","))
    return {"bytes": float(n * (kb + sum(vb)) + groups * out), "flops": 0.0}


def _reduce(codes, v, d, how):
    """v reduced by code into d places.  Rows spread over several copies of
    the places first: one popular code would serialise its atomics."""
    copies = max(1, (1 << 25) // d)
    to = torch.arange(codes.numel(), device=DEV).remainder_(copies).mul_(d).add_(codes)
    if how == "sum":
        return torch.zeros(copies * d, device=DEV, dtype=v.dtype).index_add_(0, to, v).view(copies, d).sum(0)
    out = torch.full((copies * d,), math.inf if how == "amin" else -math.inf, device=DEV, dtype=v.dtype)
    out = out.scatter_reduce_(0, to, v, how).view(copies, d)
    return out.amin(0) if how == "amin" else out.amax(0)


def exact(case, seed):
    op = case["op"]
    if op in ("batch", "sort_pair", "encode"):
        return None  # whole numbers only
    codes, vals = _table(case, seed)
    d = case["groups"]
    count = _reduce(codes, torch.ones_like(codes), d, "sum")
    here = count > 0
    out = []
    for a in case["aggs"].split(","):
        v = None if a == "count" else vals[int(a[3:])]
        if v is None or (not v.is_floating_point() and a[:3] != "avg"):
            out.append(None)
            continue
        r = _reduce(codes, v.double(), d, "sum" if a[:3] in ("sum", "avg") else "a" + a[:3])
        r = r / count.clamp(min=1) if a[:3] == "avg" else r
        # a code that no row holds: the dense column keeps its 0
        out.append(r[here] if op == "ordered" else torch.where(here, r, torch.zeros_like(r)))
    if op == "ordered":
        out.insert(0, None)
    return out if any(r is not None for r in out) else None
