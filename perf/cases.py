"""Timed workloads of the group-by library, one dict of plain values each.

Every case is one call of a public entry point (``GroupBy.aggregate`` on the
hash, pre-sorted and sort-based paths, ``BatchedGroupBy.run``,
``hash_partition``) followed by what a program does with the result.  A hash
group-by returns its groups in no particular order, so a program that keeps
per-key results stores them by key: keys are ids in ``[0, card)`` (surrogate
keys, dictionary codes), each result column is written into a table with one
row per id, and ids without rows keep zeros.  Null results become NaN in
floating tables and 0 in integer ones, as pandas shows them.  General keys
(an integer and a string column) are put in order of first appearance through
the group's smallest row number, as ``pandas.groupby(sort=False)`` orders them.
"""
import math

import torch

import cudf_amd as ca
from cudf_amd import Column, TypeId
from cudf_amd.aggregation import Aggregation, Kind
from cudf_amd.partitioning import hash_partition

DTYPE = {"int32": torch.int32, "int64": torch.int64, "float32": torch.float32, "float64": torch.float64}
TYPE_ID = {"int32": TypeId.INT32, "int64": TypeId.INT64, "float32": TypeId.FLOAT32, "float64": TypeId.FLOAT64}
TORCH = {TypeId.INT32: torch.int32, TypeId.INT64: torch.int64, TypeId.FLOAT32: torch.float32,
         TypeId.FLOAT64: torch.float64}
WIDTH = {"int32": 4, "int64": 8, "float32": 4, "float64": 8}
KIND = {"sum": Kind.SUM, "count": Kind.COUNT_VALID, "size": Kind.COUNT_ALL, "min": Kind.MIN, "max": Kind.MAX,
        "mean": Kind.MEAN, "var": Kind.VARIANCE, "median": Kind.MEDIAN, "nunique": Kind.NUNIQUE}


def listed():
    return [
        # The smallest call: a dashboard query over a day's few thousand rows.
        # Latency of one call: launches, allocations and the host path.
        {"name": "tiny_10k", "path": "hash", "rows": 10_000, "card": 100, "key": "int32", "key_nulls": 0.0,
         "include": False, "skew": 0.0, "values": "int64:sum,count,min,max", "nulls": 0.0},
        # The basic configuration: a million rows, a thousand groups, nullable values.
        {"name": "groups1k_1m", "path": "hash", "rows": 1_000_000, "card": 1_000, "key": "int32", "key_nulls": 0.0,
         "include": False, "skew": 0.0, "values": "int64:sum,count,min,max", "nulls": 0.05},
        # A fact table over a small dimension, null keys kept as their own group.
        {"name": "groups1k_40m", "path": "hash", "rows": 40_000_003, "card": 1_000, "key": "int64", "key_nulls": 0.01,
         "include": True, "skew": 0.0, "values": "float32:sum,mean,max;int32:sum,min", "nulls": 0.03},
        # Many groups in a call below a million rows (served requests): the device-wide table.
        {"name": "groups100k_300k", "path": "hash", "rows": 300_007, "card": 100_000, "key": "int64",
         "key_nulls": 0.01, "include": False, "skew": 0.0, "values": "float64:sum,mean,count,max", "nulls": 0.0},
        # High cardinality with every statistic of the headline request on two nullable columns.
        {"name": "groups800k_8m", "path": "hash", "rows": 8_000_003, "card": 800_000, "key": "int32",
         "key_nulls": 0.01, "include": False, "skew": 0.0,
         "values": "float64:sum,mean,count,min,max,var;int32:sum,mean,count,min,max,var", "nulls": 0.05},
        # The largest: 100M rows over 10M ids.
        {"name": "groups10m_100m", "path": "hash", "rows": 100_000_000, "card": 10_000_000, "key": "int64",
         "key_nulls": 0.01, "include": False, "skew": 0.0, "values": "float64:sum,count,min,max,var;int32:sum,max",
         "nulls": 0.0},
        # Skewed ids (visits per user): Zipf(1.1) over a million values.
        {"name": "zipf_20m", "path": "hash", "rows": 20_000_000, "card": 1_000_000, "key": "int64", "key_nulls": 0.0,
         "include": False, "skew": 1.1, "values": "int64:sum,count,min,max", "nulls": 0.0},
        # General keys: an integer and a string column, strings of 4..32 characters.
        {"name": "int_string_10m", "path": "general", "rows": 10_000_000, "card": 100, "pool": 10_000,
         "groups": 900_001, "values": "float32:sum,count,max;int64:sum,max", "nulls": 0.02},
        # Keys that arrive sorted (clustered tables): the runs path.
        {"name": "sorted_50m", "path": "sorted", "rows": 50_000_001, "card": 5_000_000, "key": "int64",
         "values": "float64:sum,mean,count,min,max,var;int32:sum,mean,count,min,max,var", "nulls": 0.05},
        # Shuffle before an exchange: rows regrouped by key hash.
        {"name": "partition256_50m", "path": "partition", "rows": 50_000_000, "card": 5_000_000, "parts": 256,
         "key": "int64", "values": "float64;int32", "nulls": 0.0},
        # Sort-based aggregations of keys in no order.
        {"name": "median_nunique_4m", "path": "sortbased", "rows": 4_000_003, "card": 50_000, "key": "int32",
         "values": "float64:median,max;int32:nunique", "nulls": 0.03},
        # Many independent group-bys in one plan, executed again for each refresh.
        {"name": "batch_16", "path": "batch", "instances": 16, "rows_lo": 100_000, "rows_hi": 2_000_000,
         "values": "int64:sum,count,min,max;float32:sum,max", "shape_seed": 4},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


STATS = ["sum,count,min,max", "sum,mean,max", "sum,mean,count,min,max,var", "count,min", "mean,var", "sum"]


def _draw_values(rng, most=2):
    n = rng.randint(1, most)
    return ";".join("%s:%s" % (rng.choice(list(DTYPE)), rng.choice(STATS)) for _ in range(n))


def draw(rng):
    path = rng.choice(["hash"] * 7 + ["general", "sorted", "sorted", "partition", "sortbased", "batch"])
    if path == "hash":
        rows = _log_uniform(rng, 1e4, 5e7) | 1
        skew = 1.1 if rng.random() < 0.15 else 0.0
        card = min(1_000_000, max(10, rows // 20)) if skew else _log_uniform(rng, 20, max(40, rows / 5))
        return {"path": path, "rows": rows, "card": card, "key": rng.choice(["int32", "int64"]),
                "key_nulls": rng.choice([0.0, 0.01]), "include": rng.random() < 0.2, "skew": skew,
                "values": _draw_values(rng), "nulls": rng.choice([0.0, 0.0, 0.02, 0.05])}
    if path == "general":
        rows, card, pool = _log_uniform(rng, 2e4, 1e7) | 1, rng.randint(5, 100), _log_uniform(rng, 20, 1e4)
        return {"path": path, "rows": rows, "card": card, "pool": pool,
                "groups": _log_uniform(rng, 50, min(card * pool, rows * 0.7)), "values": _draw_values(rng), "nulls": rng.choice([0.0, 0.02])}
    if path == "sorted":
        rows = _log_uniform(rng, 1e5, 5e7) | 1
        return {"path": path, "rows": rows, "card": _log_uniform(rng, 100, rows / 5),
                "key": rng.choice(["int32", "int64"]), "values": _draw_values(rng),
                "nulls": rng.choice([0.0, 0.05])}
    if path == "partition":
        return {"path": path, "rows": _log_uniform(rng, 1e5, 5e7) | 1, "card": 1_000_000,
                "parts": rng.choice([2, 7, 8, 16, 61, 64, 128, 200, 256, 500]), "key": rng.choice(["int32", "int64"]),
                "values": rng.choice(["float64", "float32;int64", "float64;int32", "int32"]),
                "nulls": rng.choice([0.0, 0.05])}
    if path == "sortbased":
        rows = _log_uniform(rng, 5e4, 8e6) | 1
        return {"path": path, "rows": rows, "card": _log_uniform(rng, 50, rows / 10),
                "key": rng.choice(["int32", "int64"]),
                "values": rng.choice(["float64:median", "float32:median,max;int64:nunique", "int32:nunique,sum"]),
                "nulls": rng.choice([0.0, 0.05])}
    return {"path": path, "instances": rng.randint(4, 32), "rows_lo": _log_uniform(rng, 2e3, 1e5),
            "rows_hi": _log_uniform(rng, 2e5, 3e6), "values": "int64:sum,count,min,max;float32:sum,max",
            "shape_seed": rng.randrange(1000)}


# -- shapes ------------------------------------------------------------------


def _spec(case):
    """[(value type, [aggregation names])]"""
    out = []
    for part in case["values"].split(";"):
        t, _, aggs = part.partition(":")
        out.append((t, aggs.split(",") if aggs else []))
    return out


def _result_type(vtype, agg):
    if agg in ("count", "size", "nunique"):
        return "int32"
    if agg in ("mean", "var", "median"):
        return "float64"
    if agg == "sum":
        return "int64" if vtype.startswith("int") else vtype
    return vtype


def _batch_shapes(case):
    """Rows log-uniform in the case's range, cardinality log-uniform up to half the rows."""
    import random
    r = random.Random(case["shape_seed"])
    shapes = []
    for _ in range(case["instances"]):
        n = _log_uniform(r, case["rows_lo"], case["rows_hi"])
        shapes.append((n, max(1, _log_uniform(r, 1, n / 2))))
    return shapes


# -- inputs ------------------------------------------------------------------


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _pack(valid):
    """LSB-first 32-bit validity words."""
    n = valid.numel()
    v = torch.nn.functional.pad(valid.to(torch.uint8), (0, (-n) % 32)).view(-1, 8)
    w = torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], dtype=torch.uint8, device=valid.device)
    return (v * w).sum(1, dtype=torch.uint8).view(torch.int32)


def _column(t, valid=None):
    tid = TYPE_ID[str(t.dtype).replace("torch.", "")]
    if valid is None:
        return Column(tid, t.numel(), t.view(torch.uint8))
    return Column(tid, t.numel(), t.view(torch.uint8), _pack(valid), int((~valid).sum().item()))


def _valid(g, n, nulls):
    return torch.rand(n, device=g.device, generator=g) >= nulls if nulls else None


def _values(g, n, vtype):
    if vtype == "int32":
        return torch.randint(0, 10_001, (n,), dtype=torch.int32, device=g.device, generator=g)
    if vtype == "int64":
        return torch.randint(-10**9, 10**9 + 1, (n,), dtype=torch.int64, device=g.device, generator=g)
    if vtype == "float32":
        return torch.rand(n, dtype=torch.float32, device=g.device, generator=g)
    return torch.randn(n, dtype=torch.float64, device=g.device, generator=g)


def _pairs(case, device):
    """The distinct pairs of a general-key case as int * pool + string."""
    most = case["card"] * case["pool"]
    step = most // 3 | 1
    while math.gcd(step, most) > 1:
        step += 2
    return torch.arange(case["groups"], device=device) * step % most


def _keys(g, case):
    n, card, dtype = case["rows"], case["card"], DTYPE[case["key"]]
    if case.get("skew"):
        w = torch.arange(1, card + 1, dtype=torch.float64, device=g.device) ** -case["skew"]
        cdf = torch.cumsum(w, 0) / w.sum()
        rank = torch.searchsorted(cdf, torch.rand(n, dtype=torch.float64, device=g.device, generator=g))
        return torch.randperm(card, device=g.device, generator=g)[rank.clamp_(max=card - 1)].to(dtype)
    key = torch.randint(0, card, (n,), dtype=dtype, device=g.device, generator=g)
    if case["path"] == "sorted":  # every id has a row
        key[:card] = torch.arange(card, device=g.device)
    return key


def _inputs(case, seed):
    """The raw tensors of a case: everything follows from the seed."""
    g = torch.Generator(device=_device()).manual_seed(seed)
    s = {}
    if case["path"] == "batch":
        s["instances"] = [(torch.randint(0, c, (n,), dtype=torch.int32, device=g.device, generator=g),
                           [(_values(g, n, t), None) for t, _ in _spec(case)]) for n, c in _batch_shapes(case)]
        return s
    n = case["rows"]
    if case["path"] == "general":
        # `groups` distinct (integer, string) pairs, each in at least one row
        pair = torch.cat([torch.arange(case["groups"], device=g.device),
                          torch.randint(0, case["groups"], (n - case["groups"],), device=g.device, generator=g)])
        pair = _pairs(case, g.device)[pair[torch.randperm(n, device=g.device, generator=g)]]
        s["k1"] = (pair // case["pool"] + 1).to(torch.int32)
        s["sid"] = pair % case["pool"]
        lens = 4 + torch.arange(case["pool"], device=g.device) * 7919 % 29
        start = torch.cumsum(lens, 0) - lens
        chars = torch.randint(33, 127, (int(lens.sum()),), dtype=torch.uint8, device=g.device, generator=g)
        code = torch.randperm(case["pool"], device=g.device, generator=g)
        for j in range(3):  # the first characters tell the pool's strings apart
            chars[start + j] = (33 + code // 94**j % 94).to(torch.uint8)
        ln = lens[s["sid"]]
        offs = torch.zeros(n + 1, dtype=torch.int64, device=g.device)
        torch.cumsum(ln, 0, out=offs[1:])
        total = int(offs[-1])
        src = torch.repeat_interleave(start[s["sid"]] - offs[:-1], ln, output_size=total)
        s["chars"] = chars[src + torch.arange(total, device=g.device)]
        s["offsets"] = offs.to(torch.int32)
        # what the exact result needs: the pool itself
        s["pool"] = (lens, start, chars)
    else:
        key = _keys(g, case)
        s["key"] = torch.sort(key).values if case["path"] == "sorted" else key
        s["key_valid"] = _valid(g, n, case.get("key_nulls", 0.0))
    s["values"] = [(_values(g, n, t), _valid(g, n, case["nulls"])) for t, _ in _spec(case)]
    return s


def prepare(case, seed):
    raw = _inputs(case, seed)
    dev = _device()
    s = {"case": case}
    spec = _spec(case)
    path = case["path"]
    if path == "batch":
        shapes = _batch_shapes(case)
        inst = [(_column(k), [_column(v) for v, _ in vs]) for k, vs in raw["instances"]]
        s["plan"] = ca.BatchedGroupBy(inst, [[Aggregation(KIND[a]) for a in aggs] for _, aggs in spec])
        base, at = [], 0
        for _, c in shapes:
            base.append(at)
            at += c
        s["base"] = base
        s["tables"] = [[torch.zeros(at, dtype=DTYPE[_result_type(t, a)], device=dev) for a in aggs]
                       for t, aggs in spec]
        return s
    s["columns"] = [_column(v, ok) for v, ok in raw["values"]]
    if path == "general":
        s["keys"] = ca.Table([_column(raw["k1"]),
                              Column(TypeId.STRING, case["rows"], raw["chars"], None, 0, 0, raw["offsets"])])
        s["rownum"] = _column(torch.arange(case["rows"], dtype=torch.int32, device=dev))
        return s
    s["keys"] = ca.Table([_column(raw["key"], raw["key_valid"])])
    if path in ("hash", "sortbased"):
        rows = case["card"] + 1  # the last row is the null key's
        s["tables"] = [[torch.zeros(rows, dtype=DTYPE[_result_type(t, a)], device=dev) for a in aggs]
                       for t, aggs in spec]
    return s


# -- one pass ----------------------------------------------------------------

_BITS = {}


def _bits(column, n):
    """Validity of a column's first n rows."""
    dev = column.mask.device
    if dev not in _BITS:
        _BITS[dev] = torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], dtype=torch.uint8, device=dev)
    return column.mask.view(torch.uint8).unsqueeze(1).bitwise_and(_BITS[dev]).view(-1)[:n].bool()


def _data(column):
    """A result column as a tensor, nulls as NaN (0 in integers)."""
    n = column.size
    dt = TORCH[column.type_id]
    t = column.data[:n * dt.itemsize].view(dt)
    if column.mask is None:
        return t
    return torch.where(_bits(column, n), t, math.nan if dt.is_floating_point else 0)


def _requests(case, columns):
    return [ca.GroupByRequest(c, [Aggregation(KIND[a]) for a in aggs]) for c, (_, aggs) in zip(columns, _spec(case))]


def run(s):
    case = s["case"]
    path = case["path"]
    if path == "partition":
        table, offsets = hash_partition(ca.Table(s["keys"].columns() + s["columns"]), [0], case["parts"])
        return {"columns": [_data(c) for c in table.columns()], "offsets": torch.tensor(offsets)}
    if path == "batch":
        plan = s["plan"]
        plan.run()
        ids, cols = [], [[[] for _ in aggs] for _, aggs in _spec(case)]
        for i in range(len(plan)):
            keys, res = plan.result(i)
            ids.append(_data(keys.columns()[0]) + s["base"][i])
            for r, t in enumerate(res):
                for a, c in enumerate(t.columns()):
                    cols[r][a].append(_data(c))
        ids = torch.cat(ids).to(torch.int64)
        for tables, results in zip(s["tables"], cols):
            for t, parts in zip(tables, results):
                t.scatter_(0, ids, torch.cat(parts))
        return s["tables"]
    if path == "sorted":
        keys, res = ca.GroupBy(s["keys"], keys_are_sorted=ca.Sorted.YES).aggregate(_requests(case, s["columns"]))
        return {"keys": _data(keys.columns()[0]), "results": [[_data(c) for c in t.columns()] for t in res]}
    if path == "general":
        reqs = _requests(case, s["columns"]) + [ca.GroupByRequest(s["rownum"], [Aggregation(Kind.MIN)])]
        keys, res = ca.GroupBy(s["keys"]).aggregate(reqs)
        order = torch.argsort(_data(res[-1].columns()[0]))
        k1, k2 = keys.columns()
        n = k1.size
        offs = k2.offsets[:n + 1]
        lens = offs.diff()[order]
        ends = torch.cumsum(lens, 0)
        total = int(ends[-1])
        src = torch.repeat_interleave(offs[:n][order] - (ends - lens), lens, output_size=total)
        chars = k2.data[src + torch.arange(total, device=src.device)]
        return {"k1": _data(k1)[order], "lengths": lens, "chars": chars,
                "results": [[_data(c)[order] for c in t.columns()] for t in res]}
    include = bool(case.get("include"))
    keys, res = ca.GroupBy(s["keys"], ca.NullPolicy.INCLUDE if include else ca.NullPolicy.EXCLUDE).aggregate(
        _requests(case, s["columns"]))
    key = keys.columns()[0]
    ids = key.data[:key.size * TORCH[key.type_id].itemsize].view(TORCH[key.type_id]).to(torch.int64)
    if include and key.mask is not None:
        ids = torch.where(_bits(key, key.size), ids, case["card"])
    for tables, t in zip(s["tables"], res):
        for table, c in zip(tables, t.columns()):
            table.scatter_(0, ids, _data(c))
    return s["tables"]


# -- what a pass cannot do without --------------------------------------------


def work(case):
    spec = _spec(case)
    if case["path"] == "batch":
        total = 0
        for n, c in _batch_shapes(case):
            groups = c * -math.expm1(-n / c)
            total += n * (4 + sum(WIDTH[t] for t, _ in spec))
            total += groups * (4 + sum(WIDTH[_result_type(t, a)] for t, aggs in spec for a in aggs))
        return {"bytes": total, "flops": 0}
    n = case["rows"]
    masks = len(spec) if case["nulls"] else 0
    masks += 1 if case.get("key_nulls") else 0
    inputs = n * sum(WIDTH[t] for t, _ in spec) + masks * n / 8
    if case["path"] == "general":
        groups = case["groups"]
        key_in, key_out = 4 + 4 + 18, 4 + 4 + 18
    else:
        groups = case["card"] * -math.expm1(-n / case["card"])
        key_in = key_out = WIDTH[case["key"]]
    if case["path"] == "partition":
        return {"bytes": 2 * (inputs + n * key_in), "flops": 0}
    out = groups * (key_out + sum(WIDTH[_result_type(t, a)] for t, aggs in spec for a in aggs))
    return {"bytes": inputs + n * key_in + out, "flops": 0}


def tolerance(case):
    if case["path"] == "partition":
        return "exact"
    spec = _spec(case)
    if any(t == "float32" and set(aggs) & {"sum", "mean", "var"} for t, aggs in spec):
        # float32 sums in another order (measured up to 4e-7 between two runs and against 64 bits)
        return {"rel": 2e-6, "max": 1e-4, "differ": 0.0}
    if any(t == "float64" and set(aggs) & {"sum", "mean", "var", "median"} for t, aggs in spec) or \
            any(set(aggs) & {"mean", "var"} for _, aggs in spec):
        # float64 sums in another order; variances from sums where that is within 1e-11
        return {"rel": 1e-11, "max": 1e-9, "differ": 0.0}
    return "exact"


# -- the same in plain torch, 64 bits ------------------------------------------


def _exact_stats(ids, groups, v, ok, aggs, vtype):
    """Per id: the statistics of its valid values (float64 / int64)."""
    if ok is not None:
        ids, v = ids[ok], v[ok]
    dev = v.device
    whole = vtype.startswith("int")
    x = v.to(torch.int64) if whole else v.double()
    cnt = torch.zeros(groups, dtype=torch.int64, device=dev).index_add_(0, ids, torch.ones_like(ids))
    total = torch.zeros(groups, dtype=x.dtype, device=dev).index_add_(0, ids, x)
    nan = torch.tensor(math.nan, dtype=torch.float64, device=dev)
    out = []
    for a in aggs:
        if a == "count":
            r = cnt
        elif a == "sum":
            r = total if whole or ok is None else torch.where(cnt > 0, total, nan)
        elif a in ("min", "max"):
            r = torch.zeros(groups, dtype=x.dtype, device=dev).scatter_reduce_(
                0, ids, x, "amin" if a == "min" else "amax", include_self=False)
            if not whole and ok is not None:
                r = torch.where(cnt > 0, r, nan)
        elif a == "mean":
            r = total.double() / cnt
        elif a == "var":
            d = x.double() - (total.double() / cnt)[ids]
            r = torch.zeros(groups, dtype=torch.float64, device=dev).index_add_(0, ids, d * d) / (cnt - 1)
            r = torch.where(cnt > 1, r, nan)
        elif a == "nunique":
            u = torch.unique(torch.stack([ids, x]), dim=1)[0] if not whole else \
                torch.unique(ids * (2 * 10**9 + 2) + x + 10**9) // (2 * 10**9 + 2)
            r = torch.zeros(groups, dtype=torch.int64, device=dev).index_add_(0, u, torch.ones_like(u))
        else:  # median
            o = torch.sort(x.double(), stable=True).indices
            o = o[torch.sort(ids[o], stable=True).indices]
            xs, first = x.double()[o], torch.cumsum(cnt, 0) - cnt
            last = xs.numel() - 1
            r = (xs[(first + (cnt - 1).clamp(min=0) // 2).clamp(max=last)] + xs[(first + cnt // 2).clamp(max=last)]) / 2
            r = torch.where(cnt > 0, r, nan)
        out.append(r)
    return out, cnt


def exact(case, seed):
    if case["path"] == "partition":
        return None  # rows are moved, not computed
    raw = _inputs(case, seed)
    spec = _spec(case)
    if case["path"] == "batch":
        cols = [[[] for _ in aggs] for _, aggs in spec]
        for (k, vs), (_, c) in zip(raw["instances"], _batch_shapes(case)):
            for r, ((t, aggs), (v, ok)) in enumerate(zip(spec, vs)):
                for a, x in enumerate(_exact_stats(k.to(torch.int64), c, v, ok, aggs, t)[0]):
                    cols[r][a].append(x)
        return [[torch.cat(p) for p in r] for r in cols]
    n = case["rows"]
    if case["path"] == "general":
        code = (raw["k1"].to(torch.int64) - 1) * case["pool"] + raw["sid"]
        uniq, ids = torch.unique(code, return_inverse=True)
        groups = uniq.numel()
        first = torch.full((groups,), n, dtype=torch.int64, device=code.device).scatter_reduce_(
            0, ids, torch.arange(n, device=code.device), "amin")
        order = torch.argsort(first)
        lens, start, chars = raw["pool"]
        sid = uniq[order] % case["pool"]
        ln = lens[sid]
        ends = torch.cumsum(ln, 0)
        src = torch.repeat_interleave(start[sid] - (ends - ln), ln) + torch.arange(int(ends[-1]), device=ln.device)
        res = [[x[order] for x in _exact_stats(ids, groups, v, ok, aggs, t)[0]]
               for (t, aggs), (v, ok) in zip(spec, raw["values"])]
        return {"k1": uniq[order] // case["pool"] + 1, "lengths": ln, "chars": chars[src], "results": res + [[first[order]]]}
    key = raw["key"].to(torch.int64)
    if case["path"] == "sorted":
        uniq, ids = torch.unique_consecutive(key, return_inverse=True)
        return {"keys": uniq, "results": [_exact_stats(ids, uniq.numel(), v, ok, aggs, t)[0]
                                          for (t, aggs), (v, ok) in zip(spec, raw["values"])]}
    groups = case["card"] + 1
    kv = raw["key_valid"]
    if kv is not None:
        key = torch.where(kv, key, case["card"]) if case.get("include") else key[kv]
    seen = torch.zeros(groups, dtype=torch.bool, device=key.device)
    seen[key] = True
    out = []
    for (t, aggs), (v, ok) in zip(spec, raw["values"]):
        if kv is not None and not case.get("include"):
            v, ok = v[kv], None if ok is None else ok[kv]
        got, _ = _exact_stats(key, groups, v, ok, aggs, t)
        out.append([torch.where(seen, x, 0) for x in got])  # ids without rows stay zero
    return out
