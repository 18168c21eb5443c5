"""The work that users have this framework do, as cases of measurable size.

Six kinds, each through the package's public entry points over columns that are already in HBM:

  sort     one column: the stable argsort alone, the argsort with the gather of a payload column (an
           ORDER BY of two columns), or the sorted values
  table    a whole table through the plan engine, ordered by one key or by two
  group    a hash group-by over one or two key columns: the keys, then one aggregate after another
  dense    a group-by over integer keys in [0, key_count), as a dictionary-encoded column has them
  unique   the keep-first distinct rows over two columns, and both columns taken at them
  batched  a plan over record batches stored back to back: every batch sorted and grouped in one run

Row counts go from a request of a thousand rows to columns of fifty million.
"""
from __future__ import annotations

import json
import math

import numpy as np
import torch

import arrowmetal_amd as am

DEV = "cuda"
WIDTH = {"i64": 8, "f64": 8, "i32": 4, "f32": 4, "i16": 2}

# ------------------------------------------------------------------ the cases


def sort_case(n, dtype, out, nulls=0.0, descending=False, nulls_first=False, order="ieee", spread="wide", **kw):
    return dict(kind="sort", n=n, dtype=dtype, out=out, nulls=nulls, descending=descending, nulls_first=nulls_first,
                order=order, spread=spread, **kw)


def group_case(n, keys, support, aggs, zipf=0.0, nulls=0.0, **kw):
    return dict(kind="group", n=n, keys=keys, support=support, aggs=aggs, zipf=zipf, nulls=nulls, **kw)


def dense_case(n, key_count, nulls):
    return dict(kind="dense", n=n, key_count=min(key_count, n // 4), nulls=nulls)


def listed():
    return [
        # A request over a small result: latency and launches count.
        sort_case(1_000, "i64", "indices", name="argsort_1k"),
        # The plain argsort of a million full-range keys.
        sort_case(1_000_000, "i64", "indices", name="argsort_1m"),
        # ORDER BY over the large table: descending, nulls last, with the gather of its payload column.
        sort_case(50_000_000, "i64", "take", nulls=0.02, descending=True, name="order_by_50m"),
        # The same in float64 with NaN and -0.0, under the total order.
        sort_case(50_000_000, "f64", "take", nulls=0.02, descending=True, order="total", name="order_by_f64_50m"),
        # A 32-bit column (dates, ids) of an odd length with nulls first: its sorted values.
        sort_case(6_000_011, "i32", "values", nulls=0.1, nulls_first=True, name="sort_i32_6m"),
        # A table ordered by a low-cardinality key, then by an amount (a report).
        dict(kind="table", n=4_000_037, by=2, nulls=0.02, columns=4, name="table_two_keys_4m"),
        # A dashboard's group-by over a small table.
        group_case(20_011, "i64", 300, "int", name="group_20k"),
        # The skewed group-by with many groups: integer sum and counts.
        group_case(50_000_000, "i64", 100_000, "int", zipf=1.1, name="group_zipf_50m"),
        # Few groups, float64 values: min, max and the correctly rounded sum.
        group_case(50_000_000, "i64", 200, "float", name="group_float_50m"),
        # Two narrower key columns with nulls, 32-bit values: sum, mean, min, max and count.
        group_case(3_000_017, "i32,i16", 40_000, "stats", zipf=1.1, nulls=0.02, name="group_two_keys_3m"),
        # DISTINCT over two columns, as a served request has it.
        dict(kind="unique", n=10_000_000, a=1_000_000, b=1_000, name="unique_10m"),
        # Record batches of uneven length, each sorted and grouped, in one run.
        dict(kind="batched", batches=512, median=20_000, cap=4_000_000, layout=7, keys=1_000, name="batched_512"),
    ]


def _log(rng, lo, hi):
    """A whole number spread over [lo, hi] on a logarithmic scale (mostly odd or ragged)."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sort", "sort", "group", "group", "table", "dense", "unique", "batched"])
    if kind == "sort":
        dtype = rng.choice(["i64", "f64", "i32", "f32"])
        out = rng.choice(["indices", "take", "values"])
        order = rng.choice(["ieee", "total", "nan_largest"]) if dtype[0] == "f" and out != "values" else "ieee"
        return sort_case(_log(rng, 1_000, 50_000_000), dtype, out, nulls=rng.choice([0.0, 0.02, 0.2]),
                         descending=rng.random() < 0.5, nulls_first=rng.random() < 0.3, order=order,
                         spread=rng.choice(["wide", "wide", "small"]))
    if kind == "group":
        keys = rng.choice(["i64", "i64", "i32", "i32,i16"])
        n = _log(rng, 1_000, 32_000_000 if "," not in keys else 4_000_000)
        support = min(_log(rng, 24, 1_000_000), n // 4)
        return group_case(n, keys, support, rng.choice(["int", "float", "stats"]), zipf=rng.choice([0.0, 1.1]),
                          nulls=rng.choice([0.0, 0.02]))
    if kind == "table":
        return dict(kind="table", n=_log(rng, 1_000, 8_000_000), by=rng.choice([1, 2]), nulls=rng.choice([0.0, 0.02]),
                    columns=rng.choice([2, 3, 4]))
    if kind == "dense":
        return dense_case(_log(rng, 1_000, 50_000_000), _log(rng, 8, 60_000), rng.choice([0.0, 0.02]))
    if kind == "unique":
        return dict(kind="unique", n=_log(rng, 1_000, 10_000_000), a=_log(rng, 100, 1_000_000), b=_log(rng, 10, 1_000))
    return dict(kind="batched", batches=_log(rng, 16, 512), median=_log(rng, 2_000, 20_000), cap=4_000_000,
                layout=rng.randrange(1 << 20), keys=_log(rng, 50, 1_000))


# ------------------------------------------------------------------ inputs


class Maker:
    """Seeded columns, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) * 1_000_003 + 17)

    def bits(self, n):
        """Full-range 64-bit integers."""
        return torch.randint(-2**63, 2**63 - 1, (n,), generator=self.g, device=DEV, dtype=torch.int64)

    def ints(self, n, lo, hi, dtype=torch.int64):
        return torch.randint(lo, hi, (n,), generator=self.g, device=DEV, dtype=dtype)

    def unit(self, n):
        return torch.rand(n, generator=self.g, device=DEV, dtype=torch.float64)

    def valid(self, n, nulls):
        return self.unit(n) >= nulls if nulls else None

    def ranks(self, n, support, zipf=0.0):
        """n numbers in [0, support), uniform or Zipf, each of them at least once, and where the first of each is."""
        if zipf:
            cdf = torch.arange(1, support + 1, device=DEV, dtype=torch.float64).pow(-zipf).cumsum(0)
            r = torch.searchsorted(cdf / cdf[-1], self.unit(n)).clamp_(max=support - 1)
        else:
            r = self.ints(n, 0, support)
        at = torch.randperm(n, generator=self.g, device=DEV)[:support]
        r[at] = torch.arange(support, device=DEV)
        return r, at


def column(values, valid=None):
    """The column as the framework holds it: imported once, resident in HBM (zeros under its nulls)."""
    if valid is not None:
        values = torch.where(valid, values, 0)
    return am.MetalArray.from_numpy(values.cpu().numpy(), None if valid is None else valid.cpu().numpy())


def sort_keys(mk, case):
    n, dtype = case["n"], case["dtype"]
    small = case["spread"] == "small"   # few distinct values: states, days, quantities
    if dtype == "i64":
        return mk.ints(n, 0, 5_000) if small else mk.bits(n) >> 1
    if dtype == "i32":
        return mk.ints(n, 0, 5_000, torch.int32) if small else mk.ints(n, -2**31, 2**31 - 1, torch.int32)
    x = mk.ints(n, 0, 10_000).double() / 100 if small else mk.unit(n) * 2e6 - 1e6
    if case["out"] != "values":
        odd = mk.unit(n)
        x[odd < 0.001] = math.nan
        x[(odd >= 0.001) & (odd < 0.002)] = -0.0
    return x if dtype == "f64" else x.float()


def batch_offsets(case):
    """Lognormal batch lengths; the layout is the plan's, so it belongs to the case."""
    z = np.random.default_rng(case["layout"]).standard_normal(case["batches"])
    lens = np.minimum(np.exp(math.log(case["median"]) + 1.78 * z), case["cap"]).astype(np.int64)
    total = np.cumsum(lens)
    lens = lens[: max(1, int(np.searchsorted(total, 60_000_000)))]
    return np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)


def table_columns(mk, case):
    """Column name -> (values, validity), in the table's order."""
    n = case["n"]
    cols = {"region": (mk.ints(n, 0, 200, torch.int32), mk.valid(n, case["nulls"])),
            "amount": (mk.unit(n) * 1e6, mk.valid(n, case["nulls"])),
            "id": (mk.bits(n), None),
            "qty": (mk.ints(n, 0, 1000, torch.int32), None)}
    return {k: cols[k] for k in list(cols)[: case["columns"]]}


def present(valid, at):
    """Validity with no null at the given rows (every group has a value)."""
    if valid is not None:
        valid[at] = True
    return valid


def group_columns(mk, case):
    """(key columns, validity of each, {value name: (values, validity)})."""
    n, support = case["n"], case["support"]
    r, at = mk.ranks(n, support, case["zipf"])
    if case["keys"] == "i64":
        keys = [mk.bits(support)[r]]
    elif case["keys"] == "i32":
        keys = [(r * 3 + 1_000_000).int()]
    else:
        keys = [(r // 12).int(), (r % 12).short()]
    # A key that is missing is one group more: of one column, or of every value of the other.
    missing = [r == 7] if len(keys) == 1 else [r // 12 == 5, r % 12 == 9]
    valid = [~m if case["nulls"] else None for m in missing]
    if case["aggs"] == "int":
        values = (mk.ints(n, -10**9, 10**9 + 1), None)
    elif case["aggs"] == "float":
        values = (mk.unit(n) * 2e6 - 1e6, None)
    else:
        values = (mk.ints(n, -10**6, 10**6, torch.int32), present(mk.valid(n, case["nulls"]), at))
    return keys, valid, values


AGGS = {"int": ("sum", "count_all", "count"), "float": ("min", "max", "sum"),
        "stats": ("sum", "mean", "min", "max", "count")}


def prepare(case, seed):
    mk, kind = Maker(seed), case["kind"]
    if kind == "sort":
        n = case["n"]
        keys = column(sort_keys(mk, case), mk.valid(n, case["nulls"]))
        return case, keys, column(mk.unit(n) * 2e6 - 1e6) if case["out"] == "take" else None
    if kind == "table":
        src = am.PlanSource("t", {k: column(*v) for k, v in table_columns(mk, case).items()})
        by = [["region", False], ["amount", True]] if case["by"] == 2 else [["amount", True]]
        return case, src, json.dumps({"op": "sort", "by": by, "input": {"op": "scan", "source": "t"}})
    if kind == "group":
        keys, valid, values = group_columns(mk, case)
        return case, [column(k, v) for k, v in zip(keys, valid)], column(*values)
    if kind == "dense":
        keys, values = dense_columns(mk, case)
        return case, column(*keys), column(*values)
    if kind == "unique":
        return case, [column(c) for c in unique_columns(mk, case)]
    offs = batch_offsets(case)
    n = int(offs[-1])
    r = mk.ints(n, 0, case["keys"])
    lens = torch.from_numpy(np.diff(offs)).to(DEV)
    pos = torch.arange(n, device=DEV) - torch.from_numpy(offs[:-1]).to(DEV).repeat_interleave(lens)
    r = torch.where(pos < case["keys"], (pos * 7919 + seed) % case["keys"], r)   # every key in every batch
    cols = column(mk.bits(n)), column(mk.bits(case["keys"])[r]), column(mk.ints(n, -10**9, 10**9 + 1))
    plan = am.Batched(offs)
    plan.tune(*cols)
    return case, plan, cols


def dense_columns(mk, case):
    n = case["n"]
    r, at = mk.ranks(n, case["key_count"])
    return (r.int(), None), (mk.ints(n, -10**6, 10**6, torch.int32), present(mk.valid(n, case["nulls"]), at))


def distinct_pairs(case):
    d = case["a"] * case["b"]
    return max(1, int(-d * math.expm1(-case["n"] / d)))   # as many as n uniform pairs hold


def unique_columns(mk, case):
    d, count = case["a"] * case["b"], distinct_pairs(case)
    step = int(mk.ints(1, d // 3, d)) | 1
    while math.gcd(step, d) > 1:
        step += 2
    code = torch.arange(count, device=DEV).mul_(step).remainder_(d)   # distinct, spread over all pairs
    code = code[mk.ranks(case["n"], count)[0]]
    return code // case["b"], code % case["b"]


# ------------------------------------------------------------------ one pass

_TYPES = {"c": "|i1", "C": "|u1", "s": "<i2", "S": "<i2", "i": "<i4", "I": "<i4", "l": "<i8", "L": "<i8", "f": "<f4", "g": "<f8"}


class _View:
    """A device buffer of a result, for torch to look at where it lies."""

    def __init__(self, owner, ptr, n, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2}


def tensors(a):
    """A result array as the tensors of its values and, where it has nulls, of its validity bitmap."""
    values, validity, offset, n, nulls, _ = a.device_buffers()
    if n == 0:
        return []
    t = [torch.as_tensor(_View(a, values, offset + n, _TYPES[a.format]), device=DEV)[offset:]]
    if validity and nulls:
        t.append(torch.as_tensor(_View(a, validity, (offset + n + 7) // 8, "|u1"), device=DEV))
    return t


def run(state):
    case, kind = state[0], state[0]["kind"]
    if kind == "sort":
        keys, payload = state[1:]
        opts = (case["descending"], "at_start" if case["nulls_first"] else "at_end", case["order"])
        if case["out"] == "values":
            return [tensors(keys.sort(*opts))]
        idx = keys.argsort(*opts)
        return [tensors(idx)] + ([tensors(payload.take(idx))] if payload is not None else [])
    if kind == "table":
        return [tensors(c) for c in am.plan_run(state[2], [state[1]]).values()]
    if kind == "group":
        g = am.group_by(state[1])
        out = g.key_arrays()
        for name in AGGS[case["aggs"]]:
            out.append(g.count_all() if name == "count_all" else getattr(g, name)(state[2]))
        return [tensors(a) for a in out]
    if kind == "dense":
        g = state[1].group_by(case["key_count"])
        v = state[2]
        return [tensors(a) for a in (g.count(), g.sum(v), g.mean(v), g.min(v), g.max(v))]
    if kind == "unique":
        rows = am.unique_rows(state[1])
        return [tensors(rows)] + [tensors(c.take(rows)) for c in state[1]]
    plan, cols = state[1:]
    plan.run(*cols)
    return [tensors(plan.result(name)) for name in ("indices", "keys", "sums", "counts", "group_offsets")]


# ------------------------------------------------------------------ what a pass cannot do without


def work(case):
    """Each input read once, each output written once; these paths move and compare, they multiply nothing."""
    kind, n = case["kind"], case.get("n", 0)
    bitmap = n / 8 if case.get("nulls") else 0
    if kind == "sort":
        w = WIDTH[case["dtype"]]
        out = {"indices": 4, "take": 4 + 16, "values": w}[case["out"]]
        b = n * (w + out) + bitmap * (2 if case["out"] == "values" else 1)
    elif kind == "table":
        widths = [4, 8, 8, 4][: case["columns"]]
        b = 2 * n * sum(widths) + 4 * bitmap
    elif kind == "group":
        widths = [WIDTH[k] for k in case["keys"].split(",")]
        v = 4 if case["aggs"] == "stats" else 8
        b = n * (sum(widths) + v) + bitmap * (len(widths) + (case["aggs"] == "stats"))
        b += case["support"] * (sum(widths) + 8 * len(AGGS[case["aggs"]]))
    elif kind == "dense":
        b = 8 * n + bitmap + case["key_count"] * 32
    elif kind == "unique":
        b = 16 * n + 20 * distinct_pairs(case)
    else:
        n = int(batch_offsets(case)[-1])
        b = 28 * n + 24 * case["batches"] * case["keys"]
    return {"bytes": float(b), "flops": 0.0}


# ------------------------------------------------------------------ the computed numbers in 64 bits


def stable_order(keys, valid, descending, nulls_first, order="ieee"):
    """Row numbers of the stable sort: values, then NaN (the ieee order), nulls at one end."""
    n = len(keys)
    if keys.is_floating_point():
        b = (keys.double() if order == "total" else torch.where(keys == 0, 0.0, keys.double())).view(torch.int64)
        k = torch.where(b < 0, b ^ 0x7FFFFFFFFFFFFFFF, b)
        nan = keys.isnan() if order != "total" else torch.zeros(n, dtype=torch.bool, device=DEV)
        if order == "nan_largest":
            k, nan = torch.where(nan, 2**63 - 1, k), torch.zeros_like(nan)
    else:
        k, nan = keys.long(), torch.zeros(n, dtype=torch.bool, device=DEV)
    k = ~k if descending else k
    null = torch.zeros_like(nan) if valid is None else ~valid
    rank = torch.where(null, -1 if nulls_first else 2, nan.long())
    o = torch.sort(torch.where(rank == 0, k, 0), stable=True).indices
    return o[torch.sort(rank[o], stable=True).indices]


def exact(case, seed):
    mk, kind = Maker(seed), case["kind"]
    if kind == "sort" and case["out"] == "take":
        n = case["n"]
        keys, valid = sort_keys(mk, case), mk.valid(case["n"], case["nulls"])
        payload = mk.unit(n) * 2e6 - 1e6
        return [None, [payload[stable_order(keys, valid, case["descending"], case["nulls_first"], case["order"])]]]
    if kind == "table":
        cols = table_columns(mk, case)
        amount, valid = cols["amount"]
        o = stable_order(amount, valid, True, False)
        if case["by"] == 2:
            region, rv = cols["region"]
            o = o[stable_order(region[o], None if rv is None else rv[o], False, False)]
        amount = amount if valid is None else torch.where(valid, amount, 0.0)
        return [[amount[o]] if k == "amount" else None
                for k in cols]
    if kind == "group" and case["aggs"] != "int":
        keys, valid, (values, ok) = group_columns(mk, case)
        code = torch.zeros(case["n"], dtype=torch.int64, device=DEV)
        for k, v in zip(keys, valid):
            u, c = torch.unique(k, return_inverse=True)
            code = code * (len(u) + 1) + (c if v is None else torch.where(v, c, len(u)))
        u, ids = torch.unique(code, return_inverse=True)
        keep = slice(None) if ok is None else ok
        x, ids = values[keep].double(), ids[keep]
        total = torch.zeros(len(u), dtype=torch.float64, device=DEV).index_add_(0, ids, x)
        if case["aggs"] == "float":
            lo, hi = (torch.zeros_like(total).scatter_reduce_(0, ids, x, how, include_self=False) for how in ("amin", "amax"))
            return [None, [lo], [hi], [total]]
        count = torch.bincount(ids, minlength=len(u))
        return [None] * len(keys) + [None, [torch.where(count > 0, total / count, 0.0)], None, None, None]
    if kind == "dense":
        (keys, _), (values, ok) = dense_columns(mk, case)
        keep = slice(None) if ok is None else ok
        ids = keys.long()[keep]
        total = torch.zeros(case["key_count"], dtype=torch.float64, device=DEV).index_add_(0, ids, values[keep].double())
        count = torch.bincount(ids, minlength=case["key_count"])
        return [None, None, [torch.where(count > 0, total / count, 0.0)], None, None]
    return None
