"""The work that programs give this library, as cases that can be timed and compared.

Every case is one call (or one short sequence of calls) of a public operator over columns that are
resident in device memory, as a query engine issues it: torch owns the columns, the operators of
craton_bolt_amd read and write them through plain device pointers, and the results stay on the device
where the operator leaves them there (scalars and served rows come back to the host).  A case is a dict of
plain values; `kind` names the operator:

  aggregate  SELECT SUM, COUNT, MIN, MAX, AVG, STDDEV ... WHERE      bolt_aggregate
  expr       fused WHERE + SUM(a * b) (the TPC-H Q6 shape)            bolt_aggregate_expr
  filter     WHERE as stream compaction of several columns            bolt_filter_compact
  groupby    GROUP BY one or two keys, groups in key order            bolt_groupby
  joinagg    hash build + fused probe and aggregates                  bolt_join_build, bolt_join_probe_aggregate
  join       equi-join to row pairs, then a take of an attribute      bolt_join, bolt_take
  sort       radix sort of (int64 key, row id) pairs                  bolt_sort_pairs_i64
  orderby    ORDER BY two columns with NULLs                          bolt_sort_indices
  topk       ORDER BY ... LIMIT ... OFFSET                            bolt_sort_limit
  serve      a mix of star queries through the request loop           Server
"""
from __future__ import annotations

import ctypes as C
import math

import torch

from craton_bolt_amd import _native as N
from craton_bolt_amd.device import DeviceBuffer, DeviceColumn
from craton_bolt_amd.ops import Program, Server, Term, scalar_value

DEV = "cuda"


# ---- the cases ---------------------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # an interactive dashboard tile over a small table: the smallest call, latency and launches count
        dict(name="aggregate_10k", kind="aggregate", rows=10_007, nulls=0.1, keep=0.7),
        # a revenue query over a large fact table, nothing materialised
        dict(name="expr_q6_150m", kind="expr", rows=150_000_001),
        # WHERE over a table with mixed widths and NULLs, the survivors kept for the next operator
        dict(name="filter_30m", kind="filter", rows=30_000_003, keep=0.3, nulls=0.05),
        # a report over a table of ordinary size: few groups, integer sums
        dict(name="groupby_1m", kind="groupby", rows=1_000_000, groups=1_000, keys="i32", skew=0.0, values="i64",
             nulls=0.0),
        # the h2o.ai groupby shape: 10M rows, 10,000 groups of two keys, float sums
        dict(name="groupby_10m_pair", kind="groupby", rows=10_000_000, groups=10_000, keys="pair", skew=0.0,
             values="f64", nulls=0.0),
        # a skewed key over a large table: millions of groups, a long tail
        dict(name="groupby_zipf_200m", kind="groupby", rows=200_000_000, groups=10_000_000, keys="i64", skew=1.1,
             values="f64", nulls=0.0),
        # the headline join: filter + join + aggregates, half of the probe rows hit
        dict(name="joinagg_16m_256m", kind="joinagg", build=16 << 20, probe=256 << 20, keys="sparse", hit=0.5),
        # fact to dimension with the dimension's attribute fetched; unmatched fact rows are kept
        dict(name="join_left_20m", kind="join", left=20_000_000, right=500_000, how="left", keys="dense", dtype="i64",
             hit=0.9),
        # a whole-table sort by a 64-bit key
        dict(name="sort_256m", kind="sort", rows=256 << 20, descending=False, bits=64),
        # a report's ORDER BY: a date with NULLs, then an amount, descending
        dict(name="orderby_5m", kind="orderby", rows=5_000_011, nulls=0.05, days=2500),
        # the newest / largest rows of a large table
        dict(name="topk_256m", kind="topk", rows=256 << 20, dtype="i64", limit=100, offset=0),
        # dashboards served together over one star schema
        dict(name="serve_60m", kind="serve", rows=60_000_000, queries=12, slots=8),
    ]


def _spread(rng, lo: int, hi: int) -> int:
    """A size between lo and hi, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["aggregate", "expr", "filter", "groupby", "groupby", "groupby", "joinagg", "join", "sort",
                       "orderby", "topk", "serve"])
    if kind == "aggregate":
        return dict(kind=kind, rows=_spread(rng, 1_000, 100_000_000), nulls=rng.choice([0.0, 0.1]),
                    keep=rng.choice([0.1, 0.7, 1.0]))
    if kind == "expr":
        return dict(kind=kind, rows=_spread(rng, 10_000, 150_000_000))
    if kind == "filter":
        return dict(kind=kind, rows=_spread(rng, 10_000, 60_000_000), keep=round(rng.uniform(0.02, 0.95), 2),
                    nulls=rng.choice([0.0, 0.05]))
    if kind == "groupby":
        rows = _spread(rng, 10_000, 100_000_000)
        return dict(kind=kind, rows=rows, groups=_spread(rng, 10, max(20, min(10_000_000, rows // 2))),
                    keys=rng.choice(["i32", "i64", "pair"]), skew=rng.choice([0.0, 1.1]),
                    values=rng.choice(["i64", "f64"]), nulls=rng.choice([0.0, 0.0, 0.05]))
    if kind == "joinagg":
        build = _spread(rng, 1_000, 16 << 20)
        return dict(kind=kind, build=build, probe=_spread(rng, 100_000, 256 << 20), keys=rng.choice(["sparse", "dense"]),
                    hit=round(rng.uniform(0.1, 1.0), 2))
    if kind == "join":
        return dict(kind=kind, left=_spread(rng, 50_000, 20_000_000), right=_spread(rng, 1_000, 5_000_000),
                    how=rng.choice(["inner", "left", "full"]), keys=rng.choice(["sparse", "dense"]),
                    dtype=rng.choice(["i64", "i32"]), hit=round(rng.uniform(0.7, 1.0), 2))
    if kind == "sort":
        return dict(kind=kind, rows=_spread(rng, 10_000, 256 << 20), descending=rng.choice([False, True]),
                    bits=rng.choice([64, 64, 40, 24]))
    if kind == "orderby":
        return dict(kind=kind, rows=_spread(rng, 10_000, 30_000_000), nulls=rng.choice([0.0, 0.05]),
                    days=rng.choice([30, 2500]))
    if kind == "topk":
        return dict(kind=kind, rows=_spread(rng, 100_000, 256 << 20), dtype=rng.choice(["i64", "i32", "f64"]),
                    limit=rng.choice([10, 100, 1000]), offset=rng.choice([0, 0, 200]))
    return dict(kind=kind, rows=_spread(rng, 5_000_000, 60_000_000), queries=rng.choice([4, 8, 12]),
                slots=rng.choice([4, 8]))


# ---- inputs ------------------------------------------------------------------------------------

class _Rng:
    """Seeded device-side draws."""

    def __init__(self, seed: int):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def ints(self, n: int, lo: int, hi: int, dtype=torch.int64) -> torch.Tensor:
        return torch.randint(lo, hi, (n,), generator=self.g, device=DEV, dtype=dtype)

    def unit(self, n: int) -> torch.Tensor:
        return torch.rand(n, generator=self.g, device=DEV, dtype=torch.float64)

    def perm(self, n: int) -> torch.Tensor:
        return torch.randperm(n, generator=self.g, device=DEV)

    def valid(self, n: int, nulls: float) -> torch.Tensor | None:
        return self.unit(n) >= nulls if nulls > 0 else None


def _scatter64(x: torch.Tensor) -> torch.Tensor:
    """A bijection of the 64-bit integers: surrogate ids that use their whole range."""
    x = (x ^ (x >> 29)) * -0x40A7B892E31B1A47
    return x ^ ((x >> 32) & 0xFFFFFFFF)


def _scatter32(x: torch.Tensor) -> torch.Tensor:
    """A bijection of the 32-bit integers, as int32."""
    return (x * 0x9E3779B1 + 0x7F4A7C15).to(torch.int32)


def _zipf(r: _Rng, n: int, ranks: int, s: float) -> torch.Tensor:
    """Ranks 0 .. ranks - 1 with P(rank k) about (k + 1)^-s, by inversion of the continuous law."""
    u = r.unit(n)
    top = float(ranks + 1) ** (1.0 - s) - 1.0
    k = u.mul_(top).add_(1.0).pow_(1.0 / (1.0 - s))
    return k.to(torch.int64).sub_(1).clamp_(0, ranks - 1)


def _bitmap(valid: torch.Tensor) -> torch.Tensor:
    """Arrow LSB-first validity bitmap, padded to whole 8-byte words."""
    n = valid.numel()
    b = torch.zeros((n + 63) // 64 * 64, dtype=torch.uint8, device=DEV)
    b[:n] = valid
    w = torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], dtype=torch.uint8, device=DEV)
    return (b.view(-1, 8) * w).sum(1, dtype=torch.uint8)


def _column(values: torch.Tensor, dtype: int, bits: torch.Tensor | None = None, scale: int = 0,
            length: int | None = None) -> N.BoltColumn:
    return N.BoltColumn(values.data_ptr(), bits.data_ptr() if bits is not None else None,
                        values.shape[0] if length is None else length, dtype, scale)


def _columns(*cols: N.BoltColumn):
    return (N.BoltColumn * len(cols))(*cols)


def _agg_list(*aggs: tuple[int, int]):
    return (N.BoltAgg * len(aggs))(*[N.BoltAgg(op, col) for op, col in aggs])


def _filter(*terms: N.BoltPredTerm):
    arr = (N.BoltPredTerm * len(terms))(*terms)
    return N.BoltFilter(arr, len(terms)), arr


def _cents(r: _Rng, n: int) -> torch.Tensor:
    """Decimal128(12, 2) amounts as (n, 2) little-endian words."""
    lo = r.ints(n, -50_000, 1_000_000)
    return torch.stack([lo, lo >> 63], 1)


# ---- kinds: inputs, the pass, and the same answer in 64 bits -------------------------------------

class Aggregate:
    AGGS = [(N.SUM, 0), (N.COUNT, 1), (N.SUM, 1), (N.MIN, 2), (N.MAX, 2), (N.AVG, 2), (N.STDDEV_SAMP, 2), (N.SUM, 3)]

    def __init__(self, c, seed):
        r, n = _Rng(seed), c["rows"]
        self.amount = r.ints(n, -1_000_000, 1_000_000)
        self.count = r.ints(n, 0, 1000, torch.int32)
        self.valid = r.valid(n, c["nulls"])
        self.price = torch.exp(r.unit(n) * 4.0)
        self.money = _cents(r, n)
        self.pick = r.ints(n, 0, 1000, torch.int32)
        self.cut = int(c["keep"] * 1000)
        self.bits = _bitmap(self.valid) if self.valid is not None else None
        self.cols = _columns(_column(self.amount, N.I64), _column(self.count, N.I32, self.bits),
                             _column(self.price, N.F64), _column(self.money, N.DEC128, scale=2),
                             _column(self.pick, N.I32))
        self.aggs = _agg_list(*self.AGGS)
        self.filter = _filter(N.BoltPredTerm(4, N.LT, self.cut, 0.0, 0))
        self.res = (N.BoltScalar * len(self.AGGS))()

    def run(self):
        N.check(N.lib().bolt_aggregate(None, self.cols, 5, self.aggs, len(self.AGGS), C.byref(self.filter[0]),
                                       self.res), "bolt_aggregate")
        return [scalar_value(x) for x in self.res]

    def exact(self):
        p = self.price[self.pick < self.cut]
        return [None, None, None, float(p.min()), float(p.max()), float(p.mean()), float(p.std()), None]


class Expr:
    def __init__(self, c, seed):
        r, n = _Rng(seed), c["rows"]
        self.price = r.unit(n).mul_(999.0).add_(1.0)
        self.disc = r.ints(n, 0, 11, torch.int32).to(torch.float64).div_(100.0)
        self.qty = r.ints(n, 1, 50, torch.int32)
        p = Program()
        pr, d, q = p.load(0, N.F64), p.load(1, N.F64), p.load(2, N.I32)
        p.store(p.binary("*", pr, d, N.F64), 0)
        c1 = p.binary("<", q, p.const(24, N.I32), N.I32)
        c2 = p.binary(">=", d, p.const(0.05, N.F64), N.F64)
        c3 = p.binary("<=", d, p.const(0.07, N.F64), N.F64)
        c4 = p.binary(">", p.binary("+", pr, p.cast(q, N.F64), N.F64), p.const(100.0, N.F64), N.F64)
        p.store(p.binary("and", p.binary("and", c1, c2, N.BOOL), p.binary("and", c3, c4, N.BOOL), N.BOOL), 1)
        self.prog, self.n_ops = p.array(N.BoltExprOp), len(p.ops)
        self.cols = _columns(_column(self.price, N.F64), _column(self.disc, N.F64), _column(self.qty, N.I32))
        self.aggs = _agg_list((N.SUM, 0), (N.COUNT_STAR, 0))
        self.res = (N.BoltScalar * 2)()

    def run(self):
        N.check(N.lib().bolt_aggregate_expr(None, self.cols, 3, self.prog, self.n_ops, 2, 1, self.aggs, 2, self.res),
                "bolt_aggregate_expr")
        return [scalar_value(x) for x in self.res]

    def exact(self):
        k = (self.qty < 24) & (self.disc >= 0.05) & (self.disc <= 0.07) & (self.price + self.qty > 100.0)
        return [float((self.price * self.disc)[k].sum()), None]


class Filter:
    def __init__(self, c, seed):
        r, n = _Rng(seed), c["rows"]
        self.ids = r.ints(n, -(1 << 62), 1 << 62)
        self.price = torch.exp(r.unit(n) * 4.0)
        self.qty = r.ints(n, 0, 1000, torch.int32)
        self.valid = r.valid(n, c["nulls"])
        self.bits = _bitmap(self.valid) if self.valid is not None else None
        self.cols = _columns(_column(self.ids, N.I64), _column(self.price, N.F64, self.bits),
                             _column(self.qty, N.I32))
        self.out = [torch.zeros_like(x) for x in (self.ids, self.price, self.qty)]
        self.out_bits = torch.zeros_like(self.bits) if self.bits is not None else None
        self.outs = _columns(_column(self.out[0], N.I64), _column(self.out[1], N.F64, self.out_bits),
                             _column(self.out[2], N.I32))
        self.cut = int(round(c["keep"] * 1000))
        self.filter = _filter(N.BoltPredTerm(2, N.LT, self.cut, 0.0, 0))
        self.n = C.c_int64()

    def run(self):
        N.check(N.lib().bolt_filter_compact(None, self.cols, 3, C.byref(self.filter[0]), None, self.outs,
                                            C.byref(self.n)), "bolt_filter_compact")
        got = [self.n.value] + self.out
        return got + [self.out_bits] if self.out_bits is not None else got

    def exact(self):
        price = torch.zeros_like(self.price)
        kept = self.price[self.qty < self.cut]
        price[: kept.numel()] = kept
        return [None, None, price, None] + ([None] if self.bits is not None else [])


class GroupBy:
    def __init__(self, c, seed):
        r, n, g = _Rng(seed), c["rows"], c["groups"]
        ids = _zipf(r, n, g, c["skew"]) if c["skew"] else r.ints(n, 0, g)
        if c["keys"] == "i64":
            self.keys = [_scatter64(ids)]
            kcols = [_column(self.keys[0], N.I64)]
        elif c["keys"] == "i32":
            self.keys = [_scatter32(ids)]
            kcols = [_column(self.keys[0], N.I32)]
        else:  # two columns, the first of about the square root of the groups
            d = max(1, math.isqrt(g))
            self.keys = [(ids % d).to(torch.int32), (ids // d).to(torch.int32)]
            kcols = [_column(k, N.I32) for k in self.keys]
        del ids
        self.valid = r.valid(n, c["nulls"])
        self.bits = _bitmap(self.valid) if self.valid is not None else None
        if c["values"] == "i64":
            self.vals = [r.ints(n, 0, 1000)]
            vcols = [_column(self.vals[0], N.I64, self.bits)]
            self.ops = [(N.SUM, 0), (N.COUNT_STAR, 0), (N.MIN, 0), (N.MAX, 0)]
            self.types = [torch.int64] * 4
        else:
            self.vals = [r.unit(n).mul_(100.0), r.ints(n, 1, 16).to(torch.float64)]
            vcols = [_column(self.vals[0], N.F64, self.bits), _column(self.vals[1], N.F64)]
            self.ops = [(N.SUM, 0), (N.SUM, 1)]
            self.types = [torch.float64] * 2
            if g > 100_000:  # the long tail is counted, not summed twice
                self.vals, vcols = self.vals[:1], vcols[:1]
                self.ops, self.types = [(N.SUM, 0), (N.COUNT_STAR, 0)], [torch.float64, torch.int64]
        self.kcols, self.vcols, self.aggs = _columns(*kcols), _columns(*vcols), _agg_list(*self.ops)
        self.types = [k.dtype for k in self.keys] + self.types
        cap = min(g, n) + 1  # and the NULL group
        self.out = [torch.zeros(cap, dtype=t, device=DEV) for t in self.types]
        self.out_bits = [torch.zeros((cap + 63) // 64 * 8, dtype=torch.uint8, device=DEV) for _ in self.types]

    def run(self):
        """GROUP BY, the groups in key order, then the result table copied into the caller's columns."""
        L, t, rows, col = N.lib(), C.c_void_p(), C.c_int64(), N.BoltColumn()
        N.check(L.bolt_groupby(None, self.kcols, len(self.keys), self.vcols, len(self.vals), self.aggs, len(self.ops),
                               None, N.GROUPBY_SORTED, C.byref(t)), "bolt_groupby")
        N.check(L.bolt_table_num_rows(t, C.byref(rows)))
        k, valid = rows.value, []
        for i, x in enumerate(self.out):
            N.check(L.bolt_table_column(t, i, C.byref(col)))
            N.check_rt(L.bolt_hip_memcpy_dtod_async(x.data_ptr(), col.data, k * x.element_size(), None), "dtod")
            if col.validity:
                b = self.out_bits[i]
                N.check_rt(L.bolt_hip_memcpy_dtod_async(b.data_ptr(), col.validity, (k + 7) // 8, None), "dtod")
                valid.append(b)
        L.bolt_table_release(t)
        return {"groups": k, "columns": self.out, "valid": valid}

    def exact(self):
        if all(t != torch.float64 for t in self.types):
            return None
        k = self.keys[0].to(torch.int64)
        if len(self.keys) == 2:
            k = (k << 32) | self.keys[1].to(torch.int64)
        k, order = torch.sort(k)
        count = torch.unique_consecutive(k, return_counts=True)[1]
        got = [None] * len(self.keys)
        for op, col in self.ops:
            if op != N.SUM:
                got.append(None)
                continue
            v = self.vals[col]
            if col == 0 and self.valid is not None:
                v = torch.where(self.valid, v, 0.0)
            x = torch.zeros_like(self.out[len(got)])
            x[: count.numel()] = torch.segment_reduce(v[order], "sum", lengths=count)
            got.append(x)
        return {"columns": got}


def _join_keys(r: _Rng, c: dict, n_dim: int, n_fact: int):
    """Unique dimension keys in shuffled order, and foreign keys of which a share `hit` is among them."""
    dim = r.perm(n_dim)
    fact = r.ints(n_fact, 0, n_dim)
    fact += (r.unit(n_fact) >= c["hit"]) * n_dim
    if c["keys"] == "sparse":
        if c.get("dtype") == "i32":
            return _scatter32(dim), _scatter32(fact)
        return _scatter64(dim), _scatter64(fact)
    t = torch.int32 if c.get("dtype") == "i32" else torch.int64
    return dim.to(t), fact.to(t)


class JoinAgg:
    def __init__(self, c, seed):
        r = _Rng(seed)
        self.dim, self.fk = _join_keys(r, c, c["build"], c["probe"])
        self.attr = r.ints(c["build"], 0, 1_000_000, torch.int32)
        self.amount = r.unit(c["probe"]).mul_(100.0)
        self.bk, self.bc = _column(self.dim, N.I64), _column(self.attr, N.I32)
        self.cols = _columns(_column(self.fk, N.I64), _column(self.amount, N.F64))
        self.filter = _filter(N.BoltPredTerm(1, N.GT, 0, 10.0, 0))
        self.aggs = _agg_list((N.SUM, N.JOIN_CARRY), (N.SUM, 1), (N.COUNT_STAR, 0))
        self.res = (N.BoltScalar * 3)()

    def run(self):
        L, t = N.lib(), C.c_void_p()
        N.check(L.bolt_join_build(None, C.byref(self.bk), C.byref(self.bc), C.byref(t)), "bolt_join_build")
        N.check(L.bolt_join_probe_aggregate(None, t, self.cols, 2, 0, C.byref(self.filter[0]), self.aggs, 3, self.res),
                "bolt_join_probe_aggregate")
        L.bolt_join_table_release(t)
        return [scalar_value(x) for x in self.res]

    def exact(self):
        s, total = torch.sort(self.dim)[0], 0.0
        for i in range(0, self.fk.numel(), 1 << 26):
            fk, amt = self.fk[i:i + (1 << 26)], self.amount[i:i + (1 << 26)]
            at = torch.searchsorted(s, fk).clamp_(max=s.numel() - 1)
            total += float(torch.where((s[at] == fk) & (amt > 10.0), amt, 0.0).sum())
        return [None, total, None]


class Join:
    def __init__(self, c, seed):
        r = _Rng(seed)
        self.right, self.left = _join_keys(r, c, c["right"], c["left"])
        dt = N.I32 if c["dtype"] == "i32" else N.I64
        self.attr = r.ints(c["right"], 0, 1_000_000, torch.int32)
        self.lk, self.rk, self.src = _column(self.left, dt), _column(self.right, dt), _column(self.attr, N.I32)
        self.how = {"inner": 0, "left": 1, "full": 3}[c["how"]]
        cap = c["left"] + c["right"]
        self.rows = [torch.zeros(cap, dtype=torch.int32, device=DEV) for _ in range(2)]
        self.got = torch.zeros(cap, dtype=torch.int32, device=DEV)
        self.got_bits = torch.zeros((cap + 63) // 64 * 8, dtype=torch.uint8, device=DEV)
        self.dst = _column(self.got, N.I32, self.got_bits)
        self.cap, self.n = cap, C.c_int64()

    def run(self):
        L = N.lib()
        N.check(L.bolt_join(None, C.byref(self.lk), C.byref(self.rk), 1, self.how, self.rows[0].data_ptr(),
                            self.rows[1].data_ptr(), self.cap, C.byref(self.n)), "bolt_join")
        k = self.n.value
        N.check(L.bolt_take(None, C.byref(self.src), self.rows[1].data_ptr(), k, C.byref(self.dst)), "bolt_take")
        return [k] + self.rows + [self.got, self.got_bits]

    def exact(self):
        return None


class Sort:
    def __init__(self, c, seed):
        r, n = _Rng(seed), c["rows"]
        if c["bits"] == 64:
            self.keys = r.ints(n, -(1 << 63), (1 << 63) - 1)
        else:
            self.keys = r.ints(n, 0, 1 << c["bits"])
        self.vals = torch.arange(n, dtype=torch.int32, device=DEV)
        self.ko, self.vo = torch.empty_like(self.keys), torch.empty_like(self.vals)
        self.n, self.desc = n, int(c["descending"])

    def run(self):
        N.check(N.lib().bolt_sort_pairs_i64(None, self.keys.data_ptr(), self.vals.data_ptr(), self.n, self.desc,
                                            self.ko.data_ptr(), self.vo.data_ptr()), "bolt_sort_pairs_i64")
        return [self.ko, self.vo]

    def exact(self):
        return None


class OrderBy:
    def __init__(self, c, seed):
        r, n = _Rng(seed), c["rows"]
        self.day = r.ints(n, 17_532, 17_532 + c["days"], torch.int32)
        self.valid = r.valid(n, c["nulls"])
        self.bits = _bitmap(self.valid) if self.valid is not None else None
        self.amount = r.unit(n).mul_(2000.0).sub_(100.0)
        self.cols = _columns(_column(self.day, N.DATE32, self.bits), _column(self.amount, N.F64))
        self.desc, self.first = (C.c_int32 * 2)(0, 1), (C.c_int32 * 2)(0, 0)
        self.rows = torch.empty(n, dtype=torch.int32, device=DEV)

    def run(self):
        N.check(N.lib().bolt_sort_indices(None, self.cols, 2, self.desc, self.first, self.rows.data_ptr()),
                "bolt_sort_indices")
        return self.rows

    def exact(self):
        return None


class TopK:
    def __init__(self, c, seed):
        r, n = _Rng(seed), c["rows"]
        if c["dtype"] == "i64":
            self.key, dt = r.ints(n, -(1 << 63), (1 << 63) - 1), N.I64
        elif c["dtype"] == "i32":
            self.key, dt = r.ints(n, -(1 << 31), (1 << 31) - 1, torch.int32), N.I32
        else:
            self.key, dt = r.unit(n).mul_(2000.0).sub_(100.0), N.F64
        self.cols = _columns(_column(self.key, dt))
        self.desc, self.first = (C.c_int32 * 1)(1), (C.c_int32 * 1)(0)
        self.limit, self.offset, self.n = c["limit"], c["offset"], C.c_int64()
        self.rows = torch.empty(self.limit, dtype=torch.int32, device=DEV)

    def run(self):
        N.check(N.lib().bolt_sort_limit(None, self.cols, 1, self.desc, self.first, self.offset, self.limit,
                                        self.rows.data_ptr(), C.byref(self.n)), "bolt_sort_limit")
        return self.rows[: self.n.value]

    def exact(self):
        return None


class Serve:
    """The star schema of the served form: a fact table (three foreign keys, a Decimal128 price, a float
    quantity, a date) and three dimensions; revenue by city over a quarter, a brand ranking of expensive
    items, and a category x zone count over three joins, in turn."""

    DIMS = ((1_000_000, (100_000,)), (100_000, (10_000, 1_000)), (2_500, (25,)))
    DAY0 = 17_532

    def __init__(self, c, seed):
        r, n = _Rng(seed), c["rows"]
        self.fk = [r.ints(n, 0, d, torch.int32) for d, _ in self.DIMS]
        cents = r.ints(n, 100, 1_000_000)
        self.price = torch.stack([cents, torch.zeros_like(cents)], 1)
        del cents
        self.qty = r.unit(n).mul_(49.0).add_(1.0)
        self.date = r.ints(n, self.DAY0, self.DAY0 + 2557, torch.int32)
        fact = [self._dev(x, dt) for x, dt in zip(self.fk + [self.price, self.qty, self.date],
                                                  [N.I32] * 3 + [N.DEC128, N.F64, N.DATE32])]
        dims = []
        for size, mods in self.DIMS:
            key = r.perm(size).to(torch.int32)
            dims.append((self._dev(key, N.I32), [self._dev(key % m, N.I32) for m in mods]))
        torch.cuda.synchronize()
        self.server = Server(fact, dims, slots=c["slots"])
        draws = r.ints(c["queries"] * 2, 0, 1 << 30).tolist()
        self.specs = [self._spec(i % 3, draws[2 * i], draws[2 * i + 1]) for i in range(c["queries"])]
        self.queries = [self.server.query(**s) for s in self.specs]

    @staticmethod
    def _dev(x: torch.Tensor, dtype: int) -> DeviceColumn:
        b = DeviceBuffer(x.numel() * x.element_size())
        N.check_rt(N.lib().bolt_hip_memcpy_dtod(b.ptr, x.data_ptr(), b.nbytes), "dtod")
        return DeviceColumn(b, x.shape[0], dtype)

    def _spec(self, t: int, a: int, b: int) -> dict:
        d0 = self.DAY0 + a % (2557 - 120)
        if t == 0:
            return dict(terms=[Term(5, N.GE, d0), Term(5, N.LT, d0 + 90)], joins=[(1, 1)], group=[(0, 0)],
                        aggs=[(N.SUM, 3), (N.SUM, 4), (N.COUNT_STAR, 0)], order_agg=0, limit=100, est_groups=10_000)
        if t == 1:
            return dict(terms=[Term(5, N.GE, d0), Term(5, N.LT, d0 + 60), Term(3, N.GE, 100_000 + b % 500_000)],
                        joins=[(0, 0)], group=[(0, 0)], aggs=[(N.SUM, 3), (N.COUNT_STAR, 0)], order_agg=0, limit=100,
                        est_groups=100_000)
        return dict(terms=[Term(5, N.GE, d0), Term(5, N.LT, d0 + 120)], joins=[(0, 0), (1, 1), (2, 2)],
                    group=[(2, 0), (1, 1)], aggs=[(N.COUNT_STAR, 0), (N.SUM, 4), (N.SUM, 3)], order_agg=2, limit=100,
                    est_groups=25_000)

    def run(self):
        tickets = [self.server.submit(q) for q in self.queries]
        out = []
        for t in tickets:
            res = self.server.wait(t)
            if res["status"] != N.BOLT_OK:
                raise RuntimeError(res["error"])
            cols = list(zip(*res["rows"]))
            out.append([res["n_groups"]] + [torch.tensor(x, dtype=torch.float64 if isinstance(x[0], float)
                                                         else torch.int64) for x in cols])
        return out

    def exact(self):
        out = []
        for s in self.specs:
            k = torch.ones_like(self.date, dtype=torch.bool)
            for t in s["terms"]:
                x = self.date if t.col == 5 else self.price[:, 0]
                k &= (x >= t.value) if t.op == N.GE else (x < t.value)
            g = torch.zeros((), dtype=torch.int64, device=DEV)
            for j, a in s["group"]:  # every foreign key is present, an attribute is its key's remainder
                dim = s["joins"][j][1]
                m = self.DIMS[dim][1][a]
                g = g * m + self.fk[dim][k].to(torch.int64) % m
            u, inv = torch.unique(g, return_inverse=True)
            cols = []
            for op, col in s["aggs"]:
                v = (torch.ones_like(inv) if op == N.COUNT_STAR else
                     self.price[k, 0] if col == 3 else self.qty[k])
                cols.append(torch.zeros(u.numel(), dtype=v.dtype, device=DEV).index_add_(0, inv, v))
            top = torch.sort(cols[s["order_agg"]], descending=True, stable=True)[1][: s["limit"]]
            out.append([None] * (1 + len(s["group"])) +
                       [x[top].cpu() if x.dtype == torch.float64 else None for x in cols])
        return out


_KINDS = {"aggregate": Aggregate, "expr": Expr, "filter": Filter, "groupby": GroupBy, "joinagg": JoinAgg,
          "join": Join, "sort": Sort, "orderby": OrderBy, "topk": TopK, "serve": Serve}


def prepare(case: dict, seed: int):
    return _KINDS[case["kind"]](case, seed)


def run(state):
    return state.run()


def exact(case: dict, seed: int):
    return prepare(case, seed).exact()


def work(case: dict) -> dict:
    """Every input column read once, every result written once."""
    k, c = case["kind"], case
    if k == "aggregate":
        b = c["rows"] * (8 + 4 + 8 + 16 + 4 + (0.125 if c["nulls"] else 0))
    elif k == "expr":
        b = c["rows"] * 20
    elif k == "filter":  # the predicate's column whole, the others where rows survive or their lines are shared
        row = 20 + (0.125 if c["nulls"] else 0)
        b = c["rows"] * row * (1 + c["keep"])
    elif k == "groupby":
        key = {"i32": 4, "i64": 8, "pair": 8}[c["keys"]]
        wide = c["values"] == "f64" and c["groups"] <= 100_000
        val = (16 if wide else 8) + (0.125 if c["nulls"] else 0)
        b = c["rows"] * (key + val) + min(c["groups"], c["rows"]) * (key + (32 if c["values"] == "i64" else 16))
    elif k == "joinagg":
        b = c["build"] * 12 + c["probe"] * 16
    elif k == "join":
        w = 4 if c["dtype"] == "i32" else 8
        pairs = c["left"] * (c["hit"] if c["how"] == "inner" else 1)
        b = (c["left"] + c["right"]) * w + c["right"] * 4 + pairs * (8 + 4 + 4.125)
    elif k == "sort":
        b = c["rows"] * 24
    elif k == "orderby":
        b = c["rows"] * (4 + 8 + 4 + (0.125 if c["nulls"] else 0))
    elif k == "topk":
        b = c["rows"] * (4 if c["dtype"] == "i32" else 8) + c["limit"] * 4
    else:  # one shared lap for every `slots` queries: date, price, quantity and the foreign keys
        b = c["rows"] * 40 * -(-c["queries"] // c["slots"])
    return {"bytes": float(b), "flops": 0.0}


def tolerance(case: dict):
    """Whole numbers and bytes are the same; sums in 64-bit floats differ by their order of addition."""
    if case["kind"] in ("filter", "join", "sort", "orderby", "topk"):
        return "exact"
    return {"rel": 1e-13, "max": 1e-12}
