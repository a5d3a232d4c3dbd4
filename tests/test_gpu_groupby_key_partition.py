"""GROUP BY through the key partition (BOLT_GB_KEY_PARTITION=1 takes it at any
size): every key form, NULL keys and inputs, filters, every aggregate, row
counts around the partition's tiles and chunks, and inputs with more groups
than the partitions' LDS tables hold (the plain path runs instead), against
the oracle with test_gpu_groupby's comparisons and tolerances."""
import ctypes as C
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from craton_bolt_amd import _native as N
from craton_bolt_amd.device import DeviceColumn
from craton_bolt_amd.ops import Term, execute_groupby, groupby_last_plan

from gpu_util import dec_array
from test_gpu_groupby import run_both

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def forced(monkeypatch):
    monkeypatch.setenv("BOLT_JIT", "1")
    monkeypatch.setenv("BOLT_GB_KEY_PARTITION", "1")


def _key(kind, n, groups, rng):
    g = rng.integers(0, groups, n)
    if kind == "i64":
        k = g * 0x9E3779B97F4A7 - 1  # the empty marker (-1) among them
        return [(k.astype(np.int64), N.I64, None)], [N.I64]
    if kind == "i32":
        return [((g * 7919 - 1).astype(np.int32), N.I32, None)], [N.I32]
    if kind == "date":
        return [(g.astype(np.int32), N.DATE32, None)], [N.DATE32]
    if kind == "f64":
        k = g.astype(np.float64) - 3.0
        k[g == 1] = np.nan
        k[(g == 3) & (rng.random(n) < 0.5)] = -0.0
        return [(k, N.F64, None)], [N.F64]
    if kind == "f32":
        return [(g.astype(np.float32), N.F32, None)], [N.F32]
    if kind == "dec":
        return [(dec_array([int(x) - 5 for x in g]), N.DEC128, None)], [N.DEC128]
    if kind in ("null_i64", "clash_i64"):  # clash: the NULL group beside a key of its packed value
        k = g * 0x9E3779B97F4A7 - 1
        if kind == "clash_i64":
            k[g == 2] = 2 ** 63 - 1
        return [(k.astype(np.int64), N.I64, rng.random(n) > 0.3)], [N.I64]
    if kind == "null_i32":
        return [(g.astype(np.int32), N.I32, rng.random(n) > 0.3)], [N.I32]
    a, b = (g % 50).astype(np.int32), (g // 50).astype(np.int32)
    if kind == "null_pair":
        return [(a, N.I32, rng.random(n) > 0.2), (b, N.I32, rng.random(n) > 0.2)], [N.I32, N.I32]
    return [(a, N.I32, None), (b, N.I32, None)], [N.I32, N.I32]


@pytest.mark.parametrize("n", [1, 4095, 4097, 100_003])
@pytest.mark.parametrize("kind", ["i64", "i32", "date", "f64", "f32", "null_i32", "null_i64", "clash_i64", "pair",
                                  "null_pair"])
def test_key_forms(gpu, n, kind):
    print(f"[case] key partition {kind} n={n}", flush=True)
    rng = np.random.default_rng(n)
    keys, kdt = _key(kind, n, max(2, n // 9), rng)
    v = rng.integers(-1000, 1000, n).astype(np.int64)
    x = rng.normal(size=n)
    run_both(keys, [(v, N.I64, None), (x, N.F64, rng.random(n) > 0.2)],
             [(N.SUM, 0), (N.COUNT_STAR, 0), (N.MIN, 0), (N.MAX, 1), (N.SUM, 1), (N.COUNT, 1)], kdt)


@pytest.mark.parametrize("nullable", [False, True])
@pytest.mark.parametrize("n", [1, 4097, 100_003])
def test_decimal_keys(gpu, n, nullable):
    """The copy keeps the low word of a Decimal128 key, the extraction widens it again (-5 to 11,000, -1 and 0
    among them; NULL rows hold high words of any value): as the same keys in 64 bits."""
    print(f"[case] key partition dec n={n} nullable={nullable}", flush=True)
    rng = np.random.default_rng(n)
    (dec, _, _), = _key("dec", n, max(2, n // 9), rng)[0]
    valid = rng.random(n) > 0.3 if nullable else None
    v = rng.integers(-1000, 1000, n).astype(np.int64)
    aggs = [(N.SUM, 0), (N.COUNT_STAR, 0), (N.MAX, 0)]
    want, _ = run_both([(dec[:, 0].copy(), N.I64, valid)], [(v, N.I64, None)], aggs, [N.I64])
    if nullable:
        dec[~valid, 1] = 77
    got = execute_groupby([DeviceColumn.from_numpy(dec, N.DEC128, valid)], [DeviceColumn.from_numpy(v)], aggs)
    assert got["n_groups"] == want["n_groups"]
    (gk, gv), (wk, wv) = got["keys"][0], want["keys"][0]
    live = np.ones(len(wk), bool) if wv is None else wv
    assert (gv is None) == (wv is None) and (gv is None or np.array_equal(gv, wv))
    assert np.array_equal(gk[live, 0], wk[live]) and np.array_equal(gk[live, 1], wk[live] >> 63)
    for (g, _), (w, _) in zip(got["aggs"], want["aggs"]):
        assert np.array_equal(g, w)


@pytest.mark.parametrize("n", [60_001])
def test_aggregates_and_filter(gpu, n):
    rng = np.random.default_rng(5)
    keys, kdt = _key("i32", n, 4000, rng)
    i32 = rng.integers(-100, 100, n).astype(np.int32)
    f32 = rng.normal(size=n).astype(np.float32)
    dec = dec_array([int(x) for x in rng.integers(-10 ** 12, 10 ** 12, n)])
    f64 = rng.normal(size=n) + 10.0
    va = rng.random(n) > 0.1
    ins = [(i32, N.I32, va), (f32, N.F32, None), (dec, N.DEC128, va), (f64, N.F64, va)]
    print("[case] key partition aggregates", flush=True)
    run_both(keys, ins, [(N.SUM, 0), (N.AVG, 0), (N.MAX, 1), (N.SUM, 2), (N.COUNT, 2), (N.MIN, 3), (N.COUNT_STAR, 0)],
             kdt, terms=[Term(3, N.GT, 9.5), Term(0, N.LT, 50)])
    print("[case] key partition variance", flush=True)
    run_both(keys, [(f64, N.F64, va)], [(N.VAR_SAMP, 0), (N.STDDEV_POP, 0), (N.AVG, 0)], kdt)
    print("[case] key partition keys only", flush=True)
    run_both(keys, [(i32, N.I32, None)], [], kdt)


def test_no_row_passes(gpu):
    rng = np.random.default_rng(6)
    keys, kdt = _key("i64", 10_000, 500, rng)
    run_both(keys, [(np.ones(10_000), N.F64, None)], [(N.SUM, 0)], kdt, terms=[Term(0, N.GT, 2.0)])


def test_more_groups_than_the_tables(gpu):
    """Every row its own group: partitions overflow, the plain path takes over."""
    n = 1_500_000
    print("[case] key partition overflow", flush=True)
    k = np.random.default_rng(7).permutation(n).astype(np.int64)
    run_both([(k, N.I64, None)], [(k.astype(np.float64), N.F64, None)], [(N.SUM, 0), (N.COUNT_STAR, 0)], [N.I64])


# SUM(f64) and COUNT(*) are two words: 256 tables of 6440 slots, of which the
# groups may take 0.6 (989,000).  At 300,000 and above a bound of 16 slots a
# probe left keys without one, and the whole call ran again on the plain path.
@pytest.mark.parametrize("kind", ["i64", "i32", "pair"])
@pytest.mark.parametrize("groups", [300_000, 500_000, 700_000, 930_000])
def test_every_group_finds_a_slot(gpu, kind, groups):
    n = 2_200_000
    print(f"[case] key partition {kind} groups={groups}", flush=True)
    rng = np.random.default_rng(groups)
    g = rng.permutation(n) % groups
    if kind == "pair":
        keys, kdt = [((g % 900).astype(np.int32), N.I32, None), ((g // 900).astype(np.int32), N.I32, None)], [N.I32] * 2
    elif kind == "i32":
        keys, kdt = [((g * 7919 - 1).astype(np.int32), N.I32, None)], [N.I32]
    else:
        keys, kdt = [(rng.integers(-2 ** 63, 2 ** 63 - 1, groups)[g], N.I64, None)], [N.I64]
    run_both(keys, [(rng.normal(size=n), N.F64, None)], [(N.SUM, 0), (N.COUNT_STAR, 0)], kdt)
    assert groupby_last_plan() == {"tier": 0, "spilled_rows": 0, "partial_records": groups, "partitions": 0}


@pytest.mark.parametrize("few", [0, 10_000])
def test_too_many_groups_are_counted(gpu, few):
    """More groups than the tables take, by themselves or behind a few frequent ones (which a sample takes
    for all): the count ends the partition, and the plain path answers."""
    n, many = 2_400_000, 1_300_000
    print(f"[case] key partition declined few={few}", flush=True)
    rng = np.random.default_rng(8)
    g = rng.permutation(n) % many
    if few:
        g = np.where(rng.random(n) < 0.3, rng.integers(0, few, n), g)
    run_both([(g * 0x9E3779B97F4A7, N.I64, None)], [(rng.normal(size=n), N.F64, None)], [(N.SUM, 0), (N.COUNT_STAR, 0)],
             [N.I64])
    assert groupby_last_plan()["spilled_rows"] > 0


@pytest.mark.parametrize("n,groups,parted", [((1 << 24) + 1, 3300, False), ((1 << 24) + 1, 4300, True),
                                             (2_200_000, 3300, True)])
def test_nearly_full_tables(gpu, monkeypatch, n, groups, parted):
    """Two words leave the plain path's tables 3752 slots: above 2^24 rows the partition begins where the groups
    fill them.  It has one partial record per group, the plain path one per workgroup and group."""
    monkeypatch.delenv("BOLT_GB_KEY_PARTITION")
    print(f"[case] key partition n={n} groups={groups}", flush=True)
    k = np.random.default_rng(groups).integers(0, groups, n).astype(np.int32)
    v = (np.arange(n) % 1000).astype(np.float64)  # sums below 2^53 are exact in any order
    got = execute_groupby([DeviceColumn.from_numpy(k)], [DeviceColumn.from_numpy(v)], [(N.SUM, 0), (N.COUNT_STAR, 0)])
    assert (groupby_last_plan()["partial_records"] == groups) == parted
    assert np.array_equal(got["keys"][0][0], np.arange(groups))
    assert np.array_equal(got["aggs"][0][0], np.bincount(k, v, groups))
    assert np.array_equal(got["aggs"][1][0], np.bincount(k, minlength=groups))


_PEAK = """
import ctypes as C, os
import numpy as np
from craton_bolt_amd import _native as N
from craton_bolt_amd.device import DeviceColumn
from craton_bolt_amd.ops import execute_groupby
def peak():
    used, high = C.c_size_t(), C.c_size_t()
    N.check_rt(N.lib().bolt_hip_pool_stats(C.byref(used), C.byref(high)))
    return high.value
n = 4_000_000
g = np.random.default_rng(9).permutation(n) % 1_300_000
k, v = DeviceColumn.from_numpy(g * 0x9E3779B97F4A7), DeviceColumn.from_numpy(np.ones(n))
for how in ("0", "1"):
    os.environ["BOLT_GB_KEY_PARTITION"] = how
    assert execute_groupby([k], [v], [(N.SUM, 0), (N.COUNT_STAR, 0)])["n_groups"] == 1_300_000
    print("peak", how, peak(), flush=True)
"""


def test_declined_attempt_holds_no_memory(gpu):
    """A call whose attempt is given up needs no more device memory at once than the plain path alone (the
    high-water mark of a process of its own: it never falls)."""
    print("[case] key partition declined, peak memory", flush=True)
    r = subprocess.run([sys.executable, "-u", "-c", _PEAK], cwd=Path(__file__).resolve().parent.parent, timeout=100,
                       env=dict(os.environ), capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    plain, tried = (int(line.split()[2]) for line in r.stdout.splitlines() if line.startswith("peak"))
    # a few hundred bytes go with the rows that the LDS tier happens to spill; the attempt's copies alone are 64 MB
    assert tried <= plain + (1 << 20), (tried, plain)


def test_compiles_what_it_runs(gpu):
    """A query shape of its own: the partition's kernel and the LDS tier over the copies, not the plain tier's."""
    def compiled():
        c, h, s = C.c_int64(), C.c_int64(), C.c_int64()
        N.lib().bolt_jit_cache_stats(C.byref(c), C.byref(h), C.byref(s))
        return c.value + h.value

    rng = np.random.default_rng(10)
    keys, kdt = _key("f32", 5000, 900, rng)
    x = rng.normal(size=5000)
    print("[case] key partition compiles", flush=True)
    before = compiled()
    run_both(keys, [(x, N.F64, rng.random(5000) > 0.2)],  # NULLs: a bitmap there, bytes in the copy
             [(N.MIN, 0), (N.COUNT, 0), (N.MAX, 0), (N.AVG, 0), (N.COUNT_STAR, 0)], kdt)
    assert compiled() - before == 2


@pytest.mark.parametrize("groups", [9_000, 300_000])
def test_chosen_by_the_sample(gpu, monkeypatch, groups):
    """Large enough to be chosen without the switch: the same result."""
    monkeypatch.delenv("BOLT_GB_KEY_PARTITION")
    n = 2_500_000
    print(f"[case] key partition sampled groups={groups}", flush=True)
    rng = np.random.default_rng(groups)
    k = rng.integers(0, groups, n).astype(np.int32)
    v = rng.integers(0, 1000, n).astype(np.int64)
    run_both([(k, N.I32, None)], [(v, N.I64, None)], [(N.SUM, 0), (N.MIN, 0)], [N.I32])
