"""ORDER BY + LIMIT through the sampled bound (BOLT_TOPK_SAMPLE_BYTES=0 takes it
above 2^20 rows): dtypes with NULLs, skewed and tied keys (the bound then
declines and the counting pass runs), limits from one row to many, two keys.
Exact against the oracle."""
import numpy as np
import pytest

import oracle as O
from craton_bolt_amd import _native as N
from craton_bolt_amd.device import DeviceColumn
from craton_bolt_amd.ops import execute_sort_limit

from gpu_util import both

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def sampled(monkeypatch):
    monkeypatch.setenv("BOLT_TOPK_SAMPLE_BYTES", "0")


def _check(cols, desc, nf, limit, offset):
    got = execute_sort_limit([d for d, _ in cols], limit, offset, desc, nf)
    assert np.array_equal(got, O.sort_limit([h for _, h in cols], desc, nf, limit, offset))


@pytest.mark.parametrize("kind", ["i64", "i32", "f64", "f32", "dec", "bool", "flag", "days", "skewed", "constant", "nulls",
                                  "f64_nulls", "f32_nulls", "dec_nulls", "bool_nulls"])
@pytest.mark.parametrize("limit,offset", [(1, 0), (100, 0), (1500, 400), (15_000, 3)])
def test_kinds(gpu, kind, limit, offset):
    print(f"[case] sampled limit {kind} {limit} {offset}", flush=True)
    n = 1_100_003
    rng = np.random.default_rng(limit)
    valid = rng.random(n) > 0.001 if kind.endswith("nulls") else None
    if kind == "i64":
        col = both(rng.integers(-(1 << 62), 1 << 62, n), N.I64)
    elif kind == "i32":
        col = both(rng.integers(-(1 << 31), 1 << 31, n).astype(np.int32), N.I32)
    elif kind == "f64":
        v = rng.standard_normal(n)
        v[rng.integers(0, n, 60)] = np.nan
        v[rng.integers(0, n, 60)] = -np.inf
        col = both(v, N.F64)
    elif kind.startswith("f32"):
        col = both(rng.standard_normal(n).astype(np.float32), N.F32, valid)
    elif kind == "f64_nulls":
        col = both(rng.standard_normal(n), N.F64, valid)
    elif kind.startswith("dec"):
        lo = rng.integers(-(1 << 62), 1 << 62, n)
        col = both(np.stack([lo, rng.integers(-3, 3, n) if kind == "dec" else rng.integers(-(1 << 40), 1 << 40, n)], 1),
                   N.DEC128, valid)
    elif kind.startswith("bool"):  # one in 200: the bound of 1900 rows holds them, the others' bounds decline
        flag = rng.random(n) < 0.005
        col = (DeviceColumn.from_numpy(flag.astype(np.uint8), N.BOOL, valid), both(flag.astype(np.int32), N.I32, valid)[1])
    elif kind == "flag":
        col = both((rng.random(n) < 0.0001).astype(np.int32), N.I32)
    elif kind == "days":
        col = both(rng.integers(0, 2500, n).astype(np.int32), N.DATE32)
    elif kind == "skewed":
        col = both((2.0 ** (rng.random(n) * 62)).astype(np.int64), N.I64)
    elif kind == "constant":
        col = both(np.full(n, 5, np.int64), N.I64)
    else:
        col = both(rng.integers(0, 1 << 40, n), N.I64, valid)
    for desc in (False, True):
        _check([col], [desc], [desc], limit, offset)


def test_two_keys(gpu):
    n = 1_200_000
    rng = np.random.default_rng(2)
    cols = [both(rng.integers(0, 300_000, n).astype(np.int32), N.I32, rng.random(n) > 0.01),
            both(rng.random(n), N.F64)]
    for desc in ([False, True], [True, False]):
        _check(cols, desc, [False, True], 200, 50)
