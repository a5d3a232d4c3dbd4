"""Edges of the batched take and compaction kernels: every operator over every
dtype (NaN among the floats), tiles and waves that end inside a row stripe,
survivor bitmaps that start at any bit, capacities inside a tile, NULL row
ids.  Expected values are numpy's; all comparisons are exact."""
import ctypes as C

import numpy as np
import pytest

from craton_bolt_amd import _native as N
from craton_bolt_amd.device import DeviceBuffer, DeviceColumn
from craton_bolt_amd.ops import NULL_ROW, Term, _filter, columns_array, compact_columns, take

pytestmark = pytest.mark.gpu

_OPS = {N.LT: np.less, N.LE: np.less_equal, N.GT: np.greater, N.GE: np.greater_equal, N.EQ: np.equal,
        N.NE: np.not_equal}


def _values(rng, n, dt):
    if dt in (N.F32, N.F64):
        a = rng.integers(-4, 5, n).astype(np.float32 if dt == N.F32 else np.float64)
        a[rng.random(n) < 0.1] = np.nan
        return a
    if dt == N.BOOL:
        return rng.integers(0, 2, n).astype(np.uint8)
    if dt == N.DEC128:
        lo = rng.integers(-3, 4, n)
        return np.stack([lo, lo >> 63], 1).astype(np.int64)
    return rng.integers(-4, 5, n).astype(np.int64 if dt == N.I64 else np.int32)


@pytest.mark.parametrize("n", [1, 257, 4097, 20_011])
@pytest.mark.parametrize("dt", [N.BOOL, N.I32, N.DATE32, N.I64, N.F32, N.F64, N.DEC128])
def test_compact_every_operator(gpu, n, dt):
    print(f"[case] compact operators n={n} dt={dt}", flush=True)
    rng = np.random.default_rng(n * 16 + dt)
    a = _values(rng, n, dt)
    valid = rng.random(n) > 0.25
    ids = np.arange(n, dtype=np.int64)
    cmp = a[:, 0] if dt == N.DEC128 else a
    for op, fn in _OPS.items():
        for v in (None, valid):
            col = DeviceColumn.from_numpy(a, dt, valid=v)
            outs, k = compact_columns([col, DeviceColumn.from_numpy(ids)], [Term(0, op, 1)])
            want = np.nonzero(fn(cmp, 1) & (True if v is None else v))[0]
            assert k == len(want)
            assert np.array_equal(outs[1].to_numpy(k), want)
            assert np.array_equal(outs[0].to_numpy(k), a[want], equal_nan=dt in (N.F32, N.F64))
            if v is not None:
                assert outs[0].valid_numpy(k).all()


@pytest.mark.parametrize("keep", [0.003, 0.5, 0.97])
def test_compact_bitmaps_start_anywhere(gpu, keep):
    """Two nullable columns beside the predicate's; tile boundaries fall on arbitrary output bits."""
    print(f"[case] compact bitmaps keep={keep}", flush=True)
    n = 70_003
    rng = np.random.default_rng(int(keep * 1000))
    pick = rng.random(n)
    cols, vals, bits = [DeviceColumn.from_numpy(pick)], [], []
    for dt in (N.I32, N.DEC128):
        a, v = _values(rng, n, dt), rng.random(n) > 0.4
        cols.append(DeviceColumn.from_numpy(a, dt, valid=v))
        vals.append(a)
        bits.append(v)
    outs, k = compact_columns(cols, [Term(0, N.LT, keep)])
    want = np.nonzero(pick < keep)[0]
    assert k == len(want)
    for o, a, v in zip(outs[1:], vals, bits):
        assert np.array_equal(o.to_numpy(k), a[want])
        assert np.array_equal(o.valid_numpy(k), v[want])
        tail = o.validity.to_numpy(np.uint8)[(k + 7) // 8:(n + 7) // 8]
        assert not tail.any()  # cleared past the survivors


@pytest.mark.parametrize("cap", [1, 31, 32, 33, 2049, 9000])
def test_compact_capacity_inside_a_tile(gpu, cap):
    n = 20_000
    rng = np.random.default_rng(cap)
    a, v = rng.integers(0, 10, n).astype(np.int64), rng.random(n) > 0.3
    want = np.nonzero(a < 5)[0]
    col = DeviceColumn.from_numpy(a, valid=v)
    f, _keep = _filter([Term(0, N.GE, 0), Term(0, N.LT, 5)], [col])
    want = np.nonzero((a < 5) & v)[0]
    out = DeviceColumn.empty(n, N.I64, with_validity=True)
    out.values.copy_from(np.full(n, -7, np.int64))
    out.validity.fill(0xFF)
    oc = (N.BoltColumn * 1)(out.c(length=cap))
    n_out = C.c_int64()
    st = N.lib().bolt_filter_compact(None, columns_array([col]), 1, C.byref(f), None, oc, C.byref(n_out))
    k = min(cap, len(want))
    assert n_out.value == len(want) and st == (N.BOLT_DECLINE if cap < len(want) else N.BOLT_OK)
    got = out.values.to_numpy(np.int64, n)
    assert np.array_equal(got[:k], a[want[:k]]) and np.all(got[k:] == -7)
    b = np.unpackbits(out.validity.to_numpy(np.uint8), bitorder="little")
    assert b[:k].all()
    assert b[(cap + 31) // 32 * 32:].all()  # words past the capacity keep their bits


@pytest.mark.parametrize("n", [1, 255, 257, 1023, 1025, 300_001])
@pytest.mark.parametrize("src_valid", [False, True])
def test_take_null_rows(gpu, n, src_valid):
    print(f"[case] take nulls n={n} {src_valid}", flush=True)
    rng = np.random.default_rng(n)
    src = rng.integers(-1000, 1000, 777).astype(np.int32)
    v = rng.random(777) > 0.5
    rows = rng.integers(0, 777, n).astype(np.uint32)
    null = rng.random(n) < 0.4
    rows[null] = NULL_ROW
    col = DeviceColumn.from_numpy(src, valid=v if src_valid else None)
    out = take(col, DeviceBuffer.from_numpy(rows), n, nullable=True)
    at = np.where(null, 0, rows)
    assert np.array_equal(out.to_numpy(n), np.where(null, 0, src[at]))
    assert np.array_equal(out.valid_numpy(n), ~null & (v[at] if src_valid else True))
    if null.any() and not src_valid:
        with pytest.raises(N.PlanError, match="NULL row id"):
            take(col, DeviceBuffer.from_numpy(rows), n)


def test_take_from_an_empty_source(gpu):
    rows = np.full(1000, NULL_ROW, np.uint32)
    out = take(DeviceColumn.empty(0, N.I64), DeviceBuffer.from_numpy(rows), 1000, nullable=True)
    assert not out.valid_numpy(1000).any() and not out.to_numpy(1000).any()
    with pytest.raises(N.PlanError, match="out of range"):
        take(DeviceColumn.empty(0, N.I64), DeviceBuffer.from_numpy(np.zeros(4, np.uint32)), 4, nullable=True)
