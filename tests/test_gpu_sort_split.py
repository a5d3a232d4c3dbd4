"""The splitter sort (up to 2^25 rows) over key distributions that put its
buckets at their limits: skewed and clustered keys, values with buckets of
their own, equal keys, keys at both ends of the range, and row counts around
the one-workgroup, one-pass and two-pass forms.  Values are a permutation, so
exact agreement with numpy's stable argsort also pins stability."""
import numpy as np
import pytest

from craton_bolt_amd.device import DeviceBuffer, DeviceColumn
from craton_bolt_amd.ops import sort_last_plan, sort_pairs_i64

pytestmark = pytest.mark.gpu

I64 = np.iinfo(np.int64)


def _keys(kind: str, n: int, rng) -> np.ndarray:
    if kind == "uniform":
        return rng.integers(I64.min, I64.max, n, endpoint=True)
    if kind == "float_bits":  # exponents make the top bytes few and uneven
        return (rng.random(n) * 2000.0 - 100.0).view(np.int64)
    if kind == "days":
        return rng.integers(17_532, 20_032, n)
    if kind == "two_values":
        return np.where(rng.random(n) < 0.3, np.int64(5), np.int64(-5))
    if kind == "constant":
        return np.full(n, 42, np.int64)
    if kind == "ends":  # both ends of the range heavy, a few keys between
        k = rng.integers(-1000, 1000, n)
        u = rng.random(n)
        return np.where(u < 0.4, I64.min, np.where(u < 0.8, I64.max, k))
    if kind == "outliers":  # a dense cluster and rare huge values
        k = rng.integers(0, 3000, n)
        k[rng.random(n) < 1e-3] = I64.max - 7
        return k
    if kind == "geometric":  # every scale from 1 to 2^62
        return (2.0 ** (rng.random(n) * 62)).astype(np.int64)
    if kind == "ascending":
        return np.arange(n, dtype=np.int64) * 977 - n
    return np.arange(n, dtype=np.int64)[::-1].copy() // 3  # descending, triples


@pytest.mark.parametrize("n", [2, 63, 2047, 6144, 6145, 32_768, 32_769, 100_003, 131_072, 131_073, 262_145, 1_500_007])
@pytest.mark.parametrize("kind", ["uniform", "float_bits", "days", "two_values", "constant", "ends", "outliers",
                                  "geometric", "ascending", "triples"])
def test_split_sort(gpu, n, kind):
    print(f"[case] split sort n={n} {kind}", flush=True)
    rng = np.random.default_rng(n)
    key = _keys(kind, n, rng).astype(np.int64)
    rid = rng.permutation(n).astype(np.uint32)
    for desc in (False, True):
        ko, vo = sort_pairs_i64(DeviceBuffer.from_numpy(key), DeviceBuffer.from_numpy(rid), n, desc)
        order = np.argsort(~key if desc else key, kind="stable")
        assert np.array_equal(ko.to_numpy(np.int64, n), key[order])
        assert np.array_equal(vo.to_numpy(np.uint32, n), rid[order])


@pytest.mark.parametrize("kind", ["uniform", "float_bits", "days", "geometric"])
@pytest.mark.parametrize("n", [9_000_001, 1 << 25, (1 << 25) + 1])
def test_split_sort_large(gpu, n, kind):
    print(f"[case] split sort n={n} {kind}", flush=True)
    rng = np.random.default_rng(n)
    key = _keys(kind, n, rng).astype(np.int64)
    rid = np.arange(n, dtype=np.uint32)
    ko, vo = sort_pairs_i64(DeviceBuffer.from_numpy(key), DeviceBuffer.from_numpy(rid), n)
    order = np.argsort(key, kind="stable")
    assert np.array_equal(ko.to_numpy(np.int64, n), key[order])
    assert np.array_equal(vo.to_numpy(np.uint32, n), order.astype(np.uint32))


_ANY = -1  # bytes that vary: all eight
_MASK = {0: 0, 1: 1, 2: 0x1FF, 3: 0x1FFFF, 4: 0x1FFFFFF, 5: 0x1FFFFFFFF}


@pytest.mark.parametrize("n,nbytes,shift,plan", [
    (131_072, 1, 0, ("sample", 0)), (131_073, 0, 0, ("copy", 0)), (131_073, 1, 56, ("bytes", 1)),
    (131_073, 2, 0, ("bytes", 2)), (131_073, 3, 0, ("sample", 0)), (262_144, 3, 8, ("bytes", 3)),
    (524_287, 4, 0, ("sample", 0)), (524_288, 4, 24, ("bytes", 4)), (1 << 23, 5, 0, ("sample", 0)),
    (1 << 23, 4, 0, ("bytes", 4)), (1 << 23, _ANY, 0, ("sample", 0)), ((1 << 23) + 1, 0, 0, ("copy", 0)),
    ((1 << 23) + 1, 1, 0, ("bytes", 1)), ((1 << 23) + 1, 3, 0, ("bytes", 3)), ((1 << 23) + 1, 5, 0, ("bytes", 5)),
    ((1 << 23) + 1, _ANY, 0, ("digits", 2))])
def test_few_varying_bytes(gpu, n, nbytes, shift, plan):
    """Keys in which few bytes vary take a pass per byte.  The top varying byte takes two values, so above 2^23
    rows the top two bytes alone do not separate the rows."""
    print(f"[case] sort n={n} bytes={nbytes} shift={shift}", flush=True)
    rng = np.random.default_rng(n + nbytes)
    key = rng.integers(I64.min, I64.max, n, endpoint=True)
    if nbytes != _ANY:
        key = (key & _MASK[nbytes]) << shift
    rid = np.arange(n, dtype=np.uint32)
    for desc in (False, True):
        ko, vo = sort_pairs_i64(DeviceBuffer.from_numpy(key), DeviceBuffer.from_numpy(rid), n, desc)
        assert sort_last_plan() == plan
        order = np.argsort(~key if desc else key, kind="stable")
        assert np.array_equal(ko.to_numpy(np.int64, n), key[order])
        assert np.array_equal(vo.to_numpy(np.uint32, n), order.astype(np.uint32))


@pytest.mark.parametrize("rows,plan", [(1, ("sample", 0)), (10, ("bytes", 8)), (400, ("bytes", 8)),
                                       (2000, ("sample", 0))])
def test_values_shared_by_rows(gpu, rows, plan):
    """Above 2^23 rows, floats whose exponents leave the top two bytes uneven: values of a few to a few hundred
    rows take passes by bytes, the sample's buckets are left with the others."""
    n = 9_000_001
    print(f"[case] sort rows per value={rows}", flush=True)
    rng = np.random.default_rng(rows)
    key = (rng.integers(0, n // rows, n) / 100.0).view(np.int64)
    rid = np.arange(n, dtype=np.uint32)
    ko, vo = sort_pairs_i64(DeviceBuffer.from_numpy(key), DeviceBuffer.from_numpy(rid), n)
    assert sort_last_plan() == plan
    order = np.argsort(key, kind="stable")
    assert np.array_equal(ko.to_numpy(np.int64, n), key[order])
    assert np.array_equal(vo.to_numpy(np.uint32, n), order.astype(np.uint32))


@pytest.mark.parametrize("n", [2, 777, 40_000, 600_001])
@pytest.mark.parametrize("shape", ["fits", "cut", "pairs", "ties", "long_ties", "one_run", "deep", "constant"])
def test_order_by_packed(gpu, n, shape):
    """ORDER BY by packed keys: all fields fit in 64 bits, the last one is cut,
    runs that agree on all packed bits, few and short (put in order in place),
    many, long, one of them too long (ranks and the next bits instead), several
    times over, and fields without a range."""
    import oracle as O
    from craton_bolt_amd import _native as N
    from craton_bolt_amd.ops import execute_sort
    from gpu_util import both, dec_array

    print(f"[case] packed order n={n} {shape}", flush=True)
    rng = np.random.default_rng(n)
    va, vb = rng.random(n) > 0.1, rng.random(n) > 0.1
    wide = rng.random(n) * 2000.0 - 100.0
    if shape == "fits":
        flag = (rng.random(n) < 0.5).astype(np.int32)  # the oracle orders it as an integer
        cols = [both(rng.integers(0, 9, n).astype(np.int32), N.I32, va),
                (DeviceColumn.from_numpy(flag.astype(np.uint8), N.BOOL, vb), both(flag, N.I32, vb)[1]),
                both(rng.integers(-5, 5, n).astype(np.float32), N.F32, None)]
    elif shape == "cut":
        cols = [both(rng.integers(0, 2500, n).astype(np.int32), N.DATE32, va), both(wide, N.F64, vb),
                both(rng.integers(0, 3, n).astype(np.int64), N.I64, None)]
    elif shape == "ties":  # the second key differs only below the packed bits
        cols = [both(wide[rng.integers(0, max(n // 8, 1), n)], N.F64, None),
                both(1.0 + rng.integers(0, 4, n) * 2.0 ** -52, N.F64, vb)]
    elif shape == "pairs":
        cols = [both(wide[rng.permutation(n) // 2], N.F64, va), both(wide[::-1].copy(), N.F64, vb)]
    elif shape == "one_run":  # 64 rows are put in order in place, 65 are not
        k = np.arange(n, dtype=np.int64) * (2 ** 62 // n)
        k[rng.permutation(n)[:65]] = 5
        cols = [both(k[rng.permutation(n)], N.I64, None), both(rng.integers(-2 ** 62, 2 ** 62, n), N.I64, vb)]
    elif shape == "deep":  # few values over all bits of every key
        few = rng.integers(-2 ** 63, 2 ** 63 - 1, 5)
        cols = [both(few[rng.integers(0, 5, n)], N.I64, v) for v in (va, None, vb)] + [both(wide, N.F64, None)]
    elif shape == "long_ties":
        cols = [both(np.where(rng.random(n) < 0.5, 1e-300, -1e300), N.F64, va),
                both(np.where(rng.random(n) < 0.5, 1e-200, -1e200), N.F64, vb)]
    else:
        cols = [both(np.full(n, 7, np.int64), N.I64, None), both(dec_array([3] * n), N.DEC128, None),
                both(wide, N.F64, np.zeros(n, bool))]
    k = len(cols)
    for desc, nf in [([False] * k, [True] * k), ([True, False, True][:k], [False, True, False][:k])]:
        got = execute_sort([x for x, _ in cols], desc, nf)
        want = O.sort_indices([h for _, h in cols], desc, nf)
        assert np.array_equal(got, want)


def test_order_by_few_values_first(gpu):
    """A float of two values, then a float: the second sort's key is the first's rank and the next bits (61 of
    them), where sorting field by field ended with the two values alone, in two bytes."""
    from craton_bolt_amd import _native as N
    from craton_bolt_amd.ops import execute_sort

    n = 600_001
    print("[case] packed order, few values first", flush=True)
    rng = np.random.default_rng(11)
    a, x = rng.integers(0, 2, n).astype(np.float64), rng.random(n)
    got = execute_sort([DeviceColumn.from_numpy(a, N.F64), DeviceColumn.from_numpy(x, N.F64)], [False, True], [True, True])
    assert sort_last_plan() == ("sample", 0)
    assert np.array_equal(got, np.lexsort((-x, a)))
