"""GPU: the pair-emitting probe at the edges of its waves and tiles, with unique
build keys (where a preserved side's pairs need no offsets from other tiles) and
with duplicates, against a direct lookup on the host: pairs in probe-row order,
a NULL or unmatched key of the preserved side padded in its place."""
import numpy as np
import pytest

from craton_bolt_amd import _native as N
from craton_bolt_amd.ops import NULL_ROW, execute_join

from gpu_util import both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dup", [False, True])
@pytest.mark.parametrize("how", ["inner", "left", "full"])
@pytest.mark.parametrize("nl", [1, 63, 64, 65, 511, 512, 513, 4095, 4096, 4097, 12_345])
@pytest.mark.parametrize("nulls", [False, True])
def test_pairs_at_tile_edges(gpu, nl, how, dup, nulls):
    nr = 200
    rng = np.random.default_rng(nl)
    rk = np.arange(nr, dtype=np.int64) * 3
    lk = rng.integers(0, 2 * nr, nl).astype(np.int64) * 3
    if dup:
        rk[nr // 2:] = rk[:nr // 2]
    if how == "inner" and nl <= nr:
        lk = np.unique(lk)  # the left side builds: unique there
    valid = rng.random(len(lk)) >= 0.1 if nulls else None
    (dl, _), (dr, _) = both(lk, N.I64, valid), both(rk, N.I64)
    l, r = execute_join([dl], [dr], how)
    pairs = set()
    for i, k in enumerate(lk):
        hits = np.nonzero(rk == k)[0] if valid is None or valid[i] else []
        pairs.update((i, int(j)) for j in hits)
        if len(hits) == 0 and how != "inner":
            pairs.add((i, NULL_ROW))
    if how == "full":
        seen = {j for _, j in pairs}
        pairs.update((NULL_ROW, j) for j in range(nr) if j not in seen)
    got = list(zip(l.tolist(), r.tolist()))
    assert len(got) == len(pairs) and set(got) == pairs
    if how != "inner" or len(lk) > nr:  # the left side probes
        assert np.all(np.diff(l[l != NULL_ROW].astype(np.int64)) >= 0)


def test_preserved_side_over_capacity(gpu):
    dl, _ = both(np.arange(9_000, dtype=np.int64), N.I64)
    dr, _ = both(np.arange(100, dtype=np.int64), N.I64)
    with pytest.raises(N.BoltError) as e:
        execute_join([dl], [dr], "left", capacity=8_191)
    assert e.value.code == N.BOLT_DECLINE
    l, r = execute_join([dl], [dr], "left", capacity=9_000)
    assert len(l) == 9_000 and np.array_equal(np.nonzero(r != NULL_ROW)[0], np.arange(100))
