"""GPU: join tables that one block builds in LDS, at the edges of their size
(18432 slots at the default load) and of the table's kinds, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def keys(kind, nr, rng):
    if kind == "dense":  # key-range table
        return (rng.permutation(nr) - nr // 2).astype(np.int32)
    if kind == "edge":  # range just past a power of two: hash-mixed unless the slots reach the next one
        k = rng.permutation(nr).astype(np.int32)
        k[k == nr - 1] = 1 << max(1, int(np.ceil(np.log2(max(nr, 2)))))
        return k
    if kind == "sparse":
        return (rng.permutation(nr).astype(np.int64) * 193939 - (1 << 31)).astype(np.int32)
    if kind == "dups":  # a dense range that loses tuples: falls back
        return rng.integers(-1, max(1, nr // 3), nr).astype(np.int32)
    return np.full(nr, 7, np.int32)[: nr]  # "one"


@pytest.mark.parametrize("kind", ["dense", "edge", "sparse", "dups", "one"])
@pytest.mark.parametrize("nr", [1, 2, 31, 1023, 1025, 8192, 9215, 9216, 9300])
def test_small_build_matches_oracle(qo, orc, kind, nr):
    if kind == "one":
        nr = min(nr, 500)  # every probe of the key matches every tuple
    rng = np.random.default_rng(nr)
    rk = keys(kind, nr, rng)
    rp = rng.integers(-(1 << 31), 1 << 31, nr).astype(np.int32)
    if kind == "dups":
        rp[rk == -1] = -1  # tuples that look like an empty slot
    ns = 3001
    sk = np.concatenate([rng.choice(rk, ns - 1000), rng.integers(-(1 << 31), 1 << 31, 990).astype(np.int32),
                         np.arange(-5, 5, dtype=np.int32)])
    sp = rng.integers(-(1 << 31), 1 << 31, ns).astype(np.int32)
    got = qo.operators.hash_join(rk, rp, sk, sp, capacity=4_000_000)
    exp = orc.hash_join(rk, rp, sk, sp)
    a, b = (np.stack([np.asarray(c, np.int64) for c in x[:3]], 1) for x in (got, exp))
    assert a.shape == b.shape
    assert np.array_equal(a[np.lexsort(a.T)], b[np.lexsort(b.T)])
