"""GPU: what qo_hj_filter_sort leaves alone.  Output rows past the match count
keep what they held, and with more rows than the outputs hold none is written
(the count is)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
INT_MIN, INT_MAX = -(1 << 31), (1 << 31) - 1
MARK = 0x5A5A5A5A


def rand32(rng, n):
    return rng.integers(INT_MIN, INT_MAX, n, dtype=np.int64, endpoint=True).astype(np.int32)


def build_keys(kind, nr, rng):
    k = rng.permutation(nr).astype(np.int64)
    if kind == "spread":
        k = ((k * 1_640_531_527 + 7) & 0x7FFFFFFF) - (1 << 30)
    elif kind == "gaps":
        k = k + k // 3
    return k.astype(np.int32)


def run(qo, rk, rp, sk, sp, cap):
    """(status, count, the three output columns whole) of a join without a filter."""
    D, lib = qo.device.DeviceBuffer, qo._lib.load()
    tb, n = lib.qo_join_table_bytes(len(rk)), len(sk) + 64
    mark = np.full(n, MARK, np.int32)
    with D(tb) as t:
        cols = [D.from_numpy(a) for a in (rk, rp, sk, sp)]
        out = [D.from_numpy(mark) for _ in range(3)]
        m = C.c_uint64()
        rc = lib.qo_hj_filter_sort(t.ptr, tb, cols[0].ptr, cols[1].ptr, len(rk), cols[2].ptr, cols[3].ptr, None,
                                   len(sk), 0, 0, *[o.ptr for o in out], cap, C.byref(m), None)
        return rc, m.value, [o.to_numpy(np.int32, n) for o in out]


@pytest.mark.parametrize("kind", ["dense", "gaps", "spread"])
@pytest.mark.parametrize("misses", [0, 1, 7, 90_000])
def test_rows_past_the_count_are_untouched(qo, orc, kind, misses):
    """Few unmatched S tuples (hardly any of them in a sample) and many, all inside the build range."""
    rng = np.random.default_rng(misses + 1)
    nr, ns = 30_011, 300_007
    rk = build_keys(kind, nr, rng)
    sk = rk[rng.integers(0, nr, ns)]
    free = np.setdiff1d(np.arange(rk.min(), min(int(rk.max()), int(rk.min()) + 60_000)), rk).astype(np.int32)
    if not len(free):                     # every key of the range is a build key
        free = np.array([int(rk.max()) + 1], np.int32)
    sk[rng.permutation(ns)[:misses]] = free[rng.integers(0, len(free), misses)]
    rp, sp = rand32(rng, nr), rand32(rng, ns)
    exp = orc.sort_join_rows(*orc.hash_join(rk, rp, sk, sp, np.zeros(ns, np.int32), 0, 0))
    rc, m, cols = run(qo, rk, rp, sk, sp, ns)
    assert rc == 0 and m == len(exp[0])
    for c, e in zip(cols, exp):
        assert np.array_equal(c[:m], e)
        assert (c[m:] == MARK).all()


@pytest.mark.parametrize("kind", ["dense", "gaps", "spread"])
@pytest.mark.parametrize("short", [1, 1000, 150_000])
def test_nothing_is_written_over_capacity(qo, orc, kind, short):
    rng = np.random.default_rng(short)
    nr, ns = 30_011, 300_007
    rk = build_keys(kind, nr, rng)
    sk = rk[rng.integers(0, nr, ns)]
    rc, m, cols = run(qo, rk, rand32(rng, nr), sk, rand32(rng, ns), ns - short)
    assert rc == 3 and m == ns            # QO_ERR_CAPACITY
    for c in cols:
        assert (c == MARK).all()


@pytest.mark.parametrize("kind", ["gaps", "spread"])
@pytest.mark.parametrize("misses", [5, 90_000])
def test_outputs_that_hold_the_matches_exactly(qo, orc, kind, misses):
    """Room for the rows but not for every S tuple in the build range."""
    rng = np.random.default_rng(misses)
    nr, ns = 30_011, 300_007
    rk = build_keys(kind, nr, rng)
    sk = rk[rng.integers(0, nr, ns)]
    free = np.setdiff1d(np.arange(rk.min(), int(rk.min()) + 60_000), rk).astype(np.int32)
    free = free[(free > rk.min()) & (free < rk.max())]
    sk[rng.permutation(ns)[:misses]] = free[rng.integers(0, len(free), misses)]
    rp, sp = rand32(rng, nr), rand32(rng, ns)
    exp = orc.sort_join_rows(*orc.hash_join(rk, rp, sk, sp, np.zeros(ns, np.int32), 0, 0))
    m = len(exp[0])
    assert m == ns - misses
    rc, got, cols = run(qo, rk, rp, sk, sp, m)
    assert rc == 0 and got == m
    for c, e in zip(cols, exp):
        assert np.array_equal(c[:m], e) and (c[m:] == MARK).all()
