"""GPU: hash group-by at the edges of its rules, against the oracle (exact)."""
import ctypes as C
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("capacity", [131_071, 131_072, 131_073])
def test_most_groups_that_a_launch_merges(qo, orc, capacity):
    """Around the number of groups from which the blocks' tables go straight to the global one."""
    n = 400_000
    k = (orc.gen_uniform_u32(n, 3, 0, 0, 100_000).astype(np.int64) * 2_654_435_761).astype(np.uint32).astype(np.int32)
    k[:5] = -1
    v = orc.gen_uniform_u32(n, 3, 1, 0, 0).astype(np.int32)
    for g, e in zip(qo.operators.groupby_agg(k, v, capacity), orc.groupby_agg(k, v)):
        assert np.array_equal(g, e)


def group_us(qo, k, v, capacity):
    """(median time, number of groups, rows) of qo_groupby_agg on device columns."""
    D, n = qo.device.DeviceBuffer, len(k)
    dk, dv = D.from_numpy(k), D.from_numpy(v)
    out = [D(4 * capacity), D(8 * capacity), D(8 * capacity), D(4 * capacity), D(4 * capacity)]
    num, t = D(8), []
    for _ in range(7):
        t0 = time.perf_counter()
        qo._lib.call("qo_groupby_agg", dk.ptr, dv.ptr, n, capacity, *[o.ptr for o in out], num.ptr, None)
        qo._lib.call("qo_device_sync")
        t.append(time.perf_counter() - t0)
    types = [np.int32, np.int64, np.int64, np.int32, np.int32]
    return sorted(t)[3] * 1e6, int(num.to_numpy(np.uint64, 1)[0]), [o.to_numpy(d, capacity) for o, d in zip(out, types)]


@pytest.mark.parametrize("n", [1 << 20, (1 << 22) + 3])
@pytest.mark.parametrize("capacity,groups", [(1025, 4000), (1025, 2049), (2000, 4096), (3072, 4100), (3072, 6000)])
def test_more_groups_than_the_capacity(qo, orc, n, capacity, groups):
    """Past the capacity but not past the table: the exact number, and rows that are true for their keys."""
    k = (orc.gen_uniform_u32(n, 4, 0, 0, groups - 1).astype(np.int64) * 40_503 - 7_000_000).astype(np.int32)
    k[::1001] = -1
    v = orc.gen_uniform_u32(n, 4, 1, 0, 0).astype(np.int32)
    _, num, rows = group_us(qo, k, v, capacity)
    exp = orc.groupby_agg(k, v)
    assert num == len(exp[0]) > capacity
    at = np.searchsorted(exp[0], rows[0])
    assert (np.diff(rows[0].astype(np.int64)) > 0).all()
    for g, e in zip(rows, exp):
        assert np.array_equal(g, np.asarray(e)[at])


@pytest.mark.parametrize("filtered", [False, True])
@pytest.mark.parametrize("aligned", [False, True])
def test_share_launch_forms(qo, orc, filtered, aligned):
    """The second launch's forms: 4-byte loads, a filter, a dominant key, a key of the empty-marker pattern."""
    n, capacity, groups = (1 << 20) + 7, 3072, 5000
    rng = np.random.default_rng(6)
    k = rng.integers(0, groups, n).astype(np.int32) * 977 - 100
    k[rng.random(n) < 0.2] = 977 * 3 - 100
    k[::997] = -1
    v, f = rng.integers(-(1 << 31), 1 << 31, n, dtype=np.int64).astype(np.int32), rng.integers(0, 10, n).astype(np.int32)
    keep = f <= 6 if filtered else np.ones(n, bool)
    exp = orc.groupby_agg(k[keep], v[keep])
    D, off = qo.device.DeviceBuffer, 0 if aligned else 1
    cols = [D.from_numpy(np.concatenate([np.zeros(off, np.int32), a])) for a in (k, v, f)]
    p = [c.ptr + 4 * off for c in cols]
    types = [np.int32, np.int64, np.int64, np.int32, np.int32]
    out, num = [D(8 * capacity) for _ in types], D(8)
    if filtered:
        qo._lib.call("qo_groupby_agg_filtered", *p, n, 0, 6, capacity, *[o.ptr for o in out], num.ptr, None)
    else:
        qo._lib.call("qo_groupby_agg", p[0], p[1], n, capacity, *[o.ptr for o in out], num.ptr, None)
    qo._lib.call("qo_device_sync")
    assert int(num.to_numpy(np.uint64, 1)[0]) == len(exp[0])
    rows = [o.to_numpy(t, capacity) for o, t in zip(out, types)]
    at = np.searchsorted(exp[0], rows[0])
    for g, e in zip(rows, exp):
        assert np.array_equal(g, np.asarray(e)[at])


def test_more_groups_than_the_capacity_cost_no_tuple_by_tuple_merge(qo, orc):
    n = 1 << 24
    k, v = orc.gen_uniform_u32(n, 5, 0, 0, 0), orc.gen_uniform_u32(n, 5, 1, 0, 0).astype(np.int32)
    fits = group_us(qo, (k % 3000).astype(np.int32), v, 3072)[0]
    more = group_us(qo, (k % 6000).astype(np.int32), v, 3072)[0]
    assert more < 6 * fits, (fits, more)
