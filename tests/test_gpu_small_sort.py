"""GPU: the one-work-group sort of small arrays and the one-launch end of a
group-by, at the edges of their size ranges, against the oracle (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SIZES = [1, 2, 63, 64, 65, 1023, 1024, 1025, 4095, 4096, 4097, 8191, 8192, 8193]


@pytest.mark.parametrize("bits", [0, 7, 20, 32])
@pytest.mark.parametrize("n", SIZES)
def test_small_sort_records(qo, orc, n, bits):
    """Stable over ties (0 bits: one key), digits that all keys share, full-range keys."""
    rec = np.empty((n, 2), np.uint32)
    rec[:, 0] = np.arange(n)
    y = orc.gen_uniform_u32(n, 5, 1, 0, 0)
    rec[:, 1] = (y & np.uint32((1 << bits) - 1 if bits < 32 else 0xFFFFFFFF)) + np.uint32(0x7F0000 if bits < 32 else 0)
    assert np.array_equal(qo.operators.sort_records(rec), orc.sort_records(rec))


@pytest.mark.parametrize("span", [1, 9, 1 << 31])
@pytest.mark.parametrize("m", SIZES)
def test_small_sort_join_rows(qo, orc, m, span):
    """Signed keys around zero, runs longer than 64 rows (span 1 and 9), repeated s_payloads."""
    k = (orc.gen_uniform_u32(m, 6, 0, 0, span).astype(np.int64) - span // 2).astype(np.int32)
    sp = orc.gen_uniform_u32(m, 6, 1, 0, 0).astype(np.int32)
    sp[::3] = -5
    rp = k * np.int32(3) + np.int32(1)  # a function of the key: rows that tie are identical
    got = qo.operators.sort_join_rows(k, rp, sp)
    exp = orc.sort_join_rows(k, rp, sp)
    for g, e in zip(got, exp):
        assert np.array_equal(g, e)


@pytest.mark.parametrize("groups,n", [(1, 5000), (1023, 5000), (1024, 40000), (1025, 40000), (2048, 70001),
                                      (2049, 70001), (2048, (1 << 20) + 3)])
def test_group_finish_edges(qo, orc, groups, n):
    """Capacities around the one-launch end's limits, with the empty-marker key; the last size takes the
    partitioned path, whose groups arrive as finished rows."""
    k = orc.gen_uniform_u32(n, 7, 0, 0, groups).astype(np.int64) * 7919 - 12345
    k[k == -12345 + 7919 * (groups - 1)] = -1
    k = k.astype(np.int32)
    v = orc.gen_uniform_u32(n, 7, 1, 0, 0).astype(np.int32)
    for g, e in zip(qo.operators.groupby_agg(k, v, groups), orc.groupby_agg(k, v)):
        assert np.array_equal(g, e)


@pytest.mark.parametrize("cap", [1, 100, 1024, 1500])
def test_group_finish_over_capacity(qo, orc, cap):
    """More keys than the outputs hold: the count says so (or that the table overflowed)."""
    k = orc.gen_uniform_u32(60000, 8, 0, 0, 50000).astype(np.int32)
    with pytest.raises(qo._lib.QoError):
        qo.operators.groupby_agg(k, k, cap)


@pytest.mark.parametrize("m,hot", [(60000, 65), (60000, 6144), (60000, 6145), (200000, 17000), (200000, 40000),
                                   (400000, 64)])
def test_join_rows_long_runs(qo, orc, m, hot):
    """Keys of more than 64 rows: sorted in LDS (to 6144 rows), by passes of one work-group, or, past its limit, on
    the full width; many long runs and several hot keys; constant and negative s_payloads."""
    rng = np.random.default_rng(m + hot)
    k = rng.integers(-m, m, m).astype(np.int32)
    k[:hot] = 12
    k[hot:hot + 300] = -7
    if hot == 64:
        k = rng.integers(0, m // 75, m).astype(np.int32)   # most keys past 64 rows: more runs than the list holds
    k = rng.permutation(k)
    sp = rng.integers(-(1 << 31), (1 << 31) - 1, m, dtype=np.int64).astype(np.int32)
    sp[k == -7] = 5
    rp = k * np.int32(3) + np.int32(1)
    for g, e in zip(qo.operators.sort_join_rows(k, rp, sp), orc.sort_join_rows(k, rp, sp)):
        assert np.array_equal(g, e)


@pytest.mark.parametrize("groups,n", [(16, 300_000), (16, 320_000), (1024, 126_000), (1024, 140_000), (5000, 40_000),
                                      (2000, 1_000_003), (70_000, 900_000)])
def test_group_merge_edges(qo, orc, groups, n):
    """Around the number of blocks from which a launch merges their tables; more groups than one table holds; the
    empty-marker key."""
    k = (orc.gen_uniform_u32(n, 9, 0, 0, groups).astype(np.int64) * 2_654_435_761).astype(np.uint32).astype(np.int32)
    k[k == k[0]] = -1
    v = orc.gen_uniform_u32(n, 9, 1, 0, 0).astype(np.int32)
    for g, e in zip(qo.operators.groupby_agg(k, v, groups), orc.groupby_agg(k, v)):
        assert np.array_equal(g, e)


@pytest.mark.parametrize("mask", [0x0, 0xFF, 0xFF00, 0xFFFFF, 0xFF00FF00, 0xFF0000FF, 0xFF000000, 0xFFFFFFFF])
@pytest.mark.parametrize("n", [8193, 70001, (1 << 20) + 4097])
def test_sort_records_skips_equal_digits(qo, orc, n, mask):
    """Keys that vary in some digits only: zero to four passes, ending in either buffer; aligned and not."""
    y = orc.gen_uniform_u32(n + 1, 10, 2, 0, 0) & np.uint32(mask) | np.uint32(0x01020304 & ~mask)
    rec = np.stack([np.arange(n + 1, dtype=np.uint32), y], 1)
    assert np.array_equal(qo.operators.sort_records(rec[:n]), orc.sort_records(rec[:n]))
    with qo.device.DeviceBuffer.from_numpy(rec) as d:  # records at an 8-byte offset
        qo._lib.call("qo_sort_records", d.ptr + 8, n, None)
        got = d.to_numpy(np.uint32, 2 * n + 2).reshape(-1, 2)
    assert np.array_equal(got[1:], orc.sort_records(rec[1:])) and np.array_equal(got[0], rec[0])
