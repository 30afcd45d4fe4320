"""GPU: sort of join rows whose keys repeat.  The rows at the edges of the ways a
long run is sorted, against the oracle, and what repeated keys may cost next to
distinct ones (a ratio within one process: sorting all rows once more on eight
digits instead of four at most triples the time)."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(qo, orc, k, seed):
    rng = np.random.default_rng(seed)
    k = rng.permutation(k).astype(np.int32)
    sp = rng.integers(-(1 << 31), (1 << 31) - 1, len(k), dtype=np.int64).astype(np.int32)
    sp[::7] = -4
    rp = np.arange(len(k), dtype=np.int32)
    for g, e in zip(qo.operators.sort_join_rows(k, rp, sp), orc.sort_join_rows(k, rp, sp)):
        assert np.array_equal(g, e)


@pytest.mark.parametrize("runs", [1, 512, 1029, 1030, 1031])
@pytest.mark.parametrize("length", [65, 90])
def test_number_of_long_runs(qo, orc, runs, length):
    """Around the number of long runs (1024 and one per 16384 rows) past which all rows are sorted on the full width."""
    m = 100_000
    k = np.arange(m) + 10
    k[: runs * length] = -(np.arange(runs * length) // length)
    check(qo, orc, k, runs + length)


@pytest.mark.parametrize("length", [6143, 6144, 6145, 6200, 30_000])
@pytest.mark.parametrize("at", ["first", "last", "middle"])
def test_length_of_a_long_run(qo, orc, length, at):
    """Around the longest run that is sorted in LDS, at either end of the rows."""
    m = 40_000
    k = np.arange(m) * 2
    k[:length] = {"first": -1, "last": 3 * m, "middle": m + 1}[at]
    check(qo, orc, k, length)


def sort_us(qo, key):
    """Median time of qo_sort_join_rows on rows with these keys (already together), s_payloads over 32 bits."""
    D, m = qo.device.DeviceBuffer, len(key)
    rng = np.random.default_rng(1)
    sp = rng.integers(-(1 << 31), (1 << 31) - 1, m, dtype=np.int64).astype(np.int32)
    src = [D.from_numpy(a) for a in (key.astype(np.int32), np.arange(m, dtype=np.int32), sp)]
    dst = [D(4 * m) for _ in range(3)]
    t = []
    for _ in range(9):
        for d, s in zip(dst, src):
            qo._lib.call("qo_memcpy_d2d", d.ptr, s.ptr, 4 * m, None)
        qo._lib.call("qo_device_sync")
        t0 = time.perf_counter()
        qo._lib.call("qo_sort_join_rows", *[d.ptr for d in dst], m, None)
        t.append(time.perf_counter() - t0)
    return sorted(t)[4] * 1e6


@pytest.mark.parametrize("m,length", [(10_000_000, 70), (10_000_000, 20_000), (12_000_000, 50_000), (100_000, 16_000)])
def test_repeated_keys_cost_no_more_than_another_sort(qo, m, length):
    unique, runs = sort_us(qo, np.arange(m)), sort_us(qo, np.arange(m) // length)
    assert runs < 2.5 * unique, (unique, runs)
