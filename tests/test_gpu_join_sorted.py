"""GPU: the key-order split of qo_hj_filter_sort (dense and spread keys, one and
two splits) and the calls that leave it for the generic path, against the
oracle (exact, rows in order)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
INT_MIN, INT_MAX = -(1 << 31), (1 << 31) - 1


def rand32(rng, n):
    return rng.integers(INT_MIN, INT_MAX, n, dtype=np.int64, endpoint=True).astype(np.int32)


def check(qo, orc, rk, rp, sk, sp, sf, lo, hi, cap=None):
    got = qo.operators.hj_filter_sort(rk, rp, sk, sp, sf, lo, hi, cap)
    exp = orc.sort_join_rows(*orc.hash_join(rk, rp, sk, sp, sf, lo, hi))
    assert len(got[0]) == len(exp[0])
    for g, e in zip(got, exp):
        assert np.array_equal(g, e)


def keys(kind, nr, rng):
    k = rng.permutation(nr).astype(np.int64)
    if kind == "spread":                      # 31-bit keys around zero, all distinct
        k = ((k * 1_640_531_527 + 7) & 0x7FFFFFFF) - (1 << 30)
    elif kind == "full":                      # both ends of int32
        k = (k * 2_654_435_761 + 99) % (1 << 32) - (1 << 31)
        k[:2] = np.array([INT_MIN, INT_MAX])[:nr]
        k = np.unique(k)
        rng.shuffle(k)
    elif kind == "gaps":                      # a key-range table with empty slots, negative base
        k = k + (k >> 1) - nr // 2
    elif kind == "clustered":                 # half the keys in a narrow interval: uneven buckets
        k = np.where(k % 2 == 0, k, k * 4001)
        k = np.unique(k)
        rng.shuffle(k)
    return k.astype(np.int32)


@pytest.mark.parametrize("kind", ["dense", "gaps", "spread", "full", "clustered"])
@pytest.mark.parametrize("nr,ns,sel", [(1, 20000, 1.0), (5, 16384, 0.5), (700, 16383, 0.5), (3000, 16385, 0.03),
                                       (4096, 65536, 1.0), (40001, 250007, 0.4)])
def test_sorted_join_matches_oracle(qo, orc, kind, nr, ns, sel):
    rng = np.random.default_rng(nr + ns)
    rk = keys(kind, nr, rng)
    nr = len(rk)
    sk = rk[rng.integers(0, nr, ns)]
    sk[::17] = rand32(rng, len(sk[::17]))      # keys without a match, most of them outside the range
    sp = rand32(rng, ns)
    sp[::5] = 3                                # ties
    sf = rng.integers(0, 1000, ns).astype(np.int32)
    check(qo, orc, rk, rand32(rng, nr), sk, sp, sf, 0, int(1000 * sel) - 1)


@pytest.mark.parametrize("kind", ["dense", "spread"])
def test_sorted_join_two_splits(qo, orc, kind):
    rng = np.random.default_rng(5)
    nr, ns = 400_003, 2_900_017
    rk = keys(kind, nr, rng)
    sk = rk[rng.integers(0, nr, ns)]
    check(qo, orc, rk, rand32(rng, nr), sk, rand32(rng, ns), rng.integers(0, 4, ns).astype(np.int32), 0, 3)


@pytest.mark.parametrize("kind", ["dense", "spread"])
@pytest.mark.parametrize("hot", [0.02, 0.3, 1.0])
def test_sorted_join_hot_key(qo, orc, kind, hot):
    """One key holds a share of S: a long run in its bucket, a bucket that overflows, or a spread the sample rejects."""
    rng = np.random.default_rng(9)
    nr, ns = 20000, 300_000
    rk = keys(kind, nr, rng)
    sk = rk[rng.integers(0, nr, ns)]
    sk[: int(hot * ns)] = rk[77]
    sk = rng.permutation(sk)
    check(qo, orc, rk, rand32(rng, nr), sk, rand32(rng, ns), np.zeros(ns, np.int32), 0, 0)


def test_sorted_join_repeated_build_keys_and_sentinel(qo, orc):
    rng = np.random.default_rng(11)
    ns = 40000
    rk = (np.arange(3000) % 2999).astype(np.int32)          # one key twice, with one payload
    sk = rng.integers(0, 3100, ns).astype(np.int32)
    check(qo, orc, rk, rk * 2, sk, rand32(rng, ns), np.zeros(ns, np.int32), 0, 0, 2 * ns)
    rk = np.arange(-1, 2999).astype(np.int32)               # (-1, -1): the empty slot's bit pattern
    sk = rng.integers(-3, 3000, ns).astype(np.int32)
    check(qo, orc, rk, rk, sk, rand32(rng, ns), np.zeros(ns, np.int32), 0, 0)


def test_sorted_join_capacity_and_no_rows(qo, orc):
    rng = np.random.default_rng(12)
    nr, ns = 5000, 50000
    rk = keys("dense", nr, rng)
    sk = rk[rng.integers(0, nr, ns)]
    sf = rng.integers(0, 10, ns).astype(np.int32)
    a = (rk, rand32(rng, nr), sk, rand32(rng, ns), sf)
    m = len(orc.hash_join(*a, 0, 4)[0])
    check(qo, orc, *a, 0, 4, m)                              # the outputs hold the rows exactly
    with pytest.raises(qo._lib.QoError):
        qo.operators.hj_filter_sort(*a, 0, 4, m - 1)
    check(qo, orc, *a, 7, 6)                                 # an empty filter range
    check(qo, orc, rk, a[1], sk + nr, a[3], sf, 0, 9)        # no S key in the build range


def test_sorted_join_unaligned_columns(qo, orc):
    """Columns at 4-byte offsets (no 16-byte loads), through the C entry point."""
    import ctypes as C
    rng = np.random.default_rng(13)
    nr, ns = 9001, 70001
    rk, D = keys("gaps", nr, rng), qo.device.DeviceBuffer
    rp, sp = rand32(rng, nr), rand32(rng, ns)
    sk, sf = rk[rng.integers(0, nr, ns)], rng.integers(0, 9, ns).astype(np.int32)
    lib = qo._lib.load()
    tb = lib.qo_join_table_bytes(nr)
    with D(tb) as t, D(4 * ns + 8) as ok, D(4 * ns + 8) as orp, D(4 * ns + 8) as osp:
        cols = [D.from_numpy(np.concatenate([np.zeros(1, np.int32), a])) for a in (rk, rp, sk, sp, sf)]
        m = C.c_uint64()
        qo._lib.call("qo_hj_filter_sort", t.ptr, tb, cols[0].ptr + 4, cols[1].ptr + 4, nr, cols[2].ptr + 4,
                     cols[3].ptr + 4, cols[4].ptr + 4, ns, 0, 5, ok.ptr + 4, orp.ptr + 4, osp.ptr + 4, ns, C.byref(m),
                     None)
        exp = orc.sort_join_rows(*orc.hash_join(rk, rp, sk, sp, sf, 0, 5))
        assert m.value == len(exp[0])
        for b, e in zip((ok, orp, osp), exp):
            assert np.array_equal(b.to_numpy(np.int32, m.value + 1)[1:], e)
