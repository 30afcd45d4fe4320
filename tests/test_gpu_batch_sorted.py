"""GPU: the batch's sorted join of small queries, the queries it leaves to the
generic stages, and replays on refreshed columns, against the oracle (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
INT_MIN, INT_MAX = -(1 << 31), (1 << 31) - 1


def rand32(rng, n):
    return rng.integers(INT_MIN, INT_MAX, n, dtype=np.int64, endpoint=True).astype(np.int32)


def query(rng, nr, ns, kind="spread", sel=0.5):
    k = np.arange(nr, dtype=np.int64)
    if kind == "spread":
        k = ((k * 1_640_531_527 + 7) & 0x7FFFFFFF) - (1 << 30)
    elif kind == "full" and nr > 1:
        k[0], k[-1] = INT_MIN, INT_MAX
    elif kind == "dups" and nr > 1:
        k[1] = k[0]
    rk = rng.permutation(k).astype(np.int32)
    sk = rk[rng.integers(0, nr, ns)] if nr else rand32(rng, ns)
    if kind == "misses":
        sk[::3] = rand32(rng, len(sk[::3]))
    if kind == "hot":
        sk[: ns // 2] = rk[0]
    rp = rk * np.int32(7) if kind == "dups" else rand32(rng, nr)
    sp = rand32(rng, ns)
    sp[::4] = 1
    if kind == "run":                        # a run too long to rank row against row, narrow payloads
        sk[:900] = rk[-1]
        sp = rng.integers(0, 50, ns).astype(np.int32)
    sf = rng.integers(0, 1000, ns).astype(np.int32)
    return rk, rp, sk, sp, sf, 0, int(1000 * sel) - 1


def expect(orc, q):
    return orc.sort_join_rows(*orc.hash_join(*q))


SHAPES = [(1, 1, "dense", 1.0), (0, 50, "dense", 1.0), (40, 0, "dense", 1.0), (1, 3000, "dense", 1.0),
          (768, 2304, "spread", 1.0), (769, 2304, "spread", 1.0), (768, 2305, "dense", 1.0), (5000, 30011, "misses", 0.7),
          (5000, 20000, "full", 0.5), (3000, 9000, "run", 1.0), (20000, 90001, "spread", 0.05), (9000, 9000, "spread", 0.0)]


@pytest.mark.parametrize("extra", [[], [(2000, 8000, "dups", 0.5)], [(500, 40000, "hot", 1.0)], [(300_000, 20000, "spread", 0.5)],
                                   [(400_001, 8, "dense", 1.0), (64, 64, "dups", 1.0)]])
def test_batch_sorted_matches_oracle(qo, orc, extra):
    """All small; with a query that repeats a build key, one whose bucket overflows, and ones too large."""
    rng = np.random.default_rng(len(extra) + 3)
    qs = [query(rng, *s) for s in SHAPES + extra]
    got = qo.operators.batch_hj_filter_sort(qs, [2 * len(q[2]) + 1 for q in qs])
    for q, g in zip(qs, got):
        for a, e in zip(g, expect(orc, q)):
            assert np.array_equal(a, e)


def test_batch_sorted_replays_on_refreshed_columns(qo, orc):
    """The same plan launched on other keys, payloads and selectivities: nothing of the first values is kept."""
    rng = np.random.default_rng(21)
    D = qo.device.DeviceBuffer
    shapes = [(3000, 24000), (700, 2000), (12000, 60000)]
    dev = []
    for nr, ns in shapes:
        d = {"nr": nr, "ns": ns, "flo": 0, "fhi": 499, "cap": 2 * ns}
        d.update({c: D(4 * nr) for c in ("rkey", "rpay")}, **{c: D(4 * ns) for c in ("skey", "spay", "sfilt")},
                 **{c: D(8 * ns) for c in ("okey", "orpay", "ospay")})
        dev.append(d)
    batch = qo.operators.JoinBatch(dev)
    try:
        for kinds in (("spread",) * 3, ("dense", "full", "misses"), ("dups", "spread", "hot"), ("spread", "dense", "run")):
            qs = [query(rng, nr, ns, k) for (nr, ns), k in zip(shapes, kinds)]
            for d, q in zip(dev, qs):
                for c, a in zip(("rkey", "rpay", "skey", "spay", "sfilt"), q):
                    d[c].write(a)
            for _ in range(2):
                batch.launch()
                counts = batch.counts()
                for d, q, m in zip(dev, qs, counts):
                    exp = expect(orc, q)
                    assert int(m) == len(exp[0])
                    for c, e in zip(("okey", "orpay", "ospay"), exp):
                        assert np.array_equal(d[c].to_numpy(np.int32, int(m)), e)
    finally:
        batch.destroy()


def test_batch_sorted_over_capacity(qo, orc):
    rng = np.random.default_rng(22)
    qs = [query(rng, 100, 5000, "dense", 1.0), query(rng, 100, 400, "dense", 1.0)]
    with pytest.raises(qo._lib.QoError):
        qo.operators.batch_hj_filter_sort(qs, [4999, 400])
