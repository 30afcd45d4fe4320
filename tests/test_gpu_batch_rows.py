"""GPU: a batch of joins writes the rows of its results and nothing past them,
whatever share of the S tuples has a match, against the oracle (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
INT_MIN, INT_MAX = -(1 << 31), (1 << 31) - 1
MARK = 0x5A5A5A5A


def rand32(rng, n):
    return rng.integers(INT_MIN, INT_MAX, n, dtype=np.int64, endpoint=True).astype(np.int32)


@pytest.mark.parametrize("misses", [0.0, 1e-4, 0.3, 1.0])
def test_batch_rows_past_the_count_are_untouched(qo, orc, misses):
    rng = np.random.default_rng(int(misses * 1e4) + 1)
    D = qo.device.DeviceBuffer
    dev, host = [], []
    for nr, ns, kind in [(1, 700, "even"), (700, 2000, "even"), (5000, 40_000, "even"), (30_011, 200_003, "even"),
                         (9000, 60_000, "dups"), (4000, 50_000, "hot")]:
        rk = (rng.permutation(nr) * 2).astype(np.int32)      # odd keys of the range have no match
        if kind == "dups":
            rk[1] = rk[0]
        sk = rk[rng.integers(0, nr, ns)]
        if kind == "hot":
            sk[: ns // 2] = rk[5]
        miss = rng.random(ns) < misses
        sk[miss] = np.maximum(sk[miss] - 1, 1) | 1
        q = (rk, rk * np.int32(3) if kind == "dups" else rand32(rng, nr), sk, rand32(rng, ns),
             rng.integers(0, 10, ns).astype(np.int32))
        cap = ns + 4096
        d = {"nr": nr, "ns": ns, "flo": 0, "fhi": 8, "cap": cap}
        d.update({c: D.from_numpy(a) for c, a in zip(("rkey", "rpay", "skey", "spay", "sfilt"), q)})
        d.update({c: D.from_numpy(np.full(cap, MARK, np.int32)) for c in ("okey", "orpay", "ospay")})
        dev.append(d)
        host.append(q)
    batch = qo.operators.JoinBatch(dev)
    try:
        batch.launch()
        for d, q, m in zip(dev, host, batch.counts()):
            exp = orc.sort_join_rows(*orc.hash_join(*q, 0, 8))
            assert int(m) == len(exp[0])
            for c, e in zip(("okey", "orpay", "ospay"), exp):
                got = d[c].to_numpy(np.int32, d["cap"])
                assert np.array_equal(got[: len(e)], e)
                assert (got[len(e):] == MARK).all()
    finally:
        batch.destroy()
