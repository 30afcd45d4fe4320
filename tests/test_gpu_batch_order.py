"""GPU: batches of as many queries as are planned together and one more, with one
bucket, a few and hundreds, some without rows and some left to the generic stages,
against the oracle (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq", [1, 255, 256, 257, 513])
def test_batch_of_uneven_queries(qo, orc, nq):
    rng = np.random.default_rng(nq)
    D = qo.device.DeviceBuffer
    dev, host = [], []
    for i in range(nq):
        # The last query of the first group of 256 and the first of the next have
        # several hundred buckets.
        nr, ns = (30_011, 600_003) if i in (0, 254, 255, 256) else [(1, 300), (800, 3000), (6000, 9000), (0, 50), (5, 0)][i % 5]
        rk = (rng.permutation(nr) * 7).astype(np.int32)
        if i % 50 == 7 and nr > 1:
            rk[1] = rk[0]  # left to the generic stages
        sk = rk[rng.integers(0, nr, ns)] if nr else rng.integers(0, 99, ns).astype(np.int32)
        sk[rng.random(ns) < 0.2] += 1
        q = (rk, np.full(nr, 9, np.int32) if i % 50 == 7 else rk ^ np.int32(5), sk,
             rng.integers(-(1 << 31), 1 << 31, ns).astype(np.int32), rng.integers(0, 10, ns).astype(np.int32))
        d = {"nr": nr, "ns": ns, "flo": 0, "fhi": 7, "cap": 2 * ns + 8}
        d.update({c: D.from_numpy(a if len(a) else np.zeros(1, np.int32)) for c, a in zip(("rkey", "rpay", "skey", "spay", "sfilt"), q)})
        d.update({c: D.from_numpy(np.zeros(d["cap"], np.int32)) for c in ("okey", "orpay", "ospay")})
        dev.append(d)
        host.append(q)
    batch = qo.operators.JoinBatch(dev)
    try:
        for _ in range(2):
            batch.launch()
            counts = batch.counts()
        for i, (d, q, m) in enumerate(zip(dev, host, counts)):
            exp = orc.sort_join_rows(*orc.hash_join(*q, 0, 7))
            assert int(m) == len(exp[0]), i
            for c, e in zip(("okey", "orpay", "ospay"), exp):
                assert np.array_equal(d[c].to_numpy(np.int32, len(e)) if len(e) else e, e), (i, c)
    finally:
        batch.destroy()
