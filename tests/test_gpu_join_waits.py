"""GPU: joins whose bounded device-side waits run out.  With no sleeps allowed a
work-group that finds a predecessor unpublished gives up at once; a synchronous
call then says so instead of returning rows at wrong places."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
QO_OK, QO_ERR_DEVICE_WAIT = 0, 9


@pytest.fixture
def no_patience(qo):
    lib = qo._lib.load()
    assert lib.qo_debug_set_spin_limit(0) == 0
    yield lib
    assert lib.qo_debug_set_spin_limit(1 << 22) == 0
    lib.qo_device_sync()                       # reads and clears the device's error word


def tables(rng, nr, ns):
    rk = (rng.permutation(nr) * 3).astype(np.int32)
    sk = rk[rng.integers(0, nr, ns)]
    sk[::5] += 1                               # no such build key
    return rk, rng.integers(0, 99, nr).astype(np.int32), sk, rng.integers(-99, 99, ns).astype(np.int32)


@pytest.mark.parametrize("nr,ns", [(3000, 40_000), (200_003, 3_000_017)])
def test_join_reports_a_wait_that_ran_out(qo, orc, no_patience, nr, ns):
    rng = np.random.default_rng(nr)
    t = tables(rng, nr, ns)
    exp = orc.sort_join_rows(*orc.hash_join(*t, np.zeros(ns, np.int32), 0, 0))
    D, lib = qo.device.DeviceBuffer, no_patience
    tb = lib.qo_join_table_bytes(nr)
    cols, table, out, m = [D.from_numpy(a) for a in t], D(tb), [D(4 * ns) for _ in range(3)], C.c_uint64()
    for _ in range(10):
        rc = lib.qo_hj_filter_sort(table.ptr, tb, cols[0].ptr, cols[1].ptr, nr, cols[2].ptr, cols[3].ptr, None, ns, 0, 0,
                                   *[o.ptr for o in out], ns, C.byref(m), None)
        if rc == QO_ERR_DEVICE_WAIT:
            continue
        assert rc == QO_OK and m.value == len(exp[0])
        for o, e in zip(out, exp):
            assert np.array_equal(o.to_numpy(np.int32, m.value), e)
    assert lib.qo_device_sync() == QO_OK       # the call reported it: nothing is left for the next one


def test_batch_counts_report_a_wait_that_ran_out(qo, orc, no_patience):
    rng = np.random.default_rng(4)
    D, dev, exp = qo.device.DeviceBuffer, [], []
    for nr, ns in [(2000, 30_000), (30_000, 400_000), (9000, 90_000)]:
        t = tables(rng, nr, ns)
        exp.append(orc.sort_join_rows(*orc.hash_join(*t, np.zeros(ns, np.int32), 0, 0)))
        d = {"nr": nr, "ns": ns, "flo": 0, "fhi": 0, "cap": ns, "sfilt": D.from_numpy(np.zeros(ns, np.int32))}
        d.update({c: D.from_numpy(a) for c, a in zip(("rkey", "rpay", "skey", "spay"), t)})
        d.update({c: D(4 * ns) for c in ("okey", "orpay", "ospay")})
        dev.append(d)
    batch = qo.operators.JoinBatch(dev)
    try:
        for _ in range(10):
            batch.launch()
            try:
                counts = batch.counts()
            except qo._lib.QoError:
                continue
            for d, e, m in zip(dev, exp, counts):
                assert int(m) == len(e[0])
                for c, x in zip(("okey", "orpay", "ospay"), e):
                    assert np.array_equal(d[c].to_numpy(np.int32, int(m)), x)
    finally:
        batch.destroy()
