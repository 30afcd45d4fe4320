"""GPU: tiny queries of a batch, whatever the span of their build keys: rows
against the oracle, and no query sent to the generic stages for its span alone
(which would cost the whole batch several times the sorted join's time)."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
INT_MIN, INT_MAX = -(1 << 31), (1 << 31) - 1


def build_keys(nr, kind, rng):
    k = rng.integers(-1000, 1000, nr * 8)
    if kind == "span over a power of two":           # 2^20 + 2 keys wide
        k = np.concatenate([[0, (1 << 20) + 1], rng.integers(1, 1 << 20, nr * 2)])
    elif kind == "span of 2^31":
        k = np.concatenate([[-5, (1 << 31) - 6], rng.integers(0, 1 << 30, nr * 2)])
    elif kind == "full":
        k = np.concatenate([[INT_MIN, INT_MAX], rng.integers(INT_MIN, INT_MAX, nr * 2)])
    k = np.unique(k)
    keep = np.r_[0, len(k) - 1, 1 + rng.permutation(len(k) - 2)[: nr - 2]] if nr > 1 else np.array([0])
    return rng.permutation(k[keep]).astype(np.int32)


def queries(kind, shapes, rng):
    for nr, ns in shapes:
        rk = build_keys(nr, kind, rng)
        sk = rk[rng.integers(0, len(rk), ns)]
        yield (rk, rng.integers(INT_MIN, INT_MAX, len(rk)).astype(np.int32), sk,
               rng.integers(INT_MIN, INT_MAX, ns).astype(np.int32), np.zeros(ns, np.int32))


@pytest.mark.parametrize("kind", ["narrow", "span over a power of two", "span of 2^31", "full"])
def test_tiny_queries_of_any_span(qo, orc, kind):
    rng = np.random.default_rng(1)
    shapes = [(1, 1), (2, 3), (2, 2304), (767, 2000), (768, 2304), (768, 5), (769, 2305), (1500, 5000)]
    qs = [(*q, 0, 0) for q in queries(kind, shapes, rng)]
    for q, got in zip(qs, qo.operators.batch_hj_filter_sort(qs, [len(q[2]) for q in qs])):
        for g, e in zip(got, orc.sort_join_rows(*orc.hash_join(*q))):
            assert np.array_equal(g, e)


def test_span_costs_a_batch_nothing(qo):
    D, us = qo.device.DeviceBuffer, {}
    for kind in ("narrow", "span over a power of two", "full"):
        rng, dev = np.random.default_rng(2), []
        for q in queries(kind, [(700, 2000)] * 64, rng):
            d = {"nr": len(q[0]), "ns": len(q[2]), "flo": 0, "fhi": 0, "cap": len(q[2])}
            d.update({c: D.from_numpy(a) for c, a in zip(("rkey", "rpay", "skey", "spay", "sfilt"), q)})
            d.update({c: D(4 * len(q[2])) for c in ("okey", "orpay", "ospay")})
            dev.append(d)
        batch, t = qo.operators.JoinBatch(dev), []
        for _ in range(9):
            t0 = time.perf_counter()
            batch.launch()
            qo._lib.call("qo_device_sync")
            t.append(time.perf_counter() - t0)
        batch.destroy()
        us[kind] = sorted(t)[4] * 1e6
    assert max(us.values()) < 1.6 * us["narrow"], us
