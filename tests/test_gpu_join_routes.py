"""GPU: what the sorted join's look at S may cost a join that then takes the
probe and the sort all the same, next to the same join sent there at once (tune
operator 5, param 4): a ratio within one process, and equal rows."""
import ctypes as C
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
JOIN_PART, AUTO, L2 = 5, 0, 4
INT_MIN, INT_MAX = -(1 << 31), (1 << 31) - 1


class Join:
    """The tables on the device and a call of qo_hj_filter_sort."""

    def __init__(self, qo, rk, sk):
        rng = np.random.default_rng(1)
        D, self.qo, self.nr, self.ns = qo.device.DeviceBuffer, qo, len(rk), len(sk)
        rand = lambda n: rng.integers(INT_MIN, INT_MAX, n, dtype=np.int64).astype(np.int32)
        self.tb = qo._lib.load().qo_join_table_bytes(self.nr)
        self.table, self.cap = D(self.tb), 2 * self.ns
        self.cols = [D.from_numpy(a.astype(np.int32)) for a in (rk, rand(self.nr), sk, rand(self.ns))]
        self.out, self.m = [D(4 * self.cap) for _ in range(3)], C.c_uint64()

    def run(self):
        r, rp, s, sp = [c.ptr for c in self.cols]
        self.qo._lib.call("qo_hj_filter_sort", self.table.ptr, self.tb, r, rp, self.nr, s, sp, None, self.ns, 0, 0,
                          *[o.ptr for o in self.out], self.cap, C.byref(self.m), None)

    def route(self, param):
        lib, cls = self.qo._lib.load(), self.ns.bit_length() - 1
        b, i, p = C.c_int(), C.c_int(), C.c_int()
        lib.qo_tune_get(JOIN_PART, cls, C.byref(b), C.byref(i), C.byref(p))
        lib.qo_tune_set(JOIN_PART, cls, b, i, param)

    def us(self):
        t = []
        for _ in range(15):
            t0 = time.perf_counter()
            self.run()
            t.append(time.perf_counter() - t0)
        return sorted(t)[7] * 1e6

    def rows(self):
        return [o.to_numpy(np.int32, self.m.value) for o in self.out]


def compare(qo, rk, sk, most):
    """Times with the sorted join's choice and without it; the same rows either way (when R's keys are distinct)."""
    j = Join(qo, rk, sk)
    off = on = float("inf")
    for i in range(9):  # in turn, so that a slow moment of the host is no one side's
        if i >= 3 and on < most * off:
            break
        j.route(L2)
        off, want = min(off, j.us()), j.rows()
        j.route(AUTO)
        on, got = min(on, j.us()), j.rows()
    print(f"{on:.0f} us, {off:.0f} sent to the probe at once: {on / off:.2f} of at most {most}", flush=True)
    if len(np.unique(rk)) == len(rk):
        for g, w in zip(got, want):
            assert np.array_equal(g, w)
    assert on < most * off, (on, off)


def keys(kind, nr, rng):
    k = rng.permutation(nr).astype(np.int64)
    return (k * 1_640_531_527 + 7) & 0x7FFFFFFF if kind == "spread" else k


@pytest.mark.parametrize("kind", ["dense", "spread"])
@pytest.mark.parametrize("nr,ns,hot", [(4096, 16384, 1.0), (20_000, 100_000, 1.0), (20_000, 100_000, 0.3)])
def test_hot_key_costs_no_serial_count(qo, kind, nr, ns, hot):
    rng = np.random.default_rng(ns)
    rk = keys(kind, nr, rng)
    sk = rk[rng.integers(0, nr, ns)]
    sk[: int(hot * ns)] = rk[3]
    compare(qo, rk, rng.permutation(sk), 1.3)


@pytest.mark.parametrize("kind", ["dense", "spread"])
@pytest.mark.parametrize("nr,ns", [(1 << 22, 1 << 14), (1 << 24, 1 << 14), (1 << 24, 1 << 18)])
def test_small_probe_of_a_large_build_side(qo, kind, nr, ns):
    """Few S tuples and many build keys: no bucket per slice of the build side for them."""
    rng = np.random.default_rng(nr + ns)
    rk = keys(kind, nr, rng)
    compare(qo, rk, rk[rng.integers(0, nr, ns)], 1.2)


@pytest.mark.parametrize("kind", ["dense", "spread"])
def test_small_probe_keeps_a_small_workspace(qo, kind):
    """The device memory that a join of 2^16 rows with 2^24 build keys leaves reserved beside its tables."""
    import torch
    rng = np.random.default_rng(5)
    nr, ns = 1 << 24, 1 << 16
    rk = keys(kind, nr, rng)
    j = Join(qo, rk, rk[rng.integers(0, nr, ns)])
    used = []
    for route in (L2, AUTO):
        j.route(route)
        qo._lib.call("qo_release_workspaces")
        free = torch.cuda.mem_get_info()[0]
        j.run()
        used.append(free - torch.cuda.mem_get_info()[0])
    assert used[1] < 1.5 * used[0] + (64 << 20), used


def cases(nr, ns, kind):
    """Joins that leave the sorted join: (name, R keys, S keys)."""
    rng = np.random.default_rng(nr)
    rk = keys(kind, nr, rng)
    sk = rk[rng.integers(0, nr, ns)]
    dup = rk.copy()
    dup[:3] = dup[-3:]
    yield "repeated build keys", dup, sk
    hot = sk.copy()
    hot[: ns // 20] = rk[5]                  # more rows than a bucket holds
    yield "hot key", rk, rng.permutation(hot)
    yield "few keys referenced", rk, np.sort(rk)[rng.integers(0, 40, ns)]


@pytest.mark.parametrize("kind", ["dense", "spread"])
@pytest.mark.parametrize("nr,ns", [(200_000, 2_000_000), (1_500_000, 6_000_000)])
def test_joins_that_leave_the_sorted_join(qo, kind, nr, ns):
    for name, rk, sk in cases(nr, ns, kind):
        print(name, flush=True)
        compare(qo, rk, sk, 1.12)
