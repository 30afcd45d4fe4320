"""GPU: what the planner measures of the device is possible on it."""
import time

import pytest

from query_on_opencl_fpga_amd import planner as P

pytestmark = pytest.mark.gpu
SORT_PASS = 1


def test_sort_pass_is_no_faster_than_a_copy(qo):
    """A radix pass reads the rows twice and writes them scattered: its bytes cannot pass faster than a copy's."""
    D, n = qo.device.DeviceBuffer, 1 << 28
    t = []
    with D(n) as a, D(n) as b:
        for _ in range(9):
            qo._lib.call("qo_device_sync")
            t0 = time.perf_counter()
            for _ in range(20):
                qo._lib.call("qo_copy", a.ptr, b.ptr, n, None)
            qo._lib.call("qo_device_sync")
            t.append((time.perf_counter() - t0) / 20)
    copy_gbps = 2 * n / min(t) / 1e9
    saved = P.cost_table()
    try:
        assert P.calibrate(24, 5)[SORT_PASS][1] < copy_gbps
    finally:
        for i, (f, g) in enumerate(saved):
            P.set_cost(i, f, g)


def test_built_in_costs_are_this_device(qo):
    """The table a plan starts from, next to a calibration at the size it was taken at: within a factor of two."""
    built_in = P.cost_table()
    try:
        measured = P.calibrate(26, 5)
    finally:
        for i, (f, g) in enumerate(built_in):
            P.set_cost(i, f, g)
    for name, (f0, g0), (f1, g1) in zip(P.COST_NAMES, built_in, measured):
        assert 0.5 < g0 / g1 < 2 and (0.5 < f0 / f1 < 2 or abs(f0 - f1) < 5), (name, f0, g0, f1, g1)
