"""GPU: per-group aggregates where a wave of the kernel holds 64 groups in registers:
group counts around that, one unit per group and several, runs of empty groups as long
as and longer than what is held, and groups far from where even ones would be, against
the oracle (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def lengths(kind):
    if kind == "one unit":  # more than 2^11 waves' first units, each its own group
        return [3] * 70_001
    if kind == "two units":
        return [129, 200] * 3001
    if kind == "held":  # empty groups up to, at and past what a wave holds
        return [5] + [0] * 62 + [5] + [0] * 63 + [5] + [0] * 64 + [300] + [0] * 500 + [1] * 70
    if kind == "late":  # nearly all units in the last groups
        return [0] * 50_000 + [1] * 3000 + [20_000] * 5
    if kind == "early":
        return [20_000] * 5 + [1] * 3000 + [0] * 50_000
    return [130] * int(kind)


@pytest.mark.parametrize("kind", ["one unit", "two units", "held", "late", "early", "31", "32", "33", "62", "4097"])
def test_groups_held_by_a_wave(qo, orc, kind):
    from query_on_opencl_fpga_amd.device import DeviceBuffer
    ln = np.array(lengths(kind), np.int64)
    n, g = int(ln.sum()), len(ln)
    sp = (np.cumsum(ln) - ln).astype(np.int32)
    rec = np.empty((n, 2), np.uint32)
    rec[:, 0] = orc.gen_uniform_u32(n, 12, 0, 0, 0)
    rec[:, 1] = np.repeat(np.arange(g, dtype=np.uint32), ln)
    with DeviceBuffer.from_numpy(rec) as ds, DeviceBuffer.from_numpy(sp) as dsp, DeviceBuffer(g * 4) as out:
        for op in range(4):
            qo._lib.call("qo_aggregate_groups", ds.ptr, n, dsp.ptr, g, op, out.ptr, None)
            got, exp = out.to_numpy(np.int32, g), orc.parallel_aggregate(rec, sp, op)
            assert np.array_equal(got, exp), (op, np.flatnonzero(got != exp)[:5])
