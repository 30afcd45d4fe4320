"""GPU: per-group aggregates over group start positions of uneven lengths, at the
edges of the work units and of the search for a unit's group, against the oracle
(exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def lengths(kind, rng):
    if kind == "one":
        return [300_001]
    if kind == "edges":  # around one unit and one load of its lanes
        return [1, 7, 8, 9, 127, 128, 129, 255, 256, 257, 0, 0, 1, 1024, 0]
    if kind == "hot":  # a group of thousands of units between single rows, runs of empty groups
        return [1] * 77 + [400_000] + [0] * 130 + [1] * 9 + [150_000, 0, 3]
    if kind == "tail":  # the last group ends mid-unit, the one before is long
        return [70_000, 1]
    if kind == "none":  # only empty groups but the first row's
        return [1] + [0] * 1000
    return rng.integers(0, 400, int(kind)).tolist()


@pytest.mark.parametrize("kind", ["one", "edges", "hot", "tail", "none", "7", "8", "9", "63", "64", "65", "513", "5000"])
def test_aggregate_uneven_groups(qo, orc, kind):
    from query_on_opencl_fpga_amd.device import DeviceBuffer
    rng = np.random.default_rng(17)
    ln = np.array(lengths(kind, rng), np.int64)
    n, g = int(ln.sum()), len(ln)
    sp = (np.cumsum(ln) - ln).astype(np.int32)
    rec = np.empty((n, 2), np.uint32)
    rec[:, 0] = orc.gen_uniform_u32(n, 11, 0, 0, 0)
    rec[:, 1] = np.repeat(np.arange(g, dtype=np.uint32), ln)
    with DeviceBuffer.from_numpy(rec) as ds, DeviceBuffer.from_numpy(sp) as dsp, DeviceBuffer(g * 4) as out:
        for op in range(4):
            qo._lib.call("qo_aggregate_groups", ds.ptr, n, dsp.ptr, g, op, out.ptr, None)
            got, exp = out.to_numpy(np.int32, g), orc.parallel_aggregate(rec, sp, op)
            assert np.array_equal(got, exp), (op, np.flatnonzero(got != exp)[:5])
