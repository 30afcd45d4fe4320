"""GPU: the direct group-by at the edges of its range of groups, and the packed
COUNT and SUM word of its tables where it is emptied, against the oracle or sums
known beforehand (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
INT_MIN, INT_MAX = -(1 << 31), (1 << 31) - 1


def check(got, exp):
    for g, e in zip(got, exp):
        assert np.array_equal(np.asarray(g, np.int64), np.asarray(e, np.int64))


@pytest.mark.parametrize("skip", [0, 1])  # 1: unaligned columns
@pytest.mark.parametrize("groups", [1023, 1024, 1025, 2048, 2049, 3071, 3072, 3073])
def test_direct_range_matches_oracle(qo, orc, groups, skip):
    from query_on_opencl_fpga_amd.device import DeviceBuffer
    n = (1 << 20) + 5
    k = (orc.gen_uniform_u32(n + skip, 31, 0, 0, groups).astype(np.int64) * 48271 - 7).astype(np.int32)
    k[::97] = -1  # the empty-marker key, in place of one of the others
    k[k == 48271 - 7] = -1
    v = orc.gen_uniform_u32(n + skip, 31, 1, 0, 0).astype(np.int32)
    v[5], v[6] = INT_MIN, INT_MAX
    if not skip:
        check(qo.operators.groupby_agg(k, v, groups), orc.groupby_agg(k, v))
        return
    exp = orc.groupby_agg(k[1:], v[1:])
    sizes = [4, 8, 8, 4, 4]
    outs = [DeviceBuffer(groups * b) for b in sizes]
    with DeviceBuffer.from_numpy(k) as dk, DeviceBuffer.from_numpy(v) as dv, DeviceBuffer(8) as num:
        qo._lib.call("qo_groupby_agg", dk.ptr + 4, dv.ptr + 4, n, groups, *[o.ptr for o in outs], num.ptr, None)
        g = int(num.to_numpy(np.uint64, 1)[0])
    assert g == len(exp[0])
    check([o.to_numpy(np.int32 if b == 4 else np.int64, g) for o, b in zip(outs, sizes)], exp)
    for o in outs:
        o.free()


def test_packed_word_is_emptied(qo):
    """Each block adds tens of thousands of one value to a group: both fields of the word would overflow."""
    from query_on_opencl_fpga_amd.device import DeviceBuffer
    groups, n = 8, 90_000_008
    vals = np.array([INT_MIN, INT_MAX, -1, 0, 1, INT_MIN + 1, INT_MAX - 1, 12345], np.int32)
    k = np.tile(np.arange(groups, dtype=np.int32), n // groups)
    v = np.tile(vals, n // groups)
    got = qo.operators.groupby_agg(k, v, groups)
    c = n // groups
    check(got, (np.arange(groups), [c] * groups, [c * int(x) for x in vals], vals, vals))
