"""GPU: record compaction where a block takes several tiles, at the edges of a
tile and of one tile per CU, against the oracle (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TILE, CUS = 16384, 256


@pytest.mark.parametrize("skip", [0, 1])  # 1: not 16-byte aligned, tiles of half the size
@pytest.mark.parametrize("n", [TILE - 1, TILE, TILE + 1, TILE * CUS - 1, TILE * CUS, TILE * CUS + 1, TILE * CUS * 2 + 4099])
def test_filter_records_many_tiles(qo, orc, n, skip):
    from query_on_opencl_fpga_amd.device import DeviceBuffer
    r = np.empty((n + skip, 2), np.uint32)
    r[:, 0] = np.arange(n + skip)
    r[:, 1] = orc.gen_uniform_u32(n + skip, 21, 0, 0, 0)
    r[n // 3:n // 2, 1] = 5  # tiles that select all
    r[n // 2:n // 2 + 3 * TILE, 1] = 0xFFFFFFF0  # tiles that select none
    with DeviceBuffer.from_numpy(r) as d, DeviceBuffer(max(n, 1) * 8) as o, DeviceBuffer(8) as c:
        qo._lib.call("qo_filter_records", d.ptr + 8 * skip, n, 0, 1 << 30, o.ptr, c.ptr, None)
        m = int(c.to_numpy(np.uint64, 1)[0])
        got = o.to_numpy(np.uint32, 2 * m).reshape(m, 2)
    assert np.array_equal(got, orc.filter_records(r[skip:], 0, 1 << 30))
