"""GPU: hash group-by at the edges of its rules, against the oracle (exact)."""
import ctypes as C
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("capacity", [131_071, 131_072, 131_073])
def test_most_groups_that_a_launch_merges(qo, orc, capacity):
    """Around the number of groups from which the blocks' tables go straight to the global one."""
    n = 400_000
    k = (orc.gen_uniform_u32(n, 3, 0, 0, 100_000).astype(np.int64) * 2_654_435_761).astype(np.uint32).astype(np.int32)
    k[:5] = -1
    v = orc.gen_uniform_u32(n, 3, 1, 0, 0).astype(np.int32)
    for g, e in zip(qo.operators.groupby_agg(k, v, capacity), orc.groupby_agg(k, v)):
        assert np.array_equal(g, e)
