"""The checks of a batch's new masks share one buffer: each instance gets the answer of its own mask."""
import numpy as np
import pytest

import xgrid_amd as xgrid
from xgrid_amd.batch import Batch

from helpers import assert_bitexact, grid_pair
from oracle.cpu_path import CpuKernel

pytestmark = pytest.mark.gpu
f2 = xgrid.grid[float, 2]


def _creep():
    @xgrid.kernel()
    def creep(u: f2, n: int) -> None:
        for it in range(0, n):
            u[0, 0] = (u[0, 1][0] + u[0, -1][0] + u[1, 0][0] + u[-1, 0][0]) * 0.25
            with xgrid.boundary(1):
                u[0, 0] = u[0, 3][0]
    return creep


@pytest.mark.parametrize("counts", [(1,), (2, 5), (5, 2, 40)])
def test_masks_of_one_check(double, counts):
    """Along a row of wall cells values move three cells an iteration, too far for a blocked launch;
    down a column of them they do not.  Members are added between steps, so the buffer grows and is used again."""
    k = _creep()
    b = Batch(k)
    rng = np.random.default_rng(4)
    trip, pairs = 12, []
    for count in counts:
        for i in range(count):
            n = 150 + 7 * i
            mask = np.full((n, n), 9, np.int32)
            mask[1:-1, 1:-1] = 0
            mask[1:-1, 0] = 1
            if i % 2:
                mask[0, :-3] = 1
            p = grid_pair(double, (n, n), float, mask, rng.random((n, n)))
            pairs.append(p)
            b.add(p[0], trip)
        b.step(1)
        ck = CpuKernel(k)
        for j, (d, h) in enumerate(pairs):
            ck(h, trip)
    assert b.counters()["validations"] == len(counts)
    for d, h in pairs:
        assert_bitexact(d, h, levels=[0])
    b.close()
