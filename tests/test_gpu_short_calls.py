"""Calls of a few launches: three are made directly (replaying a graph costs more), and a pair of interiors
inside a chain does not cut it in two."""
import numpy as np
import pytest

import xgrid_amd as xgrid

from helpers import assert_bitexact, grid_pair, run_pair

pytestmark = pytest.mark.gpu
f2 = xgrid.grid[float, 2]


def _kernel():
    @xgrid.kernel()
    def steps(u: f2, v: f2, w: f2, a: float) -> None:
        u[0, 0] = u[0, 0] + a * (u[1, 0] + u[-1, 0] + u[0, 1] + u[0, -1] - 4.0 * u[0, 0])
        v[0, 0] = v[0, 0] + a * (u[1, 0][0] - u[-1, 0][0])
        w[0, 0] = w[0, 0] * 0.5 + u[0, 0][0] * v[0, 0][0]
        with xgrid.boundary(1):
            u[0, 0] = 0.0
    return steps


@pytest.mark.parametrize("n, launches", [(45, 1), (200, 3)])
def test_launches(double, n, launches):
    """45^2: one chain (v and w are a pair, with u before and the wall after them).  200^2: u, the pair, the
    wall; no graph, however often the call repeats."""
    k = _kernel()
    rng = np.random.default_rng(1)
    mask = np.full((n, n), 9, np.int32)
    mask[1:-1, 1:-1] = 0
    mask[1:-1, 0] = 1
    pairs = [grid_pair(double, (n, n), float, mask, rng.random((n, n))) for _ in range(3)]
    dev, host = [p[0] for p in pairs], [p[1] for p in pairs]
    run_pair(k, (*dev, 0.01), (*host, 0.01), steps=12)
    for p in pairs:
        assert_bitexact(*p)
    before = k.native.counters()
    for _ in range(12):
        k(*dev, 0.01)
    after = k.native.counters()
    assert after["launches"] - before["launches"] == 12 * launches
    assert after["graph_replays"] == 0
