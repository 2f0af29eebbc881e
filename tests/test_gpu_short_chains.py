"""Chains of small statements stay one launch where their pairs and fans, as launches of their own, would take
longer: few cells per statement, several launches.  Either way the oracle's bits."""
import numpy as np
import pytest

import xgrid_amd as xgrid

from helpers import assert_bitexact, grid_pair, run_pair

pytestmark = pytest.mark.gpu
f2 = xgrid.grid[float, 2]


def _fields():
    @xgrid.kernel()
    def fields(u: f2, v: f2, w: f2, a: float) -> None:
        u[0, 0] = u[0, 0] + a * (u[1, 0] + u[-1, 0] + u[0, 1] + u[0, -1] - 4.0 * u[0, 0])
        with xgrid.boundary(1):
            u[0, 0] = 0.0
        v[0, 0] = v[0, 0] + a * (u[1, 0][0] - u[-1, 0][0])
        with xgrid.boundary(1):
            v[0, 0] = 0.0
        w[0, 0] = w[0, 0] + a * (v[1, 0][0] - v[-1, 0][0])
        with xgrid.boundary(1):
            w[0, 0] = 0.0
    return fields


def _pair():
    @xgrid.kernel()
    def pair(u: f2, v: f2, w: f2, a: float) -> None:
        v[0, 0] = v[0, 0] + a * (u[1, 0] - u[-1, 0])
        w[0, 0] = w[0, 0] + a * (u[0, 1] - u[0, -1])
        with xgrid.boundary(1):
            v[0, 0] = w[0, 1][0]
    return pair


@pytest.mark.parametrize("make, n, launches", [(_fields, 16, 1), (_fields, 45, 1), (_fields, 64, 3),
                                               (_pair, 16, 1), (_pair, 45, 1), (_pair, 64, 2)])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_launches(prec, make, n, launches, request):
    xg = request.getfixturevalue(prec)
    k = make()
    rng = np.random.default_rng(2)
    mask = np.full((n, n), 9, np.int32)
    mask[1:-1, 1:-1] = 0
    mask[1:-1, 0] = 1
    pairs = [grid_pair(xg, (n, n), float, mask, rng.random((n, n))) for _ in range(3)]
    dev, host = [p[0] for p in pairs], [p[1] for p in pairs]
    run_pair(k, (*dev, 0.01), (*host, 0.01), steps=12)
    for p in pairs:
        assert_bitexact(*p)
    before = k.native.counters()["launches"]
    for _ in range(12):
        k(*dev, 0.01)
    assert k.native.counters()["launches"] - before == 12 * launches
