"""Staged 3-D tiles on rows of any pitch: 16-byte loads and stores where neither the base of a
row nor its end is a multiple of 16 bytes, against the oracle's bits."""
import numpy as np
import pytest

import xgrid_amd as xgrid
from oracle import restate as R

from helpers import assert_bitexact, grid_pair, run_pair

pytestmark = pytest.mark.gpu
f3 = xgrid.grid[float, 3]


def _kernel():
    """Both ends of every axis, one array read at two levels and one read beside it."""
    @xgrid.kernel()
    def pitch3(u: f3, w: f3, a: float) -> None:
        u[0, 0, 0] = w[0, 0, 0] + a * (u[1, 0, 0] + u[-1, 0, 0] + u[0, 1, 0] + u[0, -1, 0] + w[0, 0, 1] +
                                       u[0, 0, -1] - 6.0 * u[0, 0, 0])
    return pitch3


# rows shorter than a lane's columns, around one lane, one tile (128 or 256 columns) and two,
# with every remainder by the four columns of an FP32 lane
@pytest.mark.parametrize("n2", [3, 4, 5, 6, 7, 9, 127, 129, 130, 131, 254, 255, 257, 258, 259, 515])
@pytest.mark.parametrize("holes", [False, True], ids=["box", "masked"])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_rows_of_any_pitch(prec, holes, n2, request):
    xg = request.getfixturevalue(prec)
    shape = (7, 11, n2)
    rng = np.random.default_rng(n2)
    mask = np.ones(shape, np.int32)
    mask[1:-1, 1:-1, 1:-1] = 0
    if holes:
        mask[1:-1, 1:-1, 1:-1][rng.random((5, 9, n2 - 2)) < 0.3] = 1
    k = _kernel()
    dw, hw = grid_pair(xg, shape, float, None, rng.random(shape))
    d, h = grid_pair(xg, shape, float, mask, rng.random(shape))
    run_pair(k, (d, dw, 0.1), (h, hw, 0.1), steps=3)
    assert_bitexact(d, h)


def test_streamed_rows_of_odd_pitch(double):
    """Non-temporal stores (a grid of more than 128 MiB) on an odd pitch."""
    from xgrid_amd import workloads as W
    n, steps, nu = 259, 2, 0.1
    assert n ** 3 * 8 > 128 << 20
    u0, mask, dx = W.heat_3d_setup(n, np.float64, seed=6)
    dt = 0.1 * dx * dx / nu
    k = W.make_heat_3d()
    g = double.Grid((n, n, n), float)
    g.now[...] = u0
    g.boundary[...] = mask
    for _ in range(steps):
        k(g, nu, dt, dx)
    want = R.heat_3d(u0, nu, dt, dx, steps, np.float64)
    assert np.array_equal(g.now.view(np.uint8), want.view(np.uint8))
