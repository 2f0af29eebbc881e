"""Flat 3-D launches (rows that leave lanes of staged tiles idle): remainders of columns, rows and
planes, walls stored beside the rows, and non-temporal stores, against the oracle's bits."""
import numpy as np
import pytest

from oracle import restate as R

from helpers import assert_bitexact, grid_pair, run_pair
from test_gpu_pitch import _kernel

pytestmark = pytest.mark.gpu


# interiors of one to five planes (two per work-item), rows of every remainder by a lane's two or
# four columns, more rows than a workgroup of 256 work-items holds, more than a band of 32 workgroups
@pytest.mark.parametrize("shape", [(3, 5, 9), (4, 6, 7), (5, 40, 6), (6, 300, 8), (7, 9, 270), (4, 1500, 37), (5, 700, 50),
                                   (6, 64, 140)])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_flat_rows(prec, shape, request):
    xg = request.getfixturevalue(prec)
    rng = np.random.default_rng(shape[2])
    mask = np.ones(shape, np.int32)
    mask[1:-1, 1:-1, 1:-1] = 0
    k = _kernel()
    dw, hw = grid_pair(xg, shape, float, None, rng.random(shape))
    d, h = grid_pair(xg, shape, float, mask, rng.random(shape))
    run_pair(k, (d, dw, 0.1), (h, hw, 0.1), steps=3)
    assert_bitexact(d, h)


@pytest.mark.parametrize("shape", [(9, 12, 45), (6, 33, 70), (5, 8, 131), (4, 90, 302)])
@pytest.mark.parametrize("prec,dtype", [("double", np.float64), ("single", np.float32)])
def test_flat_rows_with_walls(prec, dtype, shape, request):
    """The walls in the same launch: the cells beside the rows are stored with them, by either way."""
    from xgrid_amd import workloads as W
    xg = request.getfixturevalue(prec)
    rng = np.random.default_rng(shape[1])
    u0 = rng.random(shape).astype(dtype)
    g = xg.Grid(shape, float)
    g.now[...] = u0
    g.boundary[...] = W.box_walls(shape)
    k = W.make_heat_3d()
    for _ in range(3):
        k(g, 0.1, 0.01, 0.25)
    want = R.heat_3d(u0, 0.1, 0.01, 0.25, 3, dtype)
    assert np.array_equal(g.now.view(np.uint8), want.view(np.uint8))


def test_streamed_flat_rows(double):
    """Non-temporal stores (a grid of more than 128 MiB), 68 of 128 lanes' columns held."""
    from xgrid_amd import workloads as W
    shape = (430, 600, 70)
    assert np.prod(shape) * 8 > 128 << 20
    u0 = np.random.default_rng(1).random(shape)
    g = double.Grid(shape, float)
    g.now[...] = u0
    g.boundary[...] = W.box_walls(shape)
    W.make_heat_3d()(g, 0.1, 0.01, 0.25)
    want = R.heat_3d(u0, 0.1, 0.01, 0.25, 1, np.float64)
    assert np.array_equal(g.now.view(np.uint8), want.view(np.uint8))
