"""Independent statements in one launch: the oracle's bits for interiors and walls of
every rank, and where the grids passed make the statements depend on each other."""
import numpy as np
import pytest

import xgrid_amd as xgrid

from helpers import assert_bitexact, grid_pair, run_pair

pytestmark = pytest.mark.gpu
f1, f2, f3 = (xgrid.grid[float, d] for d in (1, 2, 3))


def _kernel_3d():
    """An interior, a wall of one value (a parameter), a wall that copies its neighbour."""
    @xgrid.kernel()
    def walls3(u: f3, a: float) -> None:
        u[0, 0, 0] = u[0, 0, 0] + a * (u[1, 0, 0] + u[-1, 0, 0] + u[0, 1, 0] + u[0, -1, 0] + u[0, 0, 1] +
                                       u[0, 0, -1] - 6.0 * u[0, 0, 0])
        with xgrid.boundary(1):
            u[0, 0, 0] = a * 2.0
        with xgrid.boundary(2):
            u[0, 0, 0] = u[0, 0, 0] * 0.5
    return walls3


# rows shorter than a tile, of exactly one and of two tiles, odd ones (no 16-byte rows), and
# boxes that end inside a lane's columns
@pytest.mark.parametrize("shape", [(3, 3, 3), (9, 11, 70), (6, 10, 256), (5, 7, 301), (10, 18, 518)])
@pytest.mark.parametrize("walls", ["one", "left_other", "planes_other", "holes", "inset"])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_interior_and_walls_3d(prec, walls, shape, request):
    """`one`: the rows' ends belong to the wall statement that has one value; `left_other`: some
    belong to another class; `holes`: class 0 is no box; `inset`: the box ends mid-lane."""
    xg = request.getfixturevalue(prec)
    rng = np.random.default_rng(sum(shape))
    mask = np.ones(shape, np.int32)
    mask[1:-1, 1:-1, 1:-1] = 0
    if walls == "left_other":
        mask[:, :, 0] = 2
    elif walls == "planes_other":
        mask[0] = mask[-1] = 2
    elif walls == "holes":
        mask[1:-1, 1:-1, 1:-1][rng.random([n - 2 for n in shape]) < 0.2] = 1
    elif walls == "inset" and shape[2] > 12:
        mask[:, :, :6] = 1
        mask[:, :, -5:] = 1
    k = _kernel_3d()
    d, h = grid_pair(xg, shape, float, mask, rng.random(shape))
    run_pair(k, (d, 0.1), (h, 0.1), steps=4)
    assert_bitexact(d, h)
    assert k.native.lowered.fans


@pytest.mark.parametrize("shape", [(3,), (1025,), (5000,), (3, 3), (66, 64), (70, 131)])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_interior_and_walls_1d_2d(prec, shape, request):
    from xgrid_amd import workloads as W
    xg = request.getfixturevalue(prec)
    rng = np.random.default_rng(sum(shape))
    k = W.make_diffusion_1d() if len(shape) == 1 else W.make_diffusion_2d()
    d, h = grid_pair(xg, shape, float, W.box_walls(shape), rng.random(shape))
    run_pair(k, (d, 0.1, 0.2, 1.5), (h, 0.1, 0.2, 1.5), steps=4)
    assert_bitexact(d, h)
    assert k.native.lowered.fans


@pytest.mark.parametrize("case", ["apart", "aliased", "shifted"])
def test_dependent_grids_run_in_order(double, case):
    """Statements that are independent by name but not on the grids passed (or that store
    shifted over each other's cells) run one after the other, in order."""
    if case == "shifted":
        @xgrid.kernel()
        def k(u: f2, v: f2, w: f2) -> None:
            u[0, 0] = w[0, 0] + 1.0
            with xgrid.boundary(1):
                u[0, 1] = w[0, 0] * 2.0
            with xgrid.boundary(2):
                v[0, 0] = w[0, 0] * 3.0
    else:
        @xgrid.kernel()
        def k(u: f2, v: f2, w: f2) -> None:
            u[0, 0] = w[0, 0] + 1.0
            with xgrid.boundary(1):
                v[0, 0] = w[0, 1][0] * 2.0
            with xgrid.boundary(2):
                u[0, 0] = v[0, 0] * 3.0

    rng = np.random.default_rng(8)
    shape = (70, 90)
    mask = np.zeros(shape, np.int32)
    mask[:, 2:40:3] = 1
    mask[5, :] = 2
    mask[:, -1] = 3
    du, hu = grid_pair(double, shape, float, mask, rng.random(shape))
    dv, hv = grid_pair(double, shape, float, mask, rng.random(shape))
    dw, hw = grid_pair(double, shape, float, None, rng.random(shape))
    dargs, hargs = ((du, dv, du), (hu, hv, hu)) if case == "aliased" else ((du, dv, dw), (hu, hv, hw))
    run_pair(k, dargs, hargs, steps=4)
    for d, h in zip(dargs, hargs):
        assert_bitexact(d, h)
