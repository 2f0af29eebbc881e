"""2-D tiles whose work-items hold 16 bytes of a row, at the widths where a lane's cells are
only partly its own, against the oracle's bits."""
import numpy as np
import pytest

import xgrid_amd as xgrid

from helpers import assert_bitexact, grid_pair, run_pair

pytestmark = pytest.mark.gpu
f2, i2, f1 = xgrid.grid[float, 2], xgrid.grid[int, 2], xgrid.grid[float, 1]


def _pair():
    """Two statements that run as one launch (the second takes the first's value), near and far
    columns of both sides, a grid of another element type, and a wall."""
    @xgrid.kernel()
    def rows(b: f2, u: f2, m: i2, a: float) -> None:
        b[0, 0] = a * (u[0, 1] - u[0, -1]) + u[1, 2] / 3.0 + (u[-1, -2] if m[0, 1] > 0 else b[0, -1])
        u[0, 0] = (u[0, 2] + u[0, -2] + u[1, 0] + u[-1, 1]) / 4.0 - a * b[0, 0][0]
        with xgrid.boundary(1):
            u[0, 0] = u[0, 0] + 1.0
    return rows


def _shifted():
    """A store beside the cell (no vector store) and one that reads its own cell's new value."""
    @xgrid.kernel()
    def shifted(b: f2, u: f2, a: float) -> None:
        b[0, 1] = u[0, 0] * a + u[1, 1]
        u[0, 0] = u[0, 0][0] * a + b[0, 0][0]
    return shifted


def _lower():
    """A coefficient per column of a 1-D grid: views of two shapes, so no tile is safe."""
    @xgrid.kernel()
    def lower(u: f2, c: f1, a: float) -> None:
        u[0, 0] = u[0, 0] + a * c[0] * (u[0, 1] - u[0, -1])
    return lower


# interiors narrower than a lane's columns, of one lane, around one tile (128 or 256 columns) and
# two, with every remainder by the four columns of an FP32 lane
@pytest.mark.parametrize("cols", [1, 2, 3, 4, 5, 6, 7, 9, 126, 127, 129, 130, 254, 255, 257, 258, 515])
@pytest.mark.parametrize("holes", [False, True], ids=["box", "masked"])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_rows_of_any_width(prec, holes, cols, request):
    xg = request.getfixturevalue(prec)
    shape = (10, cols + 4)
    rng = np.random.default_rng(cols)
    mask = np.ones(shape, np.int32)
    mask[2:-2, 2:-2] = 0
    if holes:
        mask[2:-2, 2:-2][rng.random((6, cols)) < 0.3] = 1
    mi = rng.integers(-3, 4, shape).astype(np.int32)
    db, hb = grid_pair(xg, shape, float, mask, rng.random(shape))
    du, hu = grid_pair(xg, shape, float, mask, rng.random(shape))
    dm, hm = grid_pair(xg, shape, int, None, mi)
    run_pair(_pair(), (db, du, dm, 0.1), (hb, hu, hm, 0.1), steps=3)
    assert_bitexact(db, hb)
    assert_bitexact(du, hu)
    run_pair(_shifted(), (db, du, 0.1), (hb, hu, 0.1), steps=2)
    assert_bitexact(db, hb)
    assert_bitexact(du, hu)


@pytest.mark.parametrize("mode", ["limit", "wrap"])
def test_rows_to_the_edge(mode):
    """Class 0 everywhere: tiles at the grid's edge clamp or wrap every read."""
    xgrid.init(precision="float", overstep=mode)
    try:
        rng = np.random.default_rng(5)
        d, h = grid_pair(xgrid, (9, 263), float, None, rng.random((9, 263)))
        dc, hc = grid_pair(xgrid, (263,), float, None, rng.random(263))
        run_pair(_lower(), (d, dc, 0.1), (h, hc, 0.1), steps=2)
        assert_bitexact(d, h)
    finally:
        xgrid.init(precision="double")
