"""A field that spreads from rest: its edge holds every size of number down to the subnormals, where
corrected quotients give way to divisions workgroup by workgroup."""
import numpy as np
import pytest

import xgrid_amd as xgrid

from helpers import assert_bitexact, grid_pair, run_pair

pytestmark = pytest.mark.gpu
f2 = xgrid.grid[float, 2]


@pytest.mark.parametrize("prec", ["double", "single"])
def test_spread_from_rest(prec, request):
    """In FP64 and in FP32 (no literal in the body: a division of FP32 numbers) the edge reaches the
    subnormals and passes through tiles row by row and column by column; 1, 9 and 16 iterations."""
    xg = request.getfixturevalue(prec)

    @xgrid.kernel()
    def spread(u: f2, b: f2, d: float, trip: int) -> None:
        for _ in range(0, trip):
            u[0, 0] = (u[0, 1][0] + u[0, -1][0] + (u[1, 0][0] + u[-1, 0][0])) / d + b[0, 0][0]
            with xgrid.boundary(1):
                u[0, 0] = u[-1, 0][0]

    shape = (150, 700)
    for at in ("wall", "middle"):
        mask = np.zeros(shape, np.int32)
        mask[0], mask[:, 0], mask[:, -1] = 9, 9, 9
        mask[-1] = 1
        u0, b0 = np.zeros(shape), np.zeros(shape)
        if at == "wall":
            u0[:, 0] = 1.0
        else:
            b0[70, 350] = 1e-3
        du, hu = grid_pair(xg, shape, float, mask, u0)
        db, hb = grid_pair(xg, shape, float, None, b0)
        small = []
        for trip in (1, 9, 16, 50, 50, 200, 300):
            run_pair(spread, (du, db, 4.3, trip), (hu, hb, 4.3, trip))
            assert_bitexact(du, hu, levels=[0])
            small.append(np.abs(hu.now[hu.now != 0]).min())
        # (the edge from the middle meets the walls, 350 columns away, before it is that small in FP64)
        assert min(small) < np.finfo(hu.now.dtype).smallest_normal or (at == "middle" and prec == "double")
    low = spread.native.lowered
    assert low.loops[0].waves and "value_rgq" in low.device_src
