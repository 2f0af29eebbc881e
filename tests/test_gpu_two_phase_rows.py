"""The first phase of a two-phase 2-D statement stores whole lanes of its temporary, at any store offset."""
import numpy as np
import pytest

import xgrid_amd as xgrid

from helpers import assert_bitexact, grid_pair, run_pair

pytestmark = pytest.mark.gpu
f2 = xgrid.grid[float, 2]


@pytest.mark.parametrize("cols", [70, 131, 141, 300])
@pytest.mark.parametrize("kind", ["box", "holes"])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_shifted_store(prec, kind, cols, request):
    @xgrid.kernel()
    def shifted(u: f2, v: f2, a: float) -> None:
        u[0, 1] = u[0, 0][0] * a + v[0, 0]

    xg = request.getfixturevalue(prec)
    rng = np.random.default_rng(cols)
    mask = np.ones((50, cols), np.int32)
    mask[1:-1, 1:-1] = 0
    if kind == "holes":
        mask[(rng.random((50, cols)) < 0.2) & (mask == 0)] = 1
    pairs = [grid_pair(xg, (50, cols), float, mask, rng.random((50, cols))) for _ in range(2)]
    run_pair(shifted, (*[p[0] for p in pairs], 0.3), (*[p[1] for p in pairs], 0.3), steps=4)
    for p in pairs:
        assert_bitexact(*p)
