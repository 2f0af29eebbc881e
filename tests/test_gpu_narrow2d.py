"""2-D tiles no wider than a wave (narrow grids, and the last tile of a row of tiles) hold one cell per
work-item, wider ones 16 bytes of a row: the oracle's bits on both sides of the line."""
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
        v[0, 0] = v[0, 0] + a * (u[0, 1] - u[0, -1])
        w[0, 0] = v[0, 0][0] * 0.5 + u[-1, 1] * a
        with xgrid.boundary(1):
            u[0, 0] = 0.25
    return steps


@pytest.mark.parametrize("cols", [3, 4, 6, 65, 66, 67, 69, 130, 131, 194, 195, 258, 259, 322, 323])
@pytest.mark.parametrize("kind", ["box", "holes"])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_columns(prec, kind, cols, request):
    """cols - 2 interior columns: 1 to 64 are one narrow tile; 65 and more a wide one, after 128 (FP64) or 256
    (FP32) the next."""
    xg = request.getfixturevalue(prec)
    k = _kernel()
    rows = 301
    rng = np.random.default_rng(cols)
    mask = np.full((rows, cols), 9, np.int32)
    mask[1:-1, 1:-1] = 0
    mask[1:-1, 0] = 1
    if kind == "holes":
        mask[(rng.random((rows, cols)) < 0.2) & (mask == 0)] = 1
    pairs = [grid_pair(xg, (rows, cols), float, mask, rng.random((rows, cols))) for _ in range(3)]
    dev, host = [p[0] for p in pairs], [p[1] for p in pairs]
    run_pair(k, (*dev, 0.1), (*host, 0.1), steps=3)
    for p in pairs:
        assert_bitexact(*p)
