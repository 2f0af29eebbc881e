"""The order in which plain launches take a blocked loop's wave tiles (edge tiles first): one, two,
three and more tiles along either axis, against the oracle's bits."""
import numpy as np
import pytest

from helpers import assert_bitexact, grid_pair, run_pair
from test_gpu_wave import _loop_kernel, _mask

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(60, 330), (150, 330), (330, 100), (330, 200), (300, 330), (420, 560)])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_wave_tiles_in_any_number(prec, shape, request):
    xg = request.getfixturevalue(prec)
    rng = np.random.default_rng(shape[0] + shape[1])
    k = _loop_kernel()
    du, hu = grid_pair(xg, shape, float, _mask("walls", shape, rng), rng.random(shape))
    dv, hv = grid_pair(xg, shape, float, None, rng.random(shape) * 0.25)
    run_pair(k, (du, dv, 0.9, 4.0, 17), (hu, hv, 0.9, 4.0, 17), steps=2)
    assert_bitexact(du, hu, levels=[0])
