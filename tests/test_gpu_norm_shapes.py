"""FP64 reductions at the sizes where the walk over a class changes: rows around the
narrow-row limit (32 cells), a chunk (64) and a turn of a wave (256), one-cell-wide
walls, lists and masked boxes with a ragged end, and fewer chunks than workgroups."""
import math

import numpy as np
import pytest

from tests.test_gpu_precision import _grid

pytestmark = pytest.mark.gpu

# Squares are added in chains of at most 8 per lane, then over 64 lanes, 8 waves, and one
# or two partials per lane of the last workgroup: fewer than 64 roundings of non-negative
# sums, one more in each square and in the root.
REL = 66 * 2.0 ** -53

SHAPES = [(1,), (63,), (4097,), (3, 1), (40, 31), (40, 32), (40, 33), (40, 64), (40, 65), (7, 255), (7, 256), (7, 257),
          (2100, 1), (5, 9, 1), (6, 5, 3), (6, 5, 17), (9, 8, 33), (12, 11, 64), (12, 11, 129)]


def _check(r, d):
    ref = math.sqrt(math.fsum((d * d).ravel().tolist()))
    assert r["linf"] == (np.abs(d).max() if d.size else 0.0)
    assert abs(r["l2"] - ref) <= REL * ref


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_diff_norm_at_the_edges_of_its_walk(double, shape):
    from xgrid_amd import norms
    rng = np.random.default_rng(sum(shape))
    av, bv = rng.standard_normal(shape), rng.standard_normal(shape)
    sparse, dense = np.zeros(shape, np.int32), np.zeros(shape, np.int32)
    sparse.ravel()[::7] = 1                               # a list
    dense[rng.random(shape) < 0.7] = 1                    # a masked box
    thin = np.zeros(shape, np.int32)
    thin[..., -1] = 1                                     # a one-cell-wide box
    for mask in (np.zeros(shape, np.int32), sparse, dense, thin):
        a, b = _grid(double, av, mask), _grid(double, bv)
        for klass in (0, 1):
            sel = mask == klass
            for other, d in ((b, av - bv), (None, av)):
                r = norms.diff_norm(a, other, klass=klass)
                assert r["cells"] == sel.sum()
                _check(r, d[sel])


@pytest.mark.parametrize("shape", [s for s in SHAPES if min(s) >= 3], ids=str)
def test_poisson_residual_at_the_edges_of_its_walk(double, shape):
    from xgrid_amd import norms
    from xgrid_amd.workloads import box_walls
    rng = np.random.default_rng(sum(shape) + 1)
    # Integers: the residual of a cell has no rounding in any order.
    pv, rv = (rng.integers(-50, 50, shape).astype(np.float64) for _ in range(2))
    mask = box_walls(shape)
    res = -2.0 * rv
    for ax in range(len(shape)):
        res += (ax + 1.0) * (np.roll(pv, -1, ax) + np.roll(pv, 1, ax) - 2.0 * pv)
    r = norms.poisson_residual(_grid(double, pv, mask), _grid(double, rv), [ax + 1.0 for ax in range(len(shape))],
                               rhs_scale=2.0)
    _check(r, res[mask == 0])
