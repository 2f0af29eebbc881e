"""A call whose iterations need a wider halo than wave tiles have runs unblocked; calls of fewer
iterations on the same mask still run blocked, whatever came before."""
import numpy as np
import pytest

import xgrid_amd as xgrid
from xgrid_amd import _lib
from xgrid_amd.batch import Batch

from helpers import assert_bitexact, grid_pair, run_pair

pytestmark = pytest.mark.gpu
f2 = xgrid.grid[float, 2]


def _creep():
    """Three cells along row 0 per iteration: 8 iterations fit a halo of 24, 9 do not."""
    @xgrid.kernel()
    def creep(u: f2, v: f2, trip: int) -> None:
        for _ in range(0, trip):
            u[0, 0] = (u[0, 1][0] + u[0, -1][0] + u[1, 0][0] + u[-1, 0][0]) * 0.25 + v[0, 0]
            with xgrid.boundary(1):
                u[0, 0] = u[0, -1][0] + 1.0
            with xgrid.boundary(2):
                u[0, 0] = u[0, -1][0] * 0.5
            with xgrid.boundary(3):
                u[0, 0] = u[0, -1][0] - 0.25
    return creep


def _mask(n):
    mask = np.zeros((n, n), np.int32)
    mask[0, :] = 1 + np.arange(n) % 3
    mask[-1, :] = mask[:, 0] = mask[:, -1] = 4
    return mask


def test_short_calls_stay_blocked(double):
    n, k = 150, _creep()
    rng = np.random.default_rng(13)
    du, hu = grid_pair(double, (n, n), float, _mask(n), rng.random((n, n)))
    dv, hv = grid_pair(double, (n, n), float, None, rng.random((n, n)) * 1e-3)
    done = 0
    for trip in (9, 8, 1, 12, 3, 30, 8, 8, 8):      # (the last ones are captured and replayed)
        run_pair(k, (du, dv, trip), (hu, hv, trip))
        assert_bitexact(du, hu)
        if trip <= 8:
            done += trip
        info = k.native.loop_info(k.native.loop_plan(0, n * n))
        assert info["state"] == (1 if trip <= 8 else -1)
        assert info["iterations"] <= done and (trip > 8 or info["iterations"] >= 8)
    lid = k.native.loop_plan(0, n * n)
    assert k.native.time_loop(lid, 8, reps=2) > 0
    with pytest.raises(_lib.BackendError):
        k.native.time_loop(lid, 12, reps=2)


def test_batched_short_calls_stay_blocked(double):
    n, k = 150, _creep()
    rng = np.random.default_rng(14)
    u0, v0 = rng.random((n, n)), rng.random((n, n)) * 1e-3
    b, members = Batch(k), []
    for trip in (12, 8, 3):
        both = []
        for _ in range(2):
            u, v = double.Grid((n, n), float), double.Grid((n, n), float)
            u.now[...], v.now[...] = u0, v0
            u.boundary[...] = _mask(n)
            both.append((u, v))
        b.add(*both[0], trip)
        members.append((trip, both))
    b.step(4)
    for trip, ((bu, _), (pu, pv)) in members:
        for _ in range(4):
            k(pu, pv, trip)
        assert np.array_equal(bu.now.view(np.uint8), pu.now.view(np.uint8))
    b.close()
