"""Wave tiles of blocked loops (the region in registers, rows per wave): the oracle's
bits at the edges of tiles, for every kind of mask, odd and even iteration counts,
and when one kernel alternates between grids."""
import numpy as np
import pytest

import xgrid_amd as xgrid
from xgrid_amd.backend import build_kernel

from helpers import assert_bitexact, grid_pair, run_pair

pytestmark = pytest.mark.gpu
f2 = xgrid.grid[float, 2]


def _loop_kernel():
    """Corner reads, another grid read beside the cell, a boundary row that reads across rows,
    one that reads along itself, and one that divides."""
    @xgrid.kernel()
    def relax(u: f2, v: f2, a: float, d: float, trip: int) -> None:
        for _ in range(0, trip):
            u[0, 0] = (u[0, 1][0] + u[0, -1][0] + (u[1, 0][0] + u[-1, 0][0])) * a / d - \
                u[1, 1][0] * 0.015625 + u[-1, -1][0] * 0.03125 - v[0, -1] * 0.5
            with xgrid.boundary(1):
                u[0, 0] = u[0, -1][0]
            with xgrid.boundary(2):
                u[0, 0] = u[1, 0][0] / d
            with xgrid.boundary(3):
                u[0, 0] = u[0, 1][0] * a
            with xgrid.boundary(4):
                u[0, 0] = 0.25
    return relax


def _mask(kind, shape, rng):
    m = np.zeros(shape, np.int32)
    if kind in ("spots", "lattice"):     # a masked class 0, members anywhere inside (or apart from each other)
        inside = rng.random(shape) < (0.1 if kind == "spots" else 0.7)
        if kind == "lattice":
            inside &= (np.arange(shape[0]) % 3 == 0)[:, None] & (np.arange(shape[1]) % 3 == 0)[None, :]
        inside[:2], inside[-2:], inside[:, :2], inside[:, -2:] = False, False, False, False
        m[inside] = rng.integers(1, 5, int(inside.sum()))
    m[:, -1] = 1
    m[0, :] = 2
    m[:, 0] = 3
    m[-1, :] = 4
    if kind == "creep":                  # data runs two cells along row 0 per iteration
        m[0, 1:-1] = 1 + 2 * (np.arange(shape[1] - 2) % 2)
    return m


# rows x columns: a single tile; one row and column beyond one; one wave's rows; tiles cut
# short in either direction; both wave tiles (the 8-row one on the last, with many workgroups)
@pytest.mark.parametrize("shape", [(3, 3), (33, 128), (64, 129), (129, 65), (40, 1000), (700, 131), (1500, 1450)])
@pytest.mark.parametrize("kind", ["walls", "lattice", "spots", "creep"])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_wave_tiles_match_oracle(prec, kind, shape, request):
    """Members of one class beside each other ("spots") read each other at time 0, which the
    reference races on: there the unblocked launches say what is right."""
    xg = request.getfixturevalue(prec)
    rng = np.random.default_rng(shape[0] * 7 + shape[1])
    k = _loop_kernel()
    unblocked = _loop_kernel()
    unblocked.native, unblocked.depth = build_kernel(unblocked)
    unblocked.native.set_options(blocked=False)
    mask = _mask(kind, shape, rng)
    big = shape[0] * shape[1] > 10 ** 6
    pairs = []
    for _ in range(1 if big else 2):     # two grids in turn on one kernel
        u0, v0 = rng.random(shape), rng.random(shape) * 0.25
        du, hu = grid_pair(xg, shape, float, mask, u0)
        dv, hv = grid_pair(xg, shape, float, None, v0)
        if kind == "spots":
            hu, hv = grid_pair(xg, shape, float, mask, u0)[0], grid_pair(xg, shape, float, None, v0)[0]
        pairs.append((du, dv, hu, hv))
    # 4: a power of two (reciprocal form); 3.7: divisions.  One iteration, odd and even counts,
    # more than a launch of several tiles runs
    for d, trip in ((4.0, 7),) if big else ((4.0, 1), (3.7, 2), (4.0, 13), (3.7, 50)):
        for du, dv, hu, hv in pairs:
            if kind == "spots":
                k(du, dv, 0.9, d, trip)
                unblocked(hu, hv, 0.9, d, trip)
                assert np.array_equal(du.now.view(np.uint8), hu.now.view(np.uint8))
                continue
            run_pair(k, (du, dv, 0.9, d, trip), (hu, hv, 0.9, d, trip))
            assert_bitexact(du, hu, levels=[0])
    assert k.native.lowered.loops[0].waves
    info = k.native.loop_info(k.native.loop_plan(0, shape[0] * shape[1]))
    assert kind != "walls" or (info["state"] == 1 and info["iterations"] > 0)


def test_wave_tiles_proofs_follow_the_mask(double):
    """A mask set anew is proven anew: the same grid first with walls, then with a boundary row
    along which data runs faster, then with walls again."""
    k = _loop_kernel()
    rng = np.random.default_rng(3)
    shape = (90, 300)
    du, hu = grid_pair(double, shape, float, None, rng.random(shape))
    dv, hv = grid_pair(double, shape, float, None, rng.random(shape) * 0.25)
    ran = []
    for kind in ("walls", "creep", "walls"):
        m = _mask(kind, shape, rng)
        du.boundary[...] = m
        hu.boundary[...] = m
        before = k.native.loop_info(1)["iterations"] if k.native else 0
        run_pair(k, (du, dv, 0.9, 3.7, 12), (hu, hv, 0.9, 3.7, 12))
        assert_bitexact(du, hu, levels=[0])
        ran.append(k.native.loop_info(1)["iterations"] - before)
    assert ran[0] == ran[2] == 12


@pytest.mark.parametrize("prec", ["double", "single"])
def test_batched_wave_tiles_match_plain(prec, request):
    """One batch over grids of one tile and of many, walls and scattered classes."""
    from xgrid_amd.batch import Batch
    xg = request.getfixturevalue(prec)
    kb, kp = _loop_kernel(), _loop_kernel()
    rng = np.random.default_rng(11)
    batch, members = Batch(kb), []
    for shape, kind in (((20, 100), "walls"), ((64, 129), "spots"), ((257, 300), "walls"), ((31, 400), "creep")):
        mask, u0, v0 = _mask(kind, shape, rng), rng.random(shape), rng.random(shape) * 0.25
        pair = []
        for _ in range(2):
            u, v = xg.Grid(shape, float), xg.Grid(shape, float)
            u.now[...] = u0
            v.now[...] = v0
            u.boundary[...] = mask
            pair.append((u, v))
        batch.add(*pair[0], 0.9, 3.7, 11)
        members.append(pair)
    batch.step(5)
    for (ub, _), (ua, va) in members:
        for _ in range(5):
            kp(ua, va, 0.9, 3.7, 11)
        assert np.array_equal(ub.now.view(np.uint8), ua.now.view(np.uint8))
    batch.close()
