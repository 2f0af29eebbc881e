"""Blocked loops whose bodies read more than the cavity's: wave tiles whose registers hold them,
or the region in LDS; the oracle's bits either way, plain and batched."""
import numpy as np
import pytest

import xgrid_amd as xgrid
from xgrid_amd.backend import compile_kernel
from xgrid_amd.compilers import kernel_scratch

from helpers import assert_bitexact, grid_pair, run_pair

f2 = xgrid.grid[float, 2]


def _kernel(body):
    if body == "one":
        @xgrid.kernel()
        def k(p: f2, a: f2, b: f2, c: f2, d: f2, e: f2, f: f2, w: float, trip: int) -> None:
            for _ in range(0, trip):
                p[0, 0] = p[0, 0][0] + w * (p[1, 0][0] + p[-1, 0][0] + p[0, 1][0] + p[0, -1][0] - 4.0 * p[0, 0][0] - b[0, 0][0])
                with xgrid.boundary(1):
                    p[0, 0] = p[0, 1][0]
    elif body == "two":
        @xgrid.kernel()
        def k(p: f2, a: f2, b: f2, c: f2, d: f2, e: f2, f: f2, w: float, trip: int) -> None:
            for _ in range(0, trip):
                p[0, 0] = p[0, 0][0] + c[0, 0][0] * ((p[1, 0][0] - 2.0 * p[0, 0][0] + p[-1, 0][0]) / (w * 3.7) + (p[0, 1][0] - 2.0 * p[0, 0][0] + p[0, -1][0]) / (w * 4.1)) - b[0, 0][0]
                with xgrid.boundary(1):
                    p[0, 0] = p[0, 1][0]
    elif body == "three":
        @xgrid.kernel()
        def k(p: f2, a: f2, b: f2, c: f2, d: f2, e: f2, f: f2, w: float, trip: int) -> None:
            for _ in range(0, trip):
                p[0, 0] = p[0, 0][0] + a[0, 0][0] * (c[0, 0][0] * (p[1, 0][0] + p[-1, 0][0] + p[0, 1][0] + p[0, -1][0] - 4.0 * p[0, 0][0]) - w * b[0, 0][0])
                with xgrid.boundary(1):
                    p[0, 0] = p[0, 1][0] + b[0, 0][0]
    elif body == "six":
        @xgrid.kernel()
        def k(p: f2, a: f2, b: f2, c: f2, d: f2, e: f2, f: f2, w: float, trip: int) -> None:
            for _ in range(0, trip):
                p[0, 0] = w * (a[0, 0][0] * p[1, 0][0] + b[0, 0][0] * p[-1, 0][0] + c[0, 0][0] * p[0, 1][0] + d[0, 0][0] * p[0, -1][0] - e[0, 0][0]) / (1.0 + f[0, 0][0])
                with xgrid.boundary(1):
                    p[0, 0] = p[0, 1][0]
    else:   # two values in a wall's statement
        @xgrid.kernel()
        def k(p: f2, a: f2, b: f2, c: f2, d: f2, e: f2, f: f2, w: float, trip: int) -> None:
            for _ in range(0, trip):
                p[0, 0] = (p[1, 0][0] + p[-1, 0][0] + p[0, 1][0] + p[0, -1][0]) * w
                with xgrid.boundary(1):
                    p[0, 0] = p[0, 1][0] * c[0, 0][0] + b[0, 0][0]
    return k


# rows of the wave tiles that each body gets, in either precision (none: the region in LDS)
TILES = {"one": [8, 4], "two": [8, 4], "three": [4], "six": [], "wall": []}


@pytest.mark.parametrize("prec", ["double", "single"])
@pytest.mark.parametrize("body", TILES)
def test_tiles_hold_the_body(body, prec, request, tmp_path):
    request.getfixturevalue(prec)
    xgrid.init(precision="double" if prec == "double" else "float", cacheroot=str(tmp_path), precompile=False)
    low, _, path = compile_kernel(_kernel(body))
    waves = low.loops[0].waves
    assert [w.rows for w in waves] == TILES[body]
    assert all(kernel_scratch(path)[w.kernel] == 0 for w in waves[-1:])


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["double", "single"])
@pytest.mark.parametrize("body", TILES)
def test_bodies_match_oracle(body, prec, request):
    """Sizes of one tile, of tiles cut short, and (last) of many workgroups; odd and even counts, more
    than one launch."""
    xg = request.getfixturevalue(prec)
    k = _kernel(body)
    rng = np.random.default_rng(9)
    for shape, trip in (((20, 70), 5), ((150, 300), 1), ((150, 300), 14), ((300, 129), 23), ((1300, 1290), 10)):
        mask = np.full(shape, 9, np.int32)
        mask[1:-1, 1:-1] = 0
        mask[1:-1, 0] = 1
        others = [grid_pair(xg, shape, float, None, rng.random(shape) * 0.2) for _ in range(6)]
        dp, hp = grid_pair(xg, shape, float, mask, rng.random(shape))
        run_pair(k, (dp, *[o[0] for o in others], 0.25, trip), (hp, *[o[1] for o in others], 0.25, trip))
        assert_bitexact(dp, hp, levels=[0])
        info = k.native.loop_info(k.native.loop_plan(0, shape[0] * shape[1]))
        assert info["state"] == 1 and info["iterations"] > 0


@pytest.mark.gpu
@pytest.mark.parametrize("body", ["two", "three", "six"])
def test_batch_equals_plain(double, body):
    from xgrid_amd.batch import Batch
    k = _kernel(body)
    rng = np.random.default_rng(4)
    b = Batch(k)
    pairs = []
    for shape in ((40, 100), (150, 300), (70, 131)):
        mask = np.full(shape, 9, np.int32)
        mask[1:-1, 1:-1] = 0
        mask[1:-1, 0] = 1
        fields = [rng.random(shape)] + [rng.random(shape) * 0.2 for _ in range(6)]
        both = []
        for _ in range(2):
            gs = [double.Grid(shape, float) for _ in fields]
            for g, v in zip(gs, fields):
                g.now[...] = v
            gs[0].boundary[...] = mask
            both.append(gs)
        b.add(*both[0], 0.25, 13)
        pairs.append(both)
    b.step(3)
    for batched, plain in pairs:
        for _ in range(3):
            k(*plain, 0.25, 13)
        assert np.array_equal(batched[0].now.view(np.uint8), plain[0].now.view(np.uint8))
    b.close()
