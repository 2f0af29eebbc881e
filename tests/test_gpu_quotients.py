"""Corrected quotients in blocked loops: a division by a divisor that is no power of two gives the
bits of IEEE division for numerators of every class, over divisors of every size and sign."""
import numpy as np
import pytest

import xgrid_amd as xgrid

pytestmark = pytest.mark.gpu
f2 = xgrid.grid[float, 2]


def _kernel():
    @xgrid.kernel()
    def shrink(u: f2, one: f2, d: float, trip: int) -> None:
        for _ in range(0, trip):
            u[0, 0] = u[0, 1][0] / d * one[0, 0][0]
    return shrink


def _numerators(kind, shape, dt, rng):
    """`plain` ones take the corrected form throughout; the others make workgroups divide."""
    n = shape[0] * shape[1]
    big = {np.float64: 300, np.float32: 30}[dt]
    x = ((rng.random(n) - 0.5) * 10.0 ** rng.integers(-12, 12, n)).astype(dt)
    x[::7] = 0.0
    x[3::7] = -0.0
    if kind == "wide":
        x = (rng.choice([-1.0, 1.0], n) * rng.random(n) * 10.0 ** rng.integers(-big, big, n)).astype(dt)
    elif kind == "bits":
        it = {np.float64: np.int64, np.float32: np.int32}[dt]
        x = rng.integers(np.iinfo(it).min, np.iinfo(it).max, n, dtype=it).view(dt).copy()
    elif kind == "one":      # a single cell, in one workgroup of many
        x[n // 2 + 17] = np.inf
        x[n // 3 + 5] = np.finfo(dt).smallest_subnormal
    return x.reshape(shape)


@pytest.mark.parametrize("kind", ["plain", "wide", "bits", "one"])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_quotients_are_ieee(prec, kind, request):
    xg = request.getfixturevalue(prec)
    dt = np.float64 if prec == "double" else np.float32
    rng = np.random.default_rng(11)
    shape = (300, 500)
    u0 = _numerators(kind, shape, dt, rng)
    mask = np.zeros(shape, np.int32)
    mask[:, -1] = 1
    k = _kernel()
    one = xg.Grid(shape, float)
    one.now[...] = 1.0
    f = np.finfo(dt)
    for d in (3.0, 0.1, 1e-5, 6.02e23, -7.25, 0.0, np.inf, np.nextafter(dt(2), dt(0)), np.nextafter(dt(1), dt(2)),
              f.max, f.max / 16 * 0.7, f.smallest_normal * 1.5, f.smallest_subnormal * 3, np.nan, 1.5):
        d = float(dt(d))
        for trip in (1, 3):
            u = xg.Grid(shape, float)
            u.now[...] = u0
            u.boundary[...] = mask
            want = u0.copy()
            with np.errstate(all="ignore"):
                for _ in range(trip):
                    want[:, :-1] = want[:, 1:] / dt(d)
            k(u, one, d, trip)
            got, nan = u.now, np.isnan(want)
            assert np.array_equal(np.isnan(got), nan), (d, trip)
            bits = {np.float64: np.uint64, np.float32: np.uint32}[dt]
            assert np.array_equal(got[~nan].view(bits), want[~nan].view(bits)), (d, trip)
    low = k.native.lowered
    assert low.loops[0].waves and "value_rgq" in low.device_src
    assert k.native.loop_info(k.native.loop_plan(0, shape[0] * shape[1]))["iterations"] > 0
