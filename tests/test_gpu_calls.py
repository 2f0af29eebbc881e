"""A kernel's written-out call against the general one: the same values, levels and errors after
every kind of change between calls."""
import numpy as np
import pytest

import xgrid_amd as xgrid

pytestmark = pytest.mark.gpu
f1 = xgrid.grid[float, 1]


def _pair(tick):
    """The same kernel twice; the second always takes the general path."""
    from xgrid_amd.backend import HipKernel, build_kernel
    out = []
    for _ in range(2):
        @xgrid.kernel(tick=tick)
        def blend(u: f1, w: f1, a: float) -> None:
            u[0] = u[0][-1] + a * w[0][-1]
        blend.native, blend.depth = build_kernel(blend)
        out.append(blend)
    assert out[0].native.call is not HipKernel._invoke
    out[1].native.call = HipKernel._invoke
    return out


@pytest.mark.parametrize("tick", [True, False])
@pytest.mark.parametrize("touch", ["nothing", "read", "write", "mask", "levels", "new grid", "same grid", "other depth"])
def test_written_out_call(double, touch, tick):
    kernels = _pair(tick)
    grids = []
    for _ in kernels:
        rng = np.random.default_rng(3)
        g = [double.Grid((100,), float) for _ in range(2)]
        for x in g:
            x.now[...] = rng.random(100)
        grids.append(g)
    for step in range(8):
        for k, g in zip(kernels, grids):
            u, w = g
            if step == 4:
                if touch == "read":
                    u.now
                elif touch == "write":
                    u.now[3] = 7.0
                    w.level(1)[5] = 2.0
                elif touch == "mask":
                    u.boundary[50:] = 1
                elif touch == "levels":
                    u._extend_time(1)
                elif touch == "other depth":
                    w._extend_time(3)
                elif touch == "new grid":
                    g[1] = w = double.Grid((100,), float)
                    w.now[...] = 0.25
            k(u, u if touch == "same grid" and step >= 4 else w, 0.5)
    for a, b in zip(*grids):
        assert a.time_levels == b.time_levels
        for t in range(a.time_levels):
            assert np.array_equal(a.level(t), b.level(t))


def test_refused_calls(double):
    kernels = _pair(True)
    left = []
    for k in kernels:
        u, w, wrong = double.Grid((8,), float), double.Grid((8,), float), double.Grid((8, 8), float)
        for g in (u, w):
            g.now[...] = np.arange(8.0)
        errors = []
        for args in ((u, w, 0.5), (u, w, 0.5), (u, w), (u, w, 0.5, 1), (u, wrong, 0.5), (u, 3.0, 0.5), (u, w, "x"), (u, w, 0.5)):
            try:
                k(*args)
                errors.append(None)
            except Exception as e:
                errors.append((type(e), str(e)))
        left.append((errors, [g.level(t).tolist() for g in (u, w) for t in range(g.time_levels)]))
    assert left[0] == left[1]
    assert [e is None for e in left[0][0]] == [True, True, False, False, False, False, False, True]
