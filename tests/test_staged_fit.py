"""Staged 3-D kernels that spill at six waves per SIMD are built for five; the others stay as they are."""
import numpy as np
import pytest

import xgrid_amd as xgrid
from xgrid_amd.backend import compile_batch, compile_kernel
from xgrid_amd.batch import Batch
from xgrid_amd.compilers import kernel_scratch
from xgrid_amd.config import get_config

from helpers import assert_bitexact, grid_pair, run_pair
from oracle.cpu_path import CpuKernel

f3 = xgrid.grid[float, 3]


def _near():
    @xgrid.kernel()
    def near(u: f3, a: float) -> None:
        u[0, 0, 0] = u[0, 0, 0] + a * (u[1, 0, 0] + u[-1, 0, 0] + u[0, 1, 0] + u[0, -1, 0] + u[0, 0, 1] + u[0, 0, -1])
        with xgrid.boundary(1):
            u[0, 0, 0] = 0.5
    return near


def _far():
    @xgrid.kernel()
    def far(u: f3, a: float) -> None:
        u[0, 0, 0] = u[0, 0, 0] + a * (u[1, 0, 0] + u[-1, 0, 0] + u[0, 1, 0] + u[0, -1, 0] + u[0, 0, 1] + u[0, 0, -1] +
                                       u[2, 0, 0] + u[-2, 0, 0] + u[0, 2, 0] + u[0, -2, 0] + u[0, 0, 2] + u[0, 0, -2])
        with xgrid.boundary(1):
            u[0, 0, 0] = 0.5
    return far


@pytest.mark.parametrize("prec", ["double", "float"])
def test_waves(prec, tmp_path):
    xgrid.init(precision=prec, cacheroot=str(tmp_path))
    for make, asked in ((_near, 6), (_far, 5)):
        low, _, path = compile_kernel(make())
        head = next(l for l in low.device_src.split("\n") if 'extern "C"' in l and " xg_k0(" in l)
        assert f"amdgpu_waves_per_eu({asked})" in head
        assert kernel_scratch(path)["xg_k0"] <= 64
        assert kernel_scratch(compile_batch(low, get_config()))["xg_k0_b"] <= 64


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(9, 10, 11), (20, 18, 133), (37, 21, 260)])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_reach_two(prec, shape, request):
    xg = request.getfixturevalue(prec)
    rng = np.random.default_rng(5)
    mask = np.ones(shape, np.int32)
    mask[2:-2, 2:-2, 2:-2] = 0
    d, h = grid_pair(xg, shape, float, mask, rng.random(shape))
    run_pair(_far(), (d, 0.05), (h, 0.05), steps=4)
    assert_bitexact(d, h)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["double", "single"])
def test_reach_two_batched(prec, request):
    xg = request.getfixturevalue(prec)
    k = _far()
    b = Batch(k)
    rng = np.random.default_rng(6)
    pairs = []
    for shape in ((9, 10, 11), (20, 18, 133), (37, 21, 260)):
        mask = np.ones(shape, np.int32)
        mask[2:-2, 2:-2, 2:-2] = 0
        pairs.append(grid_pair(xg, shape, float, mask, rng.random(shape)))
        b.add(pairs[-1][0], 0.05)
    b.step(4)
    ck = CpuKernel(k)
    for d, h in pairs:
        for _ in range(4):
            ck(h, 0.05)
        assert_bitexact(d, h)
    b.close()
