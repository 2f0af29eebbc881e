"""Pairs of interiors at the sizes where they leave the chain's workgroup (more cells than its 1024
work-items) and where the chain ends (4096 cells), against the oracle's bits."""
import numpy as np
import pytest

from oracle.cpu_path import CpuKernel, HostGrid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [33, 34, 35, 65, 66, 67])
@pytest.mark.parametrize("prec", ["double", "single"])
def test_cavity_around_the_chain(prec, n, request):
    from xgrid_amd import workloads as W
    xg = request.getfixturevalue(prec)
    k = W.make_cavity()
    cfg, masks, rng = W.cavity_config(n, dt=2e-6), W.cavity_masks(n), np.random.default_rng(n)
    dev, host = {c: xg.Grid((n, n), float) for c in "bpuv"}, {c: HostGrid((n, n), float) for c in "bpuv"}
    for c in "bpuv":
        x = rng.random((n, n)) * 0.1
        for g in (dev[c], host[c]):
            g.now[...] = x
            g.boundary[...] = masks[c]
    ck = CpuKernel(k)
    for _ in range(3):
        k(*[dev[c] for c in "bpuv"], cfg)
        ck(*[host[c] for c in "bpuv"], cfg)
    for c in "bpuv":
        assert np.array_equal(dev[c].now.view(np.uint8), host[c].now.view(np.uint8)), c
