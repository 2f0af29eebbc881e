"""Divisions by a uniform divisor that a lane may not run (an arm of a conditional, the right side
of `and`) inside blocked loops: the kernels compile, and give the bits of the oracle."""
import os
import subprocess
import sys

import numpy as np
import pytest

import xgrid_amd as xgrid

from helpers import assert_bitexact, grid_pair, run_pair

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
f2 = xgrid.grid[float, 2]


def _kernel(form):
    if form == "then":
        @xgrid.kernel()
        def k(u: f2, w: f2, d: float, e: float, trip: int) -> None:
            for _ in range(0, trip):
                u[0, 0] = u[0, 1][0] / d if w[0, 0][0] > 0.5 else u[0, -1][0]
    elif form == "else":
        @xgrid.kernel()
        def k(u: f2, w: f2, d: float, e: float, trip: int) -> None:
            for _ in range(0, trip):
                u[0, 0] = u[0, 1][0] if w[0, 0][0] > 0.5 else u[0, -1][0] / d
    elif form == "and":
        @xgrid.kernel()
        def k(u: f2, w: f2, d: float, e: float, trip: int) -> None:
            for _ in range(0, trip):
                u[0, 0] = u[0, 1][0] if w[0, 0][0] > 0.5 and u[0, 1][0] / d < 0.125 else u[1, 0][0]
    else:   # the condition divides for every cell, the arms for some
        @xgrid.kernel()
        def k(u: f2, w: f2, d: float, e: float, trip: int) -> None:
            for _ in range(0, trip):
                u[0, 0] = (u[0, 1][0] / d if w[0, 0][0] > 0.5 else u[0, -1][0] / e) if u[0, 1][0] / d < w[0, 0][0] else u[-1, 0][0]
    return k


FORMS = ["then", "else", "and", "mixed"]


@pytest.mark.parametrize("prec", ["double", "float"])
def test_compiles(tmp_path, prec):
    """In a process of its own: the device compiler ends the process where it cannot go on."""
    code = ("import sys; sys.path[:0] = [%r, %r]\n"
            "import xgrid_amd as xg, test_conditional_quotients as t\n"
            "from xgrid_amd.backend import lower_kernel\n"
            "from xgrid_amd.compilers import compile_device\n"
            "xg.init(precision=%r, cacheroot=%r, precompile=False)\n"
            "for form in t.FORMS:\n"
            "    low, _ = lower_kernel(t._kernel(form))\n"
            "    assert low.loops[0].waves and ('value_rgq' in low.device_src) == (form == 'mixed'), form\n"
            "    for src in (low.device_src, low.batch_src)[:1 + (form == 'mixed')]:\n"
            "        compile_device(src, %r)\n" % (ROOT, os.path.join(ROOT, "tests"), prec, str(tmp_path), str(tmp_path)))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("prec", ["double", "single"])
def test_match_oracle(prec, form, request):
    """Conditions that differ from lane to lane, numerators that the corrected form gets right and (a
    few cells) infinite and subnormal ones that it does not; no NaN arises."""
    xg = request.getfixturevalue(prec)
    dt = np.float64 if prec == "double" else np.float32
    shape = (150, 300)
    rng = np.random.default_rng(5)
    mask = np.zeros(shape, np.int32)
    mask[0], mask[-1], mask[:, 0], mask[:, -1] = 1, 1, 1, 1
    k = _kernel(form)
    for special in (False, True):
        u0 = ((rng.random(shape) - 0.5) * 4).astype(dt)
        if special:
            u0[::17, ::23], u0[5::31, 7::19] = np.inf, -np.inf
            u0[3::13, 11::29] = np.finfo(dt).smallest_subnormal * 5
        du, hu = grid_pair(xg, shape, float, mask, u0)
        dw, hw = grid_pair(xg, shape, float, None, rng.random(shape))
        # (twice: the first call checks the mask)
        for d, e, trip in ((3.7, 0.3, 1), (3.7, 0.3, 6), (4.0, 3.7, 5)):
            run_pair(k, (du, dw, d, e, trip), (hu, hw, d, e, trip))
            assert_bitexact(du, hu, levels=[0])
    info = k.native.loop_info(k.native.loop_plan(0, shape[0] * shape[1]))
    assert k.native.lowered.loops[0].waves and info["iterations"] > 0
