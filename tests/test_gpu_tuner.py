"""The autotuner weighs a kernel's default build (its wave tiles) against the tile shapes, keeps that choice in
its cache, and a batch tuned to it runs it."""
import pytest

import xgrid_amd as xgrid

pytestmark = pytest.mark.gpu


def test_default_build_is_a_candidate(double, tmp_path):
    from xgrid_amd import autotune, workloads as W
    from xgrid_amd.grid import Grid
    from xgrid_amd.multi import MultiSolver
    specs = [s for s in W.batch_specs(8, seed=9, lo=48, hi=200) if s.kind == "cavity"][:2]
    xgrid.init(precision="double", cacheroot=str(tmp_path), precompile=False)
    ms = MultiSolver("double")
    ms.autotune(specs, limit=2, use_cache=False)
    (tuned,) = ms.tuning.values()
    assert set(tuned["timings"]) == {"default"} | {",".join(map(str, c)) for c in autotune.CANDIDATES if c}
    best = min(tuned["timings"], key=tuned["timings"].get)
    assert tuned["shape"] == (None if best == "default" else next(c for c in autotune.CANDIDATES if c and ",".join(map(str, c)) == best))
    assert bool(ms.natives["cavity"].lowered.loops[0].waves) == (tuned["shape"] is None)
    ms.close()
    # a choice of the default build is kept and found again; it is no choice among other candidates
    tune = lambda c: autotune.tune_batch(W.make_cavity(), lambda s: W.instance_grids(s, Grid), specs, "double",
                                         candidates=c, warm=1, steps=1)
    for cached in (False, True):
        r = tune([None])
        assert r["shape"] is None and r["cached"] == cached and list(r["timings"]) == ["default"]
    assert tune([(48, 64, 1024, 10, "lds")]) == {"shape": (48, 64, 1024, 10, "lds"), "cached": False,
                                                 "timings": pytest.approx({"48,64,1024,10,lds": 1.0}, rel=1e9)}
