"""Norms taken by several threads at once are those that one thread gets: the entries share scratch
memory and one result slot each."""
import ctypes
import threading

import numpy as np
import pytest

from xgrid_amd import _lib, norms

pytestmark = pytest.mark.gpu


def _noalloc(g):
    l2, linf = ctypes.c_double(), ctypes.c_double()
    rc = _lib.load().xg_grid_norm_diff_noalloc(g._sync_for_launch(), 0, _lib.T_F64, None, 0, 0, 0, ctypes.byref(l2),
                                               ctypes.byref(linf), None)
    assert rc == 0, _lib.last_error()
    return l2.value, linf.value


def _diff(g):
    r = norms.diff_norm(g)
    return r["l2"], r["linf"]


def _poisson(g):
    r = norms.poisson_residual(g, g, (1.0, 2.0), klass=0)
    return r["l2"], r["linf"]


@pytest.mark.parametrize("entry", [_diff, _noalloc, _poisson])
def test_threads_get_their_own_norms(double, entry):
    rng = np.random.default_rng(2)
    grids = []
    for i in range(6):
        n = 40 + 300 * i
        g = double.Grid((n, n), float)
        g.now[...] = (rng.random((n, n)) - 0.5) * 3.0 ** i
        g.boundary[0], g.boundary[-1], g.boundary[:, 0], g.boundary[:, -1] = 1, 1, 1, 1
        grids.append(g)
    want = [entry(g) for g in grids]
    assert len(set(want)) == len(want)
    wrong = []

    def work(i):
        for _ in range(100):
            got = entry(grids[i])
            if got != want[i]:
                wrong.append((i, got, want[i]))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(grids))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:3]
