"""What a garbage collector releases on another thread while a call is being captured as a graph (the
interpreter runs finalizers on any thread, and calls release its lock) leaves the capture whole."""
import ctypes
import gc
import threading
import time
from ctypes import c_int, c_int32, c_int64, c_void_p

import numpy as np
import pytest

import xgrid_amd as xgrid
from xgrid_amd import _lib
from xgrid_amd.backend import HipKernel

pytestmark = pytest.mark.gpu
f1 = xgrid.grid[float, 1]


def _kernel(xg):
    @xg.kernel()
    def add(u: f1) -> None:
        u[0] = u[0][0] + 1.0
    return add


def _drop_kernel(xg):
    op = _kernel(xg)
    native = HipKernel(op)
    g = xg.Grid((64,), float)
    g.now[...] = 0.0
    return native.close


def _drop_grid(xg):
    held = [xg.Grid((64,), float)]
    held[0]._device()

    def drop():
        held.clear()
        gc.collect()
    return drop


def _drop_exported_grid(xg):
    held = [xg.Grid((64,), float)]
    held[0]._device()
    _lib.load().xg_grid_level_ptr(held[0]._handle, 0)

    def drop():
        held.clear()
        gc.collect()
    return drop


def _drop_batch(xg):
    from xgrid_amd.batch import Batch
    b = Batch(_kernel(xg))
    g = xg.Grid((64,), float)
    b.add(g)
    b.step(4)
    return b.close


@pytest.mark.parametrize("make", [_drop_kernel, _drop_grid, _drop_exported_grid, _drop_batch])
def test_release_during_capture(double, make):
    native = HipKernel(_kernel(double))
    g = double.Grid((4096,), float)
    g.now[...] = 1.0
    lib = _lib.load()
    plan = native.new_plan()
    api = _lib.Api.from_address(lib.xg_api_table())
    begin = ctypes.CFUNCTYPE(c_int, c_void_p, ctypes.POINTER(c_void_p), c_int32, c_void_p, c_int64)(api.begin)
    stmt = ctypes.CFUNCTYPE(c_int, c_void_p, c_int32, c_void_p, c_int64)(api.stmt)
    end = ctypes.CFUNCTYPE(c_int, c_void_p)(api.end)
    handles = (c_void_p * 1)(g._sync_for_launch())
    nbytes = native._descs[0].param_bytes
    params = ctypes.create_string_buffer(max(8, nbytes))

    def call(during=None):
        assert begin(plan, handles, 1, params, 0) == 0
        for i in range(4):
            assert stmt(plan, 0, params, nbytes) == 0
            if i == 1 and during:
                during()
        rc = end(plan)
        assert rc == 0, _lib.last_error()

    drop = make(double)
    thread = threading.Thread(target=drop)

    def during():
        thread.start()
        time.sleep(0.2)

    call()              # the first sighting of these arguments runs directly
    call(during)        # the second is captured
    thread.join(30)
    assert not thread.is_alive()
    call()              # and replayed
    captures = c_int64()
    assert lib.xg_kernel_counters(plan, None, None, None, ctypes.byref(captures)) == 0 and captures.value == 1
    g._device_wrote()
    assert np.array_equal(g.now, np.full(4096, 13.0))
    lib.xg_kernel_destroy(plan)
