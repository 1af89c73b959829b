"""Loops over edges at the limit of 32-bit edge counts, 2^32 - 1: no counter
wraps past it.  Every edge runs from vertex 0 to vertex 1, so the results are
known without a reference run."""
import ctypes as C

import numpy as np
import pytest

from belewitte_amd import _native as N
from belewitte_amd import device

pytestmark = pytest.mark.gpu

E = 2 ** 32 - 1


def _filled(value, n=E):
    a = device.DeviceArray(n, np.uint32)
    a.fill_u32(value)
    return a


def test_vertex_push_level(gpu):
    off = device.DeviceArray.from_host(np.array([0, E, E], np.uint32))
    levels = device.DeviceArray.from_host(np.array([0, 2 ** 31 - 1], np.int32))
    frontier = _filled(0, 1)
    cols = _filled(1)
    cfg = N.launch(block=1024)
    try:
        N.check_hip(N.hip_lib().bw_bfs_vertex_push(2, off.ptr, 4, cols.ptr, levels.ptr, 0, frontier.ptr, 0,
                                                   C.byref(cfg)))
        device.synchronize()
        assert levels.download().tolist() == [0, 1] and frontier.download().tolist() == [1]
    finally:
        for x in (off, levels, frontier, cols):
            x.free()
