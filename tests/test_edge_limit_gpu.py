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


@pytest.mark.parametrize("V", [2, (1 << 20) + 1])  # the gathered and the binned layout
def test_scatter_sums(gpu, V):
    """Vertex 1 receives E contributions of 1 / E read as FP32, 2^-32: 1 to
    two roundings (of the FP64 sum, and of the chunks' FP32 partials where
    there are several, all of them multiples of 2^-32 below 1)."""
    src, dst = _filled(0), _filled(1)
    deg, pr, out = _filled(0, V), _filled(0, V), _filled(0, V)
    N.check_hip(N.hip_lib().bw_hip_fill_u32(deg.ptr, E, 1, None))
    N.check_hip(N.hip_lib().bw_hip_fill_u32(pr.ptr, 0x3F800000, 1, None))
    layout = C.c_void_p()
    try:
        N.check_hip(N.hip_lib().bw_pr_scatter_create(C.byref(layout), 0, V, E, src.ptr, dst.ptr, 4, None))
        N.check_hip(N.hip_lib().bw_pr_scatter_iteration(layout, deg.ptr, pr.ptr, out.ptr, None))
        device.synchronize()
        got = out.download().view(np.float32)
        assert abs(float(got[1]) - 1.0) <= 2 * 2.0 ** -24
        got[1] = 0
        assert not got.any()
    finally:
        N.hip_lib().bw_pr_scatter_destroy(layout)
        for x in (src, dst, deg, pr, out):
            x.free()
