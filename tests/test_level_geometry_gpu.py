"""Every level kernel on grids that do not cover the graph at once: the rounds
of any number of workgroups visit each vertex and edge once, so depths and
counts are the oracle's."""
import ctypes as C

import numpy as np
import pytest

from belewitte_amd import _native as N
from belewitte_amd import bfs, device, graph
from oracle import binding as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", sorted(n for n in bfs.IMPLEMENTATIONS if "reduce" not in n and "bulk" not in n))
@pytest.mark.parametrize("grid", [1, 2, 3, 7, 8, 9, 17, 64])
def test_levels_on_any_grid(gpu, name, grid):
    kernel, reduction = bfs.parse(name)
    for g, block, warp, chunk in ((graph.rmat_n(5003, 40000, seed=5, undirected=True), 64, 32, 32),
                                  (graph.rmat_n(1999, 9000, seed=6, undirected=True), 128, 8, 16)):
        dg = device.DeviceGraph(g)
        dg.ensure(bfs.REPRESENTATION[kernel])
        root = g.max_out_degree_vertex()
        levels = device.DeviceArray(g.vertex_count, np.int32)
        counts, n = np.zeros(64, np.uint32), C.c_int64()
        cfg = N.launch(block=block, grid=grid, warp=warp, chunk=chunk)
        try:
            N.check_hip(N.hip_lib().bw_bfs_run(dg.ref, (C.c_int32 * 1)(kernel), 1, reduction, root, levels.ptr,
                                               counts.ctypes.data_as(N.u32p), None, 64, C.byref(n), C.byref(cfg)))
            want, _ = O.bfs_queue(O.CSR.from_graph(g), root)
            assert np.array_equal(levels.download(), want), (name, grid, g.vertex_count)
            reached = want[want < g.vertex_count]
            assert np.array_equal(counts[:n.value], np.append(np.bincount(reached)[1:], 0)), (name, grid)
        finally:
            levels.free()
            dg.free()
