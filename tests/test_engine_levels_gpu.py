"""The engine's levels at the edges of their forms: levels of up to 2048
vertices and out-edges run inside the epilogue (1024 of them per launch at
most), larger ones as their own launch with the frontier in per-workgroup
segments behind the queue, from 32 vertices per workgroup on dealt out in
runs of eight.  Depths and counts are the oracle's."""
import numpy as np
import pytest

from belewitte_amd import _native as N
from belewitte_amd import bfs_native, device, graph
from oracle import binding as O

pytestmark = pytest.mark.gpu


def _layers(*sizes):
    """Layers of the given sizes: every vertex has an in-edge from a vertex of
    the layer before, a layer's first vertex has all that its others have not."""
    src, dst, at = [], [], 0
    for a, b in zip(sizes, sizes[1:]):
        d = np.arange(at + a, at + a + b)
        src.append(at + np.where(np.arange(b) < a, np.arange(b), 0))
        dst.append(d)
        at += a
    return graph.from_edges(sum(sizes), np.concatenate(src).astype(np.uint32),
                            np.concatenate(dst).astype(np.uint32))


def _hubs(hubs, degree):
    """A vertex with `hubs` children of `degree` leaves each."""
    src = np.concatenate([np.zeros(hubs, int), np.repeat(np.arange(1, 1 + hubs), degree)])
    dst = np.concatenate([np.arange(1, 1 + hubs), np.arange(1 + hubs, 1 + hubs + hubs * degree)])
    return graph.from_edges(1 + hubs * (degree + 1), src.astype(np.uint32), dst.astype(np.uint32))


CASES = {
    "edges at the limit": _layers(1, 2048, 2048, 1, 2049, 3, 2047, 5),
    "out of it and back": _layers(1, 1, 3000, 2, 2, 4100, 1, 9000, 40, 40, 1),   # hubs of 4100 and 9000 edges too
    "more levels than a launch": graph.chain(3 * 1024 + 7),
    "many hubs out of it": _hubs(300, 257),
    "segments": _layers(1, 65535, 65535, 65536, 65537, 70000, 300, 300, 200000, 1),
    "one vertex": graph.from_edges(1, np.zeros(0, np.uint32), np.zeros(0, np.uint32)),
}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("use_graph", [False, True])
def test_level_forms(gpu, name, use_graph):
    g = CASES[name]
    csr, dg = O.CSR.from_graph(g), device.DeviceGraph(g)
    eng = bfs_native.BFSEngine(dg, edge_lists=True)
    if "hubs" in name:
        eng.set_tuning(hub_degree=256)  # every child is a hub, 256 of them in the hub queue at most
        eng.set_queues(hub_cap=256)
    roots = sorted({0, g.vertex_count // 2, g.vertex_count - 1})
    depths = {r: O.bfs_queue(csr, r)[0] for r in roots}
    runs = [("fixed", "td", None), ("fixed", "bu-wave", None), ("beamer", "td", None),
            ("schedule", "td", ["td", "td", "bu", "td", "vertex-push", "td", "td", "edge-list"])]
    try:
        for policy, variant, schedule in runs:
            for root in roots + [roots + [roots[0]]]:
                print(f"case {name} root={root} {policy} {variant} graph={use_graph}", flush=True)
                want = np.stack([depths[r] for r in np.atleast_1d(root)]).min(0)  # unreached: the largest
                reached = want[want < g.vertex_count]
                r = eng.run(root, policy, variant, schedule=schedule, use_graph=use_graph)
                counts = np.append(np.bincount(reached)[1:], 0)
                assert np.array_equal(r.levels, want), (name, root, policy)
                assert np.array_equal(r.counts, counts), (name, root, policy)
    finally:
        eng.close()
        dg.free()


@pytest.mark.parametrize("levels", [1, 2, 5, 6, 7])
def test_level_limit(gpu, levels):
    """A search of six levels (the last finds nothing) on an engine with room
    for fewer is refused."""
    g = graph.chain(5)
    csr, dg = O.CSR.from_graph(g), device.DeviceGraph(g)
    eng = bfs_native.BFSEngine(dg, max_levels=levels)
    try:
        if levels < 6:
            with pytest.raises(N.BelewitteError):
                eng.run(0)
        else:
            assert np.array_equal(eng.run(0).levels, O.bfs_queue(csr, 0)[0])
    finally:
        eng.close()
        dg.free()
