"""Multi-source search at the edges of its numbering of the frontier's edges
(tiles of 64 vertices, groups of four tiles, windows of 512 edges, the
epilogue's rounds of 4096 groups) and of its reset: depths equal the oracle's for every source and the
levels' new bits are their counts."""
import numpy as np
import pytest

from belewitte_amd import bfs_native, device, graph
from oracle import binding as O

pytestmark = pytest.mark.gpu


def _random(V, E, seed):
    rng = np.random.default_rng(seed)
    s, d = rng.integers(0, V, E), rng.integers(0, V, E)
    s = np.where(s % 7 == 0, V - 1, s)  # the last vertex is a hub; many have no out-edges
    return graph.from_edges(V, s.astype(np.uint32), d.astype(np.uint32))


@pytest.mark.parametrize("V,E", [(1, 0), (63, 100), (64, 511), (65, 600), (129, 20), (255, 900), (257, 3),
                                 (8191, 30000), (8192 * 64, 700000), (8192 * 64 + 1, 600000),
                                 (8192 * 64 * 2 + 63, 900000), (8192 * 64 * 4 + 1, 700000)])
@pytest.mark.parametrize("n", [1, 3, 64])
def test_levels(gpu, V, E, n):
    g = _random(V, E, V + n)
    csr, dg = O.CSR.from_graph(g), device.DeviceGraph(g)
    ms = bfs_native.MultiSourceBFS(dg)
    rng = np.random.default_rng(n)
    src = rng.integers(0, V, n).astype(np.uint32)
    src[-1] = V - 1
    src[n // 2] = src[0]                # a repeated source, and several in one tile
    src[n // 3] = min(V - 1, int(src[0]) + 1)
    try:
        want = np.stack([O.bfs_queue(csr, int(r))[0] for r in src])
        reached = want[want < max(V, 2)]
        bits = np.append(np.bincount(reached)[1:], 0)
        for div in (4, 1, 0, 1024):
            ms.set_tuning(topdown_divisor=div)
            for use_graph in (False, True):
                print(f"case V={V} E={g.edge_count} n={n} div={div} graph={use_graph}", flush=True)
                depths, _, got = ms.run(src, use_graph=use_graph)
                assert np.array_equal(depths, want), (V, E, n, div)
                assert np.array_equal(got, bits), (V, E, n, div)
    finally:
        ms.close()
        dg.free()
