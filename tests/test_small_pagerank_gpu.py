"""PageRank runs of small graphs (one launch for the whole run) at the edges
of the form's limits: the ranks are the fixed-point oracle's bit for bit in
DROP mode, as the binned iteration's are with one chunk per partition; in
UNIFORM mode they follow the FP64 recurrence to the rounding of FP32 ranks
(2^-24 relative per iteration's rounding, a few of which survive)."""
import numpy as np
import pytest

from belewitte_amd import device, graph, pagerank
from oracle import binding as O

pytestmark = pytest.mark.gpu


def _graph(V, E, seed):
    rng = np.random.default_rng(seed)
    s = rng.integers(0, V, E)
    d = np.where(rng.random(E) < 0.3, V - 1, rng.integers(0, V, E))  # an in-hub; some vertices without out-edges
    s = np.where(s % 5 == 0, 0, s)
    return graph.from_edges(V, s.astype(np.uint32), d.astype(np.uint32), keep_self_loops=True)


@pytest.mark.parametrize("V,E", [(1, 1), (2, 1), (63, 8191), (1024, 8192), (1025, 8193), (4097, 16384), (4100, 16385),
                                 (8191, 32768), (8192, 32700), (8192, 33500), (8193, 9000)])
@pytest.mark.parametrize("layout", ["bins", "pull"])
def test_small_run(gpu, V, E, layout):
    g = _graph(V, E, V + E)
    csr = O.CSR.from_graph(g)
    dg = device.DeviceGraph(g)
    fp = pagerank.FusedPageRank(dg, max_iterations=30)
    try:
        if layout == "bins":
            fp.bin(14, 4096, 8)
        small = V <= 8192 and g.edge_count <= 32768
        assert ("pr_small_kernel" in fp.kernel_names()) == small
        for quirk in (False, True):
            for iters in (1, 30):
                ranks, resid, _ = fp.run(iters, "drop", nodiv_quirk=quirk)
                want = O.pagerank_binned_fixed(csr, iters, nodiv_quirk=quirk)
                if small or layout == "bins":
                    assert np.array_equal(ranks.view(np.uint32), want.view(np.uint32)), (V, E, quirk, iters)
                assert np.all(np.isfinite(resid))
        ranks, resid, _ = fp.run(30, "uniform")
        x = O.pagerank_f64(csr, 30, "uniform")
        assert np.all(np.abs(ranks - x) <= 8 * 2.0 ** -24 * x), (V, E)
        again, ragain, _ = fp.run(30, "uniform")
        assert np.array_equal(ranks.view(np.uint32), again.view(np.uint32)) and np.array_equal(resid, ragain)
    finally:
        fp.close()
        dg.free()
