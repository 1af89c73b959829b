"""bw_graph_relabel_by_degree on raw arrays: both directions at once when
the reverse lists are the forward lists' transpose, each on its own
otherwise; the rows of each come out permuted, mapped and sorted."""
import numpy as np
import pytest

from belewitte_amd import _native as N
from belewitte_amd import device

pytestmark = pytest.mark.gpu


def _csr(V, rows, cols):
    o = np.lexsort((np.arange(rows.size), rows))
    return np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=V))]).astype(np.uint32), cols[o].astype(np.uint32)


def _want(V, off, cols, perm):
    rows = np.repeat(np.arange(V), np.diff(off.astype(np.int64)))
    r, c = perm[rows], perm[cols]
    o = np.lexsort((c, r))
    return np.concatenate([[0], np.cumsum(np.bincount(r, minlength=V))]).astype(np.uint32), c[o].astype(np.uint32)


@pytest.mark.parametrize("V,E", [(1, 3), (2, 1), (63, 500), (5000, 3), (5000, 40000), (70000, 4097)])
@pytest.mark.parametrize("reverse", ["transpose", "other", "columns", "none"])
def test_relabel_directions(gpu, V, E, reverse):
    rng = np.random.default_rng(V * 7 + E)
    src = np.minimum(rng.integers(0, V, E), rng.integers(0, V, E))  # skewed, with repeated edges
    dst = rng.integers(0, V, E)
    off, cols = _csr(V, src, dst)
    if reverse == "transpose":
        roff, rcols = _csr(V, dst, src)
    elif reverse == "columns":  # the transpose's in-degrees, but other columns
        roff, rcols = _csr(V, dst, rng.permutation(src))
    else:  # not the transpose: other in-degrees
        roff, rcols = _csr(V, (dst + 1) % V, src)
    order = np.argsort(-np.diff(off.astype(np.int64)), kind="stable")
    perm = np.empty(V, np.uint32)
    perm[order] = np.arange(V)
    ins = [device.DeviceArray.from_host(x) for x in (off, cols, roff, rcols)]
    outs = [device.DeviceArray(n, np.uint32) for n in (V + 1, E, V + 1, E, V)]
    rev = reverse != "none"
    try:
        N.check_hip(N.hip_lib().bw_graph_relabel_by_degree(
            V, E, ins[0].ptr, ins[1].ptr, ins[2].ptr if rev else None, ins[3].ptr if rev else None, outs[0].ptr,
            outs[1].ptr, outs[2].ptr if rev else None, outs[3].ptr if rev else None, outs[4].ptr, None))
        got = [o.download() for o in outs]
    finally:
        for x in ins + outs:
            x.free()
    assert np.array_equal(got[4], perm)
    for k, (o, c) in enumerate([(off, cols), (roff, rcols)][: 1 + rev]):
        woff, wcols = _want(V, o, c, perm)
        assert np.array_equal(got[2 * k], woff), (V, E, reverse, k)
        assert np.array_equal(got[2 * k + 1], wcols), (V, E, reverse, k)


# (row, row, column, column) whose swap an order-independent sum of hashes with
# two rounds of multiplication does not see.
@pytest.mark.parametrize("r1,r2,c1,c2", [(34456, 53208, 44788, 18958), (33183, 35060, 50385, 30693),
                                         (1794, 31874, 44307, 32023)])
def test_reverse_lists_with_two_columns_swapped(gpu, r1, r2, c1, c2):
    V = 65536
    src = np.arange(V)  # one edge each: the order stays
    dst = np.arange(V)
    dst[[c1, c2]] = r1, r2
    off, cols = _csr(V, src, dst)
    src[[c1, c2]] = c2, c1
    roff, rcols = _csr(V, dst, src)
    ins = [device.DeviceArray.from_host(x) for x in (off, cols, roff, rcols)]
    outs = [device.DeviceArray(n, np.uint32) for n in (V + 1, V, V + 1, V, V)]
    try:
        N.check_hip(N.hip_lib().bw_graph_relabel_by_degree(V, V, *(x.ptr for x in ins + outs), None))
        got = [o.download() for o in outs]
    finally:
        for x in ins + outs:
            x.free()
    for k, (o, c) in enumerate([(off, cols), (roff, rcols)]):
        woff, wcols = _want(V, o, c, np.arange(V, dtype=np.uint32))
        assert np.array_equal(got[2 * k], woff)
        assert np.array_equal(got[2 * k + 1], wcols)
