"""Row sums of the push forms' layouts (bw_pr_scatter_*), all three sources.

The sums are kept in FP64 and rounded to FP32 once per row, so a row is
within one rounding (2^-24, doubled for slack) of the exact sum of its
contributions, themselves FP32 quotients.
"""
import ctypes as C

import numpy as np
import pytest

from belewitte_amd import _native as N
from belewitte_amd import device

pytestmark = pytest.mark.gpu

EDGE_LIST, STRUCT, CSR = 0, 1, 2


def _edges(V, E, rng):
    """Random edges with a destination hub (its partition is cut into many
    chunks) and a source hub, sorted by source."""
    s = rng.integers(0, V, E)
    d = rng.integers(0, V, E)
    d[: E // 3] = V // 2
    s[E // 2: E // 2 + E // 8] = V - 1
    o = np.argsort(s, kind="stable")
    return s[o].astype(np.uint32), d[o].astype(np.uint32)


@pytest.mark.parametrize("V,E", [(1, 5), (255, 900), (256, 2048), (257, 2049), (70001, 300000), (1 << 18, 400001),
                                 ((1 << 20) + 1, 60000), ((1 << 20) + 1, 700001), (3 << 20, 1500000)])
@pytest.mark.parametrize("kind", [EDGE_LIST, STRUCT, CSR])
@pytest.mark.parametrize("offset_bytes", [4, 8])
def test_scatter_sums(gpu, V, E, kind, offset_bytes):
    if offset_bytes == 8 and kind != CSR:
        pytest.skip("only the CSR has offsets")
    rng = np.random.default_rng(V + E)
    src, dst = _edges(V, E, rng)
    deg = np.bincount(src, minlength=V).astype(np.uint32)
    pr = rng.random(V).astype(np.float32)
    bufs = [device.DeviceArray.from_host(deg), device.DeviceArray.from_host(pr)]
    d_deg, d_pr = bufs
    if kind == EDGE_LIST:
        a, b = device.DeviceArray.from_host(src), device.DeviceArray.from_host(dst)
    elif kind == STRUCT:
        a, b = device.DeviceArray.from_host(np.stack([src, dst], axis=1).reshape(-1)), None
    else:
        off = np.concatenate([[0], np.cumsum(deg, dtype=np.int64)])
        a = device.DeviceArray.from_host(off.astype(np.uint32 if offset_bytes == 4 else np.uint64))
        b = device.DeviceArray.from_host(dst)
    out = device.DeviceArray(V, np.float32)
    out.fill_u32(0)
    lib = N.hip_lib()
    layout = C.c_void_p()
    N.check_hip(lib.bw_pr_scatter_create(C.byref(layout), kind, V, E, a.ptr, b.ptr if b else None, offset_bytes, None))
    try:
        N.check_hip(lib.bw_pr_scatter_iteration(layout, d_deg.ptr, d_pr.ptr, out.ptr, None))
        device.synchronize()
        got = out.download().astype(np.float64)
    finally:
        lib.bw_pr_scatter_destroy(layout)
        for x in bufs + [a, out] + ([b] if b else []):
            x.free()
    with np.errstate(divide="ignore"):
        c = np.where(deg > 0, pr / deg.astype(np.float32), np.float32(0)).astype(np.float64)
    want = np.bincount(dst, weights=c[src], minlength=V)
    # beyond 2^20 vertices a row cut into chunks is added from FP32 partials
    chunks = 1 if V <= 1 << 20 else 1 + E // (1 << 17)
    assert np.all(np.abs(got - want) <= (1 + chunks) * 2.0 ** -24 * want), (V, E, kind)
