"""Sums of long rows in the pull iteration (bw_pr_pull_iteration).

Rows past the long-row split are summed by a wave or a workgroup each; the
thread-per-vertex variant's sum must be the reference's sequential FP32 sum
bit for bit whatever the values: ties of the rounding, binade crossings,
zeros, subnormals, negative values, infinities and NaN.  The _warp variant's
sum has no fixed order: each of its at most n partial roundings is within
2^-24 of the running sum of magnitudes, so it is within n * 2^-24 of the sum
of magnitudes (and far closer here).
"""
import ctypes as C

import numpy as np
import pytest

from belewitte_amd import _native as N
from belewitte_amd import device, pagerank

pytestmark = pytest.mark.gpu

# Around the long-row split (128), a wave's round (512), a workgroup's
# (2048), the workgroup split (8192), and long ones.
LENGTHS = (0, 1, 127, 128, 129, 300, 511, 512, 513, 1023, 2048, 8191, 8192, 8193, 10239, 10240, 10241, 20011)


def _values(kind, n, rng):
    if kind == "ranks":
        return (rng.pareto(1.2, n) * 1e-9 + 1e-9).astype(np.float32)
    if kind == "ties":  # small integers and halves of them: exact ties once the sum passes 2^24
        x = rng.integers(1, 4, n).astype(np.float32) * np.float32(0.5)
        x[:64] = 2.0 ** 18
        return x
    if kind == "wide":
        return np.ldexp(rng.random(n) + 0.5, rng.integers(-60, 60, n)).astype(np.float32)
    if kind == "rising":
        return np.ldexp(np.ones(n), np.linspace(-140, 110, n).astype(int)).astype(np.float32)
    if kind == "zeros":
        x = np.zeros(n, np.float32)
        x[n // 2:] = rng.random(n - n // 2).astype(np.float32)
        return x
    if kind == "subnormal":
        return (rng.integers(0, 1000, n).astype(np.uint32)).view(np.float32)
    if kind == "signed":
        return rng.standard_normal(n).astype(np.float32)
    x = rng.random(n).astype(np.float32)
    x[3 * n // 4] = np.inf if kind == "inf" else np.nan
    return x


@pytest.mark.parametrize("kind", ["ranks", "ties", "wide", "rising", "zeros", "subnormal", "signed", "inf", "nan"])
@pytest.mark.parametrize("offset_bytes", [4, 8])
def test_long_row_sums(gpu, kind, offset_bytes):
    rng = np.random.default_rng(11)
    pr = _values(kind, 4096, rng)
    V = pr.size
    rows = [rng.integers(0, V, n).astype(np.uint32) for n in LENGTHS]
    cols = np.concatenate(rows)
    deg = np.zeros(V, np.int64)
    deg[:len(rows)] = [r.size for r in rows]
    off = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint32 if offset_bytes == 4 else np.uint64)
    lib = N.hip_lib()
    d_off, d_cols, d_pr = (device.DeviceArray.from_host(x) for x in (off, cols, pr))
    out = device.DeviceArray(V, np.float32)
    plan = C.c_void_p()
    N.check_hip(lib.bw_pr_pull_plan_create(C.byref(plan), V, d_off.ptr, offset_bytes, None))
    try:
        for variant in ("vertex-pull-nodiv", "vertex-pull-warp-nodiv"):
            out.fill_u32(0)
            cfg = N.launch(warp=32, chunk=32)
            N.check_hip(lib.bw_pr_pull_iteration(plan, pagerank.variant_id(variant), d_cols.ptr, None, d_pr.ptr,
                                                 out.ptr, C.byref(cfg)))
            device.synchronize()
            got = out.download()[:len(rows)]
            for r, g in zip(rows, got):
                x = pr[r]
                with np.errstate(all="ignore"):
                    want = np.cumsum(x, dtype=np.float32)[-1] if r.size else np.float32(0)
                    mag = np.abs(x.astype(np.float64)).sum()
                if variant == "vertex-pull-nodiv":
                    same = np.isnan(g) and np.isnan(want) or g.view(np.uint32) == want.view(np.uint32)
                    assert same, (kind, r.size, g, want)
                elif np.isfinite(mag) and mag < 3e38:
                    exact = x.astype(np.float64).sum()
                    assert abs(float(g) - exact) <= (r.size + 1) * 2.0 ** -24 * mag + 1e-44, (kind, r.size, g, exact)
    finally:
        lib.bw_pr_pull_plan_destroy(plan)
        for a in (d_off, d_cols, d_pr, out):
            a.free()
