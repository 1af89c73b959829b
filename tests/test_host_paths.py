"""Host code of the native library without a GPU: what it allocates and
launches, and what it does when an allocation fails.  Each test runs in a
process of its own on a stand-in for the HIP runtime (native/fake_hip.cpp)
whose device memory is host memory and whose kernels do nothing."""
import subprocess
import sys
import textwrap
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

PRELUDE = f"""
import ctypes as C, sys
sys.path.insert(0, {str(ROOT)!r})
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
fake.fake_calls.restype = C.c_char_p
fake.fake_live.restype = C.c_int64
fake.fake_fail_from.argtypes = [C.c_uint64]
import numpy as np
from belewitte_amd import _native as N
from belewitte_amd import bfs, device, graph, pagerank
lib = N.hip_lib()

def calls(kind):
    return [l.split()[1:] for l in fake.fake_calls().decode().splitlines() if l.startswith(kind + " ")]
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    out = tmp_path_factory.mktemp("fake") / "libfake_hip.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", str(ROOT / "tests/native/fake_hip.cpp"), "-o",
                    str(out)], check=True)
    return out


def _run(fake, code):
    r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(code), str(fake)], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_pull_run_without_edges_or_iterations(fake):
    """A pull variant of a graph without edges: the initial ranks when no
    iteration is asked for (no column is read then), refused otherwise."""
    _run(fake, """
        off = device.DeviceArray.from_host(np.zeros(6, np.uint32))
        g = N.BwGraphDev()
        g.vertex_count, g.edge_count, g.offset_bytes = 5, 0, 4
        g.offsets = g.rev_offsets = off.ptr
        ranks = device.DeviceArray(5, np.float32)
        for variant in ("vertex-pull", "vertex-pull-nodiv", "vertex-pull-warp", "vertex-pull-warp-nodiv"):
            run = lambda n: lib.bw_pr_run(C.byref(g), pagerank.variant_id(variant), n, 0, ranks.ptr, None, None)
            assert run(0) == 0, lib.bw_hip_last_error()
            assert run(1) == 1 and b"NULL device pointer" in lib.bw_hip_last_error()
    """)
