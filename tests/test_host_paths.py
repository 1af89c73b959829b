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


PLAN = """
def binned(V, E):
    # the host's plan: nothing runs on the device
    rng = np.random.default_rng(V)
    rows = np.sort(rng.integers(0, V, E))
    off = np.searchsorted(rows, np.arange(V + 1)).astype(np.uint32)
    g = N.BwGraphDev()
    g.vertex_count, g.edge_count, g.offset_bytes = V, E, 4
    keep = [device.DeviceArray.from_host(x) for x in (off, rng.integers(0, V, E).astype(np.uint32))]
    g.rev_offsets, g.rev_cols = keep[0].ptr, keep[1].ptr
    plan = C.c_void_p()
    N.check_hip(lib.bw_pr_plan_create(C.byref(plan), V, E, g.rev_offsets, 4, g.rev_cols))
    return g, plan, keep

def run(g, plan, iterations=2):
    V = g.vertex_count
    bufs = [device.DeviceArray(V, np.float32), device.DeviceArray(V, np.float32),
            device.DeviceArray(int(lib.bw_pr_fused_acc_len(iterations)), np.float64)]
    fake.fake_clear()
    return lib.bw_pr_fused_run(C.byref(g), plan, iterations, 0, 0, *(b.ptr for b in bufs), None, None, None)
"""


def test_binned_plan_without_room_for_pieces(fake):
    """The pieces of a small graph's chunks need a buffer; without it the
    plan keeps whole chunks."""
    _run(fake, PLAN + """
grids = []
for limit in (2**64 - 1, 3 << 20):
    g, plan, keep = binned(20000, 300000)
    fake.fake_fail_from(limit)
    assert lib.bw_pr_plan_bin_host(plan, 14, 128, 8) == 0, lib.bw_hip_last_error()
    fake.fake_fail_from(2**64 - 1)
    assert run(g, plan) == 0, lib.bw_hip_last_error()
    grids.append({c[2] for c in calls("launch") if "accumulate" in c[0]})
    lib.bw_pr_plan_destroy(plan)
assert [len(x) for x in grids] == [1, 1]
whole = int(grids[1].pop()) - 1  # and one workgroup for the reduction
assert whole < 8 and int(grids[0].pop()) - 1 == 16 * whole, whole
    """)


def test_small_run_lds_limit(fake):
    """The LDS limit of a small graph's kernel is an attribute that all
    threads share: whatever the graph's size it is set to one value, which
    no launch exceeds."""
    _run(fake, PLAN + """
limits, needs = set(), set()
for V in (5400, 6000, 8192):
    g, plan, keep = binned(V, 30000)
    assert run(g, plan) == 0, lib.bw_hip_last_error()
    limits |= {(name, int(value)) for name, value in calls("attribute")}
    needs |= {(c[0], int(c[6])) for c in calls("launch") if "pr_small_kernel" in c[0]}
assert len(needs) == 3 and len(limits) == 1, (needs, limits)
name, limit = limits.pop()
assert all(n == name and lds <= limit for n, lds in needs), (needs, name, limit)
    """)


def test_engine_memory_follows_the_graph(fake):
    """An engine on a graph of a few thousand vertices holds what such a
    graph needs, and gives it back."""
    _run(fake, """
        g = N.BwGraphDev()
        g.vertex_count, g.edge_count, g.offset_bytes = 2000, 0, 4
        off = device.DeviceArray.from_host(np.zeros(2001, np.uint32))
        g.offsets = g.rev_offsets = off.ptr
        before = fake.fake_live()
        fake.fake_clear()
        e = C.c_void_p()
        N.check_hip(lib.bw_bfs_engine_create(C.byref(e), C.byref(g), None, 2001))
        held = sum(int(c[0]) for c in calls("alloc"))
        lib.bw_bfs_engine_destroy(e)
        assert held < 2 << 20, held
        assert fake.fake_live() == before
    """)


def test_short_chunks_stay_whole(fake):
    """More than 64 chunks are cut in two only if the longest one has more
    than 81920 edges."""
    _run(fake, PLAN + """
for chunk_tasks, V, E in ((16, 20000, 2400000), (64, 200000, 9000000)):
    g, plan, keep = binned(V, E)
    N.check_hip(lib.bw_pr_plan_bin_host(plan, 13, chunk_tasks, 8))
    chunks = C.c_uint32()
    N.check_hip(lib.bw_pr_plan_bin_info(plan, None, C.byref(chunks), None))
    assert 64 < chunks.value <= 128, chunks.value
    N.check_hip(run(g, plan))
    (grid,) = {int(c[2]) for c in calls("launch") if "accumulate" in c[0]}
    assert grid - 1 == chunks.value * (1 if chunk_tasks == 16 else 2), (chunk_tasks, grid, chunks.value)
    lib.bw_pr_plan_destroy(plan)
    """)


def test_contributions_only_where_gathered(fake):
    """bw_pr_run holds per-vertex contributions (the only array of 4 bytes a
    vertex besides degrees and sums) for the variants that gather them."""
    _run(fake, """
        V, E = (1 << 20) + 1, 1000  # past the gathered scatter layout
        dg = device.DeviceGraph(graph.from_edges(V, np.arange(E, dtype=np.uint32), np.arange(1, E + 1, dtype=np.uint32)))
        for name in pagerank.VARIANTS:
            dg.ensure(pagerank.REPRESENTATION[pagerank.variant_id(name)])
            ranks = device.DeviceArray(V, np.float32)
            fake.fake_clear()
            cfg = N.launch(warp=32, chunk=32)
            N.check_hip(lib.bw_pr_run(dg.ref, pagerank.variant_id(name), 2, 1, ranks.ptr, None, C.byref(cfg)))
            held = sum(int(c[0]) == 4 * V for c in calls("alloc"))
            assert held == 2 + (name.startswith("rev-") or "pull" in name), (name, held)
    """)


def test_kernel_names_are_launched(fake):
    """kernel_names() names what an iteration launches: the small-graph
    kernel, the pull kernels, the binned ones with whole and with cut chunks.
    Nothing is timed against itself for a small graph."""
    _run(fake, r"""
        import re, subprocess
        def launched():
            names = "\n".join(c[0] for c in calls("launch"))
            plain = subprocess.run(["c++filt"], input=names, capture_output=True, text=True, check=True).stdout
            plain = re.sub(r"(\d)u\b", r"\1", re.sub(r"\(anonymous namespace\)::", "", plain))
            return set(re.findall(r"bw::(\w+(?:<[^<>(]*>)?)\(", plain))
        rng = np.random.default_rng(3)
        for V, E in ((5000, 6000), (5000, 14000), (8192, 30000), (8193, 9000), (40000, 300000)):
            g = graph.from_edges(V, rng.integers(0, V, E).astype(np.uint32), rng.integers(0, V, E).astype(np.uint32))
            f = pagerank.FusedPageRank(device.DeviceGraph(g), 3)
            for shape in (None, (13, 64, 8), (14, 3, 16)):
                if shape:
                    f.bin(*shape, on_host=True)
                else:
                    f.tune(8192, 0, 2)
                fake.fake_clear()
                f.run(3)
                names = set(f.kernel_names().split(" + "))
                # one-off launches beside an iteration's
                assert names <= launched() <= names | {"pr_fused_init_kernel", "pr_reduce_kernel"}, (names, launched())
            if V <= 8192:
                fake.fake_clear()
                table = f.autotune(3)
                assert f.binning == (14, 3, 16) and list(table) == ["small"] and len(calls("launch")) == 4
    """)


def test_run_refuses_what_its_kernels_would(fake):
    """bw_pr_run refuses a block size that its passes over the vertices do not
    take, whichever variant runs (when iterations do), and asks nothing of the
    offsets of a push variant that does not iterate."""
    _run(fake, """
        dg = device.DeviceGraph(graph.rmat_n(300, 2000, seed=1))
        ranks = device.DeviceArray(dg.vertex_count, np.float32)
        def run(variant, iterations, mode=0, **launch):
            cfg = N.launch(warp=32, chunk=32, **launch)
            return lib.bw_pr_run(dg.ref, variant, iterations, mode, ranks.ptr, None, C.byref(cfg))
        for name in pagerank.VARIANTS:
            v = pagerank.variant_id(name)
            dg.ensure(pagerank.REPRESENTATION[v])
            for mode in (0, 1):
                assert run(v, 2, mode) == run(v, 2, mode, block=1024) == 0, lib.bw_hip_last_error()
                for block in (100, 2048):
                    assert run(v, 2, mode, block=block) == 1 and b"block size" in lib.bw_hip_last_error(), (name, block)
        dg.desc.offset_bytes = 5
        for name in ("vertex-push", "vertex-push-warp"):
            v = pagerank.variant_id(name)
            assert run(v, 0) == 0 and run(v, 1) == 1 and run(v, 0, 1) == 1
    """)
