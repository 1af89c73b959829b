"""The workloads this framework's speed is judged by.

Each case is one call (or the short sequence of calls) a program makes once
it holds a graph: a PageRank run of the fused iteration or of one of the
reference's variants, a BFS by the reference's level loop, by the
device-driven engine or from many sources at once, and the preparation of a
new graph on the device up to its first ranks.  Graphs are the synthetic
families of the benchmark (R-MAT, Erdos-Renyi, rewired grids), made from the
seed; sizes run from graphs where the launches count to the benchmark's
scale-22 R-MAT graph, with sizes that are no power of two among them.

Large results stay on the device (a program that goes on with them there),
as the benchmark's own timed calls leave them; the reference-shaped calls
return host arrays, as they always do.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from belewitte_amd import _native as N
from belewitte_amd import bfs, bfs_native, device, graph, pagerank, switch

DAMP = float(np.float32(0.85))
MAX_LEVELS = 4096  # levels of any case's search, and more


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # PageRank of a small graph, as run once per community, snapshot or
        # query: launches and latency are all of it.
        {"name": "fused-small", "kind": "fused", "graph": "rmat", "n": 1000, "ef": 8, "undirected": False,
         "layout": "bins", "reorder": True, "mode": "uniform", "iterations": 30},
        # An ordinary social graph, undirected, no power of two; the
        # reference's own recurrence (dangling mass dropped).
        {"name": "fused-medium", "kind": "fused", "graph": "rmat", "n": 150001, "ef": 16, "undirected": True,
         "layout": "bins", "reorder": True, "mode": "drop", "iterations": 30},
        # The benchmark's graph: R-MAT scale 22, edge factor 16, 30 iterations.
        {"name": "fused-large", "kind": "fused", "graph": "rmat", "n": 1 << 22, "ef": 16, "undirected": False,
         "layout": "bins", "reorder": True, "mode": "uniform", "iterations": 30},
        # The pull form of the fused iteration in the graph's own vertex order
        # (what a program gets that asks for neither relabelling nor bins).
        {"name": "fused-pull", "kind": "fused", "graph": "rmat", "n": 600011, "ef": 12, "undirected": False,
         "layout": "pull", "reorder": False, "mode": "uniform", "iterations": 30},
        # Two of the reference's ten variants, whole calls as a kernel study
        # makes them: a pull form and a push form.
        {"name": "variant-pull", "kind": "variant", "graph": "rmat", "n": 1 << 20, "ef": 16, "undirected": False,
         "variant": "vertex-pull", "mode": "drop", "iterations": 30},
        {"name": "variant-push", "kind": "variant", "graph": "rmat", "n": 200003, "ef": 16, "undirected": False,
         "variant": "vertex-push", "mode": "uniform", "iterations": 100},
        # The reference's BFS level loop: its benchmark workload (vertex-push,
        # R-MAT scale 16, 64-bit offsets) and an edge-list form on a larger graph.
        {"name": "levels-push", "kind": "levels", "graph": "rmat", "n": 1 << 16, "ef": 16, "undirected": False,
         "implementation": "vertex-push", "offset_bytes": 8},
        {"name": "levels-edges", "kind": "levels", "graph": "rmat", "n": 500009, "ef": 16, "undirected": True,
         "implementation": "edge-list-blockreduce", "offset_bytes": 4},
        # The BFS engine with its shipped model: few wide levels on an R-MAT
        # graph, many narrow ones on a rewired grid.
        {"name": "engine-rmat", "kind": "engine", "graph": "rmat", "n": 1 << 21, "ef": 16, "undirected": True,
         "policy": "learned"},
        {"name": "engine-grid", "kind": "engine", "graph": "grid", "n": 1 << 20, "ef": 2, "undirected": True,
         "policy": "learned"},
        # 64 searches sharing every pass over one graph.
        {"name": "multi-source", "kind": "msbfs", "graph": "rmat", "n": 1 << 19, "ef": 16, "undirected": True,
         "sources": 64},
        # A graph as it arrives on the device, relabelled, planned and ranked.
        {"name": "first-ranks", "kind": "first", "graph": "rmat", "n": 1 << 20, "ef": 16, "undirected": False,
         "mode": "uniform", "iterations": 30},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("fused", "fused", "variant", "levels", "engine", "engine", "msbfs", "first"))
    undirected = rng.random() < 0.5
    ef = rng.randint(4, 20)
    if kind == "fused":
        n = _log_uniform(rng, 1000, (1 << 25) // ef)
        return {"kind": kind, "graph": rng.choice(("rmat", "rmat", "er")), "n": n, "ef": max(2, ef // (1 + undirected)),
                "undirected": undirected, "layout": rng.choice(("bins", "bins", "pull")),
                "reorder": rng.random() < 0.7, "mode": rng.choice(("uniform", "drop")),
                "iterations": rng.randint(10, 40)}
    if kind == "variant":
        variant = rng.choice(("edge-list", "rev-edge-list", "struct-edge-list", "rev-struct-edge-list", "vertex-push",
                              "vertex-pull", "vertex-push-warp", "vertex-pull-warp"))
        return {"kind": kind, "graph": "rmat", "n": _log_uniform(rng, 1000, 600000), "ef": ef, "undirected": False,
                "variant": variant, "mode": rng.choice(("uniform", "drop")), "iterations": rng.randint(10, 100)}
    if kind == "levels":
        return {"kind": kind, "graph": rng.choice(("rmat", "er")), "n": _log_uniform(rng, 1000, 500000), "ef": ef,
                "undirected": undirected, "implementation": rng.choice(sorted(bfs.IMPLEMENTATIONS)),
                "offset_bytes": rng.choice((4, 8))}
    if kind == "engine":
        family = rng.choice(("rmat", "er", "grid"))
        return {"kind": kind, "graph": family, "n": _log_uniform(rng, 2000, 1500000), "ef": ef,
                "undirected": family != "rmat" or undirected, "policy": rng.choice(("learned", "beamer"))}
    if kind == "msbfs":
        return {"kind": kind, "graph": "rmat", "n": _log_uniform(rng, 1000, 400000), "ef": ef,
                "undirected": undirected, "sources": rng.randint(2, 64)}
    return {"kind": kind, "graph": "rmat", "n": _log_uniform(rng, 1000, 900000), "ef": ef, "undirected": False,
            "mode": rng.choice(("uniform", "drop")), "iterations": rng.randint(10, 40)}


# --------------------------------------------------------------------- inputs

def _grid_shape(n):
    h = max(2, int(math.sqrt(n)))
    return max(2, n // h), h


def _graph(case, seed):
    n, ef, und = case["n"], case["ef"], case["undirected"]
    s = 1 + int(seed) % 1000003
    if case["graph"] == "grid":
        w, h = _grid_shape(n)
        return graph.grid2d(w, h, rewire=0.01, seed=s)
    if case["graph"] == "er":
        return graph.erdos_renyi(n, n * ef, seed=s, undirected=und)
    if n & (n - 1) == 0:
        return graph.rmat(n.bit_length() - 1, ef, seed=s, undirected=und)
    return graph.rmat_n(n, n * ef, seed=s, undirected=und)


class _View:
    """A device buffer of the framework as torch sees it."""

    def __init__(self, ptr, count, typestr):
        address = ptr.value if hasattr(ptr, "value") else int(ptr)
        self.__cuda_array_interface__ = {"shape": (int(count),), "typestr": typestr, "data": (int(address), False),
                                         "version": 2}


def _tensor(owner, ptr, count, typestr):
    t = torch.as_tensor(_View(ptr, count, typestr), device="cuda")
    t.owner = owner  # frees the buffer when it goes: it stays as long as the tensor
    return t


def _padded(x, length):
    """x with zeros up to a length that does not depend on the graph."""
    if isinstance(x, np.ndarray):
        out = np.zeros(length, dtype=x.dtype)
    else:
        out = torch.zeros(length, dtype=x.dtype, device=x.device)
    out[:x.shape[0]] = x
    return out


def _stored_ef(case):
    if case["graph"] == "grid":
        return 4
    return case["ef"] * (2 if case["undirected"] else 1)


def prepare(case, seed):
    g = _graph(case, seed)
    kind = case["kind"]
    s = {"case": case, "kind": kind, "V": g.vertex_count}
    if kind == "fused":
        f = pagerank.FusedPageRank.for_graph(g, max_iterations=case["iterations"], reorder=case["reorder"])
        if case["layout"] == "bins":
            f.bin()
        s["fused"] = f
        s["ranks"] = _tensor(f, f.ranks.ptr, g.vertex_count, "<f4")
    elif kind == "variant":
        dg = device.DeviceGraph(g)
        dg.ensure(pagerank.REPRESENTATION[pagerank.variant_id(case["variant"])])
        s["dg"] = dg
    elif kind == "levels":
        k, _ = bfs.parse(case["implementation"])
        s["dg"] = device.DeviceGraph(g, offset_bytes=case["offset_bytes"], reps=(bfs.REPRESENTATION[k],))
        s["root"] = g.max_out_degree_vertex()
    elif kind == "engine":
        s["dg"] = device.DeviceGraph(g)
        eng = bfs_native.BFSEngine(s["dg"])
        eng.set_model(switch.Model.load(switch.MODEL_PATH).w)
        p = C.c_void_p()
        N.check_hip(N.hip_lib().bw_bfs_engine_levels(eng._e, C.byref(p)))
        s["engine"], s["depths"] = eng, _tensor(eng, p, g.vertex_count, "<i4")
        s["root"] = graph.random_sources(g, 1, int(seed))[0]
    elif kind == "msbfs":
        s["dg"] = device.DeviceGraph(g)
        s["ms"] = bfs_native.MultiSourceBFS(s["dg"])
        s["sources"] = np.array(graph.random_sources(g, case["sources"], int(seed)), dtype=np.uint32)
    else:
        s["dg"] = device.DeviceGraph(g)
    for v in s.values():
        if isinstance(v, device.DeviceGraph):
            v.host = None  # the device copy is all the calls need
    g.close()
    return s


# ----------------------------------------------------------------------- runs

def run(s):
    case, kind = s["case"], s["kind"]
    if kind == "fused":
        _, resid, _ = s["fused"].run(case["iterations"], case["mode"], download=False)
        return {"ranks": s["ranks"], "residuals": resid}
    if kind == "variant":
        ranks, resid = pagerank.run(s["dg"], case["variant"], case["iterations"], case["mode"])
        return {"ranks": ranks, "residuals": resid}
    if kind == "levels":
        r = bfs.run(s["dg"], s["root"], case["implementation"])
        return {"depths": r.levels, "counts": _padded(r.counts, MAX_LEVELS)}
    if kind == "engine":
        r = s["engine"].run(s["root"], case["policy"], download=False)
        return {"depths": s["depths"], "counts": _padded(r.counts, MAX_LEVELS)}
    if kind == "msbfs":
        _, _, bits = s["ms"].run(s["sources"], download=False)
        if "depths" not in s:  # the handle's depth buffer, made by its first run
            s["depths"] = _tensor(s["ms"], s["ms"]._depths.ptr, s["sources"].size * s["V"], "<i4")
        return {"depths": s["depths"], "bits": _padded(bits.view(np.int64), MAX_LEVELS)}
    dg, perm = s["dg"].relabel_by_degree()
    f = pagerank.FusedPageRank(dg, max_iterations=case["iterations"])
    f.bin()
    _, resid, _ = f.run(case["iterations"], case["mode"], download=False)
    V, E = dg.vertex_count, dg.edge_count
    return {"perm": perm.view(np.int32), "offsets": _tensor(dg, dg.array("roff").ptr, V + 1, "<i4"),
            "cols": _padded(_tensor(dg, dg.array("rcol").ptr, E, "<i4"), case["n"] * case["ef"]),
            "ranks": _tensor(f, f.ranks.ptr, V, "<f4"), "residuals": resid}


def work(case):
    V = case["n"]
    E = V * _stored_ef(case)
    kind = case["kind"]
    if kind in ("fused", "variant", "first"):
        # per iteration: offsets, columns, degrees, ranks read and written
        it = case["iterations"]
        extra = 4 * (4 * E + 4 * V) if kind == "first" else 0  # both directions read and written once
        return {"bytes": it * (4 * E + 16 * V) + extra, "flops": it * (E + 4 * V)}
    if kind == "msbfs":
        # the graph once, and every search's depths
        return {"bytes": 4 * E + 4 * V + 4 * V * case["sources"], "flops": 0}
    return {"bytes": 4 * E + 8 * V, "flops": 0}


def tolerance(case):
    # The fused iteration keeps its sums beyond 32 bits: 4e-8 off the
    # recurrence in 64 bits, the rounding of the ranks themselves.  The
    # variants hold the reference's FP32 sums in its order or in none:
    # 2e-6 off it on the largest graph.
    if case["kind"] in ("fused", "first"):
        return {"rel": 3e-7, "max": 1e-5}
    if case["kind"] == "variant":
        return {"rel": 1e-5, "max": 1e-4}
    return "exact"


# ---------------------------------------------------------------------- exact

def _exact_ranks(case, seed, relabelled):
    g = _graph(case, seed)
    V, it, uniform = g.vertex_count, case["iterations"], case["mode"] == "uniform"
    deg = torch.from_numpy(np.diff(g.offsets()).astype(np.int64)).cuda()
    roff = torch.from_numpy(g.offsets(True).astype(np.int64)).cuda()
    cols = torch.from_numpy(g.cols(True).astype(np.int64)).cuda()
    g.close()
    r = torch.full((V,), 1.0 / V, dtype=torch.float64, device="cuda")
    residuals = []
    for _ in range(it):
        c = torch.where(deg > 0, r / deg.clamp(min=1), torch.zeros_like(r))
        sums = torch.segment_reduce(c[cols], "sum", offsets=roff) if cols.numel() else torch.zeros_like(r)
        if uniform:
            sums = sums + r[deg == 0].sum() / V
        new = (1.0 - DAMP) / V + DAMP * sums
        residuals.append(float((new - r).abs().sum()))
        r = new
    if relabelled:
        order = torch.sort(deg, descending=True, stable=True).indices
        r = r[order]
    return {"ranks": r, "residuals": np.array(residuals, dtype=np.float64)}


def exact(case, seed):
    """Ranks and residuals of the recurrence in 64 bits; the other outputs
    are whole numbers."""
    if case["kind"] == "fused":
        return _exact_ranks(case, seed, case["reorder"])
    if case["kind"] == "variant":
        return _exact_ranks(case, seed, False)
    if case["kind"] == "first":
        return {**_exact_ranks(case, seed, True), "perm": None, "offsets": None, "cols": None}
    return None
