// BFS level kernels for gfx950 and their C ABI entry points.
//
// Each kernel family restates the semantics of one reference kernel
// (bfs/*.cu of merijn/Belewitte) -- same depth encoding (int32, INT_MAX =
// unvisited), same frontier count (newly discovered vertices) -- with a
// wave64 mapping: 16-byte vector loads on the edge streams, an atomic only
// when a plain load shows the neighbour still unvisited, wave64 ballots in
// place of __any_sync, and the four frontier reductions of bfs/bfs.hpp over
// 64-lane waves.

#include "common.hpp"

#include <algorithm>
#include <mutex>
#include <vector>

namespace bw {
namespace {

// A level launched by the level loop before the host knows whether the
// search goes on: it stamps its start time and returns at once when the
// level before it found nothing.  Both NULL: a launch of its own.
struct RunLevel {
    const uint32_t *prev = nullptr;  // frontier count the level starts from
    uint64_t *stamp = nullptr;

    __device__ __forceinline__ bool skip() const
    {
        if (stamp && blockIdx.x == 0 && threadIdx.x == 0) *stamp = wall_clock64();
        return prev && *prev == 0;
    }
};

// ------------------------------------------------------------ edge lists

// One edge (in, out): forward tests levels[in] and relaxes out; reverse
// (REV) tests levels[out] and relaxes in (bfs/rev_edgelist.cu:14-18).
template<int R, bool REV>
__device__ __forceinline__ void visit_edge(uint32_t in, uint32_t out, int32_t *levels,
                                           int32_t depth, FrontierCount<R> &fc)
{
    const uint32_t test = REV ? out : in;
    const uint32_t relax = REV ? in : out;
    if (levels[test] == depth && relax_depth(levels, relax, depth + 1)) fc.update();
}

// SoA EdgeList, 4 edges per thread step through uint4 loads of in[]/out[]
// (the arrays come from hipMalloc or bw_build_edge_lists and are 16-byte
// aligned; the host falls back to the scalar tail kernel otherwise).
template<int R, bool REV>
__global__ __launch_bounds__(1024) void bfs_edge_list_kernel(
    uint64_t E, const uint32_t *__restrict__ in, const uint32_t *__restrict__ out,
    int32_t *levels, int32_t depth, uint32_t *frontier, int vec, RunLevel run)
{
    if (run.skip()) return;
    FrontierCount<R> fc;
    const uint64_t stride = static_cast<uint64_t>(blockDim.x) * gridDim.x;
    const uint64_t gid = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    uint64_t done = 0;
    if (vec) {
        const uint64_t E4 = E / 4;
        const uint4 *in4 = reinterpret_cast<const uint4 *>(in);
        const uint4 *out4 = reinterpret_cast<const uint4 *>(out);
        for (uint64_t i = gid; i < E4; i += stride) {
            const uint4 a = in4[i], b = out4[i];
            visit_edge<R, REV>(a.x, b.x, levels, depth, fc);
            visit_edge<R, REV>(a.y, b.y, levels, depth, fc);
            visit_edge<R, REV>(a.z, b.z, levels, depth, fc);
            visit_edge<R, REV>(a.w, b.w, levels, depth, fc);
        }
        done = E4 * 4;
    }
    for (uint64_t i = done + gid; i < E; i += stride)
        visit_edge<R, REV>(in[i], out[i], levels, depth, fc);
    fc.finalise(frontier);
}

// AoS StructEdgeList: (in, out) pairs, two edges per uint4.
template<int R, bool REV>
__global__ __launch_bounds__(1024) void bfs_struct_edge_list_kernel(
    uint64_t E, const uint32_t *__restrict__ edges, int32_t *levels, int32_t depth,
    uint32_t *frontier, int vec, RunLevel run)
{
    if (run.skip()) return;
    FrontierCount<R> fc;
    const uint64_t stride = static_cast<uint64_t>(blockDim.x) * gridDim.x;
    const uint64_t gid = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    uint64_t done = 0;
    if (vec) {
        const uint64_t E2 = E / 2;
        const uint4 *e4 = reinterpret_cast<const uint4 *>(edges);
        for (uint64_t i = gid; i < E2; i += stride) {
            const uint4 p = e4[i];
            visit_edge<R, REV>(p.x, p.y, levels, depth, fc);
            visit_edge<R, REV>(p.z, p.w, levels, depth, fc);
        }
        done = E2 * 2;
    }
    for (uint64_t i = done + gid; i < E; i += stride)
        visit_edge<R, REV>(edges[2 * i], edges[2 * i + 1], levels, depth, fc);
    fc.finalise(frontier);
}

// ---------------------------------------------------------- vertex forms

// In-degree above which a vertex's edges are taken by its whole wave instead
// of its own thread.
constexpr uint64_t kWaveDegree = 64;
constexpr int kPushBatch = 8;                 // edges per thread in flight in the push kernel
constexpr uint32_t kNoVertex = 0xFFFFFFFFu;   // an empty slot of such a batch

// The 64-bit offset of lane `l` broadcast to the wave.
__device__ __forceinline__ uint64_t read_lane_u64(uint64_t x, int l)
{
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(x), l);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(x >> 32), l);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

// The vertex that thread t of workgroup `block` (of n, kVertexRun vertices
// in a run) takes: runs of four consecutive vertices from all over the graph,
// so that the hubs of a graph whose degrees follow the bits of the vertex id
// (R-MAT in its generated order: 256 consecutive vertices hold a ninth of the
// edges of scale 16) end up in different workgroups.  A bijection onto
// [0, n * blockDim): run i of the workgroup is run i * n + (block + i * step) % n.
constexpr uint32_t kVertexRun = 4;

__device__ __forceinline__ uint64_t spread_vertex(uint32_t block, uint32_t n, uint32_t t)
{
    const uint32_t i = t / kVertexRun;
    const uint32_t step = static_cast<uint32_t>(n * 0.618f) | 1u;
    const uint32_t at = static_cast<uint32_t>((block + static_cast<uint64_t>(i) * step) % n);
    return (static_cast<uint64_t>(i) * n + at) * kVertexRun + t % kVertexRun;
}

// bfs/vertex_push.cu: a thread per vertex finds the depth-d vertices; their
// out-edges are then expanded by the whole workgroup, blockDim x kPushBatch
// edges per step, whoever found the vertex (a prefix sum of the degrees in
// LDS gives each edge its vertex).  So neither a hub nor a workgroup's many
// hubs hold one thread or wave up (64 consecutive hubs in one wave took 406
// of the 540 us of a whole search at R-MAT scale 16; that level takes 69 us
// now).  Every out-edge of every frontier vertex is relaxed once, as in the reference, so
// depths and counts are the same: a vertex is counted by the atomic that
// lowers it, whatever the order.
template<int R, typename Off>
__global__ __launch_bounds__(1024) void bfs_vertex_push_kernel(
    uint64_t V, const Off *__restrict__ off, const uint32_t *__restrict__ cols,
    int32_t *levels, int32_t depth, uint32_t *frontier, RunLevel run)
{
    if (run.skip()) return;
    FrontierCount<R> fc;
    __shared__ Off first[1024], before[1024];  // per active vertex: its first edge, the edges of those before it
    __shared__ Off wedges[1024 / kWave];
    __shared__ uint32_t wactive[1024 / kWave];
    const int32_t nd = depth + 1;
    const uint32_t t = threadIdx.x, lane = t & (kWave - 1), wv = t / kWave, nw = blockDim.x / kWave;
    const uint64_t blocks = (V + blockDim.x - 1) / blockDim.x;
    const uint32_t n = static_cast<uint32_t>(blocks);
    for (uint32_t block = blockIdx.x; block < n; block += gridDim.x) {
        const uint64_t v = spread_vertex(block, n, t);
        Off s = 0, deg = 0;
        if (v < V && levels[v] == depth) {
            s = off[v];
            deg = off[v + 1] - s;
        }
        const uint64_t act = __ballot(deg != 0);
        const Off incl = wave_prefix_sum(deg);
        if (lane == kWave - 1) {
            wedges[wv] = incl;
            wactive[wv] = static_cast<uint32_t>(__popcll(act));
        }
        __syncthreads();
        Off e0 = incl - deg, total = 0;
        uint32_t at = static_cast<uint32_t>(__popcll(act & ((1ull << lane) - 1ull))), na = 0;
        for (uint32_t w = 0; w < nw; w++) {
            if (w < wv) {
                e0 += wedges[w];
                at += wactive[w];
            }
            total += wedges[w];
            na += wactive[w];
        }
        if (deg != 0) {
            first[at] = s;
            before[at] = e0;
        }
        __syncthreads();
        // 64 bits: the step past a total near 2^32 must not wrap.
        for (uint64_t c = 0; c < total; c += blockDim.x * kPushBatch) {
            uint32_t w[kPushBatch];
#pragma unroll
            for (int u = 0; u < kPushBatch; u++) {
                const uint64_t k = c + u * blockDim.x + t;
                w[u] = kNoVertex;
                if (k < total) {
                    uint32_t lo = 0, hi = na;  // the last active vertex with before <= k
                    while (hi - lo > 1) {
                        const uint32_t mid = (lo + hi) / 2;
                        if (before[mid] <= k) lo = mid;
                        else hi = mid;
                    }
                    w[u] = cols[first[lo] + static_cast<Off>(k - before[lo])];
                }
            }
#pragma unroll
            for (int u = 0; u < kPushBatch; u++)
                if (w[u] != kNoVertex && relax_depth(levels, w[u], nd)) fc.update();
        }
        __syncthreads();  // the lists are rebuilt by the next block
    }
    fc.finalise(frontier);
}

// bfs/vertex_pull.cu: a thread per unvisited vertex scans its in-edges
// and the first in-neighbour at depth d sets it to d+1 (a plain store:
// only this vertex's thread or wave writes levels[v]).  A vertex with more
// than kWaveDegree in-edges is probed by the whole wave, 64 in-edges per
// step, stopping at the first step where any lane finds one (a ballot);
// which in-neighbour is found does not change the depth or the count.
template<int R, typename Off>
__global__ __launch_bounds__(1024) void bfs_vertex_pull_kernel(
    uint64_t V, const Off *__restrict__ roff, const uint32_t *__restrict__ rcols,
    int32_t *levels, int32_t depth, uint32_t *frontier, RunLevel run)
{
    if (run.skip()) return;
    FrontierCount<R> fc;
    const int32_t nd = depth + 1;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint64_t stride = static_cast<uint64_t>(blockDim.x) * gridDim.x;
    const uint64_t waveFirst = static_cast<uint64_t>(spread_block(blockIdx.x, gridDim.x)) * blockDim.x + threadIdx.x - lane;
    for (uint64_t base = waveFirst; base < V; base += stride) {
        const uint64_t v = base + lane;
        const bool open = v < V && levels[v] > nd;
        uint64_t s = 0, e = 0;
        if (open) {
            s = load_off(roff, v);
            e = load_off(roff, v + 1);
        }
        const bool big = open && e - s > kWaveDegree;
        for (uint64_t m = __ballot(big); m; m &= m - 1) {
            const int l = __builtin_ctzll(m);
            const uint64_t hs = read_lane_u64(s, l), he = read_lane_u64(e, l);
            bool found = false;
            for (uint64_t j0 = hs; j0 < he && !found; j0 += kWave) {
                const uint64_t j = j0 + lane;
                found = __ballot(j < he && levels[rcols[j]] == depth) != 0;
            }
            if (found && lane == static_cast<uint32_t>(l)) {
                levels[v] = nd;
                fc.update();
            }
        }
        if (open && !big) {
            for (uint64_t j = s; j < e; j++) {
                if (levels[rcols[j]] == depth) {
                    levels[v] = nd;
                    fc.update();
                    break;
                }
            }
        }
    }
    fc.finalise(frontier);
}

// Dynamic LDS layout of the _warp kernels: per virtual warp `chunk` levels
// then `chunk + 1` offsets (the chunkMemory lambda of bfs/bfs.cpp:187-189),
// offsets 8-byte aligned.
template<typename Off>
__host__ __device__ inline uint32_t warp_lds_levels_bytes(uint32_t warps, uint32_t chunk)
{ return (warps * chunk * 4u + 7u) & ~7u; }

template<typename Off>
__host__ __device__ inline uint32_t warp_lds_bytes(uint32_t warps, uint32_t chunk)
{ return warp_lds_levels_bytes<Off>(warps, chunk) + warps * (chunk + 1) * static_cast<uint32_t>(sizeof(Off)); }

// bfs/vertex_push_warp.cu: a virtual warp of W lanes (W | 64) stages a
// chunk's levels and offsets in LDS (memcpy_SIMD) and strides over each
// depth-d vertex's neighbours.  A workgroup takes another place among the
// blocks of each round: blocks a whole round apart agree in the low bits of
// their vertex ids, and so in how many edges they hold in an R-MAT graph's
// generated order (scale 22, edge factor 8, on the 2048 workgroups that are
// in flight at once: a search's levels take 18.1 ms without, 8.3 with it).
template<int R, typename Off>
__global__ __launch_bounds__(1024) void bfs_vertex_push_warp_kernel(
    uint32_t W, uint32_t C, uint64_t V, const Off *__restrict__ off,
    const uint32_t *__restrict__ cols, int32_t *levels, int32_t depth, uint32_t *frontier, RunLevel run)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    if (run.skip()) return;
    FrontierCount<R> fc;
    const int32_t nd = depth + 1;
    const uint32_t warps = blockDim.x / W;
    const uint32_t bw = threadIdx.x / W, lane = threadIdx.x % W;
    int32_t *myLevels = reinterpret_cast<int32_t *>(lds_raw) + bw * C;
    Off *myOff = reinterpret_cast<Off *>(lds_raw + warp_lds_levels_bytes<Off>(warps, C)) + bw * (C + 1);
    const uint32_t step = static_cast<uint32_t>(gridDim.x * 0.618f) | 1u;  // at most gridDim.x
    const uint64_t round = static_cast<uint64_t>(gridDim.x) * warps * C;
    uint32_t place = spread_block(blockIdx.x, gridDim.x);

    for (uint64_t v0 = 0; v0 < V; v0 += round) {
        const uint64_t base = v0 + (static_cast<uint64_t>(place) * warps + bw) * C;
        place = place + step >= gridDim.x ? place + step - gridDim.x : place + step;
        if (base >= V) continue;
        const uint32_t end = static_cast<uint32_t>(std::min<uint64_t>(C, V - base));
        for (uint32_t i = lane; i < end; i += W) myLevels[i] = levels[base + i];
        for (uint32_t i = lane; i <= end; i += W) myOff[i] = off[base + i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        for (uint32_t v = 0; v < end; v++) {
            if (myLevels[v] != depth) continue;
            const uint64_t s = myOff[v], n = static_cast<uint64_t>(myOff[v + 1]) - s;
            for (uint64_t i = lane; i < n; i += W)
                if (relax_depth(levels, cols[s + i], nd)) fc.update();
        }
        __builtin_amdgcn_wave_barrier();
    }
    fc.finalise(frontier);
}

// bfs/vertex_pull_warp.cu: a virtual warp probes an unvisited vertex's
// in-neighbours; the lanes' hits are combined with a wave64 ballot masked to
// the virtual warp (the __any_sync of :14) and the probe stops at the first
// stride that finds one.  The chunk's new depths are counted and written
// back from LDS.
template<int R, typename Off>
__global__ __launch_bounds__(1024) void bfs_vertex_pull_warp_kernel(
    uint32_t W, uint32_t C, uint64_t V, const Off *__restrict__ roff,
    const uint32_t *__restrict__ rcols, int32_t *levels, int32_t depth, uint32_t *frontier, RunLevel run)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    if (run.skip()) return;
    FrontierCount<R> fc;
    const int32_t nd = depth + 1;
    const uint32_t warps = blockDim.x / W;
    const uint32_t bw = threadIdx.x / W, lane = threadIdx.x % W;
    int32_t *myLevels = reinterpret_cast<int32_t *>(lds_raw) + bw * C;
    Off *myOff = reinterpret_cast<Off *>(lds_raw + warp_lds_levels_bytes<Off>(warps, C)) + bw * (C + 1);
    const uint64_t warpId = (static_cast<uint64_t>(spread_block(blockIdx.x, gridDim.x)) * blockDim.x + threadIdx.x) / W;
    const uint64_t totalWarps = static_cast<uint64_t>(warps) * gridDim.x;
    const uint32_t waveLane = threadIdx.x & (kWave - 1);
    const uint32_t subBase = (waveLane / W) * W;
    const uint64_t subMask = (W >= 64) ? ~0ull : (((1ull << W) - 1ull) << subBase);

    for (uint64_t chunk = warpId; chunk * C < V; chunk += totalWarps) {
        const uint64_t base = chunk * C;
        const uint32_t end = static_cast<uint32_t>(std::min<uint64_t>(C, V - base));
        for (uint32_t i = lane; i < end; i += W) myLevels[i] = levels[base + i];
        for (uint32_t i = lane; i <= end; i += W) myOff[i] = roff[base + i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        for (uint32_t v = 0; v < end; v++) {
            if (myLevels[v] <= depth) continue;
            const uint64_t s = myOff[v], n = static_cast<uint64_t>(myOff[v + 1]) - s;
            bool found = false;
            for (uint64_t i0 = 0; i0 < n && !found; i0 += W) {
                const uint64_t i = i0 + lane;
                const bool hit = i < n && levels[rcols[s + i]] == depth;
                found = (__ballot(hit) & subMask) != 0;
            }
            if (found && lane == 0) myLevels[v] = nd;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        }
        for (uint32_t i = lane; i < end; i += W) {
            if (myLevels[i] == nd) {
                fc.update();
                levels[base + i] = nd;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    fc.finalise(frontier);
}

// ------------------------------------------------------- host dispatch

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Geometry of a level kernel: resolve_geometry's, with at most as many
// workgroups as the CUs hold at once (each ends in an atomic on the
// frontier counter).
int level_geometry(const bw_launch *cfg, uint64_t work, uint32_t &block, uint32_t &grid)
{
    BW_TRY(resolve_geometry(cfg, work, block, grid));
    if (!(cfg && cfg->grid)) grid = std::min(grid, static_cast<uint32_t>(device_cus()) * (2048u / block));
    return BW_HIP_OK;
}

template<template<int> class Launch, typename... A>
int by_reduction(int32_t reduction, A &&...args)
{
    switch (reduction) {
    case BW_RED_NORMAL: return Launch<BW_RED_NORMAL>::run(args...);
    case BW_RED_BULK: return Launch<BW_RED_BULK>::run(args...);
    case BW_RED_WAVE: return Launch<BW_RED_WAVE>::run(args...);
    case BW_RED_BLOCK: return Launch<BW_RED_BLOCK>::run(args...);
    default: return fail(BW_HIP_ERR_ARG, "unknown frontier reduction " + std::to_string(reduction));
    }
}

int check_common(const int32_t *levels, const uint32_t *frontier)
{
    if (!levels || !frontier) return fail(BW_HIP_ERR_ARG, "levels and frontier must be device pointers");
    return BW_HIP_OK;
}

template<bool REV>
struct EdgeListLaunch {
    template<int R>
    struct L {
        static int run(uint64_t E, const uint32_t *in, const uint32_t *out, int32_t *levels,
                       int32_t depth, uint32_t *frontier, const bw_launch *cfg, const RunLevel &run)
        {
            uint32_t block, grid;
            const int vec = aligned16(in) && aligned16(out);
            BW_TRY(level_geometry(cfg, vec ? (E + 3) / 4 : E, block, grid));
            hipLaunchKernelGGL((bfs_edge_list_kernel<R, REV>), dim3(grid), dim3(block), 0,
                               stream_of(cfg), E, in, out, levels, depth, frontier, vec, run);
            BW_LAUNCH_CHECK();
            return BW_HIP_OK;
        }
    };
};

template<bool REV>
struct StructLaunch {
    template<int R>
    struct L {
        static int run(uint64_t E, const uint32_t *edges, int32_t *levels, int32_t depth,
                       uint32_t *frontier, const bw_launch *cfg, const RunLevel &run)
        {
            uint32_t block, grid;
            const int vec = aligned16(edges);
            BW_TRY(level_geometry(cfg, vec ? (E + 1) / 2 : E, block, grid));
            hipLaunchKernelGGL((bfs_struct_edge_list_kernel<R, REV>), dim3(grid), dim3(block), 0,
                               stream_of(cfg), E, edges, levels, depth, frontier, vec, run);
            BW_LAUNCH_CHECK();
            return BW_HIP_OK;
        }
    };
};

enum class VertexKind { Push, Pull, PushWarp, PullWarp };

template<VertexKind K, typename Off>
struct VertexLaunch {
    template<int R>
    struct L {
        static int run(uint64_t V, const Off *off, const uint32_t *cols, int32_t *levels,
                       int32_t depth, uint32_t *frontier, const bw_launch *cfg, const RunLevel &run)
        {
            uint32_t block, grid;
            hipStream_t s = stream_of(cfg);
            if constexpr (K == VertexKind::Push || K == VertexKind::Pull) {
                BW_TRY(level_geometry(cfg, V, block, grid));
                if constexpr (K == VertexKind::Push)
                    hipLaunchKernelGGL((bfs_vertex_push_kernel<R, Off>), dim3(grid), dim3(block), 0, s,
                                       V, off, cols, levels, depth, frontier, run);
                else
                    hipLaunchKernelGGL((bfs_vertex_pull_kernel<R, Off>), dim3(grid), dim3(block), 0, s,
                                       V, off, cols, levels, depth, frontier, run);
            } else {
                const uint32_t W = (cfg && cfg->warp) ? cfg->warp : 32;
                const uint32_t C = (cfg && cfg->chunk) ? cfg->chunk : 32;
                if (W == 0 || W > 64 || (W & (W - 1)))
                    return fail(BW_HIP_ERR_ARG, "Warp size should be a power of 2 no larger than 64!");
                if (C % W != 0) return fail(BW_HIP_ERR_ARG, "Chunk size should be a multiple of warp size!");
                // A grid sized by chunks of vertices, one virtual warp each.
                const uint64_t chunks = (V + C - 1) / C;
                BW_TRY(level_geometry(cfg, chunks * W, block, grid));
                const uint32_t lds = warp_lds_bytes<Off>(block / W, C);
                if (lds > 64 * 1024)
                    return fail(BW_HIP_ERR_ARG, "Insufficient shared memory, " + std::to_string(lds)
                                                + " requested, 65536 available.");
                if constexpr (K == VertexKind::PushWarp)
                    hipLaunchKernelGGL((bfs_vertex_push_warp_kernel<R, Off>), dim3(grid), dim3(block), lds, s,
                                       W, C, V, off, cols, levels, depth, frontier, run);
                else
                    hipLaunchKernelGGL((bfs_vertex_pull_warp_kernel<R, Off>), dim3(grid), dim3(block), lds, s,
                                       W, C, V, off, cols, levels, depth, frontier, run);
            }
            BW_LAUNCH_CHECK();
            return BW_HIP_OK;
        }
    };
};

template<VertexKind K>
int vertex_entry(uint64_t V, const void *off, int32_t offset_bytes, const uint32_t *cols,
                 int32_t *levels, int32_t depth, uint32_t *frontier, int32_t reduction,
                 const bw_launch *cfg, const RunLevel &run)
{
    BW_TRY(check_common(levels, frontier));
    if (V == 0) return BW_HIP_OK;
    if (!off || !cols) return fail(BW_HIP_ERR_ARG, "CSR arrays must be device pointers");
    if (offset_bytes == 4)
        return by_reduction<VertexLaunch<K, uint32_t>::template L>(
            reduction, V, static_cast<const uint32_t *>(off), cols, levels, depth, frontier, cfg, run);
    if (offset_bytes == 8)
        return by_reduction<VertexLaunch<K, uint64_t>::template L>(
            reduction, V, static_cast<const uint64_t *>(off), cols, levels, depth, frontier, cfg, run);
    return fail(BW_HIP_ERR_ARG, "offset_bytes must be 4 or 8");
}

// ----------------------------------------------------- edge-list builder

// Edge lists from a CSR, edge-parallel: a workgroup takes kListEdges
// consecutive edges, finds the rows of the first and last by binary search
// over the offsets, and each thread finds the row of each of its edges by
// binary search within that range (a few steps over cached offsets; none
// inside one long row).  Stores are coalesced across the workgroup.
constexpr uint64_t kListEdges = 4096;

// The row of edge e: the largest r in [lo, hi] with off[r] <= e.
template<typename Off>
__device__ __forceinline__ uint64_t row_of(const Off *off, uint64_t lo, uint64_t hi, uint64_t e)
{
    while (lo < hi) {
        const uint64_t mid = lo + (hi - lo + 1) / 2;
        if (static_cast<uint64_t>(off[mid]) <= e) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

template<typename Off>
__global__ __launch_bounds__(256) void build_edge_lists_kernel(uint64_t V, uint64_t E, const Off *__restrict__ off,
                                                               const uint32_t *__restrict__ cols, uint32_t *in,
                                                               uint32_t *out, uint2 *pairs)
{
    __shared__ uint64_t range[2];
    for (uint64_t e0 = static_cast<uint64_t>(blockIdx.x) * kListEdges; e0 < E;
         e0 += static_cast<uint64_t>(gridDim.x) * kListEdges) {
        const uint64_t e1 = e0 + kListEdges < E ? e0 + kListEdges : E;
        __syncthreads();  // the previous step has read the range
        if (threadIdx.x == 0) {
            const uint64_t r0 = row_of(off, 0, V - 1, e0);
            range[0] = r0;
            range[1] = row_of(off, r0, V - 1, e1 - 1);
        }
        __syncthreads();
        const uint64_t r0 = range[0], r1 = range[1];
        for (uint64_t e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
            const uint32_t r = static_cast<uint32_t>(row_of(off, r0, r1, e));
            const uint32_t c = cols[e];
            if (in) in[e] = r;
            if (out) out[e] = c;
            if (pairs) pairs[e] = make_uint2(r, c);
        }
    }
}

__global__ void set_root_kernel(int32_t *levels, uint32_t root) { levels[root] = 0; }

}  // namespace
}  // namespace bw

using namespace bw;

namespace {

// A level kernel's launch.
template<bool REV>
int edge_list_level(uint64_t E, const uint32_t *in, const uint32_t *out, int32_t *levels, int32_t depth,
                    uint32_t *frontier, int32_t reduction, const bw_launch *cfg, const RunLevel &run)
{
    BW_TRY(check_common(levels, frontier));
    if (E == 0) return BW_HIP_OK;
    if (!in || !out) return fail(BW_HIP_ERR_ARG, "EdgeList arrays must be device pointers");
    return by_reduction<EdgeListLaunch<REV>::template L>(reduction, E, in, out, levels, depth, frontier, cfg, run);
}

template<bool REV>
int struct_level(uint64_t E, const uint32_t *edges, int32_t *levels, int32_t depth, uint32_t *frontier,
                 int32_t reduction, const bw_launch *cfg, const RunLevel &run)
{
    BW_TRY(check_common(levels, frontier));
    if (E == 0) return BW_HIP_OK;
    if (!edges) return fail(BW_HIP_ERR_ARG, "StructEdgeList must be a device pointer");
    return by_reduction<StructLaunch<REV>::template L>(reduction, E, edges, levels, depth, frontier, cfg, run);
}

int level_launch(const bw_graph_dev *g, int32_t variant, int32_t reduction, int32_t *levels, int32_t depth,
                 uint32_t *frontier, const bw_launch *cfg, const RunLevel &run)
{
    if (!g) return fail(BW_HIP_ERR_ARG, "graph is NULL");
    auto need = [&](const void *p, const char *what) {
        if (!p && g->edge_count) {
            fail(BW_HIP_ERR_ARG, std::string("variant needs the ") + what + " representation");
            return false;
        }
        return true;
    };
    const uint64_t V = g->vertex_count, E = g->edge_count;
    switch (variant) {
    case BW_BFS_EDGE_LIST:
        if (!need(g->el_in, "EdgeList") || !need(g->el_out, "EdgeList")) return BW_HIP_ERR_ARG;
        return edge_list_level<false>(E, g->el_in, g->el_out, levels, depth, frontier, reduction, cfg, run);
    case BW_BFS_REV_EDGE_LIST:
        if (!need(g->rel_in, "reverse EdgeList") || !need(g->rel_out, "reverse EdgeList")) return BW_HIP_ERR_ARG;
        return edge_list_level<true>(E, g->rel_in, g->rel_out, levels, depth, frontier, reduction, cfg, run);
    case BW_BFS_STRUCT_EDGE_LIST:
        if (!need(g->sel, "StructEdgeList")) return BW_HIP_ERR_ARG;
        return struct_level<false>(E, g->sel, levels, depth, frontier, reduction, cfg, run);
    case BW_BFS_REV_STRUCT_EDGE_LIST:
        if (!need(g->rsel, "reverse StructEdgeList")) return BW_HIP_ERR_ARG;
        return struct_level<true>(E, g->rsel, levels, depth, frontier, reduction, cfg, run);
    case BW_BFS_VERTEX_PUSH:
        return vertex_entry<VertexKind::Push>(V, g->offsets, g->offset_bytes, g->cols, levels, depth, frontier,
                                              reduction, cfg, run);
    case BW_BFS_VERTEX_PULL:
        return vertex_entry<VertexKind::Pull>(V, g->rev_offsets, g->offset_bytes, g->rev_cols, levels, depth,
                                              frontier, reduction, cfg, run);
    case BW_BFS_VERTEX_PUSH_WARP:
        return vertex_entry<VertexKind::PushWarp>(V, g->offsets, g->offset_bytes, g->cols, levels, depth, frontier,
                                                  reduction, cfg, run);
    case BW_BFS_VERTEX_PULL_WARP:
        return vertex_entry<VertexKind::PullWarp>(V, g->rev_offsets, g->offset_bytes, g->rev_cols, levels, depth,
                                                  frontier, reduction, cfg, run);
    default:
        return fail(BW_HIP_ERR_ARG, "unknown BFS variant " + std::to_string(variant));
    }
}

// A batch of levels: counts[0] is the frontier count of the level before it,
// counts[1 + i] that of its i-th level, stamps[i] when that started.
constexpr uint32_t kBatch = 4, kMaxBatch = 32;

struct Batch {
    uint64_t stamps[kMaxBatch + 1];
    uint32_t counts[kMaxBatch + 1];
};

__global__ void start_batch_kernel(Batch *b, uint32_t last, int first)
{
    const uint32_t before = first ? 1u : b->counts[last];
    __syncthreads();
    for (uint32_t i = threadIdx.x; i <= kMaxBatch; i += blockDim.x) {
        b->counts[i] = i ? 0u : before;
        b->stamps[i] = wall_clock64();  // of a level that has nothing to launch
    }
}

__global__ void end_batch_kernel(uint64_t *stamp) { *stamp = wall_clock64(); }

}  // namespace

extern "C" int bw_bfs_edge_list(uint64_t E, const uint32_t *in, const uint32_t *out, int32_t *levels,
                                int32_t depth, uint32_t *frontier, int32_t reduction, const bw_launch *cfg)
{ return edge_list_level<false>(E, in, out, levels, depth, frontier, reduction, cfg, RunLevel{}); }

extern "C" int bw_bfs_rev_edge_list(uint64_t E, const uint32_t *in, const uint32_t *out, int32_t *levels,
                                    int32_t depth, uint32_t *frontier, int32_t reduction, const bw_launch *cfg)
{ return edge_list_level<true>(E, in, out, levels, depth, frontier, reduction, cfg, RunLevel{}); }

extern "C" int bw_bfs_struct_edge_list(uint64_t E, const uint32_t *edges, int32_t *levels, int32_t depth,
                                       uint32_t *frontier, int32_t reduction, const bw_launch *cfg)
{ return struct_level<false>(E, edges, levels, depth, frontier, reduction, cfg, RunLevel{}); }

extern "C" int bw_bfs_rev_struct_edge_list(uint64_t E, const uint32_t *edges, int32_t *levels,
                                           int32_t depth, uint32_t *frontier, int32_t reduction,
                                           const bw_launch *cfg)
{ return struct_level<true>(E, edges, levels, depth, frontier, reduction, cfg, RunLevel{}); }

extern "C" int bw_bfs_vertex_push(uint64_t V, const void *off, int32_t ob, const uint32_t *cols,
                                  int32_t *levels, int32_t depth, uint32_t *frontier, int32_t reduction,
                                  const bw_launch *cfg)
{ return vertex_entry<VertexKind::Push>(V, off, ob, cols, levels, depth, frontier, reduction, cfg, RunLevel{}); }

extern "C" int bw_bfs_vertex_pull(uint64_t V, const void *off, int32_t ob, const uint32_t *cols,
                                  int32_t *levels, int32_t depth, uint32_t *frontier, int32_t reduction,
                                  const bw_launch *cfg)
{ return vertex_entry<VertexKind::Pull>(V, off, ob, cols, levels, depth, frontier, reduction, cfg, RunLevel{}); }

extern "C" int bw_bfs_vertex_push_warp(uint64_t V, const void *off, int32_t ob, const uint32_t *cols,
                                       int32_t *levels, int32_t depth, uint32_t *frontier,
                                       int32_t reduction, const bw_launch *cfg)
{ return vertex_entry<VertexKind::PushWarp>(V, off, ob, cols, levels, depth, frontier, reduction, cfg, RunLevel{}); }

extern "C" int bw_bfs_vertex_pull_warp(uint64_t V, const void *off, int32_t ob, const uint32_t *cols,
                                       int32_t *levels, int32_t depth, uint32_t *frontier,
                                       int32_t reduction, const bw_launch *cfg)
{ return vertex_entry<VertexKind::PullWarp>(V, off, ob, cols, levels, depth, frontier, reduction, cfg, RunLevel{}); }

extern "C" int bw_bfs_level(const bw_graph_dev *g, int32_t variant, int32_t reduction, int32_t *levels,
                            int32_t depth, uint32_t *frontier, const bw_launch *cfg)
{ return level_launch(g, variant, reduction, levels, depth, frontier, cfg, RunLevel{}); }

extern "C" int bw_build_edge_lists(uint64_t V, uint64_t E, const void *off, int32_t ob, const uint32_t *cols,
                                   uint32_t *in, uint32_t *out, uint32_t *pairs, void *stream)
{
    if (V == 0 || E == 0) return BW_HIP_OK;
    if (!off || !cols) return fail(BW_HIP_ERR_ARG, "CSR arrays must be device pointers");
    if (reinterpret_cast<uintptr_t>(pairs) % 8) return fail(BW_HIP_ERR_ARG, "pairs must be 8-byte aligned");
    const uint32_t grid = static_cast<uint32_t>(std::min<uint64_t>((E + kListEdges - 1) / kListEdges, 65536));
    hipStream_t s = static_cast<hipStream_t>(stream);
    uint2 *p2 = reinterpret_cast<uint2 *>(pairs);  // device allocations are 8-byte aligned
    if (ob == 4)
        hipLaunchKernelGGL(build_edge_lists_kernel<uint32_t>, dim3(grid), dim3(256), 0, s, V, E,
                           static_cast<const uint32_t *>(off), cols, in, out, p2);
    else if (ob == 8)
        hipLaunchKernelGGL(build_edge_lists_kernel<uint64_t>, dim3(grid), dim3(256), 0, s, V, E,
                           static_cast<const uint64_t *>(off), cols, in, out, p2);
    else
        return fail(BW_HIP_ERR_ARG, "offset_bytes must be 4 or 8");
    BW_LAUNCH_CHECK();
    return BW_HIP_OK;
}

extern "C" int bw_bfs_run(const bw_graph_dev *g, const int32_t *schedule, int32_t schedule_len,
                          int32_t reduction, uint32_t root, int32_t *levels, uint32_t *counts_host,
                          float *level_ms_host, int64_t max_levels, int64_t *num_levels,
                          const bw_launch *cfg)
{
    if (!g || !schedule || schedule_len <= 0 || !levels || !num_levels)
        return fail(BW_HIP_ERR_ARG, "bw_bfs_run: invalid argument");
    *num_levels = 0;
    if (root >= g->vertex_count) return BW_HIP_OK;  // bfs/bfs.cpp:53
    hipStream_t s = stream_of(cfg);

    // Levels are launched in batches, each level on its own counter and
    // returning at once when the level before it found nothing, and the
    // counts are read back once per batch: one wait for the device per batch
    // where getFrontier (bfs/bfs.cu:13-18) waits after every level.
    Batch *b = nullptr;
    struct Cleanup {
        Batch *&b;
        ~Cleanup()
        {
            if (b) (void)hipFree(b);
        }
    } cleanup{b};
    int dev = 0, rate_khz = 0;
    if (level_ms_host) {
        BW_HIP_CHECK(hipGetDevice(&dev));
        BW_HIP_CHECK(hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, dev));
        if (rate_khz <= 0) return fail(BW_HIP_ERR_RUNTIME, "device reports no wall clock rate");
    }
    BW_HIP_CHECK(hipMalloc(&b, sizeof(Batch)));
    BW_TRY(bw_hip_fill_u32(levels, static_cast<uint32_t>(kUnvisited), g->vertex_count, s));
    hipLaunchKernelGGL(set_root_kernel, dim3(1), dim3(1), 0, s, levels, root);
    BW_LAUNCH_CHECK();
    int64_t curr = 0;
    uint32_t last = 0, batch = kBatch;
    int status = BW_HIP_OK;
    for (bool done = false; !done;) {
        if (curr >= max_levels) {
            status = fail(BW_HIP_ERR_LIMIT, "BFS did not finish within max_levels launches");
            break;
        }
        const uint32_t want = static_cast<uint32_t>(std::min<int64_t>(batch, max_levels - curr));
        hipLaunchKernelGGL(start_batch_kernel, dim3(1), dim3(kWave), 0, s, b, last, curr == 0 ? 1 : 0);
        BW_LAUNCH_CHECK();
        // A level that cannot be launched only matters if the search gets there.
        uint32_t n = 0;
        int refused = BW_HIP_OK;
        for (; n < want && refused == BW_HIP_OK; n += refused == BW_HIP_OK)
            refused = level_launch(g, schedule[(curr + n) % schedule_len], reduction, levels,
                                   static_cast<int32_t>(curr + n), b->counts + 1 + n, cfg,
                                   RunLevel{b->counts + n, level_ms_host ? b->stamps + n : nullptr});
        if (level_ms_host) {
            hipLaunchKernelGGL(end_batch_kernel, dim3(1), dim3(1), 0, s, b->stamps + n);
            BW_LAUNCH_CHECK();
        }
        Batch h;
        BW_HIP_CHECK(hipMemcpyAsync(&h, b, sizeof h, hipMemcpyDeviceToHost, s));
        BW_HIP_CHECK(hipStreamSynchronize(s));
        for (uint32_t i = 0; i < n && !done; i++) {
            const uint32_t found = h.counts[1 + i];
            if (counts_host) counts_host[curr] = found;
            if (level_ms_host)
                level_ms_host[curr] = static_cast<float>(static_cast<double>(h.stamps[i + 1] - h.stamps[i]) / rate_khz);
            curr++;
            done = found == 0;
        }
        if (!done && refused != BW_HIP_OK) {
            status = refused;
            break;
        }
        last = n;
        // Graphs of many levels: batches as long as a quarter of the search so far.
        batch = std::min<uint32_t>(std::max<uint32_t>(kBatch, static_cast<uint32_t>(curr / 4)), kMaxBatch);
    }
    *num_levels = curr;
    return status;
}

// ----------------------------------------------- allocation-free level loop

// Scratch of bw_bfs_run_static: one frontier counter per level, so that a
// level's count is never reused before it is read.  Each device holds its
// own copy; its address comes from hipGetSymbolAddress, never from the
// array's name, which is only a host-side stand-in in host code.
static __device__ __align__(256) uint32_t scratch[BW_BFS_STATIC_MAX_LEVELS];

namespace {

std::mutex g_scratch_mu;
constexpr int kMaxDevices = 64;
uint32_t *g_scratch[kMaxDevices] = {};

// Device address of the current device's scratch, looked up once per device.
int static_scratch(uint32_t **out)
{
    int dev = 0;
    BW_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(BW_HIP_ERR_ARG, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void *p = nullptr;
        BW_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch[dev] = static_cast<uint32_t *>(p);
    }
    *out = g_scratch[dev];
    return BW_HIP_OK;
}

}  // namespace

extern "C" int bw_bfs_run_static(const bw_graph_dev *g, const int32_t *schedule, int32_t schedule_len,
                                 int32_t reduction, uint32_t root, int32_t *levels, uint32_t *counts_host,
                                 int64_t max_levels, int64_t *num_levels, const bw_launch *cfg)
{
    if (!g || !schedule || schedule_len <= 0 || !levels || !num_levels)
        return fail(BW_HIP_ERR_ARG, "bw_bfs_run_static: invalid argument");
    if (max_levels < 0 || max_levels > BW_BFS_STATIC_MAX_LEVELS)
        return fail(BW_HIP_ERR_ARG, "bw_bfs_run_static: max_levels " + std::to_string(max_levels) +
                                        " exceeds the " + std::to_string(BW_BFS_STATIC_MAX_LEVELS) +
                                        " frontier counters of the static scratch");
    *num_levels = 0;
    if (root >= g->vertex_count) return BW_HIP_OK;  // bfs/bfs.cpp:53
    hipStream_t s = stream_of(cfg);
    uint32_t *counters = nullptr;
    BW_TRY(static_scratch(&counters));
    // The counters of this search start at zero (a fill kernel, no memset).
    if (max_levels > 0) BW_TRY(bw_hip_fill_u32(counters, 0u, static_cast<uint64_t>(max_levels), s));
    BW_TRY(bw_hip_fill_u32(levels, static_cast<uint32_t>(kUnvisited), g->vertex_count, s));
    hipLaunchKernelGGL(set_root_kernel, dim3(1), dim3(1), 0, s, levels, root);
    BW_LAUNCH_CHECK();
    int64_t curr = 0;
    uint32_t count = 1;
    while (count != 0) {
        if (curr >= max_levels) {
            *num_levels = curr;
            return fail(BW_HIP_ERR_LIMIT, "BFS did not finish within max_levels launches");
        }
        const int32_t variant = schedule[curr % schedule_len];
        const int st = bw_bfs_level(g, variant, reduction, levels, static_cast<int32_t>(curr), counters + curr, cfg);
        if (st != BW_HIP_OK) {
            *num_levels = curr;
            return st;
        }
        // getFrontier (bfs/bfs.cu:13-18): the read-back ends the level.
        BW_HIP_CHECK(hipMemcpyAsync(&count, counters + curr, sizeof count, hipMemcpyDeviceToHost, s));
        BW_HIP_CHECK(hipStreamSynchronize(s));
        if (counts_host) counts_host[curr] = count;
        curr++;
    }
    *num_levels = curr;
    return BW_HIP_OK;
}
