// Multi-source BFS: up to 64 searches on one graph in one level loop.
//
// Each search s computes exactly the depths of the reference's BFS from its
// source (bfs/bfs.cpp:43-118 of merijn/Belewitte: INT_MAX for unreached).
// The searches share every pass over the graph: vertex v holds a 64-bit
// `visit` mask (bit s = reached by search s) and a `frontier` mask (bit s =
// at the current depth of search s).  A level runs in one of two
// directions, chosen on the device from the frontier's out-edge count:
//  - bottom-up: every vertex not yet reached by all searches ORs the
//    frontier masks of its in-neighbours, stopping as soon as that covers
//    every search still missing it.  One thread probes a vertex with few
//    in-edges, a whole wave (256 in-edges per round trip) one above the
//    tunable wave threshold; a vertex above the tunable hub degree is cut
//    into chunks of in-edges, one wave each, that OR into next[] with
//    atomics (msbfs_bu_hubs);
//  - top-down: the frontier's out-edges are numbered in vertex order (the
//    level before left their prefix sums, per 64 vertices and within), then
//    every frontier edge u -> w ORs u's mask into next[w] (edge-parallel,
//    so a hub's edges spread over the grid).  OR is order-independent, so
//    the result is the same bit for bit.
// Either way the new bits give depth + 1 in those searches.  The level loop
// runs on the device (a done flag read by every kernel), launched in
// hipGraph batches.

#include "common.hpp"

#include <algorithm>
#include <cstddef>
#include <vector>

namespace bw {
namespace {

constexpr int kBlock = 256;
constexpr int kUnroll = 4;       // bottom-up wave path: chunks of 64 in-edges per round trip
constexpr uint32_t kSlots = 2;   // top-down expand: edges per thread at a time
constexpr int kEpi = 1024;       // threads of the epilogue and the init kernel
// Bottom-up: vertices with more in-edges than the tunable hub degree are
// split into chunks of kHubChunk in-edges, one wave each (msbfs_bu_hubs),
// so that a few waves holding many such vertices do not hold up the level.
constexpr uint32_t kHubChunk = 512;
constexpr uint32_t kGroup = 4;   // tiles (64 vertices) per entry of the numbering of the frontier's edges
constexpr int kLaneUnroll = 4;   // bottom-up lane path: in-edges per round trip

struct MsState {
    uint32_t depth;
    uint32_t done;
    uint32_t num_levels;
    uint32_t topdown;                // direction of the current level (1: top-down)
    uint64_t edges;                  // out-edges of the frontier
};

// The state and the levels' counts share one allocation, so that the host
// reads the state and the first kOutFirst counts in one copy.
constexpr size_t kOutOffset = 64, kOutFirst = 64;
static_assert(sizeof(MsState) <= kOutOffset, "the counts follow the state");

struct Sources {
    uint32_t v[64];
};

struct MsArgs {
    uint64_t V;
    uint64_t E;                // forward edges
    const uint32_t *roff;      // reverse CSR (bottom-up)
    const uint32_t *rcol;
    const uint32_t *off;       // forward CSR (top-down)
    const uint32_t *col;
    uint64_t *visit;
    uint64_t *front[2];  // level d reads front[d & 1], writes front[(d & 1) ^ 1]
    uint64_t *next;      // ORed frontier masks per vertex from the top-down edges or the hub
                         // chunks (zero between levels)
    // The frontier's out-edges in vertex order: per vertex of a tile of 64
    // (one wave of msbfs_level) the edges of the frontier vertices before it
    // in the tile (only written where the tile has any), per tile its edges
    // (groups of four tiles, the last one filled up with zeros) and, on
    // top-down levels, per group the edges of the groups before it.
    uint32_t *before;
    uint4 *tile_edges;
    uint32_t *group_first;
    uint32_t groups;
    uint64_t *part;      // per workgroup of msbfs_level: newly set bits, out-edges
    const uint4 *hubs;   // bottom-up: (vertex, first in-edge, end) per hub chunk
    uint32_t nhubs;
    uint32_t hub_degree; // in-degree above which a vertex is covered by hub chunks
    int32_t *depths;     // [nsrc][V]
    uint64_t all;        // mask of the nsrc searches
    uint64_t *level_bits;  // per level: newly set bits
    MsState *st;
    uint32_t max_levels;
    uint32_t wave_degree;
    uint32_t td_div;     // top-down when next_edges * td_div <= E (0: never)
};

__device__ __forceinline__ uint64_t wave_or64(uint64_t x)
{
    for (int o = kWave / 2; o > 0; o >>= 1) x |= __shfl_xor(x, o, kWave);
    return x;
}

// Depth nd for the searches in nb (0 for lanes with nothing).  Called by all
// lanes of the wave together: the lanes store one search's row at a time,
// so the stores of one instruction go to adjacent vertices.
__device__ __forceinline__ void record(const MsArgs &a, uint64_t v, uint64_t nb, int32_t nd)
{
    uint64_t any = wave_or64(nb);
    while (any) {
        const int s = __ffsll(static_cast<unsigned long long>(any)) - 1;
        any &= any - 1;
        if ((nb >> s) & 1ull) a.depths[static_cast<uint64_t>(s) * a.V + v] = nd;
    }
}

// One level over all vertices.  Bottom-up: pulls the frontier masks of the
// in-neighbours.  Top-down: takes the masks ORed into next[] by
// the expansion (and clears them).  Then the new bits update the visit mask,
// the next frontier, the depths and the numbering of the frontier's edges;
// the workgroup's new bits and out-edges go to part[] (the epilogue adds
// them up: an atomic per workgroup on one counter would take about 3 ns
// each, one after the other, 12 us a level for the two).  Tiles go to the
// workgroups spread over the XCDs (spread_block): in generated order the
// low-numbered vertices have most of the edges.
__global__ __launch_bounds__(kBlock) void msbfs_level(MsArgs a)
{
    __shared__ uint64_t wfound[kBlock / kWave], wedges[kBlock / kWave];
    const MsState &st = *a.st;
    if (st.done) return;
    const uint32_t d = st.depth;
    const bool td = st.topdown != 0;
    const int32_t nd = static_cast<int32_t>(d) + 1;
    // Selects rather than indexes, so the argument array stays in registers.
    const uint64_t *fin = (d & 1) ? a.front[1] : a.front[0];
    uint64_t *fout = (d & 1) ? a.front[0] : a.front[1];
    const int lane = __lane_id();
    uint64_t found = 0, nedges = 0;
    for (uint64_t base = static_cast<uint64_t>(spread_block(blockIdx.x, gridDim.x)) * kBlock; base < a.V;
         base += static_cast<uint64_t>(gridDim.x) * kBlock) {
        const uint64_t v64 = base + threadIdx.x;
        const uint32_t v = static_cast<uint32_t>(v64);
        const bool live = v64 < a.V;
        const uint64_t vis = live ? a.visit[v] : a.all;
        uint64_t acc = 0;
        if (td) {
            if (live) {
                acc = a.next[v];
                if (acc) a.next[v] = 0;
            }
        } else {
            bool open = vis != a.all;
            uint32_t s = 0, e = 0;
            if (open) {
                s = a.roff[v];
                e = a.roff[v + 1];
                if (e - s > a.hub_degree) {  // covered by msbfs_bu_hubs
                    acc = a.next[v];
                    if (acc) a.next[v] = 0;
                    open = false;
                    e = s;
                }
            }
            // The lane probes the first wave_degree in-edges itself; a row
            // still missing searches after that is finished by the whole wave.
            const uint32_t lim = e - s > a.wave_degree ? s + a.wave_degree : e;
            for (uint32_t j0 = s; j0 < lim; j0 += kLaneUnroll) {
                uint32_t c[kLaneUnroll];
#pragma unroll
                for (int u = 0; u < kLaneUnroll; u++) c[u] = j0 + u < lim ? a.rcol[j0 + u] : 0xFFFFFFFFu;
#pragma unroll
                for (int u = 0; u < kLaneUnroll; u++) acc |= c[u] != 0xFFFFFFFFu ? fin[c[u]] : 0;
                if ((acc | vis) == a.all) break;
            }
            uint64_t m = __ballot(open && lim < e && (acc | vis) != a.all);
            while (m) {
                const int l = __ffsll(static_cast<unsigned long long>(m)) - 1;
                m &= m - 1;
                const uint32_t vs = __shfl(lim, l, kWave), ve = __shfl(e, l, kWave);
                const uint64_t lvis = __shfl(vis | acc, l, kWave);
                // kUnroll chunks of 64 in-edges per round trip: their loads
                // are in flight together before the coverage test.
                uint64_t wacc = 0;
                for (uint32_t k0 = vs; k0 < ve; k0 += kWave * kUnroll) {
                    uint64_t x = 0;
#pragma unroll
                    for (int u = 0; u < kUnroll; u++) {
                        const uint32_t j = k0 + u * kWave + lane;
                        x |= j < ve ? fin[a.rcol[j]] : 0;
                    }
                    wacc |= wave_or64(x);
                    if ((wacc | lvis) == a.all) break;
                }
                if (lane == l) acc |= wacc;
            }
        }
        const uint64_t nb = acc & ~vis;
        uint32_t deg = 0;
        if (live) {
            fout[v] = nb;
            if (nb) {
                a.visit[v] = vis | nb;
                found += __popcll(nb);
                deg = a.off[v + 1] - a.off[v];
            }
        }
        if (base + (threadIdx.x & ~(kWave - 1u)) < a.V) {
            const uint32_t incl = wave_prefix_sum(deg), all = __shfl(incl, kWave - 1, kWave);
            if (all) a.before[v] = incl - deg;  // past the last vertex too
            if (lane == 0) reinterpret_cast<uint32_t *>(a.tile_edges)[v / kWave] = all;
            nedges += deg;
        }
        record(a, v64, nb, nd);
    }
    for (int o = kWave / 2; o > 0; o >>= 1) {
        found += __shfl_xor(found, o, kWave);
        nedges += __shfl_xor(nedges, o, kWave);
    }
    if (lane == 0) {
        wfound[threadIdx.x / kWave] = found;
        wedges[threadIdx.x / kWave] = nedges;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t f = 0, n = 0;
        for (int w = 0; w < kBlock / kWave; w++) {
            f += wfound[w];
            n += wedges[w];
        }
        a.part[2 * blockIdx.x] = f;
        a.part[2 * blockIdx.x + 1] = n;
    }
}

// The last i of [0, n) with x[i] <= t (x ascending, x[0] <= t), for kSlots t
// at once: their loads are in flight together.
__device__ __forceinline__ void last_at_most(const uint32_t *const (&x)[kSlots], uint32_t n,
                                             const uint32_t (&t)[kSlots], uint32_t (&at)[kSlots])
{
#pragma unroll
    for (uint32_t k = 0; k < kSlots; k++) at[k] = 0;
    while (n > 1) {
        const uint32_t half = n >> 1;
#pragma unroll
        for (uint32_t k = 0; k < kSlots; k++)
            if (x[k][at[k] + half] <= t[k]) at[k] += half;
        n -= half;
    }
}

// Top-down: each frontier edge u -> w ORs u's frontier bits that w has not
// reached yet into next[w].  A workgroup takes kSlots times 256 consecutive
// edges at a time, neighbouring lanes neighbouring edges, and finds each
// one's group of tiles and vertex by binary search.  What bounds it is the
// chain of dependent loads per edge, so every thread has kSlots of them in
// flight: a level of 3.3 M edges (R-MAT scale 19) took 237 us with eight
// consecutive edges per thread one after the other, 124 us so; with plain
// stores in the atomics' place it would take 70.  Four slots leave small levels too few
// workgroups (R-MAT scale 19: 0.66 ms a search against 0.64).
__device__ __forceinline__ void td_expand(const MsArgs &a, const MsState &st)
{
    const uint64_t *fin = (st.depth & 1) ? a.front[1] : a.front[0];
    const uint64_t T = st.edges;
    constexpr uint32_t kWindow = kBlock * kSlots;
    for (uint64_t c = static_cast<uint64_t>(blockIdx.x) * kWindow; c < T;
         c += static_cast<uint64_t>(gridDim.x) * kWindow) {
        uint32_t t[kSlots], at[kSlots], w[kSlots];
        const uint32_t *x[kSlots];
        uint64_t m[kSlots], seen[kSlots], next[kSlots];
#pragma unroll
        for (uint32_t k = 0; k < kSlots; k++) {
            t[k] = static_cast<uint32_t>(min(c + k * kBlock + threadIdx.x, T - 1));
            x[k] = a.group_first;
        }
        last_at_most(x, a.groups, t, at);
        uint32_t base[kSlots];
#pragma unroll
        for (uint32_t k = 0; k < kSlots; k++) {
            // The tile of the group: the first whose edges, added to those
            // before it, pass t.
            const uint4 e = a.tile_edges[at[k]];
            const uint32_t r = t[k] - a.group_first[at[k]], e2 = e.x + e.y, e3 = e2 + e.z;
            const uint32_t tile = (r >= e.x) + (r >= e2) + (r >= e3);
            t[k] = r - (tile == 0 ? 0 : tile == 1 ? e.x : tile == 2 ? e2 : e3);
            base[k] = (at[k] * kGroup + tile) * kWave;
            x[k] = a.before + base[k];
        }
        // The last tile may hold fewer vertices: a.before has room for all.
        last_at_most(x, kWave, t, at);
#pragma unroll
        for (uint32_t k = 0; k < kSlots; k++) {
            const uint32_t u = base[k] + at[k];
            m[k] = fin[u];
            w[k] = a.col[a.off[u] + (t[k] - a.before[u])];
        }
#pragma unroll
        for (uint32_t k = 0; k < kSlots; k++) {
            seen[k] = a.visit[w[k]];
            // Past the L1, which would show what the word was when the CU
            // first read it: fewer atomics that add nothing.
            next[k] = __hip_atomic_load(&a.next[w[k]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (uint32_t k = 0; k < kSlots; k++) {
            const uint64_t nw = m[k] & ~seen[k];
            if (c + k * kBlock + threadIdx.x < T && (nw & ~next[k]))
                atomicOr(reinterpret_cast<unsigned long long *>(&a.next[w[k]]), nw);
        }
    }
}

// Bottom-up, hubs: one wave per chunk of a hub's in-edges ORs their
// frontier masks (stopping once the hub's missing searches are covered,
// counting what other chunks already found) into next[hub].
__device__ __forceinline__ void bu_hubs(const MsArgs &a, const MsState &st)
{
    const uint64_t *fin = (st.depth & 1) ? a.front[1] : a.front[0];
    const int lane = __lane_id();
    const uint32_t nwaves = gridDim.x * (kBlock / kWave);
    for (uint32_t c = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; c < a.nhubs; c += nwaves) {
        const uint4 h = a.hubs[c];
        const uint64_t vis = a.visit[h.x];
        if (vis == a.all) continue;
        uint64_t acc = 0;
        for (uint32_t k0 = h.y; k0 < h.z; k0 += kWave * kUnroll) {
            uint64_t x = 0;
#pragma unroll
            for (int u = 0; u < kUnroll; u++) {
                const uint32_t j = k0 + u * kWave + lane;
                x |= j < h.z ? fin[a.rcol[j]] : 0;
            }
            acc |= wave_or64(x);
            if ((acc | vis | a.next[h.x]) == a.all) break;
        }
        const uint64_t nb = acc & ~vis;
        if (lane == 0 && (nb & ~a.next[h.x])) atomicOr(reinterpret_cast<unsigned long long *>(&a.next[h.x]), nb);
    }
}

// The first kernel of a level, whichever its direction: the top-down
// expansion or the bottom-up hub chunks.
__global__ __launch_bounds__(kBlock) void msbfs_expand_or_hubs(MsArgs a)
{
    const MsState &st = *a.st;
    if (st.done) return;
    if (st.topdown) td_expand(a, st);
    else if (a.nhubs) bu_hubs(a, st);
}

// The edges of the groups before each group of tiles, by one workgroup: kPer
// times 64 consecutive groups per wave and round, read and written in whole
// lines, the next round's loads in flight behind this round's barrier.  One
// CU's rate bounds it: the epilogue of 131072 tiles (2^23 vertices) takes 14
// us, 4 of them for a level without numbers; tile by tile, eight consecutive
// tiles per thread, it took 121, more than every workgroup's scan of the
// frontier would have.
__device__ __forceinline__ void number_edges(const MsArgs &a, uint32_t (*wsum)[kEpi / kWave])
{
    constexpr uint32_t kPer = 4;
    const uint32_t lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    uint32_t carry = 0, buf = 0;
    uint4 y[kPer];
    auto load = [&](uint32_t r0) {
#pragma unroll
        for (uint32_t k = 0; k < kPer; k++) {
            const uint32_t i = r0 + (wid * kPer + k) * kWave + lane;
            y[k] = i < a.groups ? a.tile_edges[i] : make_uint4(0, 0, 0, 0);
        }
    };
    load(0);
    for (uint32_t r0 = 0; r0 < a.groups; r0 += kEpi * kPer, buf ^= 1) {
        uint32_t first[kPer], sum = 0;
#pragma unroll
        for (uint32_t k = 0; k < kPer; k++) {
            const uint32_t x = y[k].x + y[k].y + y[k].z + y[k].w, incl = wave_prefix_sum(x);
            first[k] = sum + incl - x;
            sum += __builtin_amdgcn_readlane(static_cast<int>(incl), kWave - 1);
        }
        load(r0 + kEpi * kPer);
        if (lane == 0) wsum[buf][wid] = sum;
        __syncthreads();  // the other half of wsum is read until the next round's barrier
        uint32_t at = carry;
        for (uint32_t w = 0; w < kEpi / kWave; w++) {
            if (w < wid) at += wsum[buf][w];
            carry += wsum[buf][w];
        }
#pragma unroll
        for (uint32_t k = 0; k < kPer; k++) {
            const uint32_t i = r0 + (wid * kPer + k) * kWave + lane;
            if (i < a.groups) a.group_first[i] = at + first[k];
        }
    }
}

// Closes level d; picks the direction of level d + 1 from its frontier's
// out-edges and numbers them if it is top-down.
__global__ __launch_bounds__(kEpi) void msbfs_epilogue(MsArgs a, uint32_t nparts)
{
    __shared__ uint64_t wfound[kEpi / kWave], wedges[kEpi / kWave];
    __shared__ uint32_t wsum[2][kEpi / kWave];
    MsState &st = *a.st;
    if (st.done) return;
    const uint32_t tid = threadIdx.x, d = st.depth;
    uint64_t found = 0, edges = 0;
    for (uint32_t i = tid; i < nparts; i += kEpi) {
        found += a.part[2 * i];
        edges += a.part[2 * i + 1];
    }
    for (int o = kWave / 2; o > 0; o >>= 1) {
        found += __shfl_xor(found, o, kWave);
        edges += __shfl_xor(edges, o, kWave);
    }
    if (tid % kWave == 0) {
        wfound[tid / kWave] = found;
        wedges[tid / kWave] = edges;
    }
    __syncthreads();  // every thread has read the state too
    found = edges = 0;
    for (uint32_t w = 0; w < kEpi / kWave; w++) {
        found += wfound[w];
        edges += wedges[w];
    }
    const bool done = found == 0 || d + 1 >= a.max_levels;
    const bool td = a.td_div != 0 && edges * a.td_div <= a.E;
    if (tid == 0) {
        a.level_bits[d] = found;
        st.num_levels = d + 1;
        st.done = done;
        if (!done) st.depth = d + 1;
        st.topdown = td;
        st.edges = edges;
    }
    if (!done && td) number_edges(a, wsum);
}

// Nothing reached, no masks, no frontier edges.
__global__ __launch_bounds__(kBlock) void msbfs_reset(MsArgs a, uint64_t ndepths)
{
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    const uint64_t t = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x;
    for (uint64_t i = t; i < a.V; i += stride) {
        a.visit[i] = 0;
        a.front[0][i] = 0;
        a.next[i] = 0;
    }
    for (uint64_t i = t; i < a.groups; i += stride) a.tile_edges[i] = make_uint4(0, 0, 0, 0);
    // The rows start at any multiple of four bytes: whole 16-byte stores from
    // the first aligned entry on.
    const uint64_t head = min(ndepths, ((16 - (reinterpret_cast<uintptr_t>(a.depths) & 15)) & 15) / 4);
    int4 *quads = reinterpret_cast<int4 *>(a.depths + head);
    const uint64_t nquads = (ndepths - head) / 4;
    for (uint64_t i = t; i < nquads; i += stride) quads[i] = make_int4(kUnvisited, kUnvisited, kUnvisited, kUnvisited);
    if (t < head) a.depths[t] = kUnvisited;
    const uint64_t tail = head + nquads * 4;
    if (t < ndepths - tail) a.depths[tail + t] = kUnvisited;
}

// Depth 0: source i gets bit i (a repeated source vertex gets several).
__global__ __launch_bounds__(kEpi) void msbfs_init(MsArgs a, Sources src, uint32_t n)
{
    __shared__ uint32_t vert[64], degree[64];
    __shared__ unsigned long long all;
    __shared__ uint32_t wsum[2][kEpi / kWave];
    const uint32_t i = threadIdx.x;
    uint32_t own = 0;
    if (i == 0) all = 0;
    if (i < n) {
        const uint32_t v = src.v[i];
        vert[i] = v;
        own = a.off[v + 1] - a.off[v];
        atomicOr(reinterpret_cast<unsigned long long *>(&a.visit[v]), 1ull << i);
        atomicOr(reinterpret_cast<unsigned long long *>(&a.front[0][v]), 1ull << i);
        a.depths[static_cast<uint64_t>(i) * a.V + v] = 0;
    }
    __syncthreads();
    // The frontier's edges: every vertex once, in vertex order.  A wave per
    // source numbers its tile, if no source before it has the same tile.
    if (i < n) {
        for (uint32_t j = 0; j < i; j++)
            if (vert[j] == vert[i]) own = 0;
        degree[i] = own;
        atomicAdd(&all, static_cast<unsigned long long>(own));
    }
    __syncthreads();
    const uint32_t lane = i % kWave;
    const uint32_t lv = lane < n ? vert[lane] : 0xFFFFFFFFu, ld = lane < n ? degree[lane] : 0;
    for (uint32_t j = i / kWave; j < n; j += kEpi / kWave) {
        const uint32_t tile = vert[j] / kWave, v = tile * kWave + lane;
        uint64_t same = __ballot(lv / kWave == tile);  // sources past n: a tile no vertex has
        if (static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(same))) - 1 < j) continue;
        uint32_t before = 0, edges = 0;
        for (; same; same &= same - 1) {
            const int k = __ffsll(static_cast<unsigned long long>(same)) - 1;
            const uint32_t kv = __shfl(lv, k, kWave), kd = __shfl(ld, k, kWave);
            edges += kd;
            before += kv < v ? kd : 0;
        }
        a.before[v] = before;
        if (lane == 0) reinterpret_cast<uint32_t *>(a.tile_edges)[tile] = edges;
    }
    __syncthreads();
    const bool td = a.td_div != 0 && all * a.td_div <= a.E;
    if (i == 0) {
        a.st->depth = 0;
        a.st->done = 0;
        a.st->num_levels = 0;
        a.st->topdown = td;
        a.st->edges = all;
    }
    if (td) number_edges(a, wsum);
}

}  // namespace
}  // namespace bw

using namespace bw;

struct bw_msbfs {
    uint64_t V = 0, E = 0;
    const uint32_t *roff = nullptr, *rcol = nullptr;
    const uint32_t *off = nullptr, *col = nullptr;
    uint64_t *visit = nullptr, *front[2] = {nullptr, nullptr};
    uint64_t *next = nullptr;
    uint32_t *before = nullptr, *group_first = nullptr;
    uint4 *tile_edges = nullptr;
    uint32_t groups = 0;
    uint64_t *part = nullptr;
    uint4 *hubs = nullptr;
    uint32_t nhubs = 0;
    uint32_t hub_degree = 0;  // the hub chunks are built for this degree (0: none yet)
    MsState *st = nullptr;  // and the levels' counts behind it
    uint32_t max_levels = 0;
    uint32_t wave_degree = BW_MSBFS_DEFAULT_WAVE_DEGREE;
    uint32_t td_div = BW_MSBFS_DEFAULT_TOPDOWN_DIVISOR;
    uint32_t grid = 0;
    hipStream_t own_stream = nullptr;
    hipGraphExec_t exec = nullptr;
    int32_t *exec_depths = nullptr;
    uint64_t exec_all = 0;
    int32_t exec_lps = 0;
    uint32_t exec_wave = 0;
    uint32_t exec_td = 0;
    const uint4 *exec_hubs = nullptr;
    uint32_t exec_nhubs = 0;
    void *exec_stream = nullptr;

    ~bw_msbfs()
    {
        if (exec) (void)hipGraphExecDestroy(exec);
        void *bufs[] = {visit, front[0], front[1], next, before, tile_edges, group_first, part, hubs, st};
        for (void *p : bufs)
            if (p) (void)hipFree(p);
        if (own_stream) (void)hipStreamDestroy(own_stream);
    }
};

namespace {

MsArgs make_args(const bw_msbfs *m, int32_t *depths, uint32_t n)
{
    MsArgs a;
    a.V = m->V;
    a.E = m->E;
    a.roff = m->roff;
    a.rcol = m->rcol;
    a.off = m->off;
    a.col = m->col;
    a.visit = m->visit;
    a.front[0] = m->front[0];
    a.front[1] = m->front[1];
    a.next = m->next;
    a.before = m->before;
    a.tile_edges = m->tile_edges;
    a.group_first = m->group_first;
    a.groups = m->groups;
    a.part = m->part;
    a.hubs = m->hubs;
    a.nhubs = m->nhubs;
    a.hub_degree = m->hub_degree;
    a.depths = depths;
    a.all = n >= 64 ? ~0ull : ((1ull << n) - 1ull);
    a.level_bits = reinterpret_cast<uint64_t *>(reinterpret_cast<char *>(m->st) + kOutOffset);
    a.st = m->st;
    a.max_levels = m->max_levels;
    a.wave_degree = m->wave_degree;
    a.td_div = m->td_div;
    return a;
}

// Hub chunks of the bottom-up levels for vertices with more than
// hub_degree in-edges, from the reverse offsets.
int build_hubs(bw_msbfs *m, uint32_t hub_degree)
{
    std::vector<uint32_t> roff(m->V + 1);
    BW_HIP_CHECK(hipMemcpy(roff.data(), m->roff, 4 * (m->V + 1), hipMemcpyDeviceToHost));
    std::vector<uint4> hubs;
    for (uint64_t v = 0; v < m->V; v++)
        if (roff[v + 1] - roff[v] > hub_degree)
            for (uint32_t j = roff[v]; j < roff[v + 1]; j += kHubChunk)
                hubs.push_back(make_uint4(static_cast<uint32_t>(v), j, std::min(j + kHubChunk, roff[v + 1]), 0));
    uint4 *d = nullptr;
    if (!hubs.empty() && (hipMalloc(&d, sizeof(uint4) * hubs.size()) != hipSuccess ||
                          hipMemcpy(d, hubs.data(), sizeof(uint4) * hubs.size(), hipMemcpyHostToDevice) != hipSuccess)) {
        if (d) (void)hipFree(d);
        return fail(BW_HIP_ERR_NOMEM, "device allocation of the hub chunks failed");
    }
    if (m->hubs) (void)hipFree(m->hubs);
    m->hubs = d;
    m->nhubs = static_cast<uint32_t>(hubs.size());
    m->hub_degree = hub_degree;
    return BW_HIP_OK;
}

int launch_levels(const bw_msbfs *m, const MsArgs &a, int32_t count, hipStream_t s)
{
    for (int32_t i = 0; i < count; i++) {
        hipLaunchKernelGGL(msbfs_expand_or_hubs, dim3(m->grid), dim3(kBlock), 0, s, a);
        BW_LAUNCH_CHECK();
        hipLaunchKernelGGL(msbfs_level, dim3(m->grid), dim3(kBlock), 0, s, a);
        BW_LAUNCH_CHECK();
        hipLaunchKernelGGL(msbfs_epilogue, dim3(1), dim3(kEpi), 0, s, a, m->grid);
        BW_LAUNCH_CHECK();
    }
    return BW_HIP_OK;
}

}  // namespace

extern "C" int bw_msbfs_create(bw_msbfs **out, const bw_graph_dev *g, uint32_t max_levels)
{
    if (!out || !g || max_levels == 0) return fail(BW_HIP_ERR_ARG, "bw_msbfs_create: invalid argument");
    *out = nullptr;
    if (g->offset_bytes != 4 || !g->rev_offsets || !g->offsets || (g->edge_count && (!g->rev_cols || !g->cols)))
        return fail(BW_HIP_ERR_ARG, "multi-source BFS needs the forward and reverse CSR with uint32 offsets");
    if (g->edge_count >= 0xFFFFFFFFull) return fail(BW_HIP_ERR_ARG, "multi-source BFS needs E < 2^32 - 1");
    if (g->vertex_count == 0 || g->vertex_count >= 0x7FFFFFFFull)
        return fail(BW_HIP_ERR_ARG, "multi-source BFS needs 0 < V < 2^31");
    auto m = new bw_msbfs();
    m->V = g->vertex_count;
    m->E = g->edge_count;
    m->roff = static_cast<const uint32_t *>(g->rev_offsets);
    m->rcol = g->rev_cols;
    m->off = static_cast<const uint32_t *>(g->offsets);
    m->col = g->cols;
    m->max_levels = max_levels;
    // As many workgroups as are in flight at once, or as have vertices or a
    // window of edges: the epilogue reads a partial of each (20000-vertex
    // chain, one source: 54 ms with 2048, 47.5 with 79).
    m->grid = std::min(static_cast<uint32_t>(device_cus()) * 8,
                       static_cast<uint32_t>(std::max<uint64_t>((m->V + kBlock - 1) / kBlock,
                                                                m->E / (kBlock * kSlots) + 1)));
    m->groups = static_cast<uint32_t>((m->V + kGroup * kWave - 1) / (kGroup * kWave));
    bool ok = hipMalloc(&m->visit, 8 * m->V) == hipSuccess && hipMalloc(&m->front[0], 8 * m->V) == hipSuccess &&
              hipMalloc(&m->front[1], 8 * m->V) == hipSuccess && hipMalloc(&m->next, 8 * m->V) == hipSuccess &&
              hipMalloc(&m->before, 4ull * kWave * kGroup * m->groups) == hipSuccess &&
              hipMalloc(&m->tile_edges, sizeof(uint4) * m->groups) == hipSuccess &&
              hipMalloc(&m->group_first, 4ull * m->groups) == hipSuccess &&
              hipMalloc(&m->part, 16ull * m->grid) == hipSuccess &&
              hipMalloc(&m->st, kOutOffset + 8 * std::max<size_t>(max_levels, kOutFirst)) == hipSuccess;
    if (!ok) {
        delete m;
        return fail(BW_HIP_ERR_NOMEM, "device allocation of the multi-source BFS failed");
    }
    const int hs = build_hubs(m, BW_MSBFS_DEFAULT_HUB_DEGREE);
    if (hs != BW_HIP_OK) {
        delete m;
        return hs;
    }
    *out = m;
    return BW_HIP_OK;
}

extern "C" int bw_msbfs_destroy(bw_msbfs *m)
{
    delete m;
    return BW_HIP_OK;
}

extern "C" int bw_msbfs_set_tuning(bw_msbfs *m, uint32_t wave_degree, uint32_t topdown_divisor,
                                   uint32_t hub_degree)
{
    if (!m) return fail(BW_HIP_ERR_ARG, "NULL handle");
    if (topdown_divisor > 1024) return fail(BW_HIP_ERR_ARG, "topdown_divisor must be 0..1024");
    if (hub_degree < 16) return fail(BW_HIP_ERR_ARG, "hub_degree must be at least 16");
    if (hub_degree != m->hub_degree) BW_TRY(build_hubs(m, hub_degree));
    m->wave_degree = wave_degree;
    m->td_div = topdown_divisor;
    return BW_HIP_OK;
}

extern "C" int bw_msbfs_run(bw_msbfs *m, const uint32_t *sources, uint32_t n, int32_t *depths,
                            int32_t levels_per_sync, int32_t use_graph, uint64_t *level_bits_host,
                            uint32_t *num_levels, float *total_ms, void *stream)
{
    if (!m || !sources || !depths || !num_levels || levels_per_sync < 1)
        return fail(BW_HIP_ERR_ARG, "bw_msbfs_run: invalid argument");
    if (n < 1 || n > 64) return fail(BW_HIP_ERR_ARG, "multi-source BFS takes 1..64 sources");
    for (uint32_t i = 0; i < n; i++)
        if (sources[i] >= m->V) return fail(BW_HIP_ERR_ARG, "source " + std::to_string(sources[i]) + " out of range");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (use_graph && !s) {
        if (!m->own_stream) BW_HIP_CHECK(hipStreamCreateWithFlags(&m->own_stream, hipStreamNonBlocking));
        s = m->own_stream;
    }
    const MsArgs a = make_args(m, depths, n);
    if (use_graph && (!m->exec || m->exec_depths != depths || m->exec_all != a.all ||
                      m->exec_lps != levels_per_sync || m->exec_wave != m->wave_degree || m->exec_td != m->td_div ||
                      m->exec_hubs != m->hubs || m->exec_nhubs != m->nhubs || m->exec_stream != s)) {
        if (m->exec) (void)hipGraphExecDestroy(m->exec);
        m->exec = nullptr;
        hipGraph_t graph = nullptr;
        BW_HIP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        const int cst = launch_levels(m, a, levels_per_sync, s);
        const hipError_t ce = hipStreamEndCapture(s, &graph);
        if (cst != BW_HIP_OK) {
            if (graph) (void)hipGraphDestroy(graph);
            return cst;
        }
        if (ce != hipSuccess) return hip_fail(ce, "hipStreamEndCapture", __FILE__, __LINE__);
        const hipError_t ie = hipGraphInstantiate(&m->exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (ie != hipSuccess) {
            m->exec = nullptr;
            return hip_fail(ie, "hipGraphInstantiate", __FILE__, __LINE__);
        }
        m->exec_depths = depths;
        m->exec_all = a.all;
        m->exec_lps = levels_per_sync;
        m->exec_wave = m->wave_degree;
        m->exec_td = m->td_div;
        m->exec_hubs = m->hubs;
        m->exec_nhubs = m->nhubs;
        m->exec_stream = s;
    }
    hipEvent_t ev0, ev1;
    BW_HIP_CHECK(hipEventCreate(&ev0));
    BW_HIP_CHECK(hipEventCreate(&ev1));
    int st = BW_HIP_OK;
    if (hipEventRecord(ev0, s) != hipSuccess) st = fail(BW_HIP_ERR_RUNTIME, "event record failed");
    if (st == BW_HIP_OK) {
        Sources src{};
        std::copy(sources, sources + n, src.v);
        hipLaunchKernelGGL(msbfs_reset, dim3(device_cus() * 8), dim3(kBlock), 0, s, a, n * m->V);
        hipError_t le = hipGetLastError();
        if (le == hipSuccess) {
            hipLaunchKernelGGL(msbfs_init, dim3(1), dim3(kEpi), 0, s, a, src, n);
            le = hipGetLastError();
        }
        if (le != hipSuccess) st = hip_fail(le, "msbfs_init", __FILE__, __LINE__);
    }
    struct {
        MsState st;
        char pad[kOutOffset - sizeof(MsState)];
        uint64_t bits[kOutFirst];
    } host{};
    static_assert(offsetof(decltype(host), bits) == kOutOffset, "as on the device");
    uint32_t batches = 0;
    const uint32_t max_batches = m->max_levels / static_cast<uint32_t>(levels_per_sync) + 2;
    while (st == BW_HIP_OK && !host.st.done) {
        if (batches++ > max_batches) {
            st = fail(BW_HIP_ERR_LIMIT, "multi-source BFS exceeded its level bound");
            break;
        }
        if (use_graph) {
            const hipError_t le = hipGraphLaunch(m->exec, s);
            if (le != hipSuccess) st = hip_fail(le, "hipGraphLaunch", __FILE__, __LINE__);
        } else {
            st = launch_levels(m, a, levels_per_sync, s);
        }
        if (st != BW_HIP_OK) break;
        if (hipMemcpyAsync(&host, m->st, sizeof host, hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            st = fail(BW_HIP_ERR_RUNTIME, "reading the multi-source BFS state failed");
    }
    if (st == BW_HIP_OK) {
        if (hipEventRecord(ev1, s) != hipSuccess || hipEventSynchronize(ev1) != hipSuccess)
            st = fail(BW_HIP_ERR_RUNTIME, "event failed");
        else if (total_ms)
            (void)hipEventElapsedTime(total_ms, ev0, ev1);
    }
    (void)hipEventDestroy(ev0);
    (void)hipEventDestroy(ev1);
    if (st != BW_HIP_OK) return st;
    *num_levels = host.st.num_levels;
    const size_t k = std::min(host.st.num_levels, m->max_levels);
    std::vector<uint64_t> more;
    const uint64_t *bits = host.bits;
    if (k > kOutFirst) {
        more.resize(k);
        BW_HIP_CHECK(hipMemcpy(more.data(), a.level_bits, 8 * k, hipMemcpyDeviceToHost));
        bits = more.data();
    }
    if (k && bits[k - 1] != 0) return fail(BW_HIP_ERR_LIMIT, "multi-source BFS reached max_levels with work left");
    if (level_bits_host) std::copy(bits, bits + k, level_bits_host);
    return BW_HIP_OK;
}
