// PageRank iteration, degree and consolidate kernels for gfx950 and their
// C ABI entry points.
//
// Each kernel computes one reference kernel of pagerank/*.cu (merijn/
// Belewitte) with the same FP32 arithmetic per contribution: IEEE division
// pr/deg, the double/float base terms of the two consolidate kernels.  The
// mapping is MI355X's own:
//   - pull forms: a workgroup stages its rows' in-edge contributions in LDS
//     in rounds of 2048, gathered with every load in flight; long rows are
//     summed one wave or one workgroup each in the same launch (the pull
//     plan).  vertex-pull and vertex-pull-nodiv keep
//     the reference's sequential FP32 sum in CSR order, bit for bit; the
//     _warp forms combine lane-strided partials by shuffles where the
//     reference adds them atomically.  The dividing forms gather
//     per-vertex quotients computed once per iteration (the same IEEE
//     values);
//   - reverse edge lists: a segmented reduction over destination runs, one
//     store per run, atomics only for runs cut by a workgroup's range;
//   - forward edge lists and push forms: propagation blocking
//     (pagerank_scatter.hip) in bw_pr_run and the plugin; the per-call
//     entry points keep one atomic per edge;
//   - FP64 reductions of the residual and dangling mass: partials per
//     workgroup that the next launch adds up in a fixed order in bw_pr_run;
//     the per-call entry points add with one atomic per workgroup on a grid
//     of two workgroups per CU.

#include "common.hpp"
#include "pagerank_scatter.hpp"

#include <algorithm>
#include <memory>
#include <vector>

namespace bw {
namespace {

constexpr float kDamp = 0.85f;  // pagerank/pagerank.hpp:9

__device__ __forceinline__ void add_f32(float *p, float v) { unsafeAtomicAdd(p, v); }
__device__ __forceinline__ void add_f64(double *p, double v) { unsafeAtomicAdd(p, v); }

// ---------------------------------------------------------------- degrees

// Occurrence counts of values[i * STRIDE + off] (the degree kernels'
// atomicAdd(&deg[x], 1) per edge).  Each wave reads 64 consecutive entries
// and adds every run of equal values inside them with one atomic from the
// run's last lane: a source-sorted edge list, whose lanes would otherwise
// all add to one counter, takes an atomic per run instead of per edge.
// Values below kHotIds are counted in LDS and added to deg once per
// workgroup: a graph relabelled by degree has its hubs there, whose
// counters would otherwise take one global atomic per edge, one after the
// other.
constexpr uint32_t kHotIds = 16384;

template<int STRIDE>
__global__ __launch_bounds__(256) void pr_degrees_runs_kernel(uint64_t E, const uint32_t *__restrict__ values,
                                                              int off, uint32_t *deg)
{
    __shared__ uint32_t hot[kHotIds];
    for (uint32_t i = threadIdx.x; i < kHotIds; i += blockDim.x) hot[i] = 0;
    __syncthreads();
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint64_t waves = static_cast<uint64_t>(gridDim.x) * (blockDim.x / kWave);
    for (uint64_t w = (static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / kWave; w * kWave < E;
         w += waves) {
        const uint64_t i = w * kWave + lane;
        const bool valid = i < E;
        const uint32_t x = valid ? values[i * STRIDE + off] : 0xFFFFFFFFu;
        const uint32_t prev = __shfl_up(x, 1, kWave), next = __shfl_down(x, 1, kWave);
        const bool head = lane == 0 || prev != x;
        const bool tail = lane == kWave - 1 || next != x;
        const uint64_t heads = __ballot(head);
        const uint64_t upto = lane == kWave - 1 ? ~0ull : ((2ull << lane) - 1ull);
        const uint32_t h = 63u - static_cast<uint32_t>(__builtin_clzll(heads & upto));
        if (valid && tail) {
            if (x < kHotIds) atomicAdd(&hot[x], lane - h + 1u);
            else atomicAdd(&deg[x], lane - h + 1u);
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kHotIds; i += blockDim.x)
        if (hot[i]) atomicAdd(&deg[i], hot[i]);
}

// Workgroups of the degree count: two per CU (the LDS counters take 64 KB),
// fewer for a short list, so that each flushes its counters after a long
// stretch of entries.
inline uint32_t degree_grid(uint64_t E)
{
    const uint64_t need = (E + 255) / 256;
    return static_cast<uint32_t>(std::max<uint64_t>(1, std::min<uint64_t>(need, 2ull * device_cus())));
}

template<typename Off>
__global__ __launch_bounds__(1024) void pr_degrees_csr_kernel(uint64_t V, const Off *__restrict__ off, uint32_t *deg)
{
    const uint64_t stride = static_cast<uint64_t>(blockDim.x) * gridDim.x;
    for (uint64_t v = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; v < V; v += stride)
        atomicAdd(&deg[v], static_cast<uint32_t>(off[v + 1] - off[v]));
}

// ------------------------------------------------------------- iteration

template<bool REV>
__device__ __forceinline__ void push_edge(uint32_t in, uint32_t out, const uint32_t *deg, const float *pr,
                                          float *np)
{
    // pagerank/edgelist.cu:15-21 (forward: origin = in) and
    // rev_edgelist.cu:15-21 (reverse list: origin = out).
    const uint32_t origin = REV ? out : in, dest = REV ? in : out;
    const uint32_t d = deg[origin];
    float r = 0.0f;
    if (d != 0) r = pr[origin] / static_cast<float>(d);
    add_f32(&np[dest], r);
}

template<bool REV>
__global__ __launch_bounds__(1024) void pr_edge_list_kernel(uint64_t E, const uint32_t *__restrict__ in,
                                                            const uint32_t *__restrict__ out,
                                                            const uint32_t *__restrict__ deg,
                                                            const float *__restrict__ pr, float *np, int vec)
{
    const uint64_t stride = static_cast<uint64_t>(blockDim.x) * gridDim.x;
    const uint64_t gid = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    uint64_t done = 0;
    if (vec) {
        const uint64_t E4 = E / 4;
        const uint4 *in4 = reinterpret_cast<const uint4 *>(in);
        const uint4 *out4 = reinterpret_cast<const uint4 *>(out);
        for (uint64_t i = gid; i < E4; i += stride) {
            const uint4 a = in4[i], b = out4[i];
            push_edge<REV>(a.x, b.x, deg, pr, np);
            push_edge<REV>(a.y, b.y, deg, pr, np);
            push_edge<REV>(a.z, b.z, deg, pr, np);
            push_edge<REV>(a.w, b.w, deg, pr, np);
        }
        done = E4 * 4;
    }
    for (uint64_t i = done + gid; i < E; i += stride) push_edge<REV>(in[i], out[i], deg, pr, np);
}

template<bool REV>
__global__ __launch_bounds__(1024) void pr_struct_edge_list_kernel(uint64_t E, const uint32_t *__restrict__ edges,
                                                                   const uint32_t *__restrict__ deg,
                                                                   const float *__restrict__ pr, float *np,
                                                                   int vec)
{
    const uint64_t stride = static_cast<uint64_t>(blockDim.x) * gridDim.x;
    const uint64_t gid = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    uint64_t done = 0;
    if (vec) {
        const uint64_t E2 = E / 2;
        const uint4 *e4 = reinterpret_cast<const uint4 *>(edges);
        for (uint64_t i = gid; i < E2; i += stride) {
            const uint4 p = e4[i];
            push_edge<REV>(p.x, p.y, deg, pr, np);
            push_edge<REV>(p.z, p.w, deg, pr, np);
        }
        done = E2 * 2;
    }
    for (uint64_t i = done + gid; i < E; i += stride) push_edge<REV>(edges[2 * i], edges[2 * i + 1], deg, pr, np);
}

// ------------------------------------------------- reverse edge lists

constexpr uint32_t kSegThreads = 256;
constexpr uint32_t kSegPerThread = 16;
constexpr uint32_t kSegBlockEdges = kSegThreads * kSegPerThread;
constexpr uint32_t kNoKey = 0xFFFFFFFFu;

// Destination and source of reverse edge e: the SoA lists hold the
// destination in in[] and the source in out[]; the AoS pairs (in, out).
template<bool AOS>
__device__ __forceinline__ void rev_edge(const uint32_t *__restrict__ a, const uint32_t *__restrict__ b, uint64_t e,
                                         uint32_t &dst, uint32_t &src)
{
    if constexpr (AOS) {
        dst = a[2 * e];
        src = a[2 * e + 1];
    } else {
        dst = a[e];
        src = b[e];
    }
}

// revEdgeListPageRank / revStructEdgeListPageRank (pagerank/rev_edgelist.cu:
// 3-23, rev_struct_edgelist.cu:3-24) for wave64.  The reverse lists are
// grouped by destination, so the per-edge atomic adds of the reference
// become a segmented reduction: a workgroup takes 4096 consecutive edges, 16
// per thread; each thread sums its runs of equal destination, a block-wide
// segmented scan carries a run's partial sum across threads, and the thread
// holding a run's last edge writes the run's total once.  A run cut by the
// workgroup's edge range (its destination continues in the neighbouring
// workgroup) is added atomically; every other run is stored, since no other
// workgroup touches its destination.  The sum order within a destination
// differs from the reference's (whose atomics have no fixed order).
template<bool AOS, bool PRE>
__global__ __launch_bounds__(kSegThreads) void pr_rev_segmented_kernel(uint64_t E, const uint32_t *__restrict__ a,
                                                                       const uint32_t *__restrict__ b,
                                                                       const uint32_t *__restrict__ deg,
                                                                       const float *__restrict__ pr, float *np,
                                                                       int vec, ReducePrev prev)
{
    __shared__ ReduceLds red;
    if (reduce_prev<kSegThreads>(prev, red)) return;
    __shared__ uint32_t firstKeys[kSegThreads], lastKeys[kSegThreads];
    __shared__ float sums[kSegThreads];
    __shared__ float waveTotal[kSegThreads / kWave];
    __shared__ int waveHead[kSegThreads / kWave];
    const uint32_t t = threadIdx.x, lane = t & (kWave - 1), wv = t / kWave;
    const uint64_t b0 = static_cast<uint64_t>(blockIdx.x) * kSegBlockEdges;
    const uint64_t bEnd = b0 + kSegBlockEdges < E ? b0 + kSegBlockEdges : E;
    const uint64_t base = b0 + static_cast<uint64_t>(t) * kSegPerThread;

    uint32_t key[kSegPerThread], src[kSegPerThread];
    if (vec && base + kSegPerThread <= E) {
        if constexpr (AOS) {
            const uint4 *p = reinterpret_cast<const uint4 *>(a + 2 * base);
#pragma unroll
            for (uint32_t q = 0; q < kSegPerThread / 2; q++) {
                const uint4 x = p[q];
                key[2 * q] = x.x;
                src[2 * q] = x.y;
                key[2 * q + 1] = x.z;
                src[2 * q + 1] = x.w;
            }
        } else {
            const uint4 *pk = reinterpret_cast<const uint4 *>(a + base);
            const uint4 *ps = reinterpret_cast<const uint4 *>(b + base);
#pragma unroll
            for (uint32_t q = 0; q < kSegPerThread / 4; q++) {
                const uint4 x = pk[q], y = ps[q];
                key[4 * q] = x.x, key[4 * q + 1] = x.y, key[4 * q + 2] = x.z, key[4 * q + 3] = x.w;
                src[4 * q] = y.x, src[4 * q + 1] = y.y, src[4 * q + 2] = y.z, src[4 * q + 3] = y.w;
            }
        }
    } else {
#pragma unroll
        for (uint32_t k = 0; k < kSegPerThread; k++) {
            key[k] = kNoKey;
            src[k] = 0;
            if (base + k < E) rev_edge<AOS>(a, b, base + k, key[k], src[k]);
        }
    }
    // Contributions (rev_edgelist.cu:15-21: origin = out[], zero for a
    // vertex without out-edges), then the running sum of each run inside the
    // thread.
    // The gathers are unconditional (a missing edge reads source 0 and is
    // masked afterwards), so all of them are in flight together.
    // PRE: pr already holds each source's contribution (pr_contrib_kernel).
    uint32_t dg[kSegPerThread];
    float pv[kSegPerThread], c[kSegPerThread];
    if constexpr (!PRE) {
#pragma unroll
        for (uint32_t k = 0; k < kSegPerThread; k++) dg[k] = deg[src[k]];
    }
#pragma unroll
    for (uint32_t k = 0; k < kSegPerThread; k++) pv[k] = pr[src[k]];
#pragma unroll
    for (uint32_t k = 0; k < kSegPerThread; k++) {
        if constexpr (PRE) c[k] = key[k] != kNoKey ? pv[k] : 0.0f;
        else c[k] = (key[k] != kNoKey && dg[k] != 0) ? pv[k] / static_cast<float>(dg[k]) : 0.0f;
    }
#pragma unroll
    for (uint32_t k = 1; k < kSegPerThread; k++)
        if (key[k] == key[k - 1]) c[k] += c[k - 1];
    const uint32_t firstKey = key[0], lastKey = key[kSegPerThread - 1];
    firstKeys[t] = firstKey;
    lastKeys[t] = lastKey;
    __syncthreads();

    // Segmented inclusive scan over the threads of (carry out, head): a
    // thread whose edges are one run continuing the previous thread's last
    // run adds the previous carry; any other thread starts a new segment.
    const bool chained = t > 0 && firstKey == lastKey && lastKeys[t - 1] == firstKey;
    float x = c[kSegPerThread - 1];
    int h = chained ? 0 : 1;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const float px = __shfl_up(x, off, kWave);
        const int ph = __shfl_up(h, off, kWave);
        if (static_cast<int>(lane) >= off) {
            if (!h) x += px;
            h |= ph;
        }
    }
    if (lane == kWave - 1) {
        waveTotal[wv] = x;
        waveHead[wv] = h;
    }
    __syncthreads();
    if (!h) {
        // No segment head from the wave's start to here: the segment comes in
        // from the previous waves.
        float inc = 0.0f;
        for (uint32_t w = 0; w < wv; w++) inc = waveTotal[w] + (waveHead[w] ? 0.0f : inc);
        x += inc;
    }
    sums[t] = x;
    __syncthreads();
    const float carryIn = (t > 0 && lastKeys[t - 1] == firstKey) ? sums[t - 1] : 0.0f;

    // The key after this thread's last edge, and the runs the workgroup's
    // edge range cuts.
    uint32_t nextKey = kNoKey;
    if (t + 1 < kSegThreads) nextKey = firstKeys[t + 1];
    uint32_t prevEdgeKey = kNoKey, nextEdgeKey = kNoKey, blockFirst = kNoKey, blockLast = kNoKey, unused = 0;
    if (b0 > 0) rev_edge<AOS>(a, b, b0 - 1, prevEdgeKey, unused);
    if (bEnd < E) rev_edge<AOS>(a, b, bEnd, nextEdgeKey, unused);
    rev_edge<AOS>(a, b, b0, blockFirst, unused);
    rev_edge<AOS>(a, b, bEnd - 1, blockLast, unused);
    const bool leftOpen = prevEdgeKey == blockFirst, rightOpen = nextEdgeKey == blockLast;
#pragma unroll
    for (uint32_t k = 0; k < kSegPerThread; k++) {
        if (key[k] == kNoKey) continue;
        const uint32_t after = k + 1 < kSegPerThread ? key[k + 1] : nextKey;
        if (after == key[k]) continue;  // not the last edge of its run here
        const float total = c[k] + (key[k] == firstKey ? carryIn : 0.0f);
        if ((leftOpen && key[k] == blockFirst) || (rightOpen && key[k] == blockLast)) add_f32(&np[key[k]], total);
        else np[key[k]] = total;
    }
}

// pagerank/vertex_push.cu:16-30
template<typename Off>
__global__ __launch_bounds__(1024) void pr_vertex_push_kernel(uint64_t V, const Off *__restrict__ off,
                                                              const uint32_t *__restrict__ cols,
                                                              const float *__restrict__ pr, float *np)
{
    const uint64_t stride = static_cast<uint64_t>(blockDim.x) * gridDim.x;
    for (uint64_t v = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; v < V; v += stride) {
        const uint64_t s = off[v], e = off[v + 1];
        const uint32_t d = static_cast<uint32_t>(e - s);
        if (d == 0) continue;
        const float r = pr[v] / static_cast<float>(d);
        for (uint64_t j = s; j < e; j++) add_f32(&np[cols[j]], r);
    }
}

// ------------------------------------------------------------ pull forms

// Rows per workgroup of the pull kernels (one thread per row), and the
// in-edges whose contributions are staged in LDS per round.
constexpr uint32_t kPullRows = 256;
constexpr uint32_t kPullChunk = 2048;
constexpr uint32_t kPullPerThread = kPullChunk / kPullRows;
constexpr uint32_t kSumBatch = 32;     // LDS reads in flight in a short row's sequential sum
constexpr uint32_t kStrideBatch = 8;   // the same for a lane of a virtual warp

// The contribution one in-edge from u brings: pr[u] / deg[u] for the
// dividing variants (vertex_pull.cu:25, the warp form dividing by the
// degree read as int, vertex_pull_warp.cu:40), pr[u] itself for nodiv.
template<int DIV>
__device__ __forceinline__ float pull_contribution(const float *__restrict__ pr, const uint32_t *__restrict__ deg,
                                                  uint32_t u)
{
    if constexpr (DIV == 1) return pr[u] / static_cast<float>(deg[u]);
    else if constexpr (DIV == 2) return pr[u] / static_cast<float>(static_cast<int32_t>(deg[u]));
    else return pr[u];
}

// The pull iteration of pagerank/vertex_pull.cu:16-30, vertex_pull_nodiv.cu,
// vertex_pull_warp.cu:4-49 and vertex_pull_warp_nodiv.cu:4-47 for wave64:
// a workgroup owns kPullRows consecutive rows of the reverse CSR and streams
// their in-edges in rounds of kPullChunk.  All 256 threads gather a round's
// contributions (coalesced column reads, independent gathers) into LDS while
// the previous round is being summed, so a hub row no longer walks its
// in-list with one dependent load after another.
//
// W = 1 (vertex-pull, vertex-pull-nodiv): thread t sums row t alone, in CSR
// order, carrying its running sum from round to round -- the reference's
// sequential FP32 sum, bit for bit.  W > 1 (the _warp variants): the W lanes
// of a virtual warp take the row's in-edges in lane-strided order (lane l
// the edges at positions l, l + W, ... of the row, as the reference's lanes
// do) and their partials are combined by a shuffle tree where the reference
// adds them atomically, in no fixed order.  Rows go round-robin to the
// virtual warps; a round boundary cuts at most one row, whose partials the
// owning warp carries to the next round.
//
// Rows with more than long_degree in-edges are summed elsewhere
// (pull_long_rows).  The rounds run over the other rows' edges only: a
// compacted position c is the edge e0 + c + the long rows' edges before it,
// found among the workgroup's few long rows by binary search.  (Rounds over
// the stored edges that jumped from long row to long row held up R-MAT's
// first workgroups, where long and short rows alternate: at scale 20, edge
// factor 16, the short rows alone took 246 us per launch and 162 us since;
// spread_block took the whole launch from 192 to 137 us, the splits below to
// 113: 142 G gathers/s, where a table of the size of one XCD's L2 allows
// between 76 (16 MiB) and 216 (2 MiB).)
template<typename Off>
struct PullShortLds {
    float vals[2][kPullChunk];
    Off rowC[kPullRows + 1];  // compacted position of each row's first edge
    Off lpos[kPullRows];      // per long row: the compacted position it stands before,
    Off lskip[kPullRows];     // and the edges of the long rows up to and including it
    Off wsum[kPullRows / kWave];
    uint32_t wlong[kPullRows / kWave];
};

template<int DIV, int W, typename Off>
__device__ __forceinline__ void pull_short_rows(uint32_t block, PullShortLds<Off> &lds, uint64_t V,
                                                const Off *__restrict__ roff, const uint32_t *__restrict__ rcols,
                                                const uint32_t *__restrict__ deg, const float *__restrict__ pr,
                                                float *np, uint64_t long_degree)
{
    auto &vals = lds.vals;
    const Off *rowC = lds.rowC;
    constexpr uint32_t kWarps = kPullRows / W;
    const uint32_t t = threadIdx.x, wv = t / kWave;
    const uint64_t r0 = static_cast<uint64_t>(block) * kPullRows;
    const uint32_t nrows = static_cast<uint32_t>(V - r0 < kPullRows ? V - r0 : kPullRows);
    const uint32_t warp = t / W, lane = t % W;
    const Off e0 = roff[r0];
    Off rs = 0, re = 0;
    if (t < nrows) {
        rs = roff[r0 + t];
        re = roff[r0 + t + 1];
    }
    const bool isLong = static_cast<uint64_t>(re - rs) > long_degree;
    const Off len = isLong ? Off{0} : static_cast<Off>(re - rs);
    const Off incl = wave_prefix_sum(len);
    const uint64_t longs = __ballot(isLong);
    if ((t & (kWave - 1)) == kWave - 1) {
        lds.wsum[wv] = incl;
        lds.wlong[wv] = static_cast<uint32_t>(__popcll(longs));
    }
    __syncthreads();
    Off before = incl - len, total = 0;
    uint32_t nlong = 0;
    uint32_t li = static_cast<uint32_t>(__popcll(longs & ((1ull << (t & (kWave - 1))) - 1ull)));
#pragma unroll
    for (uint32_t w = 0; w < kPullRows / kWave; w++) {
        if (w < wv) {
            before += lds.wsum[w];
            li += lds.wlong[w];
        }
        total += lds.wsum[w];
        nlong += lds.wlong[w];
    }
    lds.rowC[t] = before;
    if (t == kPullRows - 1) lds.rowC[kPullRows] = total;
    if (isLong) {
        lds.lpos[li] = before;
        lds.lskip[li] = re - e0 - before;
    }
    // Rows without in-edges get an empty sum.
    if (t < nrows && rs == re) np[r0 + t] = 0.0f;
    __syncthreads();
    auto edge_of = [&](Off c) {
        uint32_t lo = 0, hi = nlong;  // the long rows standing before position c
        while (lo < hi) {
            const uint32_t m = (lo + hi) / 2;
            if (lds.lpos[m] <= c) lo = m + 1;
            else hi = m;
        }
        return static_cast<Off>(e0 + c + (lo ? lds.lskip[lo - 1] : Off{0}));
    };

    // Loads of one round into registers; stored to LDS after the previous
    // round's sums, so those sums overlap the gathers' latency.  The loads
    // are unconditional (positions past the round repeat its last edge) so
    // that all column loads, then all gathers, are in flight together.
    float reg[kPullPerThread];
    auto gather = [&](Off c0, Off c1) {
        uint32_t u[kPullPerThread];
#pragma unroll
        for (uint32_t k = 0; k < kPullPerThread; k++) {
            const Off c = c0 + k * kPullRows + t;
            u[k] = rcols[edge_of(c < c1 ? c : c1 - 1)];
        }
#pragma unroll
        for (uint32_t k = 0; k < kPullPerThread; k++) reg[k] = pull_contribution<DIV>(pr, deg, u[k]);
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (uint32_t k = 0; k < kPullPerThread; k++) vals[buf][k * kPullRows + t] = reg[k];
    };

    float carry = 0.0f;  // partial of this lane's row cut by the round boundary
    Off c0 = 0, c1 = min(static_cast<Off>(kPullChunk), total);
    if (c0 < total) {
        gather(c0, c1);
        stage(0);
    }
    __syncthreads();
    int buf = 0;
    while (c0 < total) {
        const Off n0 = c1, n1 = c1 + min(static_cast<Off>(kPullChunk), static_cast<Off>(total - c1));
        if (n0 < total) gather(n0, n1);
        const float *v = vals[buf];
        if constexpr (W == 1) {
            // Thread t owns row t.
            {
                const Off s = rowC[t], e = rowC[t + 1];
                const Off lo = s > c0 ? s : c0, hi = e < c1 ? e : c1;
                if (lo < hi) {
                    // In CSR order; the LDS reads of a batch are issued
                    // together, the adds stay sequential.
                    float acc = carry;
                    uint32_t j = static_cast<uint32_t>(lo - c0);
                    const uint32_t end = static_cast<uint32_t>(hi - c0);
                    for (; j + kSumBatch <= end; j += kSumBatch) {
                        float x[kSumBatch];
#pragma unroll
                        for (uint32_t k = 0; k < kSumBatch; k++) x[k] = v[j + k];
#pragma unroll
                        for (uint32_t k = 0; k < kSumBatch; k++) acc += x[k];
                    }
                    for (; j < end; j++) acc += v[j];
                    if (hi == e) np[r0 + t] = acc;
                    carry = hi == e ? 0.0f : acc;
                }
            }
        } else {
            // Rows overlapping the round: the first row whose end passes c0
            // up to the last row starting before c1 (binary searches in LDS).
            uint32_t lo = 0, hi = nrows;
            while (lo < hi) {
                const uint32_t m = (lo + hi) / 2;
                if (rowC[m + 1] <= c0) lo = m + 1;
                else hi = m;
            }
            const uint32_t ra = lo;
            hi = nrows;
            while (lo < hi) {
                const uint32_t m = (lo + hi) / 2;
                if (rowC[m] < c1) lo = m + 1;
                else hi = m;
            }
            const uint32_t rb = lo;  // rows [ra, rb) overlap the round
            const uint32_t first = ra + (warp + kWarps - ra % kWarps) % kWarps;
            for (uint32_t i = first; i < rb; i += kWarps) {
                const Off s = rowC[i], e = rowC[i + 1];
                if (s == e) continue;
                const Off a = s > c0 ? s : c0, b = e < c1 ? e : c1;
                // Lane l takes the row positions congruent to l modulo W.
                const uint32_t p0 = static_cast<uint32_t>((a - s) % W);
                uint32_t j = static_cast<uint32_t>(a - c0) + (lane + W - p0) % W;
                const uint32_t end = static_cast<uint32_t>(b - c0);
                float part = (a == s) ? 0.0f : carry;
                for (; j + (kStrideBatch - 1) * W < end; j += kStrideBatch * W) {
                    float x[kStrideBatch];
#pragma unroll
                    for (uint32_t k = 0; k < kStrideBatch; k++) x[k] = v[j + k * W];
#pragma unroll
                    for (uint32_t k = 0; k < kStrideBatch; k++) part += x[k];
                }
                for (; j < end; j += W) part += v[j];
                if (b == e) {
#pragma unroll
                    for (int o = W / 2; o > 0; o >>= 1) part += __shfl_xor(part, o, W);
                    if (lane == 0) np[r0 + i] = part;
                    carry = 0.0f;
                } else {
                    carry = part;
                }
            }
        }
        if (n0 < total) stage(buf ^ 1);
        __syncthreads();
        c0 = n0;
        c1 = n1;
        buf ^= 1;
    }
}

// ------------------------------------- sequential FP32 sums in parallel
//
// The reference adds a row's contributions one after another in FP32, and
// vertex-pull and vertex-pull-nodiv keep that sum bit for bit.  Written as
// a loop it is one dependent add per in-edge, and the longest rows of an
// R-MAT graph hold up the whole iteration (scale 20, edge factor 16: a row
// of 39585).  The same bits come out of a parallel sum: while the running sum stays in one binade [2^k, 2^(k+1)) it is an
// integer m of units u = 2^(k-23), and adding x >= 0 rounds to
// m + rne(x / u), where x's rounded quotient depends on m only when x / u
// is exactly halfway between two integers, and then only on m's parity.  So
// a group of values maps the parity p of the incoming m to an increment
// d[p], and such maps compose associatively.  The lanes hold consecutive
// values; a wave scan of their maps gives every lane's m, the first lane
// whose m leaves the binade (m >= 2^24) is added value by value, and the
// scan goes on behind it in the new binade.  A sum leaves its binade at most
// once per doubling, so the scans are about as many as the rounds.
// Values that are negative or NaN, and a running sum that is zero,
// subnormal or not finite, are added value by value too.

__device__ __forceinline__ float lane_f32(float x, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

constexpr int kSeqPerLane = 8;
constexpr uint32_t kSeqLimit = 1u << 24;  // m at which a sum has left its binade

// The increment of m (units 2^(e - 150) for a sum with exponent field e) by
// a lane's values, for an even and an odd incoming m.
struct SeqMap {
    uint32_t d0, d1;
};

__device__ __forceinline__ bool seq_normal(uint32_t bits)
{
    const uint32_t e = bits >> 23;  // the sign bit makes it >= 256
    return e >= 1 && e <= 254;
}

// The inclusive scan over the wave of the lanes' maps for the incoming sum's
// exponent field e; lanes below `first` add nothing.  Each value's quotient
// is capped at 2^24 and each lane's increment at 2^25: past the cap the sum
// has left the binade anyway, and 64 capped increments fit 32 bits.
__device__ __forceinline__ SeqMap seq_scan(const float (&x)[kSeqPerLane], uint32_t e, uint32_t first)
{
    const uint32_t lane = __lane_id();
    uint32_t q[kSeqPerLane];
    uint32_t ties = 0, sum = 0;
#pragma unroll
    for (int k = 0; k < kSeqPerLane; k++) {
        const float y = fminf(ldexpf(x[k], 150 - static_cast<int>(e)), 16777216.0f);
        const float f = floorf(y), r = y - f;  // exact
        q[k] = static_cast<uint32_t>(f) + (r > 0.5f ? 1u : 0u);
        ties |= (r == 0.5f ? 1u : 0u) << k;
        sum += q[k];
    }
    const bool live = lane >= first;
    if (__ballot(live && ties != 0) == 0) {
        const uint32_t d = wave_prefix_sum(live ? min(sum, 1u << 25) : 0u);
        return SeqMap{d, d};
    }
    SeqMap m{0, 0};
    if (live) {
#pragma unroll
        for (int k = 0; k < kSeqPerLane; k++) {
            const uint32_t tie = (ties >> k) & 1u;
            m.d0 += q[k] + (tie & ((m.d0 + q[k]) & 1u));
            m.d1 += q[k] + (tie & ((m.d1 + q[k] + 1u) & 1u));
        }
        m.d0 = min(m.d0, 1u << 25);
        m.d1 = min(m.d1, 1u << 25);
    }
    for (int o = 1; o < kWave; o <<= 1) {
        // the lanes before this one first: p -> a[p], then this one's map at
        // the parity p + a[p]
        const uint32_t a0 = __shfl_up(m.d0, static_cast<unsigned>(o), kWave);
        const uint32_t a1 = __shfl_up(m.d1, static_cast<unsigned>(o), kWave);
        if (static_cast<int>(lane) >= o)
            m = SeqMap{a0 + ((a0 & 1u) ? m.d1 : m.d0), a1 + ((a1 & 1u) ? m.d0 : m.d1)};
    }
    return m;
}

// acc after adding the wave's 512 values one by one in lane order, each
// lane's kSeqPerLane in theirs.  acc is the same in every lane, and every
// lane takes part.
__device__ __forceinline__ float seq_add_wave(float acc, const float (&x)[kSeqPerLane])
{
    bool plain = true;
#pragma unroll
    for (int k = 0; k < kSeqPerLane; k++) plain = plain && x[k] >= 0.0f;
    const bool allPlain = __ballot(!plain) == 0;
    uint32_t first = 0;
    while (first < kWave) {
        const uint32_t bits = __builtin_amdgcn_readfirstlane(__float_as_uint(acc));
        uint32_t serial = first;  // the lane to add value by value
        if (allPlain && seq_normal(bits)) {
            const uint32_t m = (bits & 0x7FFFFFu) | 0x800000u;
            const SeqMap f = seq_scan(x, bits >> 23, first);
            const uint32_t incl = (m & 1u) ? f.d1 : f.d0;
            const uint64_t over = __ballot(m + incl >= kSeqLimit);
            serial = over ? static_cast<uint32_t>(__builtin_ctzll(over)) : kWave;
            const uint32_t before =
                serial ? static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl), static_cast<int>(serial) - 1)) : 0u;
            acc = __uint_as_float((bits & 0xFF800000u) | ((m + before) & 0x7FFFFFu));
            if (serial == kWave) return acc;
        }
#pragma unroll
        for (int k = 0; k < kSeqPerLane; k++) acc += lane_f32(x[k], static_cast<int>(serial));
        first = serial + 1;
    }
    return acc;
}

// Rows with more than long_degree in-edges (listed by the pull plan), so
// that the hubs of a skewed graph are summed side by side rather than one
// after another by the workgroup owning their rows: one wave per row, or a
// whole workgroup for a row of more than kHugeDegree in-edges, whose four
// waves gather 2048 contributions per round where one wave's 512 would leave
// the row waiting on the latency of its rounds.  SEQ: the sum is the
// reference's sequential one, bit for bit (seq_add_wave).  Otherwise (the
// _warp variants) each lane keeps a partial and the partials meet in a
// tree -- the reference's per-lane partials and atomic adds in another,
// equally valid order.
constexpr uint32_t kLongWaves = 4;
constexpr uint32_t kLongPerLane = kSeqPerLane;
constexpr uint32_t kLongRound = kWave * kLongPerLane;
constexpr uint32_t kHugeRound = kLongWaves * kLongRound;

// Rows listed by the pull plan.
struct RowList {
    const uint32_t *rows = nullptr;
    uint32_t n = 0;
};

struct PullLongLds {
    float vals[kLongWaves][kLongRound];  // a wave's round, or the four waves' parts of a workgroup's
    uint32_t d0[kLongWaves], d1[kLongWaves], plain[kLongWaves];
    float sums[kLongWaves];
};

// The contributions of in-edges c0 + k * stride + t (k < kLongPerLane) of a
// row ending at e, all in flight together; 0 past the end (adding it
// changes no sum: the running sum is never -0).
template<int DIV>
__device__ __forceinline__ void long_gather(float (&x)[kLongPerLane], uint64_t c0, uint64_t e, uint32_t t,
                                            uint32_t stride, const uint32_t *__restrict__ rcols,
                                            const uint32_t *__restrict__ deg, const float *__restrict__ pr)
{
    uint32_t u[kLongPerLane];
#pragma unroll
    for (uint32_t k = 0; k < kLongPerLane; k++) {
        const uint64_t j = c0 + k * stride + t;
        u[k] = rcols[j < e ? j : e - 1];
    }
#pragma unroll
    for (uint32_t k = 0; k < kLongPerLane; k++) {
        const uint64_t j = c0 + k * stride + t;
        const float v = pull_contribution<DIV>(pr, deg, u[k]);
        x[k] = j < e ? v : 0.0f;
    }
}

// The lane's kSeqPerLane consecutive values of a staged round.
__device__ __forceinline__ void seq_values(float (&y)[kSeqPerLane], const float *v)
{
    const float4 *v4 = reinterpret_cast<const float4 *>(v + __lane_id() * kSeqPerLane);
    const float4 a = v4[0], b = v4[1];
    y[0] = a.x, y[1] = a.y, y[2] = a.z, y[3] = a.w;
    y[4] = b.x, y[5] = b.y, y[6] = b.z, y[7] = b.w;
}

template<int DIV, bool SEQ, typename Off>
__device__ __forceinline__ void pull_huge_row(uint32_t row, PullLongLds &lds, const Off *__restrict__ roff,
                                              const uint32_t *__restrict__ rcols, const uint32_t *__restrict__ deg,
                                              const float *__restrict__ pr, float *np)
{
    const uint32_t t = threadIdx.x, wv = t / kWave, lane = t & (kWave - 1);
    const uint64_t s = static_cast<uint64_t>(roff[row]), e = static_cast<uint64_t>(roff[row + 1]);
    float x[kLongPerLane];
    if constexpr (!SEQ) {
        float part = 0.0f;
        for (uint64_t c0 = s; c0 < e; c0 += kHugeRound) {
            long_gather<DIV>(x, c0, e, t, kPullRows, rcols, deg, pr);
#pragma unroll
            for (uint32_t k = 0; k < kLongPerLane; k++) part += x[k];
        }
        part = wave_sum_f32(part);
        if (lane == 0) lds.sums[wv] = part;
        __syncthreads();
        if (t == 0) {
            float total = 0.0f;
            for (uint32_t w = 0; w < kLongWaves; w++) total += lds.sums[w];
            np[row] = total;
        }
    } else {
        float *flat = lds.vals[0];
        float acc = 0.0f;  // the same in every thread
        long_gather<DIV>(x, s, e, t, kPullRows, rcols, deg, pr);
        for (uint64_t c0 = s; c0 < e; c0 += kHugeRound) {
#pragma unroll
            for (uint32_t k = 0; k < kLongPerLane; k++) flat[k * kPullRows + t] = x[k];
            __syncthreads();
            // The next round's gathers run under this round's sums.
            if (c0 + kHugeRound < e) long_gather<DIV>(x, c0 + kHugeRound, e, t, kPullRows, rcols, deg, pr);
            float y[kSeqPerLane];
            seq_values(y, lds.vals[wv]);
            // Each wave's map in the binade of the round's incoming sum.
            const uint32_t bits = __builtin_amdgcn_readfirstlane(__float_as_uint(acc));
            bool plain = true;
#pragma unroll
            for (int k = 0; k < kSeqPerLane; k++) plain = plain && y[k] >= 0.0f;
            const bool allPlain = __ballot(!plain) == 0 && seq_normal(bits);
            SeqMap f{0, 0};
            if (allPlain) f = seq_scan(y, bits >> 23, 0);
            if (lane == kWave - 1) {
                lds.d0[wv] = f.d0;
                lds.d1[wv] = f.d1;
                lds.plain[wv] = allPlain ? 1u : 0u;
            }
            __syncthreads();
            uint32_t m = (bits & 0x7FFFFFu) | 0x800000u;
            bool stays = true;
#pragma unroll
            for (uint32_t w = 0; w < kLongWaves; w++) {
                m += (m & 1u) ? lds.d1[w] : lds.d0[w];
                stays = stays && lds.plain[w] && m < kSeqLimit;
                m = min(m, kSeqLimit);
            }
            if (stays) {
                acc = __uint_as_float((bits & 0xFF800000u) | (m & 0x7FFFFFu));
            } else {
                // Every wave adds the four parts in order: the same sum in all.
                for (uint32_t w = 0; w < kLongWaves; w++) {
                    seq_values(y, lds.vals[w]);
                    acc = seq_add_wave(acc, y);
                }
            }
            __syncthreads();  // the staged round and the maps have been read
        }
        if (t == 0) np[row] = acc;
    }
}

template<int DIV, bool SEQ, typename Off>
__device__ __forceinline__ void pull_long_rows(uint32_t block, PullLongLds &lds, RowList huge, RowList longs,
                                               const Off *__restrict__ roff,
                                               const uint32_t *__restrict__ rcols, const uint32_t *__restrict__ deg,
                                               const float *__restrict__ pr, float *np)
{
    if (block < huge.n) {
        pull_huge_row<DIV, SEQ>(huge.rows[block], lds, roff, rcols, deg, pr, np);
        return;
    }
    const uint32_t wv = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const uint32_t i = (block - huge.n) * kLongWaves + wv;
    if (i >= longs.n) return;
    const uint32_t row = longs.rows[i];
    const uint64_t s = static_cast<uint64_t>(roff[row]), e = static_cast<uint64_t>(roff[row + 1]);
    float x[kLongPerLane];
    if constexpr (!SEQ) {
        float part = 0.0f;
        for (uint64_t c0 = s; c0 < e; c0 += kLongRound) {
            long_gather<DIV>(x, c0, e, lane, kWave, rcols, deg, pr);
#pragma unroll
            for (uint32_t k = 0; k < kLongPerLane; k++) part += x[k];
        }
        part = wave_sum_f32(part);
        if (lane == 0) np[row] = part;
    } else {
        float *v = lds.vals[wv];
        float acc = 0.0f;
        long_gather<DIV>(x, s, e, lane, kWave, rcols, deg, pr);
        for (uint64_t c0 = s; c0 < e; c0 += kLongRound) {
#pragma unroll
            for (uint32_t k = 0; k < kLongPerLane; k++) v[k * kWave + lane] = x[k];
            if (c0 + kLongRound < e) long_gather<DIV>(x, c0 + kLongRound, e, lane, kWave, rcols, deg, pr);
            // The wave's LDS writes ordered before its reads, and the reads
            // before the next round's writes.
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            float y[kSeqPerLane];
            seq_values(y, v);
            acc = seq_add_wave(acc, y);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        }
        if (lane == 0) np[row] = acc;
    }
}

// c[v] = pr[v] / deg[v] (zero without out-edges): the value every
// out-edge of v carries in the dividing variants.  Computing it once per
// vertex instead of once per edge gives the same IEEE quotient, so the sums
// that gather it are the reference's bit for bit, with one gather per edge
// instead of two.  INT: the degree read as int (vertex_pull_warp.cu:40).
template<bool INT>
__global__ __launch_bounds__(256) void pr_contrib_kernel(uint64_t V, const uint32_t *__restrict__ deg,
                                                         const float *__restrict__ pr, float *c)
{
    const uint64_t stride = static_cast<uint64_t>(blockDim.x) * gridDim.x;
    for (uint64_t v = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; v < V; v += stride) {
        const uint32_t d = deg[v];
        const float q = INT ? pr[v] / static_cast<float>(static_cast<int32_t>(d)) : pr[v] / static_cast<float>(d);
        c[v] = d != 0 ? q : 0.0f;
    }
}

// One launch of a pull iteration: workgroups [0, long_blocks) sum the long
// rows (those of a whole workgroup first, each class in any order), so that
// they start at once; the others one block of kPullRows rows each.
template<int DIV, int W, typename Off>
__global__ __launch_bounds__(kPullRows) void pr_pull_kernel(uint64_t V, const Off *__restrict__ roff,
                                                             const uint32_t *__restrict__ rcols,
                                                             const uint32_t *__restrict__ deg,
                                                             const float *__restrict__ pr, float *np,
                                                             uint64_t long_degree, RowList huge, RowList longs,
                                                             uint32_t long_blocks, ReducePrev prev)
{
    static_assert(kLongWaves * kWave == kPullRows, "both parts use the same workgroup");
    __shared__ union alignas(16) {
        PullShortLds<Off> s;
        PullLongLds l;
        ReduceLds r;
    } lds;
    if (reduce_prev<kPullRows>(prev, lds.r)) return;
    const uint32_t blocks = gridDim.x - (prev.part ? 1u : 0u);
    if (blockIdx.x < long_blocks)
        pull_long_rows<DIV, W == 1, Off>(blockIdx.x, lds.l, huge, longs, roff, rcols, deg, pr, np);
    else
        pull_short_rows<DIV, W, Off>(spread_block(blockIdx.x - long_blocks, blocks - long_blocks), lds.s, V, roff,
                                     rcols, deg, pr, np, long_degree);
}

// The long rows of a reverse CSR, rows whose in-degree exceeds `threshold`:
// those past `huge` from the front of rows[0, cap), the others from its
// back, in any order; count[0] and count[1] of them.  A workgroup takes
// 1024 consecutive vertices and reserves its slots with one atomic per list.
constexpr uint32_t kListRows = 1024;

template<typename Off>
__global__ __launch_bounds__(256) void pr_long_rows_kernel(uint64_t V, const Off *__restrict__ roff,
                                                           uint64_t threshold, uint64_t huge, uint64_t cap,
                                                           uint32_t *rows, uint32_t *count)
{
    __shared__ uint32_t n[2], base[2];
    if (threadIdx.x < 2) n[threadIdx.x] = 0;
    __syncthreads();
    constexpr int kPer = kListRows / 256;
    uint32_t pos[kPer];
    int list[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const uint64_t v = static_cast<uint64_t>(blockIdx.x) * kListRows + k * 256 + threadIdx.x;
        list[k] = -1;
        if (v < V) {
            const uint64_t d = static_cast<uint64_t>(roff[v + 1]) - static_cast<uint64_t>(roff[v]);
            if (d > threshold) list[k] = d > huge ? 0 : 1;
        }
        if (list[k] >= 0) pos[k] = atomicAdd(&n[list[k]], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 2 && n[threadIdx.x]) base[threadIdx.x] = atomicAdd(&count[threadIdx.x], n[threadIdx.x]);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const uint32_t v = static_cast<uint32_t>(static_cast<uint64_t>(blockIdx.x) * kListRows + k * 256 + threadIdx.x);
        if (list[k] == 0) rows[base[0] + pos[k]] = v;
        if (list[k] == 1) rows[cap - 1 - (base[1] + pos[k])] = v;
    }
}

template<typename Off>
__host__ __device__ inline uint32_t pr_warp_vals_bytes(uint32_t warps, uint32_t chunk)
{ return (warps * chunk * 4u + 7u) & ~7u; }

template<typename Off>
__host__ __device__ inline uint32_t pr_warp_lds_bytes(uint32_t warps, uint32_t chunk)
{ return pr_warp_vals_bytes<Off>(warps, chunk) + warps * (chunk + 1) * static_cast<uint32_t>(sizeof(Off)); }

// pagerank/vertex_push_warp.cu:4-49: chunk ranks and offsets staged in LDS,
// lanes stride over each vertex's out-edges with float atomics.
template<typename Off>
__global__ __launch_bounds__(1024) void pr_vertex_push_warp_kernel(uint32_t W, uint32_t C, uint64_t V,
                                                                   const Off *__restrict__ off,
                                                                   const uint32_t *__restrict__ cols,
                                                                   const float *__restrict__ pr, float *np)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const uint32_t warps = blockDim.x / W;
    const uint32_t bw = threadIdx.x / W, lane = threadIdx.x % W;
    float *myRanks = reinterpret_cast<float *>(lds_raw) + bw * C;
    Off *myOff = reinterpret_cast<Off *>(lds_raw + pr_warp_vals_bytes<Off>(warps, C)) + bw * (C + 1);
    const uint64_t warpId = (static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / W;
    const uint64_t totalWarps = static_cast<uint64_t>(warps) * gridDim.x;
    for (uint64_t chunk = warpId; chunk * C < V; chunk += totalWarps) {
        const uint64_t base = chunk * C;
        const uint32_t end = static_cast<uint32_t>(std::min<uint64_t>(C, V - base));
        for (uint32_t i = lane; i < end; i += W) myRanks[i] = pr[base + i];
        for (uint32_t i = lane; i <= end; i += W) myOff[i] = off[base + i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        for (uint32_t v = 0; v < end; v++) {
            const uint64_t s = myOff[v];
            const uint32_t n = static_cast<uint32_t>(myOff[v + 1] - s);
            if (n == 0) continue;
            const float r = myRanks[v] / static_cast<float>(n);
            for (uint32_t i = lane; i < n; i += W) add_f32(&np[cols[s + i]], r);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// ------------------------------------------------------------ consolidate

__global__ __launch_bounds__(1024) void pr_consolidate_kernel(uint64_t V, const uint32_t *__restrict__ deg,
                                                              float *pr, float *np, int notLast, int nodiv,
                                                              int mode, const double *__restrict__ dangling,
                                                              double *resid)
{
    __shared__ double lds[1024 / kWave];
    const uint64_t stride = static_cast<uint64_t>(blockDim.x) * gridDim.x;
    const double d = static_cast<double>(kDamp);
    const double D = (mode == BW_PR_DANGLING_UNIFORM && dangling) ? *dangling : 0.0;
    // pagerank/pagerank.cu:154: (1 - dampening) / size in float.
    const float baseF = (1.0f - kDamp) / static_cast<float>(V);
    // pagerank/pagerank.cu:132: (1.0 - dampening) / size in double.
    const double baseD = (1.0 - d) / static_cast<double>(V);
    double diff = 0.0;
    for (uint64_t v = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; v < V; v += stride) {
        const float acc = np[v];
        float nr;
        if (mode == BW_PR_DANGLING_DROP) {
            if (nodiv) nr = __builtin_fmaf(kDamp, acc, baseF);
            else nr = static_cast<float>(baseD + static_cast<double>(kDamp * acc));
        } else {
            nr = static_cast<float>(baseD + d * (static_cast<double>(acc) + D / static_cast<double>(V)));
        }
        const float old = pr[v];
        const uint32_t dv = (nodiv || mode == BW_PR_DANGLING_UNIFORM) && deg ? deg[v] : 0u;
        double oldRank = static_cast<double>(old);
        if (nodiv && mode == BW_PR_DANGLING_UNIFORM && dv != 0) oldRank *= static_cast<double>(dv);
        diff += fabs(static_cast<double>(nr) - oldRank);
        pr[v] = (nodiv && dv != 0 && notLast) ? nr / static_cast<float>(dv) : nr;
        np[v] = 0.0f;
    }
    if (resid) {
        const double t = block_sum_f64(diff, lds);
        if (threadIdx.x == 0) add_f64(resid, t);
    }
}

__global__ __launch_bounds__(1024) void pr_dangling_kernel(uint64_t V, const uint32_t *__restrict__ deg,
                                                           const float *__restrict__ pr, double *out)
{
    __shared__ double lds[1024 / kWave];
    const uint64_t stride = static_cast<uint64_t>(blockDim.x) * gridDim.x;
    double acc = 0.0;
    for (uint64_t v = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; v < V; v += stride)
        if (deg[v] == 0) acc += static_cast<double>(pr[v]);
    const double t = block_sum_f64(acc, lds);
    if (threadIdx.x == 0 && t != 0.0) add_f64(out, t);
}

// What bw_pr_run does between two iterations' sums, in one pass over the
// vertices: consolidateRank / consolidateRankNoDiv (the arithmetic of
// pr_consolidate_kernel), the contributions the next iteration gathers
// (pr_contrib_kernel) and the dangling mass of the new ranks
// (pr_dangling_kernel).  Each workgroup leaves its (residual, dangling mass)
// in part[]; the next launch's extra workgroup adds them up in a fixed
// order, where one atomic per workgroup on one address took most of a pass
// (R-MAT scale 20: consolidate 11.0 us, contributions 5.4 us, now 8.1 us
// together; 20 bytes per vertex are 4.3 us of HBM).
struct FinishArgs {
    uint64_t V;
    const uint32_t *deg;      // out-degrees; NULL: nothing reads the dangling mass or the contributions
    float *pr;
    float *np;                // the sums
    float *contrib;           // NULL: nothing gathers contributions
    const double *dangling;   // UNIFORM: the mass of the ranks just gathered
    double2 *part;
    int not_last, nodiv, mode;
    int zero_np;              // the next sums are added to np
    int int_degree;           // contributions divide by the degree read as int (vertex_pull_warp.cu:40)
};

constexpr uint32_t kFinishThreads = 256;
constexpr uint32_t kFinishGrid = 4096;  // most workgroups (and partials)

// Vertices per thread and step: four, whose loads are in flight together;
// one where each vertex's sum is a chain of its own.
constexpr int finish_per_thread(bool gathered) { return gathered ? 1 : 4; }

__device__ __forceinline__ float contribution_of(float rank, uint32_t d, int int_degree)
{
    if (d == 0) return 0.0f;
    return int_degree ? rank / static_cast<float>(static_cast<int32_t>(d)) : rank / static_cast<float>(d);
}

// The workgroup's partial, in a fixed order.
__device__ __forceinline__ void store_partial(double2 *part, double resid, double dangl, ReduceLds &lds)
{
    resid = wave_sum_f64(resid);
    dangl = wave_sum_f64(dangl);
    if ((threadIdx.x & (kWave - 1)) == 0) {
        lds.red[threadIdx.x / kWave][0] = resid;
        lds.red[threadIdx.x / kWave][1] = dangl;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = 0.0, g = 0.0;
        for (uint32_t w = 0; w < kFinishThreads / kWave; w++) {
            r += lds.red[w][0];
            g += lds.red[w][1];
        }
        part[blockIdx.x] = make_double2(r, g);
    }
}

// GATHERED: the sums are the scatter layout's partials, not np.
template<bool GATHERED>
__global__ __launch_bounds__(kFinishThreads) void pr_finish_kernel(FinishArgs a, ScatterSums sums)
{
    __shared__ ReduceLds red;
    const double d = static_cast<double>(kDamp);
    const double D = a.mode == BW_PR_DANGLING_UNIFORM ? *a.dangling : 0.0;
    const float baseF = (1.0f - kDamp) / static_cast<float>(a.V);
    const double baseD = (1.0 - d) / static_cast<double>(a.V);
    double resid = 0.0, dangl = 0.0;
    constexpr int kPer = finish_per_thread(GATHERED);
    for (uint64_t b0 = static_cast<uint64_t>(blockIdx.x) * kPer * kFinishThreads; b0 < a.V;
         b0 += static_cast<uint64_t>(gridDim.x) * kPer * kFinishThreads) {
        float acc[kPer], old[kPer];
        uint32_t dv[kPer];
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const uint64_t v = b0 + k * kFinishThreads + threadIdx.x;
            const uint64_t w = v < a.V ? v : a.V - 1;
            old[k] = a.pr[w];
            dv[k] = a.deg ? a.deg[w] : 1u;
            acc[k] = GATHERED ? sums.row_sum(static_cast<uint32_t>(w)) : a.np[w];
        }
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const uint64_t v = b0 + k * kFinishThreads + threadIdx.x;
            if (v >= a.V) continue;
            float nr;
            if (a.mode == BW_PR_DANGLING_DROP) {
                if (a.nodiv) nr = __builtin_fmaf(kDamp, acc[k], baseF);
                else nr = static_cast<float>(baseD + static_cast<double>(kDamp * acc[k]));
            } else {
                nr = static_cast<float>(baseD + d * (static_cast<double>(acc[k]) + D / static_cast<double>(a.V)));
            }
            double oldRank = static_cast<double>(old[k]);
            if (a.nodiv && a.mode == BW_PR_DANGLING_UNIFORM && dv[k] != 0) oldRank *= static_cast<double>(dv[k]);
            resid += fabs(static_cast<double>(nr) - oldRank);
            if (dv[k] == 0) dangl += static_cast<double>(nr);
            a.pr[v] = (a.nodiv && dv[k] != 0 && a.not_last) ? nr / static_cast<float>(dv[k]) : nr;
            if (a.contrib && a.not_last) a.contrib[v] = contribution_of(nr, dv[k], a.int_degree);
            if (a.zero_np) a.np[v] = 0.0f;
        }
    }
    store_partial(a.part, resid, dangl, red);
}

// The initial ranks (1/V, pagerank/pagerank.cpp:88), divided by the
// out-degree when the nodiv variants start so, their contributions and the
// dangling mass partials; np starts at zero.
__global__ __launch_bounds__(kFinishThreads) void pr_start_kernel(FinishArgs a, int predivide)
{
    __shared__ ReduceLds red;
    const float init = 1.0f / static_cast<float>(a.V);
    double dangl = 0.0;
    for (uint64_t v = static_cast<uint64_t>(blockIdx.x) * kFinishThreads + threadIdx.x; v < a.V;
         v += static_cast<uint64_t>(gridDim.x) * kFinishThreads) {
        const uint32_t d = a.deg ? a.deg[v] : 1u;
        a.pr[v] = (predivide && d != 0) ? init / static_cast<float>(d) : init;
        if (a.contrib) a.contrib[v] = contribution_of(init, d, a.int_degree);
        a.np[v] = 0.0f;
        if (d == 0) dangl += static_cast<double>(init);
    }
    store_partial(a.part, 0.0, dangl, red);
}

// The reduction of an extra workgroup as a launch: after the last iteration,
// and before a pass over the vertices when no launch went before it.
__global__ __launch_bounds__(256) void pr_reduce_prev_kernel(ReducePrev p)
{
    __shared__ ReduceLds red;
    (void)reduce_prev<256>(p, red);
}

// ------------------------------------------------------------ host glue

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Workgroups of the kernels that end in one FP64 atomic add per workgroup
// (residual, dangling mass): two per CU unless the caller fixed the grid.
// Those adds all hit one address and serialise; 16384 of them cost 200 us
// on MI355X, the grid-stride loop over more vertices per thread almost
// nothing.
uint32_t reduction_grid(const bw_launch *cfg, uint32_t grid)
{
    if (cfg && cfg->grid) return grid;
    return std::min<uint32_t>(grid, 2u * static_cast<uint32_t>(device_cus()));
}

template<typename F>
int with_offsets(const void *off, int32_t ob, F &&f)
{
    if (ob == 4) return f(static_cast<const uint32_t *>(off));
    if (ob == 8) return f(static_cast<const uint64_t *>(off));
    return fail(BW_HIP_ERR_ARG, "offset_bytes must be 4 or 8");
}

int warp_params(const bw_launch *cfg, uint32_t &W, uint32_t &C)
{
    W = (cfg && cfg->warp) ? cfg->warp : 32;
    C = (cfg && cfg->chunk) ? cfg->chunk : 32;
    if (W == 0 || W > 64 || (W & (W - 1)))
        return fail(BW_HIP_ERR_ARG, "Warp size should be a power of 2 no larger than 64!");
    if (C % W != 0) return fail(BW_HIP_ERR_ARG, "Chunk size should be a multiple of warp size!");
    return BW_HIP_OK;
}

}  // namespace
}  // namespace bw

using namespace bw;

extern "C" int bw_pr_zero_degrees(uint64_t V, uint32_t *deg, const bw_launch *cfg)
{
    if (V && !deg) return fail(BW_HIP_ERR_ARG, "degrees must be a device pointer");
    return bw_hip_fill_u32(deg, 0u, V, cfg ? cfg->stream : nullptr);
}

extern "C" int bw_pr_degrees_edge_list(uint64_t E, const uint32_t *origins, uint32_t *deg, const bw_launch *cfg)
{
    if (E == 0) return BW_HIP_OK;
    if (!origins || !deg) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    const uint32_t block = 256, grid = degree_grid(E);
    hipLaunchKernelGGL(pr_degrees_runs_kernel<1>, dim3(grid), dim3(block), 0, stream_of(cfg), E, origins, 0, deg);
    BW_LAUNCH_CHECK();
    return BW_HIP_OK;
}

extern "C" int bw_pr_degrees_struct_edge_list(uint64_t E, const uint32_t *edges, int32_t reverse, uint32_t *deg,
                                              const bw_launch *cfg)
{
    if (E == 0) return BW_HIP_OK;
    if (!edges || !deg) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    const uint32_t block = 256, grid = degree_grid(E);
    hipLaunchKernelGGL(pr_degrees_runs_kernel<2>, dim3(grid), dim3(block), 0, stream_of(cfg), E, edges,
                       reverse ? 1 : 0, deg);
    BW_LAUNCH_CHECK();
    return BW_HIP_OK;
}

extern "C" int bw_pr_degrees_csr(uint64_t V, const void *off, int32_t ob, uint32_t *deg, const bw_launch *cfg)
{
    if (V == 0) return BW_HIP_OK;
    if (!off || !deg) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    uint32_t block, grid;
    BW_TRY(resolve_geometry(cfg, V, block, grid));
    return with_offsets(off, ob, [&](auto *o) {
        using Off = std::remove_const_t<std::remove_pointer_t<decltype(o)>>;
        hipLaunchKernelGGL((pr_degrees_csr_kernel<Off>), dim3(grid), dim3(block), 0, stream_of(cfg), V, o, deg);
        BW_LAUNCH_CHECK();
        return BW_HIP_OK;
    });
}

extern "C" int bw_pr_degrees_rev_csr(uint64_t V, const void *roff, int32_t ob, const uint32_t *rcols,
                                     uint32_t *deg, const bw_launch *cfg)
{
    // reverseCSRComputeDegrees counts each source once per reverse-CSR
    // entry; the entries are rcols[0 .. roff[V]), so the count runs over the
    // column array directly, edge-parallel.
    if (V == 0) return BW_HIP_OK;
    if (!roff || !rcols || !deg) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    uint64_t E = 0;
    if (ob == 4) {
        uint32_t e32 = 0;
        BW_HIP_CHECK(hipMemcpy(&e32, static_cast<const uint32_t *>(roff) + V, 4, hipMemcpyDeviceToHost));
        E = e32;
    } else if (ob == 8) {
        BW_HIP_CHECK(hipMemcpy(&E, static_cast<const uint64_t *>(roff) + V, 8, hipMemcpyDeviceToHost));
    } else {
        return fail(BW_HIP_ERR_ARG, "offset_bytes must be 4 or 8");
    }
    return bw_pr_degrees_edge_list(E, rcols, deg, cfg);
}

extern "C" int bw_pr_edge_list(uint64_t E, const uint32_t *in, const uint32_t *out, const uint32_t *deg,
                               const float *pr, float *np, const bw_launch *cfg)
{
    if (E == 0) return BW_HIP_OK;
    if (!in || !out || !deg || !pr || !np) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    const int vec = aligned16(in) && aligned16(out);
    uint32_t block, grid;
    BW_TRY(resolve_geometry(cfg, vec ? (E + 3) / 4 : E, block, grid));
    hipLaunchKernelGGL(pr_edge_list_kernel<false>, dim3(grid), dim3(block), 0, stream_of(cfg), E, in, out, deg, pr,
                       np, vec);
    BW_LAUNCH_CHECK();
    return BW_HIP_OK;
}

// Launches the segmented reverse edge-list kernel: one 256-thread workgroup
// per 4096 edges (its fixed geometry; cfg's block and grid do not apply).
template<bool AOS, bool PRE = false>
static int launch_rev_segmented(uint64_t E, const uint32_t *a, const uint32_t *b, const uint32_t *deg,
                                const float *pr, float *np, hipStream_t s, const ReducePrev &prev = {})
{
    const uint64_t blocks = (E + kSegBlockEdges - 1) / kSegBlockEdges;
    if (blocks >= 0x7FFFFFFFull) return fail(BW_HIP_ERR_ARG, "too many edges for the reverse edge-list kernel");
    const int vec = aligned16(a) && (AOS || aligned16(b));
    hipLaunchKernelGGL((pr_rev_segmented_kernel<AOS, PRE>), dim3(static_cast<uint32_t>(blocks) + (prev.part ? 1u : 0u)),
                       dim3(kSegThreads), 0, s, E, a, b, deg, pr, np, vec, prev);
    BW_LAUNCH_CHECK();
    return BW_HIP_OK;
}

extern "C" int bw_pr_rev_edge_list(uint64_t E, const uint32_t *in, const uint32_t *out, const uint32_t *deg,
                                   const float *pr, float *np, const bw_launch *cfg)
{
    if (E == 0) return BW_HIP_OK;
    if (!in || !out || !deg || !pr || !np) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    return launch_rev_segmented<false>(E, in, out, deg, pr, np, stream_of(cfg));
}

static int struct_entry(bool rev, uint64_t E, const uint32_t *edges, const uint32_t *deg, const float *pr,
                        float *np, const bw_launch *cfg)
{
    if (E == 0) return BW_HIP_OK;
    if (!edges || !deg || !pr || !np) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    if (rev) return launch_rev_segmented<true>(E, edges, nullptr, deg, pr, np, stream_of(cfg));
    const int vec = aligned16(edges);
    uint32_t block, grid;
    BW_TRY(resolve_geometry(cfg, vec ? (E + 1) / 2 : E, block, grid));
    hipLaunchKernelGGL(pr_struct_edge_list_kernel<false>, dim3(grid), dim3(block), 0, stream_of(cfg), E, edges, deg,
                       pr, np, vec);
    BW_LAUNCH_CHECK();
    return BW_HIP_OK;
}

extern "C" int bw_pr_struct_edge_list(uint64_t E, const uint32_t *edges, const uint32_t *deg, const float *pr,
                                      float *np, const bw_launch *cfg)
{ return struct_entry(false, E, edges, deg, pr, np, cfg); }

extern "C" int bw_pr_rev_struct_edge_list(uint64_t E, const uint32_t *edges, const uint32_t *deg, const float *pr,
                                          float *np, const bw_launch *cfg)
{ return struct_entry(true, E, edges, deg, pr, np, cfg); }

extern "C" int bw_pr_vertex_push(uint64_t V, const void *off, int32_t ob, const uint32_t *cols, const float *pr,
                                 float *np, const bw_launch *cfg)
{
    if (V == 0) return BW_HIP_OK;
    if (!off || !cols || !pr || !np) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    uint32_t block, grid;
    BW_TRY(resolve_geometry(cfg, V, block, grid));
    return with_offsets(off, ob, [&](auto *o) {
        using Off = std::remove_const_t<std::remove_pointer_t<decltype(o)>>;
        hipLaunchKernelGGL((pr_vertex_push_kernel<Off>), dim3(grid), dim3(block), 0, stream_of(cfg), V, o, cols, pr,
                           np);
        BW_LAUNCH_CHECK();
        return BW_HIP_OK;
    });
}

// Launches the chunked pull kernel: one 256-thread workgroup per 256 rows
// (the kernel's fixed geometry; cfg's block and grid do not apply), W lanes
// per row.
template<int DIV, int W>
static int launch_pull(uint64_t V, const void *roff, int32_t ob, const uint32_t *rcols, const uint32_t *deg,
                       const float *pr, float *np, hipStream_t s, uint64_t long_degree = ~0ull,
                       RowList huge = {}, RowList longs = {}, const ReducePrev &prev = {})
{
    const uint64_t blocks = (V + kPullRows - 1) / kPullRows;
    if (blocks > 0x7FFFFFFFull) return fail(BW_HIP_ERR_ARG, "too many vertices for the pull kernel");
    return with_offsets(roff, ob, [&](auto *o) {
        using Off = std::remove_const_t<std::remove_pointer_t<decltype(o)>>;
        const uint64_t long_blocks = static_cast<uint64_t>(huge.n) + (longs.n + kLongWaves - 1) / kLongWaves;
        if (blocks + long_blocks >= 0x7FFFFFFFull) return fail(BW_HIP_ERR_ARG, "too many vertices for the pull kernel");
        hipLaunchKernelGGL((pr_pull_kernel<DIV, W, Off>), dim3(static_cast<uint32_t>(blocks + long_blocks) + (prev.part ? 1u : 0u)), dim3(kPullRows), 0, s, V, o, rcols, deg, pr, np, long_degree, huge, longs,
                           static_cast<uint32_t>(long_blocks), prev);
        BW_LAUNCH_CHECK();
        return BW_HIP_OK;
    });
}

template<bool DIV>
static int pull_entry(uint64_t V, const void *roff, int32_t ob, const uint32_t *rcols, const uint32_t *deg,
                      const float *pr, float *np, const bw_launch *cfg)
{
    if (V == 0) return BW_HIP_OK;
    if (!roff || !rcols || !pr || !np || (DIV && !deg)) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    return launch_pull<DIV ? 1 : 0, 1>(V, roff, ob, rcols, deg, pr, np, stream_of(cfg));
}

// Rows with more in-edges than this are summed one wave each
// (pull_long_rows): beyond it, one thread's sequential sum of a row would
// hold up the workgroup owning it (R-MAT scale 20, edge factor 16: a pull
// launch takes 137 us with a split at 64, 119 at 128, 139 at 256).
constexpr uint64_t kLongDegree = 128;
// Rows with more in-edges than this get a whole workgroup (pull_huge_row;
// the same launch: 120 us with a split at 2048, 119 at 4096, 113 at 8192).
constexpr uint64_t kHugeDegree = 8192;

struct bw_pr_pull_plan {
    uint64_t V = 0;
    const void *roff = nullptr;
    int32_t ob = 4;
    uint32_t *rows = nullptr;
    RowList huge, longs;       // rows past kHugeDegree, and the others past kLongDegree
    float *contrib = nullptr;  // per-vertex contributions of the dividing variants
    ~bw_pr_pull_plan()
    {
        if (rows) (void)hipFree(rows);
        if (contrib) (void)hipFree(contrib);
    }
};

extern "C" int bw_pr_pull_plan_create(bw_pr_pull_plan **out, uint64_t V, const void *roff, int32_t ob, void *stream)
{
    if (!out) return fail(BW_HIP_ERR_ARG, "bw_pr_pull_plan_create: out is NULL");
    *out = nullptr;
    if (V && !roff) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    if (ob != 4 && ob != 8) return fail(BW_HIP_ERR_ARG, "offset_bytes must be 4 or 8");
    if (V > 0xFFFFFFFFull) return fail(BW_HIP_ERR_ARG, "the pull plan holds 32-bit row ids");
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto plan = std::make_unique<bw_pr_pull_plan>();
    plan->V = V, plan->roff = roff, plan->ob = ob;
    if (V) {
        uint64_t E = 0;
        if (ob == 4) {
            uint32_t e32 = 0;
            BW_HIP_CHECK(hipMemcpyAsync(&e32, static_cast<const uint32_t *>(roff) + V, 4, hipMemcpyDeviceToHost, s));
            BW_HIP_CHECK(hipStreamSynchronize(s));
            E = e32;
        } else {
            BW_HIP_CHECK(hipMemcpyAsync(&E, static_cast<const uint64_t *>(roff) + V, 8, hipMemcpyDeviceToHost, s));
            BW_HIP_CHECK(hipStreamSynchronize(s));
        }
        // At most E / (kLongDegree + 1) rows can exceed the threshold; the
        // two counts live in the slots after them.
        const uint64_t cap = E / (kLongDegree + 1);
        const uint64_t blocks = (V + kListRows - 1) / kListRows;
        if (blocks > 0x7FFFFFFFull) return fail(BW_HIP_ERR_ARG, "too many vertices for the pull plan");
        if (cap) {
            BW_HIP_CHECK(hipMalloc(&plan->rows, sizeof(uint32_t) * (cap + 2)));
            uint32_t *count = plan->rows + cap;
            BW_TRY(bw_hip_fill_u32(count, 0u, 2, s));
            BW_TRY(with_offsets(roff, ob, [&](auto *o) {
                hipLaunchKernelGGL(pr_long_rows_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, s, V, o,
                                   kLongDegree, kHugeDegree, cap, plan->rows, count);
                BW_LAUNCH_CHECK();
                return BW_HIP_OK;
            }));
            uint32_t n[2] = {0, 0};
            BW_HIP_CHECK(hipMemcpyAsync(n, count, sizeof n, hipMemcpyDeviceToHost, s));
            BW_HIP_CHECK(hipStreamSynchronize(s));
            plan->huge = RowList{plan->rows, n[0]};
            plan->longs = RowList{plan->rows + (cap - n[1]), n[1]};
        }
    }
    if (V) BW_HIP_CHECK(hipMalloc(&plan->contrib, sizeof(float) * V));
    *out = plan.release();
    return BW_HIP_OK;
}

extern "C" int bw_pr_pull_plan_destroy(bw_pr_pull_plan *plan)
{
    delete plan;
    return BW_HIP_OK;
}

extern "C" int bw_pr_pull_plan_info(const bw_pr_pull_plan *plan, uint32_t *long_rows)
{
    if (!plan) return fail(BW_HIP_ERR_ARG, "plan is NULL");
    if (long_rows) *long_rows = plan->huge.n + plan->longs.n;
    return BW_HIP_OK;
}

static bool pull_variant(int32_t variant)
{
    return variant == BW_PR_VERTEX_PULL || variant == BW_PR_VERTEX_PULL_NODIV || variant == BW_PR_VERTEX_PULL_WARP ||
           variant == BW_PR_VERTEX_PULL_WARP_NODIV;
}

// The sums of one pull iteration: np[v] = the sum of c over v's in-neighbours.
static int pull_sums(const bw_pr_pull_plan *plan, int32_t variant, const uint32_t *rcols, const float *c, float *np,
                     const bw_launch *cfg, const ReducePrev &prev)
{
    const uint64_t V = plan->V;
    hipStream_t s = stream_of(cfg);
    const void *ro = plan->roff;
    const int32_t ob = plan->ob;
    const RowList huge = plan->huge, longs = plan->longs;
    uint32_t W = 1, C = 1;
    if (variant == BW_PR_VERTEX_PULL_WARP || variant == BW_PR_VERTEX_PULL_WARP_NODIV) BW_TRY(warp_params(cfg, W, C));
    switch (W) {
    case 1: return launch_pull<0, 1>(V, ro, ob, rcols, nullptr, c, np, s, kLongDegree, huge, longs, prev);
    case 2: return launch_pull<0, 2>(V, ro, ob, rcols, nullptr, c, np, s, kLongDegree, huge, longs, prev);
    case 4: return launch_pull<0, 4>(V, ro, ob, rcols, nullptr, c, np, s, kLongDegree, huge, longs, prev);
    case 8: return launch_pull<0, 8>(V, ro, ob, rcols, nullptr, c, np, s, kLongDegree, huge, longs, prev);
    case 16: return launch_pull<0, 16>(V, ro, ob, rcols, nullptr, c, np, s, kLongDegree, huge, longs, prev);
    case 32: return launch_pull<0, 32>(V, ro, ob, rcols, nullptr, c, np, s, kLongDegree, huge, longs, prev);
    default: return launch_pull<0, 64>(V, ro, ob, rcols, nullptr, c, np, s, kLongDegree, huge, longs, prev);
    }
}

extern "C" int bw_pr_pull_iteration(const bw_pr_pull_plan *plan, int32_t variant, const uint32_t *rcols,
                                    const uint32_t *deg, const float *pr, float *np, const bw_launch *cfg)
{
    if (!plan) return fail(BW_HIP_ERR_ARG, "plan is NULL");
    const uint64_t V = plan->V;
    if (V == 0) return BW_HIP_OK;
    const bool div = variant == BW_PR_VERTEX_PULL || variant == BW_PR_VERTEX_PULL_WARP;
    if (!rcols || !pr || !np || (div && !deg)) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    if (!pull_variant(variant)) return fail(BW_HIP_ERR_ARG, "bw_pr_pull_iteration takes the four pull variants");
    if (div) {
        // The dividing variants gather per-vertex contributions computed here.
        hipStream_t s = stream_of(cfg);
        const uint64_t blocks = std::min<uint64_t>((V + 255) / 256, 8ull * device_cus());
        if (variant == BW_PR_VERTEX_PULL)
            hipLaunchKernelGGL(pr_contrib_kernel<false>, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, s, V, deg,
                               pr, plan->contrib);
        else
            hipLaunchKernelGGL(pr_contrib_kernel<true>, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, s, V, deg,
                               pr, plan->contrib);
        BW_LAUNCH_CHECK();
        pr = plan->contrib;
    }
    return pull_sums(plan, variant, rcols, pr, np, cfg, ReducePrev{});
}

extern "C" int bw_pr_vertex_pull(uint64_t V, const void *roff, int32_t ob, const uint32_t *rcols,
                                 const uint32_t *deg, const float *pr, float *np, const bw_launch *cfg)
{ return pull_entry<true>(V, roff, ob, rcols, deg, pr, np, cfg); }

extern "C" int bw_pr_vertex_pull_nodiv(uint64_t V, const void *roff, int32_t ob, const uint32_t *rcols,
                                       const float *pr, float *np, const bw_launch *cfg)
{ return pull_entry<false>(V, roff, ob, rcols, nullptr, pr, np, cfg); }

extern "C" int bw_pr_vertex_push_warp(uint64_t V, const void *off, int32_t ob, const uint32_t *cols,
                                      const float *pr, float *np, const bw_launch *cfg)
{
    if (V == 0) return BW_HIP_OK;
    if (!off || !cols || !pr || !np) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    uint32_t W, C, block, grid;
    BW_TRY(warp_params(cfg, W, C));
    BW_TRY(resolve_geometry(cfg, (V + C - 1) / C * W, block, grid));
    return with_offsets(off, ob, [&](auto *o) {
        using Off = std::remove_const_t<std::remove_pointer_t<decltype(o)>>;
        const uint32_t lds = pr_warp_lds_bytes<Off>(block / W, C);
        if (lds > 64 * 1024) return fail(BW_HIP_ERR_ARG, "Insufficient shared memory for warp/chunk sizes");
        hipLaunchKernelGGL((pr_vertex_push_warp_kernel<Off>), dim3(grid), dim3(block), lds, stream_of(cfg), W, C, V,
                           o, cols, pr, np);
        BW_LAUNCH_CHECK();
        return BW_HIP_OK;
    });
}

template<bool DIV>
static int pull_warp_entry(uint64_t V, const void *roff, int32_t ob, const uint32_t *rcols, const uint32_t *deg,
                           const float *pr, float *np, const bw_launch *cfg)
{
    if (V == 0) return BW_HIP_OK;
    if (!roff || !rcols || !pr || !np || (DIV && !deg)) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    uint32_t W, C;
    BW_TRY(warp_params(cfg, W, C));
    constexpr int D = DIV ? 2 : 0;
    hipStream_t s = stream_of(cfg);
    switch (W) {
    case 1: return launch_pull<D, 1>(V, roff, ob, rcols, deg, pr, np, s);
    case 2: return launch_pull<D, 2>(V, roff, ob, rcols, deg, pr, np, s);
    case 4: return launch_pull<D, 4>(V, roff, ob, rcols, deg, pr, np, s);
    case 8: return launch_pull<D, 8>(V, roff, ob, rcols, deg, pr, np, s);
    case 16: return launch_pull<D, 16>(V, roff, ob, rcols, deg, pr, np, s);
    case 32: return launch_pull<D, 32>(V, roff, ob, rcols, deg, pr, np, s);
    default: return launch_pull<D, 64>(V, roff, ob, rcols, deg, pr, np, s);
    }
}

extern "C" int bw_pr_vertex_pull_warp(uint64_t V, const void *roff, int32_t ob, const uint32_t *rcols,
                                      const uint32_t *deg, const float *pr, float *np, const bw_launch *cfg)
{ return pull_warp_entry<true>(V, roff, ob, rcols, deg, pr, np, cfg); }

extern "C" int bw_pr_vertex_pull_warp_nodiv(uint64_t V, const void *roff, int32_t ob, const uint32_t *rcols,
                                            const float *pr, float *np, const bw_launch *cfg)
{ return pull_warp_entry<false>(V, roff, ob, rcols, nullptr, pr, np, cfg); }

extern "C" int bw_pr_consolidate(uint64_t V, const uint32_t *deg, float *pr, float *np, int32_t not_last,
                                 int32_t nodiv, int32_t mode, const double *dangling, double *resid,
                                 const bw_launch *cfg)
{
    if (V == 0) return BW_HIP_OK;
    if (!pr || !np) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    if (mode != BW_PR_DANGLING_DROP && mode != BW_PR_DANGLING_UNIFORM)
        return fail(BW_HIP_ERR_ARG, "unknown PageRank mode");
    if ((nodiv || mode == BW_PR_DANGLING_UNIFORM) && !deg)
        return fail(BW_HIP_ERR_ARG, "consolidate needs out-degrees in this mode");
    if (mode == BW_PR_DANGLING_UNIFORM && !dangling)
        return fail(BW_HIP_ERR_ARG, "UNIFORM mode needs the dangling mass");
    uint32_t block, grid;
    BW_TRY(resolve_geometry(cfg, V, block, grid, 1024));
    grid = reduction_grid(cfg, grid);
    hipLaunchKernelGGL(pr_consolidate_kernel, dim3(grid), dim3(block), 0, stream_of(cfg), V, deg, pr, np,
                       not_last ? 1 : 0, nodiv ? 1 : 0, mode, dangling, resid);
    BW_LAUNCH_CHECK();
    return BW_HIP_OK;
}

namespace bw {
namespace {
__global__ void pr_predivide_kernel(uint64_t V, const uint32_t *__restrict__ deg, float *pr)
{
    const uint64_t stride = static_cast<uint64_t>(blockDim.x) * gridDim.x;
    for (uint64_t v = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; v < V; v += stride)
        if (deg[v] != 0) pr[v] = pr[v] / static_cast<float>(deg[v]);
}
}  // namespace
}  // namespace bw

extern "C" int bw_pr_predivide(uint64_t V, const uint32_t *deg, float *pr, const bw_launch *cfg)
{
    if (V == 0) return BW_HIP_OK;
    if (!deg || !pr) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    uint32_t block, grid;
    BW_TRY(resolve_geometry(cfg, V, block, grid));
    hipLaunchKernelGGL(pr_predivide_kernel, dim3(grid), dim3(block), 0, stream_of(cfg), V, deg, pr);
    BW_LAUNCH_CHECK();
    return BW_HIP_OK;
}

extern "C" int bw_pr_dangling_mass(uint64_t V, const uint32_t *deg, const float *pr, double *out,
                                   const bw_launch *cfg)
{
    if (V == 0) return BW_HIP_OK;
    if (!deg || !pr || !out) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
    uint32_t block, grid;
    BW_TRY(resolve_geometry(cfg, V, block, grid, 1024));
    grid = reduction_grid(cfg, grid);
    hipLaunchKernelGGL(pr_dangling_kernel, dim3(grid), dim3(block), 0, stream_of(cfg), V, deg, pr, out);
    BW_LAUNCH_CHECK();
    return BW_HIP_OK;
}

namespace {

// Device scratch of one bw_pr_run call.
struct RunBuffers {
    uint32_t *deg = nullptr;
    float *np = nullptr;
    float *contrib = nullptr;  // per-vertex contributions (the variants that gather them without a pull plan)
    double *acc = nullptr;     // [iterations] residuals, [iterations + 1] dangling masses, one spare
    double2 *part = nullptr;   // per workgroup of a pass over the vertices: (residual, dangling mass)
    ~RunBuffers()
    {
        for (void *p : {static_cast<void *>(deg), static_cast<void *>(np), static_cast<void *>(contrib),
                        static_cast<void *>(acc), static_cast<void *>(part)})
            if (p) (void)hipFree(p);
    }
};

}  // namespace

extern "C" int bw_pr_run(const bw_graph_dev *g, int32_t variant, int32_t iterations, int32_t mode,
                         float *ranks, double *resid_host, const bw_launch *cfg_in)
{
    if (!g || !ranks || iterations < 0) return fail(BW_HIP_ERR_ARG, "bw_pr_run: invalid argument");
    if (variant < 0 || variant >= BW_PR_NUM_REFERENCE_VARIANTS)
        return fail(BW_HIP_ERR_ARG, "unknown PageRank variant " + std::to_string(variant));
    if (mode != BW_PR_DANGLING_DROP && mode != BW_PR_DANGLING_UNIFORM)
        return fail(BW_HIP_ERR_ARG, "unknown PageRank mode");
    const uint64_t V = g->vertex_count, E = g->edge_count;
    if (V == 0) return BW_HIP_OK;
    bw_launch cfg{};
    if (cfg_in) cfg = *cfg_in;
    cfg.grid = 0;  // every kernel sizes its own grid
    hipStream_t s = static_cast<hipStream_t>(cfg.stream);
    const bool nodiv = variant == BW_PR_VERTEX_PULL_NODIV || variant == BW_PR_VERTEX_PULL_WARP_NODIV;

    auto need = [&](const void *p, const char *what) -> int {
        if (!p && E) return fail(BW_HIP_ERR_ARG, std::string("variant needs the ") + what + " representation");
        return BW_HIP_OK;
    };
    switch (variant) {
    case BW_PR_EDGE_LIST: BW_TRY(need(g->el_in, "EdgeList")); BW_TRY(need(g->el_out, "EdgeList")); break;
    case BW_PR_REV_EDGE_LIST: BW_TRY(need(g->rel_in, "reverse EdgeList")); BW_TRY(need(g->rel_out, "reverse EdgeList")); break;
    case BW_PR_STRUCT_EDGE_LIST: BW_TRY(need(g->sel, "StructEdgeList")); break;
    case BW_PR_REV_STRUCT_EDGE_LIST: BW_TRY(need(g->rsel, "reverse StructEdgeList")); break;
    case BW_PR_VERTEX_PUSH:
    case BW_PR_VERTEX_PUSH_WARP:
        if (!g->offsets || (E && !g->cols)) return fail(BW_HIP_ERR_ARG, "variant needs the CSR representation");
        break;
    default:
        if (!g->rev_offsets || (E && !g->rev_cols))
            return fail(BW_HIP_ERR_ARG, "variant needs the reverse CSR representation");
    }

    // The passes over the vertices have a geometry of their own; the caller's
    // is held to the same bounds as in the per-call entries.
    uint32_t block = 0, grid = 0;
    if (iterations > 0) BW_TRY(resolve_geometry(&cfg, V, block, grid));

    RunBuffers buf;
    const uint64_t iters = static_cast<uint64_t>(std::max(iterations, 1));
    BW_HIP_CHECK(hipMalloc(&buf.deg, sizeof(uint32_t) * V));
    BW_HIP_CHECK(hipMalloc(&buf.np, sizeof(float) * V));
    BW_HIP_CHECK(hipMalloc(&buf.acc, sizeof(double) * (2 * iters + 2)));
    BW_HIP_CHECK(hipMalloc(&buf.part, sizeof(double2) * kFinishGrid));
    const bool push = variant == BW_PR_EDGE_LIST || variant == BW_PR_STRUCT_EDGE_LIST || variant == BW_PR_VERTEX_PUSH ||
                      variant == BW_PR_VERTEX_PUSH_WARP;
    // The binned scatter and the atomic kernels divide for themselves, and a
    // pull plan holds contributions of its own.
    const bool gathers = push && E > 0 && iterations > 0 && scatter_gathers(V);
    if (gathers || variant == BW_PR_REV_EDGE_LIST || variant == BW_PR_REV_STRUCT_EDGE_LIST)
        BW_HIP_CHECK(hipMalloc(&buf.contrib, sizeof(float) * V));
    double *resid = buf.acc, *dang = buf.acc + iters, *spare = buf.acc + 2 * iters + 1;

    // Degrees once per run (pagerank/pagerank.cpp:102-112).  With the forward
    // CSR resident, every variant's out-degrees come from its offsets: the
    // same integers the variant's own degree kernel counts
    // (pagerank/pagerank.cu:40-123), without an atomic per edge; the push
    // variants, which have no degree kernel, read the same offsets, and only for
    // the contributions or the dangling mass.
    BW_TRY(bw_pr_zero_degrees(V, buf.deg, &cfg));
    const bool degrees = gathers || mode == BW_PR_DANGLING_UNIFORM ||
                         !(variant == BW_PR_VERTEX_PUSH || variant == BW_PR_VERTEX_PUSH_WARP);
    if (!degrees) {
        // nothing to count
    } else if (g->offsets) {
        BW_TRY(bw_pr_degrees_csr(V, g->offsets, g->offset_bytes, buf.deg, &cfg));
    } else switch (variant) {
    case BW_PR_EDGE_LIST: BW_TRY(bw_pr_degrees_edge_list(E, g->el_in, buf.deg, &cfg)); break;
    case BW_PR_REV_EDGE_LIST: BW_TRY(bw_pr_degrees_edge_list(E, g->rel_out, buf.deg, &cfg)); break;
    case BW_PR_STRUCT_EDGE_LIST: BW_TRY(bw_pr_degrees_struct_edge_list(E, g->sel, 0, buf.deg, &cfg)); break;
    case BW_PR_REV_STRUCT_EDGE_LIST: BW_TRY(bw_pr_degrees_struct_edge_list(E, g->rsel, 1, buf.deg, &cfg)); break;
    default:
        BW_TRY(bw_pr_degrees_rev_csr(V, g->rev_offsets, g->offset_bytes, g->rev_cols, buf.deg, &cfg));
    }

    // The push forms scatter through a binned layout (propagation blocking)
    // instead of one global atomic per edge; a graph the layout refuses
    // (beyond 2^25 vertices or 2^32 - 1 edges) keeps the atomic kernels.
    bw_pr_scatter *scatter = nullptr;
    struct ScatterGuard {
        bw_pr_scatter *&p;
        ~ScatterGuard() { bw_pr_scatter_destroy(p); }
    } scatter_guard{scatter};
    if (E > 0 && push) {
        int st = BW_HIP_OK;
        if (variant == BW_PR_EDGE_LIST)
            st = bw_pr_scatter_create(&scatter, BW_PR_SCATTER_EDGE_LIST, V, E, g->el_in, g->el_out, 4, s);
        else if (variant == BW_PR_STRUCT_EDGE_LIST)
            st = bw_pr_scatter_create(&scatter, BW_PR_SCATTER_STRUCT, V, E, g->sel, nullptr, 4, s);
        else
            st = bw_pr_scatter_create(&scatter, BW_PR_SCATTER_CSR, V, E, g->offsets, g->cols, g->offset_bytes, s);
        if (st != BW_HIP_OK && st != BW_HIP_ERR_ARG) return st;
    }

    // The pull forms split off their long rows once per run.
    bw_pr_pull_plan *pull = nullptr;
    struct PullGuard {
        bw_pr_pull_plan *&p;
        ~PullGuard() { bw_pr_pull_plan_destroy(p); }
    } pull_guard{pull};
    if (pull_variant(variant)) {
        if (iterations > 0 && !g->rev_cols) return fail(BW_HIP_ERR_ARG, "NULL device pointer");
        BW_TRY(bw_pr_pull_plan_create(&pull, V, g->rev_offsets, g->offset_bytes, s));
    }

    const bool gathered = scatter && gathers;
    FinishArgs fin{};
    fin.V = V;
    fin.deg = degrees ? buf.deg : nullptr;
    fin.pr = ranks;
    fin.np = buf.np;
    fin.part = buf.part;
    fin.nodiv = nodiv;
    fin.mode = mode;
    fin.contrib = pull && !nodiv ? pull->contrib : buf.contrib;
    const uint64_t passVerts = static_cast<uint64_t>(finish_per_thread(gathered)) * kFinishThreads;
    const uint32_t passGrid = static_cast<uint32_t>(std::min<uint64_t>((V + passVerts - 1) / passVerts, kFinishGrid));
    fin.zero_np = !pull && !gathered;  // these store every row's sum
    fin.int_degree = variant == BW_PR_VERTEX_PULL_WARP;
    hipLaunchKernelGGL(pr_start_kernel, dim3(passGrid), dim3(kFinishThreads), 0, s, fin,
                       (nodiv && mode == BW_PR_DANGLING_UNIFORM) ? 1 : 0);
    BW_LAUNCH_CHECK();

    // Per iteration the sums, whose launch also reduces the partials of the
    // pass before it, and one pass over the vertices.
    for (int32_t it = 1; it <= iterations; it++) {
        const ReducePrev prev{buf.part, passGrid, it > 1 ? &resid[it - 2] : spare, &dang[it - 1]};
        bool reduced = false;  // the sums' launch reduced `prev`
        if (pull) {
            BW_TRY(pull_sums(pull, variant, g->rev_cols, nodiv ? ranks : fin.contrib, buf.np, &cfg, prev));
            reduced = true;
        } else if (E && variant == BW_PR_REV_EDGE_LIST) {
            BW_TRY((launch_rev_segmented<false, true>(E, g->rel_in, g->rel_out, nullptr, buf.contrib, buf.np, s,
                                                      prev)));
            reduced = true;
        } else if (E && variant == BW_PR_REV_STRUCT_EDGE_LIST) {
            BW_TRY((launch_rev_segmented<true, true>(E, g->rsel, nullptr, nullptr, buf.contrib, buf.np, s, prev)));
            reduced = true;
        } else if (gathered) {
            BW_TRY(scatter_gather(scatter, buf.contrib, prev, s));
            reduced = true;
        } else if (scatter) {
            BW_TRY(scatter_bins(scatter, buf.deg, ranks, buf.np, prev, s));
            reduced = true;
        } else if (variant == BW_PR_EDGE_LIST) {
            BW_TRY(bw_pr_edge_list(E, g->el_in, g->el_out, buf.deg, ranks, buf.np, &cfg));
        } else if (variant == BW_PR_STRUCT_EDGE_LIST) {
            BW_TRY(bw_pr_struct_edge_list(E, g->sel, buf.deg, ranks, buf.np, &cfg));
        } else if (variant == BW_PR_VERTEX_PUSH) {
            BW_TRY(bw_pr_vertex_push(V, g->offsets, g->offset_bytes, g->cols, ranks, buf.np, &cfg));
        } else if (variant == BW_PR_VERTEX_PUSH_WARP) {
            BW_TRY(bw_pr_vertex_push_warp(V, g->offsets, g->offset_bytes, g->cols, ranks, buf.np, &cfg));
        }
        if (!reduced) {
            hipLaunchKernelGGL(pr_reduce_prev_kernel, dim3(1), dim3(256), 0, s, prev);
            BW_LAUNCH_CHECK();
        }
        fin.not_last = iterations > it;
        fin.dangling = &dang[it - 1];
        if (gathered)
            hipLaunchKernelGGL(pr_finish_kernel<true>, dim3(passGrid), dim3(kFinishThreads), 0, s, fin,
                               scatter_sums(scatter));
        else
            hipLaunchKernelGGL(pr_finish_kernel<false>, dim3(passGrid), dim3(kFinishThreads), 0, s, fin,
                               ScatterSums{});
        BW_LAUNCH_CHECK();
    }
    if (iterations > 0) {
        const ReducePrev prev{buf.part, passGrid, &resid[iterations - 1], spare};
        hipLaunchKernelGGL(pr_reduce_prev_kernel, dim3(1), dim3(256), 0, s, prev);
        BW_LAUNCH_CHECK();
    }
    if (resid_host && iterations > 0) {
        BW_HIP_CHECK(hipMemcpyAsync(resid_host, resid, sizeof(double) * iterations, hipMemcpyDeviceToHost, s));
    }
    BW_HIP_CHECK(hipStreamSynchronize(s));
    return BW_HIP_OK;
}
