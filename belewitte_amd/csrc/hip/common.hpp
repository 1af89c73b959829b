// Shared host/device helpers of libbelewitte_hip (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>
#include <string>

#include "belewitte_hip.h"

namespace bw {

// ------------------------------------------------------------ errors

void set_error(const std::string &msg);
int fail(int code, const std::string &msg);
int hip_fail(hipError_t e, const char *what, const char *file, int line);

#define BW_HIP_CHECK(call)                                                   \
    do {                                                                     \
        hipError_t bw_e_ = (call);                                           \
        if (bw_e_ != hipSuccess)                                             \
            return ::bw::hip_fail(bw_e_, #call, __FILE__, __LINE__);         \
    } while (0)

// Checks the launch that was just enqueued.
#define BW_LAUNCH_CHECK() BW_HIP_CHECK(hipGetLastError())

#define BW_TRY(call)                                                         \
    do {                                                                     \
        int bw_s_ = (call);                                                  \
        if (bw_s_ != BW_HIP_OK) return bw_s_;                                \
    } while (0)

constexpr int kWave = 64;
constexpr int32_t kUnvisited = INT_MAX;

inline hipStream_t stream_of(const bw_launch *cfg)
{ return cfg ? static_cast<hipStream_t>(cfg->stream) : nullptr; }

// Resolves block/grid for `work` items of a grid-stride kernel; the block
// must be a multiple of the wave size so every wave is full (the wave
// reductions rely on it).
int resolve_geometry(const bw_launch *cfg, uint64_t work, uint32_t &block,
                     uint32_t &grid, uint32_t default_block = 256);

// Number of compute units of the current device (cached per device).
int device_cus();

// -------------------------------------------------------- device side

// The block of vertices (of n equal blocks) that workgroup b takes.
// Workgroups go to the eight XCDs round robin, and the degrees of an R-MAT
// graph in its generated order follow the bits of the vertex id (each zero
// bit makes a vertex about three times heavier), so block b for workgroup b
// gives one XCD 2.5 to 3.4 times its share of the edges (scales 16 to 21,
// 256-vertex blocks).  Each run of eight blocks is rotated by the sum of the
// octal digits of its index instead: no low bit of the id stays tied to an
// XCD (1.02 to 1.14 times the share at scales 19 to 21).  A bijection; the
// last, incomplete run keeps its order.
__device__ __forceinline__ uint32_t spread_block(uint32_t b, uint32_t n)
{
    const uint32_t q = b >> 3;
    if ((q << 3) + 8 > n) return b;
    return (q << 3) | ((b + q + (q >> 3) + (q >> 6) + (q >> 9) + (q >> 12) + (q >> 15)) & 7u);
}

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v)
{
    // xor butterfly over the 64 lanes; every lane ends with the total.
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

__device__ __forceinline__ double wave_sum_f64(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

__device__ __forceinline__ float wave_sum_f32(float v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// Inclusive prefix sum over the wave by DPP row shifts and row broadcasts.
template<int kCtrl, int kRowMask, bool kBound>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t v)
{
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), kCtrl, kRowMask, 0xF, kBound));
}

__device__ __forceinline__ uint32_t wave_prefix_sum(uint32_t x)
{
    x += dpp_or_zero<0x111, 0xF, true>(x);
    x += dpp_or_zero<0x112, 0xF, true>(x);
    x += dpp_or_zero<0x114, 0xF, true>(x);
    x += dpp_or_zero<0x118, 0xF, true>(x);
    x += dpp_or_zero<0x142, 0xA, false>(x);
    x += dpp_or_zero<0x143, 0xC, false>(x);
    return x;
}

__device__ __forceinline__ uint64_t wave_prefix_sum(uint64_t x)
{
    for (int o = 1; o < kWave; o <<= 1) {
        const uint64_t y = __shfl_up(static_cast<unsigned long long>(x), static_cast<unsigned>(o), kWave);
        if (static_cast<int>(__lane_id()) >= o) x += y;
    }
    return x;
}

// Block-wide sum of a double; result valid in thread 0.  `lds` holds one
// slot per wave (16 for a 1024-thread block).
__device__ __forceinline__ double block_sum_f64(double v, double *lds)
{
    v = wave_sum_f64(v);
    const int lane = threadIdx.x & (kWave - 1);
    const int wid = threadIdx.x / kWave;
    if (lane == 0) lds[wid] = v;
    __syncthreads();
    double t = 0.0;
    if (wid == 0) {
        const int nw = blockDim.x / kWave;
        t = lane < nw ? lds[lane] : 0.0;
        t = wave_sum_f64(t);
    }
    return t;
}

// Sum of n (residual, dangling) partials in a fixed order: thread t adds
// partials t, t + kThreads, ...; then a fixed tree.  Results in thread 0.
template<int kThreads>
__device__ __forceinline__ void reduce_partials(const double2 *p, uint32_t n, double &r, double &g, double (*red)[2])
{
    r = 0.0;
    g = 0.0;
    for (uint32_t i = threadIdx.x; i < n; i += kThreads) {
        const double2 t = p[i];
        r += t.x;
        g += t.y;
    }
    r = wave_sum_f64(r);
    g = wave_sum_f64(g);
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    if (lane == 0) {
        red[wid][0] = r;
        red[wid][1] = g;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        r = 0.0;
        g = 0.0;
        for (int w = 0; w < kThreads / kWave; w++) {
            r += red[w][0];
            g += red[w][1];
        }
    }
}

// Frontier counters: the four Reduction strategies of bfs/bfs.hpp:32-116,
// with wave64 in place of the 32-wide warp.  Each adds to a counter of the
// workgroup in LDS -- per discovery, per thread, per wave or by the block --
// and the workgroup adds that to the global counter once: atomics on one
// address run one after another (the discoveries of the widest vertex-push
// level of an R-MAT scale-16 search: 473 us with a global atomic each, 406
// with this).
// Every thread of the workgroup constructs and finalises its counter.
__device__ __forceinline__ uint32_t *workgroup_count()
{
    __shared__ uint32_t count;
    return &count;
}

struct WorkgroupCount {
    __device__ __forceinline__ WorkgroupCount()
    {
        if (threadIdx.x == 0) *workgroup_count() = 0;
        __syncthreads();
    }
    __device__ __forceinline__ void flush(uint32_t *frontier)
    {
        __syncthreads();
        if (threadIdx.x == 0) {
            const uint32_t total = *workgroup_count();
            if (total) atomicAdd(frontier, total);
        }
    }
};

template<int R>
struct FrontierCount;

template<>
struct FrontierCount<BW_RED_NORMAL> : WorkgroupCount {
    __device__ __forceinline__ void update() { atomicAdd(workgroup_count(), 1u); }
    __device__ __forceinline__ void finalise(uint32_t *frontier) { flush(frontier); }
};

template<>
struct FrontierCount<BW_RED_BULK> : WorkgroupCount {
    uint32_t count = 0;
    __device__ __forceinline__ void update() { count++; }
    __device__ __forceinline__ void finalise(uint32_t *frontier)
    {
        if (count) atomicAdd(workgroup_count(), count);
        flush(frontier);
    }
};

template<>
struct FrontierCount<BW_RED_WAVE> : WorkgroupCount {
    uint32_t count = 0;
    __device__ __forceinline__ void update() { count++; }
    __device__ __forceinline__ void finalise(uint32_t *frontier)
    {
        const uint32_t total = wave_sum_u32(count);
        if ((threadIdx.x & (kWave - 1)) == 0 && total) atomicAdd(workgroup_count(), total);
        flush(frontier);
    }
};

template<>
struct FrontierCount<BW_RED_BLOCK> {
    uint32_t count = 0;
    __device__ __forceinline__ void update() { count++; }
    __device__ __forceinline__ void finalise(uint32_t *frontier)
    {
        __shared__ uint32_t partial[1024 / kWave];
        uint32_t total = wave_sum_u32(count);
        const int lane = threadIdx.x & (kWave - 1);
        const int wid = threadIdx.x / kWave;
        if (lane == 0) partial[wid] = total;
        __syncthreads();
        if (wid == 0) {
            const int nw = blockDim.x / kWave;
            uint32_t t = lane < nw ? partial[lane] : 0u;
            t = wave_sum_u32(t);
            if (lane == 0 && t) atomicAdd(frontier, t);
        }
    }
};

// atomicMin on a depth that only ever decreases within a level: a plain
// load that already shows <= nd proves the atomic would not change the
// value nor count it, so the atomic is skipped.  A stale cached copy can
// only be larger than the current value, which merely costs the atomic.
__device__ __forceinline__ bool relax_depth(int32_t *levels, uint32_t v, int32_t nd)
{
    if (levels[v] <= nd) return false;
    return atomicMin(&levels[v], nd) > nd;
}

template<typename Off>
__device__ __forceinline__ uint64_t load_off(const Off *o, uint64_t i)
{ return static_cast<uint64_t>(o[i]); }

}  // namespace bw
