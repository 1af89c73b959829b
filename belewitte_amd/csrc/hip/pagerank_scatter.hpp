// What the scatter layout (pagerank_scatter.hip) shares with the PageRank
// run loop (pagerank.hip).
#pragma once

#include "common.hpp"

namespace bw {

// A run's iteration launches reduce the (residual, dangling mass) partials
// of the launch before them in one extra workgroup, their last: a launch of
// its own would cost more than the reduction.
struct ReducePrev {
    const double2 *part = nullptr;  // NULL: no extra workgroup
    uint32_t n = 0;
    double *resid = nullptr;
    double *dangl = nullptr;
};

struct ReduceLds {
    double red[16][2];
};

// Whether this workgroup is the extra one; it has done the reduction then.
template<int kThreads>
__device__ __forceinline__ bool reduce_prev(const ReducePrev &p, ReduceLds &lds)
{
    if (!p.part || blockIdx.x != gridDim.x - 1) return false;
    double r, g;
    reduce_partials<kThreads>(p.part, p.n, r, g, lds.red);
    if (threadIdx.x == 0) {
        *p.resid = r;
        *p.dangl = g;
    }
    return true;
}

// Row sums of a gathered layout's iteration: one FP64 vector per chunk of a
// partition's bin.
struct ScatterSums {
    const double *partials;
    const uint32_t *chunk_base;  // per partition: its first chunk
    uint32_t rows_log;

    // sum += x's entries q .. q + N - 1 below n, their loads in flight together.
    template<uint32_t N>
    __device__ __forceinline__ void add_batch(const double *x, uint32_t q, uint32_t n, double &sum) const
    {
        double y[N];
#pragma unroll
        for (uint32_t k = 0; k < N; k++)
            if (q + k < n) y[k] = x[static_cast<uint64_t>(q + k) << rows_log];
#pragma unroll
        for (uint32_t k = 0; k < N; k++)
            if (q + k < n) sum += y[k];
    }

    __device__ __forceinline__ float row_sum(uint32_t v) const
    {
        const uint32_t p = v >> rows_log, c0 = chunk_base[p], n = chunk_base[p + 1] - c0;
        const double *x = partials + ((static_cast<uint64_t>(c0) << rows_log) + (v & ((1u << rows_log) - 1u)));
        double sum = 0.0;
        if (n <= 4) add_batch<4>(x, 0, n, sum);
        else
            for (uint32_t q = 0; q < n; q += 16) add_batch<16>(x, q, n, sum);
        return static_cast<float>(sum);
    }
};

bool scatter_gathers(uint64_t V);  // whether a layout of V vertices is a gathered one
ScatterSums scatter_sums(const bw_pr_scatter *sc);
int scatter_gather(const bw_pr_scatter *sc, const float *contrib, const ReducePrev &prev, hipStream_t s);
int scatter_bins(const bw_pr_scatter *sc, const uint32_t *deg, const float *pr, float *np, const ReducePrev &prev,
                 hipStream_t s);

}  // namespace bw
