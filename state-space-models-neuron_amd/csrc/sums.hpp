// Sums of partial rows of parameter gradients, in a fixed order: the bodies that their own kernels and param_sums_kernel share.
#pragma once
#include "common.hpp"

namespace m2 {

// Sum over the partial rows of partial[row][c]: 32 channels (one cache line of a row) per workgroup of 1024 threads, V to a lane,
// 32 V row phases whose sums meet in LDS; store(c, sum) by one thread per channel.  Few workgroups read little each: what bounds it
// is the chain of loads of one thread, hence many phases with wide loads (32 phases of one channel per thread: 11.2 us at 1668
// rows of 2048).
constexpr int kSumCols = 32;
template <int V, typename F>
__device__ __forceinline__ void column_sum_body(const float* __restrict__ partial, int64_t nrows, int64_t ncols, int64_t blk, F&& store) {
    constexpr int LANES = kSumCols / V, PHASES = 1024 / LANES;
    typedef float vec __attribute__((ext_vector_type(V)));
    __shared__ float red[PHASES][kSumCols + 4];
    const int l = threadIdx.x % LANES, ph = threadIdx.x / LANES;
    const int64_t col = blk * kSumCols + l * V;
    vec s = 0.f;
    if (col < ncols) {
#pragma unroll 4
        for (int64_t r = ph; r < nrows; r += PHASES) s += *reinterpret_cast<const vec*>(partial + r * ncols + col);
    }
    *reinterpret_cast<vec*>(&red[ph][l * V]) = s;
    __syncthreads();
    // 32 threads per channel, then one
    const int c = threadIdx.x & 31, q = threadIdx.x >> 5;
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < PHASES / 32; ++k) t += red[q * (PHASES / 32) + k][c];
    __syncthreads();
    red[q][c] = t;
    __syncthreads();
    if (q == 0 && blk * kSumCols + c < ncols) {
        float u[32];
#pragma unroll
        for (int k = 0; k < 32; ++k) u[k] = red[k][c];
#pragma unroll
        for (int w = 16; w >= 1; w >>= 1)
#pragma unroll
            for (int k = 0; k < w; ++k) u[k] += u[k + w];
        store(blk * kSumCols + c, u[0]);
    }
}

__device__ __forceinline__ void st_param(void* p, int pd, int64_t i, float v) {
    if (pd == M2_F32) reinterpret_cast<float*>(p)[i] = v;
    else reinterpret_cast<bf16_t*>(p)[i] = from_f32<bf16_t>(v);
}

// The per-block partials of a conv's weight and bias gradients, part[slot][channel][k + 1].  Four adjacent lanes per (channel,
// tap-or-bias), each a quarter of the slots (fixed order), combined by two shuffles; t: the thread's index over all of them.
__device__ __forceinline__ void conv_sum_body(const float* __restrict__ part, int64_t nslots, int64_t C, int k, void* __restrict__ dw, void* __restrict__ db,
                                              int pd, int64_t t) {
    const int64_t e = t >> 2;
    const int q = (int)(t & 3);
    const int kk = k + 1;
    const bool live = e < C * kk;
    const int64_t c = live ? e / kk : 0;
    const int i = live ? (int)(e % kk) : 0;
    float s = 0.f;
    if (live) {
#pragma unroll 4
        for (int64_t r = q; r < nslots; r += 4) s += part[(r * C + c) * kk + i];
    }
    s = lane_xor_add<1>(s);
    s = lane_xor_add<2>(s);
    if (!live || q != 0) return;
    if (i < k) st_param(dw, pd, c * k + i, s);
    else if (db) st_param(db, pd, c, s);
}

}  // namespace m2
