// Sum of the chunk partials of one output, shared by the reductions.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace hmx {
namespace dev {

// Workgroups of kSumParts waves, 64 outputs each: every wave sums its share of
// the chunks in order, the shares are added in order.  A serial sum over all
// chunks is bound by the latency of its loads (one component of a magnetic
// field at 544 points, 1024 chunks: 237 us with a thread per output).
constexpr int kSumParts = 16;
constexpr int kSumThreads = 64 * kSumParts;

// The sum over chunks c of partial[c * total + idx], idx = 64 blockIdx.x +
// lane; returns whether this thread holds it (the first wave, idx < total).
// All threads of the workgroup call it.
__device__ __forceinline__ bool chunk_sum(const double *__restrict__ partial, int64_t chunks,
                                          int64_t total, int64_t idx, double &sum) {
    __shared__ double part[kSumParts][64];
    const int lane = threadIdx.x & 63, p = threadIdx.x >> 6;
    const int64_t c0 = chunks * p / kSumParts, c1 = chunks * (p + 1) / kSumParts;
    sum = 0.0;
    if (idx < total) {
#pragma unroll 8
        for (int64_t c = c0; c < c1; ++c) sum += partial[c * total + idx];
    }
    part[p][lane] = sum;
    __syncthreads();
    if (p || idx >= total) return false;
    for (int q = 1; q < kSumParts; ++q) sum += part[q][lane];
    return true;
}

}  // namespace dev
}  // namespace hmx
