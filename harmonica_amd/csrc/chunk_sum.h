// Sum of the chunk partials of one output, shared by the reductions.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace hmx {
namespace dev {

// Threads that share an output's chunks, and the outputs of a workgroup: one
// wave's, 64, by P waves, each summing its share of the chunks in order and the
// shares added in order; or (P = 1) 256 with a thread each.
template <int P>
struct SumShape {
    static constexpr int parts = P, outputs = P > 1 ? 64 : 256, threads = P * outputs;
};

// Parts for a reduction of `total` outputs.  A serial sum over the chunks is
// bound by the latency of its loads: one component of a magnetic field at 544
// points, 1024 chunks, took 237 us with a thread per output.  From 2^18
// outputs on (16 waves on each of 256 CUs) other outputs hide that latency,
// chunks are few, and further waves would have nothing to do but start and
// end: a magnetic field of one prism at 10,000,000 points, 30,000,000 outputs of
// one chunk each, spent 1.5 of its 2.3 ms in 480,000 workgroups of 16 waves, and
// from 2^28 outputs on their threads passed the 2^32 of a launch.
inline int sum_parts(int64_t chunks, int64_t total, int most) {
    return chunks == 1 || total >= ((int64_t)1 << 18) ? 1 : most;
}

// The output of this thread and, summed over chunks c, partial[c * total +
// idx]; returns whether this thread holds the sum (the first part's threads,
// idx < total).  All threads of the workgroup call it.
template <int P>
__device__ __forceinline__ bool chunk_sum(const double *__restrict__ partial, int64_t chunks,
                                          int64_t total, int64_t &idx, double &sum) {
    using S = SumShape<P>;
    const int lane = threadIdx.x % S::outputs, p = threadIdx.x / S::outputs;
    idx = (int64_t)blockIdx.x * S::outputs + lane;
    const int64_t c0 = chunks * p / P, c1 = chunks * (p + 1) / P;
    sum = 0.0;
    if (idx < total) {
#pragma unroll 8
        for (int64_t c = c0; c < c1; ++c) sum += partial[c * total + idx];
    }
    if constexpr (P > 1) {
        __shared__ double part[P][S::outputs];
        part[p][lane] = sum;
        __syncthreads();
        if (p || idx >= total) return false;
        for (int q = 1; q < P; ++q) sum += part[q][lane];
    }
    return idx < total;
}

}  // namespace dev
}  // namespace hmx
