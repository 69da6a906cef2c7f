// Magnetic field of uniformly magnetised prisms (explicit prisms).
//
// For a prism with magnetisation M (A/m) the field at a point is
//   b_i = c_m sum_j M_j K_ij,   c_m = mu_0 / (4 pi),  mu_0 = 4 pi 1e-7 H/m,
// with K_ij the vertex sums of the second-derivative kernels of the gravity
// tensor in the east-north-up frame (the same grouped closed forms as the
// gravity kernels, prism_device.h): b_e uses K_ee, K_en, K_eu; b_n uses
// K_en, K_nn, K_nu; b_u uses K_eu, K_nu, K_uu.  Every component is NaN on any
// edge or vertex of a prism.  This replaces the per-pair calls of
// src/harmonica/_forward/prisms/magnetic.py:319-331 (field "b") and
// :384-397 (one component) and the nT conversion of :195-197 and :271.
//
// Launch and forms as the gravity kernels (prism_fields_far.h): 256 points per
// workgroup, one per lane, tiles of 32 prisms in LDS, far form or closed form
// by distance, one chunk of the prism list per workgroup column, chunk
// partial sums reduced in order by a second kernel (deterministic results).
#include "chunk_sum.h"
#include "hmx_internal.h"
#include "prism_fields_far.h"

namespace hmx {
namespace {

using dev::FieldSet;

constexpr double kPi = 3.141592653589793;
// mu_0 / 4 / pi with mu_0 = 4 pi 1e-7, evaluated in that order.
constexpr double kCm = 4.0 * kPi * 1e-7 / 4.0 / kPi;

// Components selected by bit c of C (0 = b_e, 1 = b_n, 2 = b_u) and the
// tensor kernels (gravity field bits 4..9) they need.
template <unsigned C>
struct MagSet {
    static constexpr unsigned tensor =
        ((C & 1u) ? 0x190u : 0u) | ((C & 2u) ? 0x2a0u : 0u) | ((C & 4u) ? 0x340u : 0u);
    static constexpr int count = __builtin_popcount(C & 7u);
};

// Prisms and magnetisations as given, for the field chunks.
struct MagSource {
    const double *prisms, *me, *mn, *mu;
    __device__ bool get(int64_t p, double (&b)[6], double (&weight)[3]) const {
#pragma unroll
        for (int c = 0; c < 6; ++c) b[c] = prisms[6 * p + c];
        weight[0] = kCm * me[p];
        weight[1] = kCm * mn[p];
        weight[2] = kCm * mu[p];
        return false;
    }
};

// The components' sums from K[f - 4] for gravity field bit f: ee 4, nn 5, uu
// 6, en 7, eu 8, nu 9.
template <unsigned C>
__device__ __forceinline__ void magnetic_terms(const double *weight, const double (&K)[6],
                                               double (&out)[MagSet<C>::count]) {
    const double me = weight[0], mn = weight[1], mu = weight[2];
    int s = 0;
    if constexpr ((C & 1u) != 0) out[s++] = me * K[0] + mn * K[3] + mu * K[4];
    if constexpr ((C & 2u) != 0) out[s++] = me * K[3] + mn * K[1] + mu * K[5];
    if constexpr ((C & 4u) != 0) out[s++] = me * K[4] + mn * K[5] + mu * K[2];
}

// Add the selected components of one prism at (e, n, u) to acc[].  Without
// kGeneral, dev::needs_general<MagSet<C>::tensor> must be false for the
// point (it is then on no face plane, so on no edge).
template <unsigned C, bool kGeneral>
__device__ __forceinline__ void magnetic_pair(double e, double n, double u, const double *b,
                                              const double *weight,
                                              double (&acc)[MagSet<C>::count],
                                              const dm::Tables &tab) {
    constexpr unsigned M = MagSet<C>::tensor;
    using F = FieldSet<M>;
    const double x0 = b[1] - e, x1 = b[0] - e, y0 = b[3] - n, y1 = b[2] - n;
    const double z0 = b[5] - u, z1 = b[4] - u;
    double K[6];
    if constexpr (kGeneral) {
        double vs[F::count];
        uint32_t sflags = 0;
        dev::prism_fields<M, true>(x0, x1, y0, y1, z0, z1, vs, sflags, tab);
#pragma unroll
        for (int f = 4; f < 10; ++f)
            if ((M >> f) & 1u) K[f - 4] = vs[F::slot(f)];
    } else {
        dev::tensor_lean<M>(x0, x1, y0, y1, z0, z1, K, tab);
    }
    double terms[MagSet<C>::count];
    magnetic_terms<C>(weight, K, terms);
#pragma unroll
    for (int c = 0; c < MagSet<C>::count; ++c) acc[c] += terms[c];
    if constexpr (kGeneral) {
        // On an edge: two coordinates on a bound of the prism, the third
        // between its bounds (vertices included).
        const bool in_e = x1 <= 0.0 && 0.0 <= x0, in_n = y1 <= 0.0 && 0.0 <= y0;
        const bool in_u = z1 <= 0.0 && 0.0 <= z0;
        const bool at_e = x0 == 0.0 || x1 == 0.0, at_n = y0 == 0.0 || y1 == 0.0;
        const bool at_u = z0 == 0.0 || z1 == 0.0;
        const bool edge = (in_e && at_n && at_u) || (in_n && at_e && at_u) || (in_u && at_e && at_n);
        if (edge) {
#pragma unroll
            for (int c = 0; c < MagSet<C>::count; ++c) acc[c] = __builtin_nan("");
        }
    }
}

// The sums of field_far_chunk and field_close_chunk: the selected components.
template <unsigned C>
struct MagneticOp {
    static constexpr unsigned fields = MagSet<C>::tensor;
    static constexpr int weights = 3, values = MagSet<C>::count;
    __device__ static void combine(const double *weight, const double (&vs)[FieldSet<fields>::count],
                                   double (&out)[values]) {
        double K[6];
#pragma unroll
        for (int f = 4; f < 10; ++f)
            if ((fields >> f) & 1u) K[f - 4] = vs[FieldSet<fields>::slot(f)];
        magnetic_terms<C>(weight, K, out);
    }
    template <bool kGeneral>
    __device__ static void closed(double e, double n, double u, const double *b,
                                  const double *weight, double (&acc)[values], uint32_t &,
                                  const dm::Tables &tab) {
        magnetic_pair<C, kGeneral>(e, n, u, b, weight, acc, tab);
    }
};

// The far pairs into the partial sums.
template <unsigned C>
__global__ __launch_bounds__(dev::kGzThreads, 3) void magnetic_far_kernel(
    const double *__restrict__ oe, const double *__restrict__ on, const double *__restrict__ ou,
    int n_obs, MagSource src, int64_t n_src, int64_t chunk_len, double *__restrict__ partial) {
    using Op = MagneticOp<C>;
    __shared__ dev::FieldFarShared<Op> sh;
    // rotated from chunk to chunk over the XCDs, as prism_gz_kernel
    const unsigned bx = (blockIdx.x + blockIdx.y) % gridDim.x;
    const int64_t base = (int64_t)bx * dev::kGzThreads, i = base + threadIdx.x;
    const int64_t c0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t c1 = c0 + chunk_len < n_src ? c0 + chunk_len : n_src;
    double acc[Op::values] = {};
    dev::field_far_chunk<Op>(src, oe, on, ou, base, n_obs, c0, c1, acc, sh);
    if (i < n_obs) {
#pragma unroll
        for (int s = 0; s < Op::values; ++s)
            partial[((int64_t)blockIdx.y * Op::values + s) * n_obs + i] = acc[s];
    }
}

// The close pairs, added to the partial sums of magnetic_far_kernel.
template <unsigned C>
__global__ __launch_bounds__(dev::kGzThreads, 3) void magnetic_close_kernel(
    const double *__restrict__ oe, const double *__restrict__ on, const double *__restrict__ ou,
    int n_obs, MagSource src, int64_t n_src, int64_t chunk_len, double *__restrict__ partial) {
    using Op = MagneticOp<C>;
    __shared__ dev::FieldCloseShared<Op> sh;
    const unsigned bx = (blockIdx.x + blockIdx.y) % gridDim.x;
    const int64_t base = (int64_t)bx * dev::kGzThreads, i = base + threadIdx.x;
    const int64_t c0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t c1 = c0 + chunk_len < n_src ? c0 + chunk_len : n_src;
    double acc[Op::values] = {};
    uint32_t flags = 0;
    if (!dev::field_close_chunk<Op>(src, oe, on, ou, base, n_obs, c0, c1, acc, flags, sh)) return;
    if (i < n_obs) {
#pragma unroll
        for (int s = 0; s < Op::values; ++s)
            partial[((int64_t)blockIdx.y * Op::values + s) * n_obs + i] += acc[s];
    }
}

// Every pair by the closed form (use_closed says for which calls).
template <unsigned C>
__global__ __launch_bounds__(dev::kGzThreads) void magnetic_closed_kernel(
    const double *__restrict__ oe, const double *__restrict__ on, const double *__restrict__ ou,
    int n_obs, MagSource src, int64_t n_src, int64_t chunk_len, double *__restrict__ partial) {
    using Op = MagneticOp<C>;
    __shared__ dev::FieldClosedShared<Op> sh;
    const int64_t base = (int64_t)blockIdx.x * dev::kGzThreads, i = base + threadIdx.x;
    const int64_t c0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t c1 = c0 + chunk_len < n_src ? c0 + chunk_len : n_src;
    double acc[Op::values] = {};
    uint32_t flags = 0;
    dev::field_closed_chunk<Op>(src, oe, on, ou, base, n_obs, c0, c1, acc, flags, sh);
    if (i < n_obs) {
#pragma unroll
        for (int s = 0; s < Op::values; ++s)
            partial[((int64_t)blockIdx.y * Op::values + s) * n_obs + i] = acc[s];
    }
}

// out[s][perm[i]] = 1e9 * (sum over chunks in order of partial[c][s][i])
// (T -> nT; perm NULL: the identity).
template <int P>
__global__ __launch_bounds__(dev::SumShape<P>::threads) void reduce_magnetic_kernel(
    const double *__restrict__ partial, int64_t chunks, int nc, int64_t n_obs,
    const int *__restrict__ perm, double *__restrict__ out) {
    int64_t idx;
    double sum;
    if (!dev::chunk_sum<P>(partial, chunks, (int64_t)nc * n_obs, idx, sum)) return;
    const int s = (int)(idx / n_obs);
    const int64_t i = idx - (int64_t)s * n_obs;
    out[(int64_t)s * n_obs + (perm ? perm[i] : i)] = 1e9 * sum;
}

__global__ void fill_zero_mag_kernel(double *__restrict__ out, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = 0.0;
}

template <unsigned C>
int launch_magnetic(const double *oe, const double *on, const double *ou, int64_t n_obs,
                    const double *prisms, const double *me, const double *mn, const double *mu,
                    int64_t n_src, int64_t chunks, bool sorted, double *partial,
                    hipStream_t stream) {
    const int64_t chunk_len = (n_src + chunks - 1) / chunks;
    dim3 grid((unsigned)((n_obs + dev::kGzThreads - 1) / dev::kGzThreads), (unsigned)chunks);
    const MagSource src{prisms, me, mn, mu};
    if (use_closed(MagSet<C>::tensor, n_obs, n_src, sorted)) {
        hipLaunchKernelGGL((magnetic_closed_kernel<C>), grid, dim3(dev::kGzThreads), 0, stream, oe,
                           on, ou, (int)n_obs, src, n_src, chunk_len, partial);
        HMX_LAUNCHED("magnetic_closed_kernel");
        return HMX_OK;
    }
    hipLaunchKernelGGL((magnetic_far_kernel<C>), grid, dim3(dev::kGzThreads), 0, stream, oe, on, ou,
                       (int)n_obs, src, n_src, chunk_len, partial);
    HMX_LAUNCHED("magnetic_far_kernel");
    hipLaunchKernelGGL((magnetic_close_kernel<C>), grid, dim3(dev::kGzThreads), 0, stream, oe, on,
                       ou, (int)n_obs, src, n_src, chunk_len, partial);
    HMX_LAUNCHED("magnetic_close_kernel");
    return HMX_OK;
}

template <int P>
int launch_reduce_parts(const double *partial, int64_t chunks, int nc, int64_t n_obs,
                        const int *perm, double *out, hipStream_t stream) {
    using S = dev::SumShape<P>;
    const int64_t blocks = ((int64_t)nc * n_obs + S::outputs - 1) / S::outputs;
    hipLaunchKernelGGL((reduce_magnetic_kernel<P>), dim3((unsigned)blocks), dim3(S::threads), 0,
                       stream, partial, chunks, nc, n_obs, perm, out);
    HMX_LAUNCHED("reduce_magnetic_kernel");
    return HMX_OK;
}

int launch_reduce(const double *partial, int64_t chunks, int nc, int64_t n_obs, const int *perm,
                  double *out, hipStream_t stream) {
    return dev::sum_parts(chunks, (int64_t)nc * n_obs, 16) == 1
               ? launch_reduce_parts<1>(partial, chunks, nc, n_obs, perm, out, stream)
               : launch_reduce_parts<16>(partial, chunks, nc, n_obs, perm, out, stream);
}

bool valid_components(uint32_t mask) { return mask != 0 && (mask & ~7u) == 0; }

}  // namespace
}  // namespace hmx

extern "C" {

int hmx_prism_magnetic_workspace_bytes(int64_t n_obs, int64_t n_prisms, uint32_t component_mask,
                                       size_t *bytes) {
    hmx::clear_error();
    if (!bytes) return hmx::fail(HMX_ERR_ARG, "bytes is NULL");
    if (n_obs < 0 || n_prisms < 0) return hmx::fail(HMX_ERR_ARG, "negative size");
    if (n_obs > INT32_MAX || n_prisms > INT32_MAX)
        return hmx::fail(HMX_ERR_ARG, "more than 2^31-1 observation points or prisms");
    if (!hmx::valid_components(component_mask))
        return hmx::fail(HMX_ERR_ARG, "invalid component mask 0x%x", component_mask);
    const int cu = hmx::device_cu_count();
    if (cu < 0) return cu;
    const int64_t chunks = hmx::prism_chunks(n_obs, n_prisms, cu);
    *bytes = (size_t)chunks * (size_t)__builtin_popcount(component_mask) * (size_t)n_obs *
             sizeof(double);
    // the point order, after the partial sums
    if (hmx::use_point_order(n_obs, n_prisms))
        *bytes = hmx::point_order_offset(*bytes) + hmx::point_order_bytes(n_obs);
    return HMX_OK;
}

int hmx_prism_magnetic(const double *easting, const double *northing, const double *upward,
                       int64_t n_obs, const double *prisms, const double *magnetization_e,
                       const double *magnetization_n, const double *magnetization_u,
                       int64_t n_prisms, uint32_t component_mask, double *out, void *workspace,
                       size_t workspace_bytes, void *stream) {
    hmx::clear_error();
    if (n_obs < 0 || n_prisms < 0) return hmx::fail(HMX_ERR_ARG, "negative size");
    if (n_obs > INT32_MAX || n_prisms > INT32_MAX)
        return hmx::fail(HMX_ERR_ARG, "more than 2^31-1 observation points or prisms");
    if (!hmx::valid_components(component_mask))
        return hmx::fail(HMX_ERR_ARG, "invalid component mask 0x%x", component_mask);
    if (n_obs == 0) return HMX_OK;
    if (!out) return hmx::fail(HMX_ERR_ARG, "out is NULL");
    if (!easting || !northing || !upward) return hmx::fail(HMX_ERR_ARG, "NULL coordinate array");
    hipStream_t st = (hipStream_t)stream;
    const int nc = __builtin_popcount(component_mask);
    if (n_prisms == 0) {  // no prisms: zeros, as the reference's accumulators
        const int64_t total = (int64_t)nc * n_obs;
        hipLaunchKernelGGL(hmx::fill_zero_mag_kernel, dim3((unsigned)((total + 255) / 256)),
                           dim3(256), 0, st, out, total);
        HMX_LAUNCHED("fill_zero_mag_kernel");
        return HMX_OK;
    }
    if (!prisms || !magnetization_e || !magnetization_n || !magnetization_u)
        return hmx::fail(HMX_ERR_ARG, "NULL prism or magnetization array");
    const int cu = hmx::device_cu_count();
    if (cu < 0) return cu;
    const int64_t chunks = hmx::prism_chunks(n_obs, n_prisms, cu);
    const size_t partial_bytes = (size_t)chunks * (size_t)nc * (size_t)n_obs * sizeof(double);
    const size_t order_at = hmx::point_order_offset(partial_bytes);
    const size_t with_order = order_at + hmx::point_order_bytes(n_obs);
    const size_t need = hmx::need_point_order(n_obs, n_prisms) ? with_order : partial_bytes;
    const bool order = hmx::use_point_order(n_obs, n_prisms) && workspace_bytes >= with_order;
    if (!workspace || workspace_bytes < need)
        return hmx::fail(HMX_ERR_ARG, "workspace too small: %zu < %zu bytes", workspace_bytes,
                         need);
    double *partial = static_cast<double *>(workspace);
    // points in wavefront-coherent order (see point_order.hip)
    const int *perm = nullptr;
    if (order) {
        hmx::PointOrder po;
        const int ost = hmx::point_order(easting, northing, upward, n_obs,
                                         static_cast<char *>(workspace) + order_at, &po, st);
        if (ost) return ost;
        easting = po.e;
        northing = po.n;
        upward = po.u;
        perm = po.perm;
    }
    int rc;
    switch (component_mask) {
#define HMX_MAG_CASE(C)                                                                       \
    case C:                                                                                   \
        rc = hmx::launch_magnetic<C>(easting, northing, upward, n_obs, prisms,                \
                                     magnetization_e, magnetization_n, magnetization_u,       \
                                     n_prisms, chunks, order, partial, st);                   \
        break;
        HMX_MAG_CASE(1u)
        HMX_MAG_CASE(2u)
        HMX_MAG_CASE(3u)
        HMX_MAG_CASE(4u)
        HMX_MAG_CASE(5u)
        HMX_MAG_CASE(6u)
        HMX_MAG_CASE(7u)
#undef HMX_MAG_CASE
    default:
        return hmx::fail(HMX_ERR_ARG, "invalid component mask 0x%x", component_mask);
    }
    if (rc) return rc;
    return hmx::launch_reduce(partial, chunks, nc, n_obs, perm, out, st);
}

}  // extern "C"
