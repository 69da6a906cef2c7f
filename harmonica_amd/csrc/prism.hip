// Prism forward-modelling kernels (explicit prisms and prism layers).
//
// Launch shape: a workgroup owns 256 observation points (4 wavefronts, one
// point per lane, FP64 accumulators in VGPRs) and one chunk of the prism
// list.  Prisms are staged tile by tile into LDS and read back as
// wave-uniform broadcasts; each wavefront evaluates them in the far form or
// the closed form (prism_far.h, prism_fields_far.h).  Each chunk writes its
// partial sums to the workspace; a second kernel reduces the chunks in
// order and applies harmonica's units, so results are deterministic.
#include <mutex>

#include "chunk_sum.h"
#include "hmx_internal.h"
#include "prism_device.h"
#include "prism_fields_far.h"

namespace hmx {
namespace {

using dev::FieldSet;

// Sums the fields of FieldSet<M>, weight G * density.
template <unsigned M>
struct GravityOp {
    static constexpr unsigned fields = M;
    static constexpr int weights = 1, values = FieldSet<M>::count;
    __device__ static void combine(const double *weight, const double (&vs)[values],
                                   double (&out)[values]) {
#pragma unroll
        for (int s = 0; s < values; ++s) out[s] = weight[0] * vs[s];
    }
    template <bool kGeneral>
    __device__ static void closed(double e, double n, double u, const double *b,
                                  const double *weight, double (&acc)[values], uint32_t &flags,
                                  const dm::Tables &tab) {
        dev::prism_pair_path<M, kGeneral>(e, n, u, b[0], b[1], b[2], b[3], b[4], b[5], weight[0],
                                          acc, flags, tab);
    }
};

struct ExplicitSource : dev::GzExplicit {
    ExplicitSource(const double *p, const double *d) : dev::GzExplicit{p, d} {}
    using dev::GzExplicit::get;
    __device__ bool get(int64_t p, double (&b)[6], double (&weight)[1]) const {
        const bool skip = get(p, b, weight[0]);
        weight[0] *= dev::kG;
        return skip;
    }
};

// Prisms of a layer, enumerated easting-major as the reference loops
// (layer.py:590-594): p = j * n_north + k.  Bounds are centre -/+ half the
// first spacing (layer.py:584-585,592-593,609-610); skip rules of
// layer.py:595-607.
struct LayerSource {
    const double *ce, *cn, *bottom, *top, *density;
    int n_east, n_north;
    double threshold;
    __device__ bool get(int64_t p, double (&b)[6], double &rho) const {
        const unsigned j = (unsigned)p / (unsigned)n_north, k = (unsigned)p - j * (unsigned)n_north;
        const int64_t idx = (int64_t)k * n_east + j;
        const double half_e = (ce[1] - ce[0]) / 2, half_n = (cn[1] - cn[0]) / 2;
        b[0] = ce[j] - half_e;
        b[1] = ce[j] + half_e;
        b[2] = cn[k] - half_n;
        b[3] = cn[k] + half_n;
        b[4] = bottom[idx];
        b[5] = top[idx];
        rho = density[idx];
        return rho == 0.0 || rho != rho || (b[5] - b[4] < threshold) || b[5] != b[5] || b[4] != b[4];
    }
    __device__ bool get(int64_t p, double (&b)[6], double (&weight)[1]) const {
        const bool skip = get(p, b, weight[0]);
        weight[0] *= dev::kG;
        return skip;
    }
};

// The far pairs of any field set into the partial sums.
template <unsigned M, class Src>
__global__ __launch_bounds__(dev::kGzThreads, FieldSet<M>::count <= 3 ? 3 : 2) void
prism_far_kernel(const double *__restrict__ oe, const double *__restrict__ on,
                 const double *__restrict__ ou, int n_obs, Src src, int64_t n_src,
                 int64_t chunk_len, double *__restrict__ partial) {
    using Op = GravityOp<M>;
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

// The close pairs, added to the partial sums of prism_far_kernel.
template <unsigned M, class Src>
__global__ __launch_bounds__(dev::kGzThreads, FieldSet<M>::count <= 3 ? 4 : 3) void
prism_close_kernel(const double *__restrict__ oe, const double *__restrict__ on,
                   const double *__restrict__ ou, int n_obs, Src src, int64_t n_src,
                   int64_t chunk_len, double *__restrict__ partial,
                   uint32_t *__restrict__ flags) {
    using Op = GravityOp<M>;
    __shared__ dev::FieldCloseShared<Op> sh;
    const unsigned bx = (blockIdx.x + blockIdx.y) % gridDim.x;
    const int64_t base = (int64_t)bx * dev::kGzThreads, i = base + threadIdx.x;
    const int64_t c0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t c1 = c0 + chunk_len < n_src ? c0 + chunk_len : n_src;
    double acc[Op::values] = {};
    uint32_t found = 0;
    if (!dev::field_close_chunk<Op>(src, oe, on, ou, base, n_obs, c0, c1, acc, found, sh)) return;
    if (i < n_obs) {
#pragma unroll
        for (int s = 0; s < Op::values; ++s)
            partial[((int64_t)blockIdx.y * Op::values + s) * n_obs + i] += acc[s];
    }
    if (FieldSet<M>::tensor && flags && found) atomicOr(flags, found);
}

// Every pair by the closed form (use_closed says for which calls).
template <unsigned M, class Src>
__global__ __launch_bounds__(dev::kGzThreads) void prism_closed_kernel(
    const double *__restrict__ oe, const double *__restrict__ on, const double *__restrict__ ou,
    int n_obs, Src src, int64_t n_src, int64_t chunk_len, double *__restrict__ partial,
    uint32_t *__restrict__ flags) {
    using Op = GravityOp<M>;
    __shared__ dev::FieldClosedShared<Op> sh;
    const int64_t base = (int64_t)blockIdx.x * dev::kGzThreads, i = base + threadIdx.x;
    const int64_t c0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t c1 = c0 + chunk_len < n_src ? c0 + chunk_len : n_src;
    double acc[Op::values] = {};
    uint32_t found = 0;
    dev::field_closed_chunk<Op>(src, oe, on, ou, base, n_obs, c0, c1, acc, found, sh);
    if (i < n_obs) {
#pragma unroll
        for (int s = 0; s < Op::values; ++s)
            partial[((int64_t)blockIdx.y * Op::values + s) * n_obs + i] = acc[s];
    }
    if (FieldSet<M>::tensor && flags && found) atomicOr(flags, found);
}

// g_u alone, each prism in the far form or the closed form (prism_far.h).
template <class Src>
__global__ __launch_bounds__(dev::kGzThreads, 4) void prism_gz_kernel(
    const double *__restrict__ oe, const double *__restrict__ on, const double *__restrict__ ou,
    int n_obs, Src src, int64_t n_src, int64_t chunk_len, double *__restrict__ partial) {
    __shared__ dev::GzShared sh;
    dm::load_tables(&sh.tables);
    // Consecutive workgroups go to the 8 XCDs in turn: with a multiple of 8
    // point blocks, rotate them from chunk to chunk, or the XCD of a block in
    // the middle of the model gets its near prisms chunk after chunk.
    const unsigned bx = (blockIdx.x + blockIdx.y) % gridDim.x;
    const int64_t base = (int64_t)bx * dev::kGzThreads, i = base + threadIdx.x;
    const bool valid = i < n_obs;
    const int64_t ii = valid ? i : n_obs - 1;
    dev::GzPoint pt{oe[ii], on[ii], ou[ii], 0.0, 0.0, oe[base], on[base]};
    pt.x = pt.e - pt.xo;
    pt.y = pt.n - pt.yo;
    double acc = 0.0;
    bool sure = false;
    const int64_t c0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t c1 = c0 + chunk_len < n_src ? c0 + chunk_len : n_src;
    if (c0 < c1) dev::gz_table(src, c0, sh);
    dev::point_box(pt, sh.box);
    for (int64_t t0 = c0; t0 < c1; t0 += dev::kGzTile) {
        const int cnt = (int)(c1 - t0 < dev::kGzTile ? c1 - t0 : dev::kGzTile);
        dev::gz_stage(src, t0, cnt, pt.xo, pt.yo, sh);
        if (t0 == c0) sure = dev::gz_sure(sh);
        dev::gz_tile(cnt, sure, pt, acc, sh);
    }
    if (valid) partial[(int64_t)blockIdx.y * n_obs + i] = acc;
}

// Singular-point scan: bit f of *flags is set when some (point, prism)
// pair is a singular point of tensor field f (replaces the serial scans
// _any_singular_point_g_* of gravity.py:272-449).  Singular points lie in the
// prism's closed box: a lane tests a prism's box against the box of its
// wave's points, and only prisms that pass are tested point by point (20,011
// bodies below 2999 stations: 100 -> 9 us).
__global__ __launch_bounds__(kObsPerBlock) void singular_scan_kernel(
    const double *__restrict__ oe, const double *__restrict__ on, const double *__restrict__ ou,
    int n_obs, const double *__restrict__ prisms, int64_t n_src, int64_t chunk_len,
    uint32_t mask, uint32_t *__restrict__ flags) {
    const int i = blockIdx.x * kObsPerBlock + threadIdx.x, lane = threadIdx.x & 63;
    const int ii = i < n_obs ? i : n_obs - 1;
    const double e = oe[ii], n = on[ii], u = ou[ii];
    const dev::FarBox box{dev::wave_min(e), dev::wave_max(e), dev::wave_min(n),
                          dev::wave_max(n), dev::wave_min(u), dev::wave_max(u),
                          0.0};
    uint32_t found = 0;
    const int64_t c0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t c1 = c0 + chunk_len < n_src ? c0 + chunk_len : n_src;
    for (int64_t t0 = c0; t0 < c1; t0 += 64) {
        bool meets = false;
        if (t0 + lane < c1) {
            const double *b = prisms + 6 * (t0 + lane);
            meets = fmin(b[0], b[1]) <= box.x1 && box.x0 <= fmax(b[0], b[1]) &&
                    fmin(b[2], b[3]) <= box.y1 && box.y0 <= fmax(b[2], b[3]) &&
                    fmin(b[4], b[5]) <= box.u1 && box.u0 <= fmax(b[4], b[5]);
        }
        dev::for_bits((uint64_t)__ballot(meets), [&](int p) {
            const double *b = prisms + 6 * (t0 + p);
            const bool in_e = b[0] <= e && e <= b[1], in_n = b[2] <= n && n <= b[3];
            const bool in_u = b[4] <= u && u <= b[5];
            const bool at_e = e == b[0] || e == b[1], at_n = n == b[2] || n == b[3];
            const bool at_u = u == b[4] || u == b[5];
            const bool edge_e = in_e && at_n && at_u, edge_n = in_n && at_e && at_u;
            const bool edge_u = in_u && at_e && at_n;
            found |= (edge_n || edge_u) ? 1u << 4 : 0u;
            found |= (edge_e || edge_u) ? 1u << 5 : 0u;
            found |= (edge_e || edge_n) ? 1u << 6 : 0u;
            found |= edge_u ? 1u << 7 : 0u;
            found |= edge_n ? 1u << 8 : 0u;
            found |= edge_e ? 1u << 9 : 0u;
        });
    }
    found &= mask;
    if (found) atomicOr(flags, found);
}

// out[s][perm[i]] = units(sum over chunks of partial[c][s][i]) (perm NULL: the
// identity), four waves per 64 outputs (4096 points: 79 chunks took 11 us with a
// thread per output, 313 chunks take 9) or a thread each (sum_parts).
template <int P>
__global__ __launch_bounds__(dev::SumShape<P>::threads) void reduce_chunks_kernel(
    const double *__restrict__ partial, int64_t chunks, int nf, int64_t n_obs, uint32_t mask,
    const int *__restrict__ perm, double *__restrict__ out) {
    int64_t idx;
    double sum;
    if (!dev::chunk_sum<P>(partial, chunks, (int64_t)nf * n_obs, idx, sum)) return;
    const int s = (int)(idx / n_obs);
    const int64_t i = idx - (int64_t)s * n_obs;
    int f = 0, seen = -1;
    for (; f < 10; ++f)
        if ((mask >> f) & 1u)
            if (++seen == s) break;
    out[(int64_t)s * n_obs + (perm ? perm[i] : i)] = dev::to_harmonica_units(f, sum);
}

// Zero fill with a kernel (stays valid inside captured HIP graphs).
__global__ void fill_zero_kernel(double *__restrict__ out, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = 0.0;
}

template <unsigned M, class Src>
int launch_forward(const double *oe, const double *on, const double *ou, int64_t n_obs,
                   const Src &src, int64_t n_src, int64_t chunks, bool sorted, double *partial,
                   uint32_t *flags, hipStream_t stream) {
    const int64_t chunk_len = (n_src + chunks - 1) / chunks;
    dim3 grid((unsigned)((n_obs + dev::kGzThreads - 1) / dev::kGzThreads), (unsigned)chunks);
    if (use_closed(M, n_obs, n_src, sorted)) {
        hipLaunchKernelGGL((prism_closed_kernel<M, Src>), grid, dim3(dev::kGzThreads), 0, stream,
                           oe, on, ou, (int)n_obs, src, n_src, chunk_len, partial, flags);
        HMX_LAUNCHED("prism_closed_kernel");
        return HMX_OK;
    }
    if constexpr (M == 0x8u) {
        hipLaunchKernelGGL((prism_gz_kernel<Src>), grid, dim3(dev::kGzThreads), 0, stream, oe, on,
                           ou, (int)n_obs, src, n_src, chunk_len, partial);
        HMX_LAUNCHED("prism_gz_kernel");
    } else {
        hipLaunchKernelGGL((prism_far_kernel<M, Src>), grid, dim3(dev::kGzThreads), 0, stream, oe,
                           on, ou, (int)n_obs, src, n_src, chunk_len, partial);
        HMX_LAUNCHED("prism_far_kernel");
        hipLaunchKernelGGL((prism_close_kernel<M, Src>), grid, dim3(dev::kGzThreads), 0, stream, oe,
                           on, ou, (int)n_obs, src, n_src, chunk_len, partial, flags);
        HMX_LAUNCHED("prism_close_kernel");
    }
    return HMX_OK;
}

template <int P>
int launch_reduce_parts(const double *partial, int64_t chunks, int nf, int64_t n_obs, uint32_t mask,
                        const int *perm, double *out, hipStream_t stream) {
    using S = dev::SumShape<P>;
    const int64_t blocks = ((int64_t)nf * n_obs + S::outputs - 1) / S::outputs;
    hipLaunchKernelGGL((reduce_chunks_kernel<P>), dim3((unsigned)blocks), dim3(S::threads), 0,
                       stream, partial, chunks, nf, n_obs, mask, perm, out);
    HMX_LAUNCHED("reduce_chunks_kernel");
    return HMX_OK;
}

int launch_reduce(const double *partial, int64_t chunks, int nf, int64_t n_obs, uint32_t mask,
                  const int *perm, double *out, hipStream_t stream) {
    return dev::sum_parts(chunks, (int64_t)nf * n_obs, 4) == 1
               ? launch_reduce_parts<1>(partial, chunks, nf, n_obs, mask, perm, out, stream)
               : launch_reduce_parts<4>(partial, chunks, nf, n_obs, mask, perm, out, stream);
}

// Field sets with their own kernel instantiation: each single field, the
// three accelerations, the six tensor terms and all ten.
template <class Src>
int dispatch_mask(uint32_t mask, const double *oe, const double *on, const double *ou,
                  int64_t n_obs, const Src &src, int64_t n_src, int64_t chunks, bool sorted,
                  double *partial, uint32_t *flags, hipStream_t stream) {
#define HMX_CASE(MASK)                                                                          \
    case MASK:                                                                                  \
        return launch_forward<MASK, Src>(oe, on, ou, n_obs, src, n_src, chunks, sorted, partial, \
                                         flags, stream);
    switch (mask) {
        HMX_CASE(0x001u)
        HMX_CASE(0x002u)
        HMX_CASE(0x004u)
        HMX_CASE(0x008u)
        HMX_CASE(0x010u)
        HMX_CASE(0x020u)
        HMX_CASE(0x040u)
        HMX_CASE(0x080u)
        HMX_CASE(0x100u)
        HMX_CASE(0x200u)
        HMX_CASE(0x00eu)
        HMX_CASE(0x3f0u)
        HMX_CASE(0x3ffu)
    }
#undef HMX_CASE
    return fail(HMX_ERR_ARG, "no kernel for field mask 0x%x", mask);
}

bool has_kernel(uint32_t mask) {
    return __builtin_popcount(mask) == 1 || mask == 0x00eu || mask == 0x3f0u || mask == 0x3ffu;
}

// Run the forward model for any field mask: one launch when the mask has
// its own kernel, else one launch per field reusing the workspace.
// chunk_cap > 0 limits the number of source chunks (so that the partial
// sums fit a fixed scratch buffer; the point order then depends on what is
// left of it).  Calls that pass
// use_point_order evaluate the points in wavefront-coherent order, sorted
// into the workspace after the room for all fields' partial sums (the
// layout hmx_forward_workspace_bytes sizes).
template <class Src>
int run_forward(const double *oe, const double *on, const double *ou, int64_t n_obs,
                const Src &src, int64_t n_src, uint32_t mask, double *out, uint32_t *flags,
                void *workspace, size_t workspace_bytes, hipStream_t stream,
                int64_t chunk_cap = 0) {
    if (n_obs <= 0) return HMX_OK;
    int cu = device_cu_count();
    if (cu < 0) return cu;
    const int nf = popcount10(mask);
    int64_t chunks = prism_chunks(n_obs, n_src, cu);
    if (chunk_cap > 0 && chunks > chunk_cap) chunks = chunk_cap;
    if (n_src == 0) {
        // No sources: the reference returns zeros.
        int64_t total = (int64_t)nf * n_obs;
        hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                           stream, out, total);
        HMX_LAUNCHED("fill_zero_kernel");
        return HMX_OK;
    }
    const size_t need_one = (size_t)chunks * (size_t)n_obs * sizeof(double);
    double *partial = static_cast<double *>(workspace);
    const size_t order_at = point_order_offset(need_one * nf);
    const size_t with_order = order_at + point_order_bytes(n_obs);
    const size_t need = chunk_cap == 0 && need_point_order(n_obs, n_src) ? with_order
                        : has_kernel(mask)                          ? need_one * nf
                                                                    : need_one;
    const bool order = use_point_order(n_obs, n_src) && workspace_bytes >= with_order;
    if (!workspace || workspace_bytes < need)
        return fail(HMX_ERR_ARG, "workspace too small: %zu < %zu bytes", workspace_bytes, need);
    const int *perm = nullptr;
    if (order) {
        PointOrder po;
        int st = point_order(oe, on, ou, n_obs, static_cast<char *>(workspace) + order_at, &po,
                             stream);
        if (st) return st;
        oe = po.e;
        on = po.n;
        ou = po.u;
        perm = po.perm;
    }
    if (has_kernel(mask)) {
        int st = dispatch_mask<Src>(mask, oe, on, ou, n_obs, src, n_src, chunks, order, partial,
                                    flags, stream);
        if (st) return st;
        return launch_reduce(partial, chunks, nf, n_obs, mask, perm, out, stream);
    }
    int s = 0;
    for (int f = 0; f < 10; ++f) {
        if (!((mask >> f) & 1u)) continue;
        uint32_t m = 1u << f;
        int st = dispatch_mask<Src>(m, oe, on, ou, n_obs, src, n_src, chunks, order, partial,
                                    flags, stream);
        if (st) return st;
        st = launch_reduce(partial, chunks, 1, n_obs, m, perm, out + (int64_t)s * n_obs, stream);
        if (st) return st;
        ++s;
    }
    return HMX_OK;
}

int check_common(int64_t n_obs, int64_t n_src, uint32_t mask, const void *out) {
    if (n_obs < 0 || n_src < 0) return fail(HMX_ERR_ARG, "negative size");
    if (n_obs > INT32_MAX || n_src > INT32_MAX)
        return fail(HMX_ERR_ARG, "more than 2^31-1 observation points or sources");
    if (mask == 0 || (mask & ~HMX_ALL_FIELDS)) return fail(HMX_ERR_ARG, "invalid field mask 0x%x", mask);
    if (n_obs > 0 && !out) return fail(HMX_ERR_ARG, "out is NULL");
    return HMX_OK;
}

// Scratch of hmx_prism_gravity_static: the chunk partial sums, in a
// file-scope device array (one per device, held until the process ends).
// Host code uses its per-device address from hipGetSymbolAddress, never the
// array's name.
constexpr int64_t kStaticScratchDoubles = (int64_t)1 << 22;  // 32 MiB
__device__ __align__(256) double scratch[kStaticScratchDoubles];

std::mutex g_scratch_mutex;
double *g_scratch_ptr[kMaxDevices] = {};

// Address of the current device's scratch array (looked up once per
// device, with that device current).
int static_scratch(double **out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(HMX_ERR_NODEV, "no HIP device: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return fail(HMX_ERR_NODEV, "device index %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(HMX_ERR_HIP, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                        hipGetErrorString(e));
        g_scratch_ptr[dev] = static_cast<double *>(p);
    }
    *out = g_scratch_ptr[dev];
    return HMX_OK;
}

}  // namespace
}  // namespace hmx

extern "C" {

int hmx_prism_gravity_static(const double *easting, const double *northing,
                             const double *upward, int64_t n_obs, const double *prisms,
                             const double *density, int64_t n_prisms, uint32_t field_mask,
                             double *out, uint32_t *singular_flags, void *stream) {
    using namespace hmx;
    clear_error();
    int st = check_common(n_obs, n_prisms, field_mask, out);
    if (st) return st;
    if (n_obs > 0 && (!easting || !northing || !upward))
        return fail(HMX_ERR_ARG, "NULL coordinate array");
    if (n_prisms > 0 && (!prisms || !density)) return fail(HMX_ERR_ARG, "NULL prism array");
    // one launch holds the partial sums of all its fields for at least one
    // chunk: n_obs x (fields of one launch) doubles
    const int64_t per_chunk = n_obs * (has_kernel(field_mask) ? popcount10(field_mask) : 1);
    if (per_chunk > kStaticScratchDoubles)
        return fail(HMX_ERR_ARG,
                    "hmx_prism_gravity_static: %lld observation points x fields exceed its scratch "
                    "of %lld doubles (use hmx_prism_gravity with a workspace)",
                    (long long)per_chunk, (long long)kStaticScratchDoubles);
    if (n_obs == 0) return HMX_OK;
    double *ws = nullptr;
    st = static_scratch(&ws);
    if (st) return st;
    ExplicitSource src{prisms, density};
    return run_forward(easting, northing, upward, n_obs, src, n_prisms, field_mask, out,
                       singular_flags, ws, (size_t)kStaticScratchDoubles * sizeof(double),
                       (hipStream_t)stream, kStaticScratchDoubles / per_chunk);
}

int hmx_prism_gravity(const double *easting, const double *northing, const double *upward,
                      int64_t n_obs, const double *prisms, const double *density,
                      int64_t n_prisms, uint32_t field_mask, double *out,
                      uint32_t *singular_flags, void *workspace, size_t workspace_bytes,
                      void *stream) {
    hmx::clear_error();
    int st = hmx::check_common(n_obs, n_prisms, field_mask, out);
    if (st) return st;
    if (n_obs > 0 && (!easting || !northing || !upward))
        return hmx::fail(HMX_ERR_ARG, "NULL coordinate array");
    if (n_prisms > 0 && (!prisms || !density)) return hmx::fail(HMX_ERR_ARG, "NULL prism array");
    hmx::ExplicitSource src{prisms, density};
    return hmx::run_forward(easting, northing, upward, n_obs, src, n_prisms, field_mask, out,
                            singular_flags, workspace, workspace_bytes, (hipStream_t)stream);
}

int hmx_prism_singular_scan(const double *easting, const double *northing, const double *upward,
                            int64_t n_obs, const double *prisms, int64_t n_prisms,
                            uint32_t field_mask, uint32_t *flags, void *stream) {
    hmx::clear_error();
    int st = hmx::check_common(n_obs, n_prisms, field_mask, flags);
    if (st) return st;
    if (n_obs == 0 || n_prisms == 0) return HMX_OK;
    if (!easting || !northing || !upward || !prisms)
        return hmx::fail(HMX_ERR_ARG, "NULL input array");
    int cu = hmx::device_cu_count();
    if (cu < 0) return cu;
    const int64_t chunks = hmx::forward_chunks(n_obs, n_prisms, cu);
    const int64_t chunk_len = (n_prisms + chunks - 1) / chunks;
    dim3 grid((unsigned)((n_obs + hmx::kObsPerBlock - 1) / hmx::kObsPerBlock), (unsigned)chunks);
    hipLaunchKernelGGL(hmx::singular_scan_kernel, grid, dim3(hmx::kObsPerBlock), 0,
                       (hipStream_t)stream, easting, northing, upward, (int)n_obs, prisms,
                       n_prisms, chunk_len, field_mask, flags);
    HMX_LAUNCHED("singular_scan_kernel");
    return HMX_OK;
}

int hmx_prism_layer_gravity(const double *easting, const double *northing, const double *upward,
                            int64_t n_obs, const double *centre_easting, int64_t n_east,
                            const double *centre_northing, int64_t n_north,
                            const double *bottom, const double *top, const double *density,
                            double thickness_threshold, uint32_t field_mask, double *out,
                            uint32_t *singular_flags, void *workspace, size_t workspace_bytes,
                            void *stream) {
    hmx::clear_error();
    if (n_east < 2 || n_north < 2)
        return hmx::fail(HMX_ERR_ARG, "a prism layer needs at least 2 centres per direction");
    int st = hmx::check_common(n_obs, n_east * n_north, field_mask, out);
    if (st) return st;
    if (n_obs > 0 && (!easting || !northing || !upward))
        return hmx::fail(HMX_ERR_ARG, "NULL coordinate array");
    if (!centre_easting || !centre_northing || !bottom || !top || !density)
        return hmx::fail(HMX_ERR_ARG, "NULL layer array");
    hmx::LayerSource src{centre_easting, centre_northing, bottom, top, density,
                         (int)n_east, (int)n_north, thickness_threshold};
    return hmx::run_forward(easting, northing, upward, n_obs, src, n_east * n_north, field_mask,
                            out, singular_flags, workspace, workspace_bytes, (hipStream_t)stream);
}

}  // extern "C"
