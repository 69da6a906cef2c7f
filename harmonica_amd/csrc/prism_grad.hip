// Derivatives of the prism g_z forward model with respect to prism
// densities and prism top heights (no counterpart in the reference, whose
// path is forward-only).
//
// With S(i, p) = sum over the 8 vertices of (-1)^(i+j+k) K_u (the g_u vertex
// sum of prism p at point i, without G rho) and
// F(i, p) = sum over the 4 top vertices of (-1)^(i+j) A_z (x, y, T - u),
//   d g_u(i) / d rho_p = G S(i, p),   d g_u(i) / d T_p = G rho_p F(i, p):
// only the top vertices depend on T, and summed over them with their signs
// d K_u / d z reduces to A_z (the other terms cancel pairwise across the
// east/west and north/south bounds).  F reuses the top-vertex arctangents
// of S, so one pass yields both.
//
//   gz_jvp: out_i = sum_p a_p S(i, p) + b_p F(i, p)     (point per lane,
//           prisms staged in LDS, chunk partials reduced in order)
//   gz_vjp: ga_p = sum_i v_i S(i, p),  gb_p = sum_i v_i F(i, p)
//           (prism per lane, points staged in LDS, partials per point chunk
//           reduced in order)
// Outputs are the raw sums; the caller applies G and harmonica's -1e5
// (g_z in mGal points down).
#include "hmx_internal.h"
#include "prism_far.h"

namespace hmx {
namespace {

// S and F of one prism at one point.
__device__ __forceinline__ void gz_sums(double e, double n, double u, double W, double E, double S,
                                        double N, double B, double T, const dm::Tables &tab,
                                        double &s_out, double &f_out) {
    s_out = dev::gu_sum_paired<true>(E - e, W - e, N - n, S - n, T - u, B - u, tab, &f_out);
}

struct alignas(16) StagedGradPrism {
    double w, e, s, n, b, t, a, c;  // bounds, weights (a: S, c: F)
};

// Bounds of prism p and whether it is skipped (layer rules minus the zero
// density rule: the derivative with respect to a zero density is not zero).
struct ExplicitGeom {
    const double *prisms;
    __device__ bool get(int64_t p, double (&bnd)[6]) const {
        for (int c = 0; c < 6; ++c) bnd[c] = prisms[6 * p + c];
        return false;
    }
    // index of prism p in the per-prism arrays
    __device__ int64_t index(int64_t p) const { return p; }
};

struct LayerGeom {
    const double *ce, *cn, *bottom, *top, *density;
    int n_east, n_north;
    double threshold;
    __device__ bool get(int64_t p, double (&bnd)[6]) const {
        const unsigned j = (unsigned)p / (unsigned)n_north, k = (unsigned)p - j * (unsigned)n_north;
        const int64_t idx = (int64_t)k * n_east + j;
        const double half_e = (ce[1] - ce[0]) / 2, half_n = (cn[1] - cn[0]) / 2;
        bnd[0] = ce[j] - half_e;
        bnd[1] = ce[j] + half_e;
        bnd[2] = cn[k] - half_n;
        bnd[3] = cn[k] + half_n;
        bnd[4] = bottom[idx];
        bnd[5] = top[idx];
        const double d = density[idx];
        return d != d || (bnd[5] - bnd[4] < threshold) || bnd[5] != bnd[5] || bnd[4] != bnd[4];
    }
    // layer arrays are (n_north, n_east) row-major
    __device__ int64_t index(int64_t p) const {
        const int j = (int)(p / n_north), k = (int)(p - (int64_t)j * n_north);
        return (int64_t)k * n_east + j;
    }
};

template <class Geom>
__global__ __launch_bounds__(kObsPerBlock) void gz_jvp_kernel(
    const double *__restrict__ oe, const double *__restrict__ on, const double *__restrict__ ou,
    int n_obs, Geom geom, const double *__restrict__ wa, const double *__restrict__ wb,
    int64_t n_src, int64_t chunk_len, double *__restrict__ partial) {
    __shared__ StagedGradPrism tile[kTile];
    __shared__ dm::Tables tables;
    dm::load_tables(&tables);
    const int i = blockIdx.x * kObsPerBlock + threadIdx.x;
    const bool valid = i < n_obs;
    const int ii = valid ? i : n_obs - 1;
    const double e = oe[ii], n = on[ii], u = ou[ii];
    double acc = 0.0;
    const int64_t c0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t c1 = c0 + chunk_len < n_src ? c0 + chunk_len : n_src;
    for (int64_t t0 = c0; t0 < c1; t0 += kTile) {
        const int cnt = (int)(c1 - t0 < kTile ? c1 - t0 : kTile);
        __syncthreads();
        for (int q = threadIdx.x; q < cnt; q += blockDim.x) {
            double bnd[6];
            const bool skip = geom.get(t0 + q, bnd);
            const int64_t idx = geom.index(t0 + q);
            StagedGradPrism sp;
            sp.w = bnd[0];
            sp.e = bnd[1];
            sp.s = bnd[2];
            sp.n = bnd[3];
            sp.b = bnd[4];
            sp.t = bnd[5];
            sp.a = skip ? 0.0 : wa[idx];
            sp.c = skip ? 0.0 : (wb ? wb[idx] : 0.0);
            tile[q] = sp;
        }
        __syncthreads();
        for (int p = 0; p < cnt; ++p) {
            const StagedGradPrism sp = tile[p];
            if (sp.a == 0.0 && sp.c == 0.0) continue;
            double S, F;
            gz_sums(e, n, u, sp.w, sp.e, sp.s, sp.n, sp.b, sp.t, tables, S, F);
            acc = fma(sp.a, S, fma(sp.c, F, acc));
        }
    }
    if (valid) partial[(int64_t)blockIdx.y * n_obs + i] = acc;
}

// Points staged per pass of the VJP kernel: one per lane of a wave, so that a
// wave sorts a tile into the forms with one comparison and one ballot.
constexpr int kVjpTile = 64;

// A lane's prism: bounds, and its rectangle's centre from the origin.
struct VjpPrism {
    double b[6];
    double x, y, area;
};

// v S and v F at the staged point o (x and y from the origin) by order 2I of
// the far form (prism_far.h): F = area z <1/r^3> at the top face.
template <int I, class Consts>
__device__ __forceinline__ void vjp_far(const VjpPrism &p, const Consts &c, const double4 &o,
                                        double &ga, double &gb) {
    const double x = p.x - o.x, y = p.y - o.y, zt = p.b[5] - o.z;
    const double X = x * x, Y = y * y, s = X + Y;
    double C[2 * I + 1], ft, f3;
    dev::far_coefs<I>(X, Y, c, C);
    const double fb = dev::far_face<I>(s, p.b[4] - o.z, C);
    dev::far_face_top<I>(s, zt, C, ft, f3);
    const double w = o.w * p.area;
    ga = fma(w, fb - ft, ga);
    gb = fma(w * zt, f3, gb);
}

// One prism per lane, points in LDS.  Workgroups whose prisms have equal
// rectangles (every layer) take the far form wherever it serves all prisms of
// a wave (by the bounding boxes of their centres, tops and bottoms), its
// constants in scalar registers up to order 6; nearer points go lane by lane
// as in the forward kernel, order 12 or the closed form by the lane's own
// distance.  200 x 200 layer and 128 x 128
// points: 7.06 -> 2.2 ms (every pair in the closed form before), bound by FP64
// issue (85% of the issue cycles while the CUs are busy).
template <class Geom>
__global__ __launch_bounds__(kObsPerBlock, 3) void gz_vjp_kernel(
    const double *__restrict__ oe, const double *__restrict__ on, const double *__restrict__ ou,
    const double *__restrict__ v, int64_t n_obs, Geom geom, int64_t n_src, int64_t chunk_len,
    double *__restrict__ partial_a, double *__restrict__ partial_b) {
    __shared__ double4 tile[kVjpTile];
    __shared__ alignas(16) double consts[dev::kFarStride];
    __shared__ int same[kObsPerBlock / 64];
    __shared__ dm::Tables tables;
    dm::load_tables(&tables);
    const int lane = threadIdx.x & 63;
    const int64_t p0 = (int64_t)blockIdx.x * kObsPerBlock, p = p0 + threadIdx.x;
    const bool valid = p < n_src;
    VjpPrism pr;
    const bool live = !geom.get(valid ? p : n_src - 1, pr.b) && valid;
    double first[6];
    geom.get(p0, first);
    const double xo = first[0], yo = first[2];
    pr.x = 0.5 * ((pr.b[0] - xo) + (pr.b[1] - xo));
    pr.y = 0.5 * ((pr.b[2] - yo) + (pr.b[3] - yo));
    pr.area = (pr.b[1] - pr.b[0]) * (pr.b[3] - pr.b[2]);
    double A, B, A0, B0;
    dev::half_sides2(pr.b, A, B);
    dev::half_sides2(first, A0, B0);
    const bool like = dev::far_alike(A, B, A0, B0);
    const bool all_like = !dev::any_lane(live && !like);
    if (lane == 0) same[threadIdx.x >> 6] = all_like;
    if (threadIdx.x < 3) dev::far_consts(A0, B0, threadIdx.x, consts);
    // boxes of the wave's live prisms: centres and tops, and bottoms
    const double inf = __builtin_inf();
    const dev::FarBox box{dev::wave_min(live ? pr.x : inf),    dev::wave_max(live ? pr.x : -inf),
                          dev::wave_min(live ? pr.y : inf),    dev::wave_max(live ? pr.y : -inf),
                          dev::wave_min(live ? pr.b[5] : inf), dev::wave_max(live ? pr.b[5] : -inf),
                          0.0};
    const double b0 = dev::wave_min(live ? pr.b[4] : inf);
    const double b1 = dev::wave_max(live ? pr.b[4] : -inf);
    const bool any_live = dev::any_lane(live);
    const double h2 = dev::far_half2(A0, B0);
    __syncthreads();
    bool use_far = true;
#pragma unroll
    for (int w = 0; w < kObsPerBlock / 64; ++w) use_far = use_far && same[w] != 0;
    double ga = 0.0, gb = 0.0;
    const int64_t c0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t c1 = c0 + chunk_len < n_obs ? c0 + chunk_len : n_obs;
    for (int64_t t0 = c0; t0 < c1; t0 += kVjpTile) {
        const int cnt = (int)(c1 - t0 < kVjpTile ? c1 - t0 : kVjpTile);
        __syncthreads();
        for (int q = threadIdx.x; q < cnt; q += blockDim.x)
            tile[q] = make_double4(oe[t0 + q], on[t0 + q], ou[t0 + q], v[t0 + q]);
        __syncthreads();
        if (!any_live) continue;
        uint64_t rest = cnt == 64 ? ~0ull : (1ull << cnt) - 1ull;
        double point_h2 = h2;  // of the lane's point
        uint64_t m2 = 0, m3 = 0, m4 = 0, m5 = 0, m6 = 0;
        if (use_far) {
            const double4 o = tile[lane < cnt ? lane : 0];
            const double x = o.x - xo, y = o.y - yo;
            const double guard = ((x - box.x0) + (y - box.y0) + (o.z - box.u0) + (o.z - b0)) * 0.0;
            const double dx = fmax(fmax(box.x0 - x, x - box.x1), 0.0);
            const double dy = fmax(fmax(box.y0 - y, y - box.y1), 0.0);
            const double dt = fmax(fmax(box.u0 - o.z, o.z - box.u1), 0.0);
            const double db = fmax(fmax(b0 - o.z, o.z - b1), 0.0);
            const double d = fmin(dt, db);
            const double d2 = fma(dx, dx, fma(dy, dy, d * d)) + guard;
            point_h2 = dev::far_sure_half2<dev::kFarMax>(h2, dev::far_reach(fma(x, x, y * y)));
            auto take = [&](bool far) {
                const uint64_t m = __ballot(far) & rest;
                rest &= ~m;
                return m;
            };
            m2 = take(dev::far_enough<2>(d2, point_h2));
            m3 = take(dev::far_enough<3>(d2, point_h2));
            m4 = take(dev::far_enough<4>(d2, point_h2));
            m5 = take(dev::far_enough<5>(d2, point_h2));
            m6 = take(dev::far_enough<6>(d2, point_h2));
        }
        auto point = [&](int q) {
            const double4 o = tile[q];
            return make_double4(o.x - xo, o.y - yo, o.z, o.w);
        };
        const dev::FarLds lds{consts};
        if (m2) {
            const dev::FarScalar<2> c(consts);
            dev::for_bits(m2, [&](int q) { vjp_far<2>(pr, c, point(q), ga, gb); });
        }
        if (m3) {
            const dev::FarScalar<3> c(consts);
            dev::for_bits(m3, [&](int q) { vjp_far<3>(pr, c, point(q), ga, gb); });
        }
        dev::for_bits(m4, [&](int q) { vjp_far<4>(pr, lds, point(q), ga, gb); });
        dev::for_bits(m5, [&](int q) { vjp_far<5>(pr, lds, point(q), ga, gb); });
        dev::for_bits(m6, [&](int q) { vjp_far<6>(pr, lds, point(q), ga, gb); });
        dev::for_bits(rest, [&](int q) {
            const double4 o = tile[q];
            bool close = true;
            if (use_far) {
                const double x = pr.x - (o.x - xo), y = pr.y - (o.y - yo);
                const double t = pr.b[5] - o.z, z = pr.b[4] - o.z;
                close = !dev::far_enough<dev::kFarMax>(fma(x, x, fma(y, y, fmin(t * t, z * z))),
                                                       dev::lane_value(point_h2, q));
                if (dev::any_lane(live && !close)) {
                    double sa = 0.0, sb = 0.0;
                    vjp_far<dev::kFarMax>(pr, lds, point(q), sa, sb);
                    ga += close ? 0.0 : sa;
                    gb += close ? 0.0 : sb;
                }
            }
            if (!dev::any_lane(live && close)) return;
            double S, F;
            gz_sums(o.x, o.y, o.z, pr.b[0], pr.b[1], pr.b[2], pr.b[3], pr.b[4], pr.b[5], tables, S,
                    F);
            ga = close ? fma(o.w, S, ga) : ga;
            gb = close ? fma(o.w, F, gb) : gb;
        });
    }
    if (valid) {
        const int64_t idx = geom.index(p);
        partial_a[(int64_t)blockIdx.y * n_src + idx] = live ? ga : 0.0;
        partial_b[(int64_t)blockIdx.y * n_src + idx] = live ? gb : 0.0;
    }
}

__global__ void reduce_scaled_kernel(const double *__restrict__ partial, int64_t chunks, int64_t n,
                                     double *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double sum = 0.0;
    for (int64_t c = 0; c < chunks; ++c) sum += partial[c * n + i];
    out[i] = sum;
}

// Chunks of the point dimension for the VJP: enough workgroups over the
// prism dimension times point chunks to fill the device, of at least 128
// points each (2500 prisms, 9801 points: a step of 627 us; with 32 points
// 716 us) unless that leaves CUs without one; those calls split down to 16
// points (841 prisms at 1156 points: a step of 425 us with 128 points).
inline int64_t vjp_chunks(int64_t n_src, int64_t n_obs, int n_cu) {
    const int64_t chunks = forward_chunks(n_src, n_obs, n_cu);
    const int64_t blocks = n_src > kObsPerBlock ? (n_src + kObsPerBlock - 1) / kObsPerBlock : 1;
    const int64_t cu = n_cu > 0 ? n_cu : 256;
    if (blocks * chunks >= cu) return chunks;
    const int64_t most = (n_obs + 15) / 16, wanted = (2 * cu + blocks - 1) / blocks;
    return most < wanted ? most : wanted;
}

template <class Geom>
int run_jvp(const double *e, const double *n, const double *u, int64_t n_obs, const Geom &g,
            const double *wa, const double *wb, int64_t n_src, double *out, void *ws,
            size_t ws_bytes, hipStream_t s) {
    if (n_obs <= 0) return HMX_OK;
    const int cu = device_cu_count();
    if (cu < 0) return cu;
    const int64_t chunks = n_src > 0 ? forward_chunks(n_obs, n_src, cu) : 0;
    const size_t need = (size_t)chunks * (size_t)n_obs * sizeof(double);
    if (chunks > 0) {
        if (!ws || ws_bytes < need)
            return fail(HMX_ERR_ARG, "workspace too small: %zu < %zu bytes", ws_bytes, need);
        const int64_t chunk_len = (n_src + chunks - 1) / chunks;
        dim3 grid((unsigned)((n_obs + kObsPerBlock - 1) / kObsPerBlock), (unsigned)chunks);
        hipLaunchKernelGGL(gz_jvp_kernel<Geom>, grid, dim3(kObsPerBlock), 0, s, e, n, u, (int)n_obs,
                           g, wa, wb, n_src, chunk_len, static_cast<double *>(ws));
        HMX_LAUNCHED("gz_jvp_kernel");
    }
    hipLaunchKernelGGL(reduce_scaled_kernel, dim3((unsigned)((n_obs + 255) / 256)), dim3(256), 0, s,
                       static_cast<const double *>(ws), chunks, n_obs, out);
    HMX_LAUNCHED("reduce_scaled_kernel");
    return HMX_OK;
}

template <class Geom>
int run_vjp(const double *e, const double *n, const double *u, const double *v, int64_t n_obs,
            const Geom &g, int64_t n_src, double *ga, double *gb, void *ws, size_t ws_bytes,
            hipStream_t s) {
    if (n_src <= 0) return HMX_OK;
    const int cu = device_cu_count();
    if (cu < 0) return cu;
    const int64_t chunks = n_obs > 0 ? vjp_chunks(n_src, n_obs, cu) : 0;
    const size_t need = 2 * (size_t)chunks * (size_t)n_src * sizeof(double);
    double *pa = static_cast<double *>(ws);
    double *pb = pa + chunks * n_src;
    if (chunks > 0) {
        if (!ws || ws_bytes < need)
            return fail(HMX_ERR_ARG, "workspace too small: %zu < %zu bytes", ws_bytes, need);
        const int64_t chunk_len = (n_obs + chunks - 1) / chunks;
        dim3 grid((unsigned)((n_src + kObsPerBlock - 1) / kObsPerBlock), (unsigned)chunks);
        hipLaunchKernelGGL(gz_vjp_kernel<Geom>, grid, dim3(kObsPerBlock), 0, s, e, n, u, v, n_obs, g,
                           n_src, chunk_len, pa, pb);
        HMX_LAUNCHED("gz_vjp_kernel");
    }
    const unsigned rb = (unsigned)((n_src + 255) / 256);
    hipLaunchKernelGGL(reduce_scaled_kernel, dim3(rb), dim3(256), 0, s, pa, chunks, n_src, ga);
    HMX_LAUNCHED("reduce_scaled_kernel");
    hipLaunchKernelGGL(reduce_scaled_kernel, dim3(rb), dim3(256), 0, s, pb, chunks, n_src, gb);
    HMX_LAUNCHED("reduce_scaled_kernel");
    return HMX_OK;
}

int check_sizes(int64_t n_obs, int64_t n_src) {
    if (n_obs < 0 || n_src < 0) return fail(HMX_ERR_ARG, "negative size");
    if (n_obs > INT32_MAX || n_src > INT32_MAX)
        return fail(HMX_ERR_ARG, "more than 2^31-1 observation points or prisms");
    return HMX_OK;
}

}  // namespace
}  // namespace hmx

extern "C" {

int hmx_gz_grad_workspace_bytes(int64_t n_obs, int64_t n_prisms, size_t *bytes) {
    using namespace hmx;
    if (!bytes) return fail(HMX_ERR_ARG, "bytes is NULL");
    int st = check_sizes(n_obs, n_prisms);
    if (st) return st;
    const int cu = device_cu_count();
    if (cu < 0) return cu;
    const size_t jvp = (size_t)forward_chunks(n_obs, n_prisms, cu) * (size_t)n_obs;
    const size_t vjp = 2 * (size_t)vjp_chunks(n_prisms, n_obs, cu) * (size_t)n_prisms;
    *bytes = (jvp > vjp ? jvp : vjp) * sizeof(double);
    return HMX_OK;
}

int hmx_prism_gz_jvp(const double *easting, const double *northing, const double *upward,
                     int64_t n_obs, const double *prisms, const double *weight_s,
                     const double *weight_f, int64_t n_prisms, double *out, void *workspace,
                     size_t workspace_bytes, void *stream) {
    using namespace hmx;
    clear_error();
    int st = check_sizes(n_obs, n_prisms);
    if (st) return st;
    if (n_obs > 0 && (!easting || !northing || !upward || !out))
        return fail(HMX_ERR_ARG, "NULL array");
    if (n_prisms > 0 && (!prisms || !weight_s)) return fail(HMX_ERR_ARG, "NULL prism array");
    ExplicitGeom g{prisms};
    return run_jvp(easting, northing, upward, n_obs, g, weight_s, weight_f, n_prisms, out,
                   workspace, workspace_bytes, (hipStream_t)stream);
}

int hmx_prism_gz_vjp(const double *easting, const double *northing, const double *upward,
                     const double *v, int64_t n_obs, const double *prisms, int64_t n_prisms,
                     double *grad_s, double *grad_f, void *workspace, size_t workspace_bytes,
                     void *stream) {
    using namespace hmx;
    clear_error();
    int st = check_sizes(n_obs, n_prisms);
    if (st) return st;
    if (n_obs > 0 && (!easting || !northing || !upward || !v)) return fail(HMX_ERR_ARG, "NULL array");
    if (n_prisms > 0 && (!prisms || !grad_s || !grad_f)) return fail(HMX_ERR_ARG, "NULL prism array");
    ExplicitGeom g{prisms};
    return run_vjp(easting, northing, upward, v, n_obs, g, n_prisms, grad_s, grad_f, workspace,
                   workspace_bytes, (hipStream_t)stream);
}

int hmx_prism_layer_gz_jvp(const double *easting, const double *northing, const double *upward,
                           int64_t n_obs, const double *centre_easting, int64_t n_east,
                           const double *centre_northing, int64_t n_north, const double *bottom,
                           const double *top, const double *density, double thickness_threshold,
                           const double *weight_s, const double *weight_f, double *out,
                           void *workspace, size_t workspace_bytes, void *stream) {
    using namespace hmx;
    clear_error();
    if (n_east < 2 || n_north < 2)
        return fail(HMX_ERR_ARG, "a prism layer needs at least 2 centres per direction");
    int st = check_sizes(n_obs, n_east * n_north);
    if (st) return st;
    if (n_obs > 0 && (!easting || !northing || !upward || !out))
        return fail(HMX_ERR_ARG, "NULL array");
    if (!centre_easting || !centre_northing || !bottom || !top || !density || !weight_s)
        return fail(HMX_ERR_ARG, "NULL layer array");
    LayerGeom g{centre_easting, centre_northing, bottom, top, density,
                (int)n_east, (int)n_north, thickness_threshold};
    return run_jvp(easting, northing, upward, n_obs, g, weight_s, weight_f, n_east * n_north, out,
                   workspace, workspace_bytes, (hipStream_t)stream);
}

int hmx_prism_layer_gz_vjp(const double *easting, const double *northing, const double *upward,
                           const double *v, int64_t n_obs, const double *centre_easting,
                           int64_t n_east, const double *centre_northing, int64_t n_north,
                           const double *bottom, const double *top, const double *density,
                           double thickness_threshold, double *grad_s, double *grad_f,
                           void *workspace, size_t workspace_bytes, void *stream) {
    using namespace hmx;
    clear_error();
    if (n_east < 2 || n_north < 2)
        return fail(HMX_ERR_ARG, "a prism layer needs at least 2 centres per direction");
    int st = check_sizes(n_obs, n_east * n_north);
    if (st) return st;
    if (n_obs > 0 && (!easting || !northing || !upward || !v)) return fail(HMX_ERR_ARG, "NULL array");
    if (!centre_easting || !centre_northing || !bottom || !top || !density || !grad_s || !grad_f)
        return fail(HMX_ERR_ARG, "NULL layer array");
    LayerGeom g{centre_easting, centre_northing, bottom, top, density,
                (int)n_east, (int)n_north, thickness_threshold};
    return run_vjp(easting, northing, upward, v, n_obs, g, n_east * n_north, grad_s, grad_f,
                   workspace, workspace_bytes, (hipStream_t)stream);
}

}  // extern "C"
