// Internal helpers shared by the libhmx translation units: error reporting,
// device queries and the launch-shape rules of the pairwise kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "../../include/hmx.h"

namespace hmx {

// Record a printf-style message for hmx_last_error() and return `code`.
int fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));

// Clear the calling thread's last error.
void clear_error();

// Devices the per-device caches of the library cover.
constexpr int kMaxDevices = 64;

// Number of compute units of the current device (cached per device), or a
// negative status if no device is usable.
int device_cu_count();

}  // namespace hmx

#define HMX_HIP(expr)                                                              \
    do {                                                                           \
        hipError_t hmx_e_ = (expr);                                                \
        if (hmx_e_ != hipSuccess)                                                  \
            return ::hmx::fail(HMX_ERR_HIP, "%s failed: %s", #expr,                \
                               hipGetErrorString(hmx_e_));                         \
    } while (0)

// After a kernel launch: report launch-configuration errors.
#define HMX_LAUNCHED(name)                                                         \
    do {                                                                           \
        hipError_t hmx_e_ = hipGetLastError();                                     \
        if (hmx_e_ != hipSuccess)                                                  \
            return ::hmx::fail(HMX_ERR_HIP, "launch of %s failed: %s", name,       \
                               hipGetErrorString(hmx_e_));                         \
    } while (0)

namespace hmx {

// Observation points per workgroup of the pairwise kernels: 4 wavefronts of
// 64 lanes, one observation point per lane.
constexpr int kObsPerBlock = 256;
// Sources staged in LDS per pass.
constexpr int kTile = 128;

// Split of the source dimension into chunks so that a launch has enough
// workgroups to fill all compute units several times over.  Each chunk's
// partial sums go to the workspace and are reduced in chunk order, so the
// result does not depend on scheduling.
inline int64_t forward_chunks(int64_t n_obs, int64_t n_src, int n_cu) {
    int64_t obs_blocks = (n_obs + kObsPerBlock - 1) / kObsPerBlock;
    if (obs_blocks < 1) obs_blocks = 1;
    int64_t target = 40LL * (n_cu > 0 ? n_cu : 256);
    int64_t chunks = (target + obs_blocks - 1) / obs_blocks;
    int64_t max_by_src = (n_src + kTile - 1) / kTile;
    if (chunks > max_by_src) chunks = max_by_src;
    if (chunks > 1024) chunks = 1024;
    if (chunks < 1) chunks = 1;
    return chunks;
}

// forward_chunks for the prism field kernels, whose pairs differ several
// times in cost (far and closed forms): chunks down to 32 prisms even out the
// workgroups, and calls that cannot give every CU a workgroup that way split
// down to 8 prisms (24 bodies at 501 points, the pair kernel: 29 -> 16 us).
inline int64_t prism_chunks(int64_t n_obs, int64_t n_src, int n_cu) {
    const int64_t obs_blocks = n_obs > kObsPerBlock ? (n_obs + kObsPerBlock - 1) / kObsPerBlock : 1;
    const int64_t cu = n_cu > 0 ? n_cu : 256;
    int64_t chunks = (40 * cu + obs_blocks - 1) / obs_blocks;
    int64_t max_by_src = (n_src + 31) / 32;
    if (obs_blocks * max_by_src < cu) max_by_src = (n_src + 7) / 8;
    if (chunks > max_by_src) chunks = max_by_src;
    if (chunks > 1024) chunks = 1024;
    return chunks < 1 ? 1 : chunks;
}

inline int popcount10(uint32_t m) { return __builtin_popcount(m & HMX_ALL_FIELDS); }

// Wavefront-coherent point order of the prism kernels (point_order.hip):
// gathered copies of the coordinates in boustrophedon strip order and the
// permutation perm (sorted position -> caller's index) for the reduction.
struct PointOrder {
    const double *e, *n, *u;
    const int *perm;
};

// Points one workgroup orders in one launch.
constexpr int kSmallOrder = 8192;

// Whether a prism call sorts its points: enough points for the strips to
// matter and enough pairs that the sort costs little next to the pair loop.
// Up to kSmallOrder points it is one launch of 25-30 us.  Scattered points
// over 20,000 bodies, g_z with and without the sort: 1000 points 165 / 170 us,
// 3000 points 352 / 417 us, 8000 points 794 / 992 us; over 2000 bodies 3000
// points 73 / 57 us; six tensor fields of 58 x 64 cells at 8085 points (3e7
// pairs) 766 / 827 us.  Beyond, it is a dozen launches (0.1 ms) and 1.2 ns a
// point, which scattered points get back from a few hundred prisms on and a
// raster's hardly ever: 1e6 points, g_z, 128 prisms 1.55 / 1.17 ms scattered
// and 1.50 / 0.35 as a raster, 512 prisms 2.5 / 4.4 and 2.4 / 1.2 ms; 200,000
// points, 1024 prisms 0.67 / 1.82 and 0.66 / 0.51 ms.  (1e7 points over 28
// prisms spent 15 of 17 ms in it.)
inline bool use_point_order(int64_t n_obs, int64_t n_src) {
    if (n_obs > kSmallOrder && n_src < 512) return false;
    const int64_t pairs = n_obs <= kSmallOrder ? (int64_t)1 << 24 : (int64_t)1 << 28;
    // n_obs * n_src >= pairs, without forming the product
    return n_obs >= 512 && n_src >= (pairs + n_obs - 1) / n_obs;
}

// Whether a call with a workspace too small for the order is refused; below
// this it evaluates the points in the caller's order.
inline bool need_point_order(int64_t n_obs, int64_t n_src) {
    return use_point_order(n_obs, n_src) && n_obs >= 2048 &&
           n_src >= (((int64_t)1 << 30) + n_obs - 1) / n_obs;
}

// Whether a call of many points in the caller's order takes the closed form for
// every pair.  Over few prisms: one kernel with little to prepare, where the far form stages constants
// for each workgroup and, but for g_z, runs a second kernel for the close pairs.
// `sorted`: the points are in wavefront-coherent order.  Times per call (us, far
// / closed), points scattered over 40 km, and as a raster:
//                         scattered                      raster
//   20,000 points, 16     g_z 23 / 18,    b 33 / 26      19 / 18,   28 / 27
//   1e6, 1                g_z 42 / 24,    b 128 / 46     32 / 23,   83 / 38
//   1e6, 7                g_z 98 / 85,    b 230 / 151    47 / 82,   134 / 114
//   1e6, 16               g_z 176 / 180,  b 364 / 316    65 / 175,  204 / 234
//   1e6, 32               g_zz 300 / 217, b 613 / 627    130 / 194, 321 / 444
// The line depends on what the closed form costs, most with the potential or g_z
// among the fields.  And g_ee, g_nn or g_en alone, whose closed form is the
// cheapest and whose far form the dearest of a single field: 1e6 points, 256
// prisms, g_ee 2.83 / 1.57 ms scattered and 1.43 / 1.39 as a raster.  Otherwise
// the far form stays, for a tenth of the closed form's error and less: in calls
// of fewer points, which it costs a few us (256 points, 3 prisms: 22 / 21), and
// over more prisms also where scattered points mix far and close lanes (1e6
// points, 256 prisms: g_zz 2.03 / 1.57 ms; as a raster 0.80 / 1.40).
inline bool use_closed(uint32_t mask, int64_t n_obs, int64_t n_src, bool sorted) {
    if (sorted || n_obs <= kSmallOrder) return false;
    if (mask == HMX_G_EE || mask == HMX_G_NN || mask == HMX_G_EN) return true;
    if (!(mask & (HMX_POTENTIAL | HMX_G_Z))) return n_src < 32;
    return n_src < (n_obs > ((int64_t)1 << 17) ? 4 : 16);
}

// Bytes of the order's workspace region for n_obs points.
size_t point_order_bytes(int64_t n_obs);

// Sort the points into the region `ws` (point_order_bytes(n_obs) bytes,
// 256-byte aligned) on stream s.
int point_order(const double *e, const double *n, const double *u, int64_t n_obs, void *ws,
                PointOrder *po, hipStream_t s);

// Offset of the order region in a forward workspace whose partial sums take
// partial_bytes.
inline size_t point_order_offset(size_t partial_bytes) { return (partial_bytes + 255) & ~(size_t)255; }

// Least squares min |G c - y|^2 (+ alpha |c|^2, per filter) through the
// one-sided Jacobi SVD (lsq_svd.hip) of A (L x k, column-major, L >= k,
// overwritten): A = G (n x m, transposed = 0) or A = G^T (transposed = 1).
// W (k x k), vec (3 k doubles), counters (2 ints); y has n entries and
// coef m.  Returns the sweeps taken (negative if max_sweeps stopped them)
// and the number of kept components.  Synchronous.
int svd_lsq(double *A, int64_t L, int64_t k, int transposed, const double *y, double alpha,
            int filter, double cutoff, double *W, double *vec, int *counters, double *coef,
            int max_sweeps, int *sweeps, int *rank, hipStream_t s);
constexpr int kSvdMaxSweeps = 60;

// One window of the gradient-boosted fit, gathered on the device: its data
// (w may be NULL) and its sources.
struct EqsWindow {
    const double *e, *n, *u, *w;
    int64_t nd;
    const double *pe, *pn, *pu;
    int64_t m;
};
// Bytes of the buffers of a batch of `batch` windows of at most n_max data
// and m_max sources (FP64 mode, damping > 0; eqs_fit.hip).
size_t eqs_batch_bytes(int64_t n_max, int64_t m_max, int64_t batch);
// Forms and factorises the normal matrices of a batch of windows; status
// (host, batch ints) receives 0 or the 1-based column of a failed pivot,
// seconds (host, 2) the times of the normal matrices and of the factors.
int eqs_factor_batch(const EqsWindow *wins, int64_t batch, int64_t n_max, int64_t m_max,
                     double damping, void *buffer, size_t buffer_bytes, int *status,
                     double *seconds, hipStream_t s);
// The coefficients of window b of a factorised batch for the data `data`
// (the window's residue): right-hand side, solve and CG refinement as
// hmx_eqs_fit; info (host, 11 doubles) as hmx_eqs_fit's.
int eqs_solve_factored(const EqsWindow &w, const double *data, double damping, void *buffer,
                       int64_t b, int64_t batch, int64_t n_max, int64_t m_max, int max_iter,
                       double rtol, double *coefs, double *info, hipStream_t s);
// Largest fits that take the SVD route when the Cholesky route cannot match
// the reference's solver: at most this many sources and matrix entries.
constexpr int64_t kSvdMaxSrc = 8192;
constexpr int64_t kSvdMaxElems = (int64_t)1 << 27;

}  // namespace hmx
