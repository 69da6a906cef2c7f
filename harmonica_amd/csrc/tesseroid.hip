// Gravitational potential and g_z of tesseroids (spherical prisms) by
// adaptive discretisation and Gauss-Legendre quadrature, as
// src/harmonica/_forward/tesseroid_gravity.py:236-336 and
// _tesseroid_utils.py do on the CPU:
//  * per (point, tesseroid), a stack of tesseroids starts with the
//    tesseroid; a popped tesseroid whose distance to the point (from its
//    centre) is below `ratio` times its longitudinal, latitudinal (or, with
//    radial discretisation, radial) size is bisected along those
//    directions and its parts pushed, else it is integrated;
//  * integration: 2 x 2 x 2 Gauss-Legendre nodes as point masses
//    rho(node) * a * r'^2 cos(lat') with the spherical point-mass kernels
//    (point.py:324-354) and the distance of _forward/utils.py:163-201.
// Launch shape as the prism kernels: 256 points per workgroup, one per lane,
// tesseroids staged in LDS tiles and read as wave-uniform broadcasts, one
// chunk of the tesseroid list per workgroup column, chunk partials reduced in
// order by a second kernel.  Most pairs leave the tesseroid undivided: they
// are integrated in place, from the geocentric positions of its nodes.  The
// few that divide it cost up to hundreds of times more, at different
// tesseroids for different lanes: a wave lists them and its lanes take them
// from the list one after the other (each with its stack in private memory).
// 3000 tesseroids of 0.5 degrees at 4087 points 10 km above: 6.9 -> 0.65 ms; the
// global 1-degree layer (64,800 at 65,160 points), whole call, 165 -> 49 ms.
// Overflows of the stack (100 entries) or of the number of small
// tesseroids per pair (100000) set a flag the host turns into the
// reference's OverflowError.
#include "devmath.h"
#include "chunk_sum.h"
#include "hmx_internal.h"

namespace hmx {
namespace {

constexpr int kTessStack = 100;
constexpr int kTessMaxSmall = 100000;
constexpr double kDegT = 3.14159265358979323846 / 180.0;
constexpr double kGT = 6.6743e-11;  // harmonica/constants.py:12
// numpy.polynomial.legendre.leggauss(2): nodes -+this, weights 1.
constexpr double kGlqNode = 0x1.279a74590331cp-1;

// Constants of one undivided tesseroid, computed once per tesseroid by
// tess_root_kernel and staged in LDS: the box and the densities at the
// radial nodes, the dimensions and centre of the discretisation test, and
// the trigonometry, radii and masses of the 2 x 2 x 2 quadrature nodes.
// Most pairs never divide the tesseroid: for them these leave three cosines
// of longitude differences per pair (the centre's and the two longitude
// nodes'), taken as the reference does, cos(lambda - lambda_p): where the
// point is close, 1 - cos(psi) is small and any other rounding of it would
// show in the result.
struct alignas(16) TessRoot {
    double t[6];    // w, e, s, n (degrees), bottom, top (m)
    double rho[2];  // density at the lower and upper radial node
    double l_lon, l_lat, l_rad;
    double sin_lat_c, cos_lat_c, lon_c, r_c;   // centre (lon_c in radians)
    double sin_lat_n[2], cos_lat_n[2], lon_n[2], radius_n[2];  // nodes (lon_n in radians)
    double mass[2][2];  // [latitude node][radial node]: rho a r^2 cos(lat)
};
static_assert(sizeof(TessRoot) == 28 * sizeof(double), "TessRoot is 28 doubles");

struct TessPoint {
    double lon, lat, r;            // degrees, degrees, m
    double lon_rad, cosphi, sinphi;
};

// _tesseroid_dimensions (_tesseroid_utils.py): the longitudinal,
// latitudinal and radial sizes of a tesseroid at its top.
__device__ __forceinline__ void tess_dimensions(const double (&t)[6], double &l_lon,
                                                double &l_lat, double &l_rad) {
    const double w = t[0] * kDegT, e = t[1] * kDegT, s = t[2] * kDegT, n = t[3] * kDegT;
    double sn, cn, ss, cs, sc, cc;
    sincos(n, &sn, &cn);
    sincos(s, &ss, &cs);
    sincos((n + s) / 2, &sc, &cc);
    l_lat = t[5] * acos(sn * ss + cn * cs);
    l_lon = t[5] * acos(sc * sc + cc * cc * cos(e - w));
    l_rad = t[5] - t[4];
}

// distance_spherical (_forward/utils.py:121-201) from precomputed point
// quantities to (lon_p [deg], lat_p [deg], r_p).
__device__ __forceinline__ double tess_distance(const TessPoint &P, double lon_p, double lat_p,
                                                double r_p) {
    double sp, cp;
    sincos(lat_p * kDegT, &sp, &cp);
    const double coslambda = cos(lon_p * kDegT - P.lon_rad);
    const double cospsi = sp * P.sinphi + cp * P.cosphi * coslambda;
    const double dr = P.r - r_p;
    return sqrt(dr * dr + 2.0 * P.r * r_p * (1.0 - cospsi));
}

// 2 x 2 x 2 Gauss-Legendre quadrature of one tesseroid (_tesseroid_utils.py
// gauss_legendre_quadrature; the density at the radial nodes as
// _tesseroid_variable_density.py).
template <bool kPot>
__device__ __forceinline__ double tess_glq(const TessPoint &P, const double (&t)[6],
                                           const double (&rho)[2]) {
    const double w = t[0], e = t[1], s = t[2], n = t[3], bottom = t[4], top = t[5];
    const double a_factor = 1.0 / 8.0 * ((e - w) * kDegT) * ((n - s) * kDegT) * (top - bottom);
    const double node[2] = {-kGlqNode, kGlqNode};
    double result = 0.0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        double sinphi_p, cosphi_p;
        sincos((0.5 * (n - s) * node[j] + 0.5 * (n + s)) * kDegT, &sinphi_p, &cosphi_p);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const double radius_p = 0.5 * (top - bottom) * node[k] + 0.5 * (top + bottom);
            const double kappa = radius_p * radius_p * cosphi_p;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const double lon_p = (0.5 * (e - w) * node[i] + 0.5 * (e + w)) * kDegT;
                const double mass = rho[k] * a_factor * kappa;
                const double coslambda = cos(lon_p - P.lon_rad);
                const double cospsi = sinphi_p * P.sinphi + cosphi_p * P.cosphi * coslambda;
                const double dr = P.r - radius_p;
                const double dist = sqrt(dr * dr + 2.0 * P.r * radius_p * (1.0 - cospsi));
                double kv;
                if constexpr (kPot) {
                    kv = 1.0 / dist * kGT;
                } else {
                    const double dz = P.r - radius_p * cospsi;
                    kv = -kGT * dz / (dist * dist * dist);
                }
                result += mass * kv;
            }
        }
    }
    return result;
}

// tess_glq of an undivided tesseroid from its precomputed constants (the
// same nodes, masses and order of summation).
template <bool kPot>
__device__ __forceinline__ double tess_glq_root(const TessPoint &P, const TessRoot &R) {
    double coslambda[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) coslambda[i] = cos(R.lon_n[i] - P.lon_rad);
    double result = 0.0;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const double radius_p = R.radius_n[k];
            const double dr = P.r - radius_p;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const double cospsi = R.sin_lat_n[j] * P.sinphi + R.cos_lat_n[j] * P.cosphi * coslambda[i];
                const double dist = sqrt(dr * dr + 2.0 * P.r * radius_p * (1.0 - cospsi));
                double kv;
                if constexpr (kPot) {
                    kv = 1.0 / dist * kGT;
                } else {
                    const double dz = P.r - radius_p * cospsi;
                    kv = -kGT * dz / (dist * dist * dist);
                }
                result += R.mass[j][k] * kv;
            }
        }
    return result;
}

// The parts of tesseroid t for a split into n_lon x n_lat x n_rad, pushed
// on the stack (false if the stack would overflow).
__device__ __forceinline__ bool tess_push_parts(double (&stk)[kTessStack][6], int &top,
                                                const double (&t)[6], int n_lon, int n_lat,
                                                int n_rad) {
    if ((top + 1) + n_lon * n_lat * n_rad > kTessStack) return false;
    const double d_lon = (t[1] - t[0]) / n_lon, d_lat = (t[3] - t[2]) / n_lat;
    const double d_rad = (t[5] - t[4]) / n_rad;
    for (int i = 0; i < n_lon; ++i)
        for (int j = 0; j < n_lat; ++j)
            for (int k = 0; k < n_rad; ++k) {
                ++top;
                stk[top][0] = t[0] + d_lon * i;
                stk[top][1] = t[0] + d_lon * (i + 1);
                stk[top][2] = t[2] + d_lat * j;
                stk[top][3] = t[2] + d_lat * (j + 1);
                stk[top][4] = t[4] + d_rad * k;
                stk[top][5] = t[4] + d_rad * (k + 1);
            }
    return true;
}

// Density of a tesseroid's radial profile from its Chebyshev coefficients
// c[0..kChebN) over [B, T] (the undivided tesseroid's radial extent):
// sum_k c_k T_k(x), x = (2 r - (B + T)) / (T - B), by Clenshaw's recurrence.
constexpr int kChebN = 32;
__device__ __forceinline__ double cheb_density(const double *__restrict__ c, double r, double B,
                                               double T) {
    double x = (2.0 * r - (B + T)) / (T - B);
    x = fmin(1.0, fmax(-1.0, x));
    double b1 = 0.0, b2 = 0.0;
#pragma unroll
    for (int k = kChebN - 1; k >= 1; --k) {
        const double b0 = fma(2.0 * x, b1, c[k] - b2);
        b2 = b1;
        b1 = b0;
    }
    return fma(x, b1, c[0] - b2);
}

// Whether the undivided tesseroid is divided, by the reference's distance
// (_distance_tesseroid_point from the centre) and in which directions.
template <bool kRadial>
__device__ __forceinline__ bool tess_divided(const TessPoint &P, const TessRoot &R, double ratio,
                                             int &n_lon, int &n_lat, int &n_rad) {
    const double coslambda = cos(R.lon_c - P.lon_rad);
    const double cospsi = R.sin_lat_c * P.sinphi + R.cos_lat_c * P.cosphi * coslambda;
    const double dr = P.r - R.r_c;
    const double d = sqrt(dr * dr + 2.0 * P.r * R.r_c * (1.0 - cospsi));
    n_lon = d / R.l_lon < ratio ? 2 : 1;
    n_lat = d / R.l_lat < ratio ? 2 : 1;
    n_rad = (kRadial && d / R.l_rad < ratio) ? 2 : 1;
    return n_lon * n_lat * n_rad > 1;
}

// Geocentric constants of one undivided tesseroid for the pairs that leave it
// so: node positions [latitude][radius][longitude], masses [latitude][radius],
// centre, and the squared distances of the centre from which the pair is
// integrated from the positions (far2) and below which it is divided
// (near2).  Between them (rounding of the reference's distance criterion, and
// nearer than 0.02 radii, where the reference's 1 - cos(psi) loses digits
// that the positions keep) the reference's own formulas decide and integrate.
struct alignas(16) TessFar {
    double node[2][2][2][3];
    double mass[2][2];
    double c[3];
    double far2, near2, pad;
};
constexpr int kFarDoubles = sizeof(TessFar) / sizeof(double);
static_assert(sizeof(TessFar) == 34 * sizeof(double), "TessFar is 34 doubles");

__device__ __forceinline__ void geocentric(double lon, double sin_lat, double cos_lat, double r,
                                           double (&x)[3]) {
    double sl, cl;
    sincos(lon, &sl, &cl);
    x[0] = r * cos_lat * cl;
    x[1] = r * cos_lat * sl;
    x[2] = r * sin_lat;
}

__device__ __forceinline__ void tess_far(const TessRoot &R, double ratio, bool radial,
                                         TessFar &F) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            F.mass[j][k] = R.mass[j][k];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                geocentric(R.lon_n[i], R.sin_lat_n[j], R.cos_lat_n[j], R.radius_n[k],
                           F.node[j][k][i]);
        }
    geocentric(R.lon_c, R.sin_lat_c, R.cos_lat_c, R.r_c, F.c);
    const double l_rad = radial ? R.l_rad : 0.0;
    const double thr = ratio * fmax(fmax(R.l_lon, R.l_lat), l_rad), thr2 = thr * thr;
    const double rc2 = R.r_c * R.r_c;
    F.far2 = fmax(fma(1e-9, thr2, thr2) + 1e-14 * rc2, 4e-4 * rc2);
    F.near2 = fma(-1e-9, thr2, thr2) - 1e-14 * rc2;
    // negative sizes (boundaries in the wrong order, without checks) divide at
    // any distance: leave the decision to the reference's formula
    if (R.l_lon < 0.0 || R.l_lat < 0.0 || l_rad < 0.0 || !(thr2 < 1e300))
        F.far2 = F.near2 = __builtin_nan("");
    F.pad = 0.0;
}

// A lane's point in geocentric coordinates: position and direction.
struct TessXyz {
    double x[3], up[3];
};

// 2 x 2 x 2 quadrature of an undivided tesseroid from its node positions:
// l^2 = |X - X'|^2 and r - r' cos(psi) = (X - X') . X / r, one reciprocal
// square root per node and no trigonometry (22 operations per node; the
// reference's distance takes a square root, two divisions and, once per two
// nodes, a cosine).
template <bool kPot>
__device__ __forceinline__ double tess_glq_far(const TessXyz &X, const TessFar &F) {
    double result = 0.0;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            double sum = 0.0;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const double dx = X.x[0] - F.node[j][k][i][0], dy = X.x[1] - F.node[j][k][i][1];
                const double dz = X.x[2] - F.node[j][k][i][2];
                const double inv = dm::rsqrt_pos(fma(dx, dx, fma(dy, dy, dz * dz)));
                if constexpr (kPot) {
                    sum += inv;
                } else {
                    const double dot = fma(dx, X.up[0], fma(dy, X.up[1], dz * X.up[2]));
                    sum = fma(dot, inv * (inv * inv), sum);
                }
            }
            result = fma(F.mass[j][k], sum, result);
        }
    return kPot ? kGT * result : -kGT * result;
}

constexpr int kTessTile = 32;   // tesseroids staged per pass: a lane's mask of divided ones
constexpr int kTessList = 256;  // pairs a wave lists at a time

struct TessShared {
    TessFar tile[kTessTile];
    TessPoint point[kObsPerBlock];
    double value[kObsPerBlock / 64][kTessList];
    uint16_t list[kObsPerBlock / 64][kTessList];
};

// Orders a wave's own LDS writes before its reads.
__device__ __forceinline__ void tess_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Adds the pairs in `mask` (bit p: tesseroid t0 + p at the lane's point, to be
// divided): listed by lane and tesseroid, taken by the lanes in list order as
// each gets free, one piece per turn, so that the wave is full whatever the
// pairs' depths; each lane then adds the values of its own pairs in order.
// A piece is tested and, if small enough, integrated in the reference's order.
// With radial discretisation and a variable density (cheb: 32 Chebyshev
// coefficients per tesseroid, else NULL), the parts' radial nodes take their
// densities from the coefficients; otherwise they share the undivided
// tesseroid's nodes (radially undivided parts) or its constant density.
template <bool kPot, bool kRadial>
__device__ void tess_divide(TessShared &sh, unsigned mask, const TessRoot *__restrict__ roots,
                            double ratio, const double *__restrict__ cheb, double &acc, int &ovf) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint16_t *list = sh.list[wave];
    double *value = sh.value[wave];
    double stk[kTessStack][6];
    while (__any(mask != 0)) {
        const int count = __popc(mask);
        int incl = count;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o);
            if (lane >= o) incl += v;
        }
        const int total = __builtin_amdgcn_readlane(incl, 63);
        const int n = total < kTessList ? total : kTessList;
        const int at = incl - count < kTessList ? incl - count : kTessList;
        int end = at;
        while (mask && end < kTessList) {
            list[end++] = (uint16_t)((unsigned)__builtin_ctz(mask) | lane << 5);
            mask &= mask - 1;
        }
        tess_sync();
        int next = 0, mine = 0, top = -1, small = 0;
        bool have = false;
        double result = 0.0;
        TessPoint P = sh.point[wave * 64];
        const TessRoot *R = roots;
        for (;;) {
            if (have && top < 0) {
                value[mine] = result;
                have = false;
            }
            const uint64_t idle = __ballot(!have);
            if (next < n) {
                const int k = next + __popcll(idle & ((1ull << lane) - 1ull));
                if (!have && k < n) {
                    have = true;
                    mine = k;
                    const unsigned pair = list[k];
                    P = sh.point[wave * 64 + (pair >> 5)];
                    R = roots + (pair & 31u);
                    result = 0.0;
                    small = 0;
                    int n_lon, n_lat, n_rad;
                    if (!tess_divided<kRadial>(P, *R, ratio, n_lon, n_lat, n_rad))
                        result = tess_glq_root<kPot>(P, *R);
                    else
                        (void)tess_push_parts(stk, top, R->t, n_lon, n_lat, n_rad);  // at most 8
                }
                next += __popcll(idle);
            }
            if (!__any(have)) break;
            if (top >= 0) {
                double t[6];
#pragma unroll
                for (int c = 0; c < 6; ++c) t[c] = stk[top][c];
                --top;
                double l_lon, l_lat, l_rad;
                tess_dimensions(t, l_lon, l_lat, l_rad);
                // _distance_tesseroid_point
                const double d =
                    tess_distance(P, (t[0] + t[1]) / 2, (t[2] + t[3]) / 2, (t[4] + t[5]) / 2);
                const int m_lon = d / l_lon < ratio ? 2 : 1;
                const int m_lat = d / l_lat < ratio ? 2 : 1;
                const int m_rad = (kRadial && d / l_rad < ratio) ? 2 : 1;
                if (m_lon * m_lat * m_rad > 1) {
                    if (!tess_push_parts(stk, top, t, m_lon, m_lat, m_rad)) {
                        ovf = 1;
                        top = -1;
                    }
                } else if (++small > kTessMaxSmall) {
                    ovf = 2;
                    top = -1;
                } else if (kRadial && cheb) {
                    double rho_p[2];
                    const double node[2] = {-kGlqNode, kGlqNode};
#pragma unroll
                    for (int k = 0; k < 2; ++k)
                        rho_p[k] = cheb_density(cheb + (R - roots) * kChebN,
                                                0.5 * (t[5] - t[4]) * node[k] + 0.5 * (t[5] + t[4]),
                                                R->t[4], R->t[5]);
                    result += tess_glq<kPot>(P, t, rho_p);
                } else {
                    result += tess_glq<kPot>(P, t, R->rho);
                }
            }
        }
        tess_sync();
        for (int k = at; k < end; ++k) acc += value[k];
        tess_sync();
        if (__any(ovf)) return;  // the host raises: what is left does not matter
    }
}

// The TessRoot constants of each tesseroid (one per thread).
__global__ __launch_bounds__(256) void tess_root_kernel(const double *__restrict__ tess,
                                                        const double *__restrict__ rho,
                                                        int64_t n, double ratio, int radial,
                                                        TessRoot *__restrict__ roots,
                                                        TessFar *__restrict__ fars) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= n) return;
    TessRoot R;
#pragma unroll
    for (int c = 0; c < 6; ++c) R.t[c] = tess[6 * q + c];
    R.rho[0] = rho[2 * q];
    R.rho[1] = rho[2 * q + 1];
    tess_dimensions(R.t, R.l_lon, R.l_lat, R.l_rad);
    const double w = R.t[0], e = R.t[1], s = R.t[2], n_ = R.t[3], bottom = R.t[4], top = R.t[5];
    sincos((s + n_) / 2 * kDegT, &R.sin_lat_c, &R.cos_lat_c);
    R.lon_c = (w + e) / 2 * kDegT;
    R.r_c = (bottom + top) / 2;
    const double a_factor = 1.0 / 8.0 * ((e - w) * kDegT) * ((n_ - s) * kDegT) * (top - bottom);
    const double node[2] = {-kGlqNode, kGlqNode};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        sincos((0.5 * (n_ - s) * node[j] + 0.5 * (n_ + s)) * kDegT, &R.sin_lat_n[j], &R.cos_lat_n[j]);
        R.lon_n[j] = (0.5 * (e - w) * node[j] + 0.5 * (e + w)) * kDegT;
        R.radius_n[j] = 0.5 * (top - bottom) * node[j] + 0.5 * (top + bottom);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int k = 0; k < 2; ++k)
            R.mass[j][k] = R.rho[k] * a_factor * (R.radius_n[k] * R.radius_n[k] * R.cos_lat_n[j]);
    roots[q] = R;
    TessFar F;
    tess_far(R, ratio, radial != 0, F);
    fars[q] = F;
}

template <bool kPot, bool kRadial>
__global__ __launch_bounds__(kObsPerBlock, 3) void tesseroid_kernel(
    const double *__restrict__ lon, const double *__restrict__ lat,
    const double *__restrict__ rad, int n_obs, const TessRoot *__restrict__ roots,
    const TessFar *__restrict__ fars, int64_t n_src, int64_t chunk_len, double ratio,
    const double *__restrict__ cheb, double *__restrict__ partial, int *__restrict__ overflow) {
    __shared__ TessShared sh;
    const int i = blockIdx.x * kObsPerBlock + threadIdx.x;
    const bool valid = i < n_obs;
    const int ii = valid ? i : n_obs - 1;
    TessPoint P;
    P.lon = lon[ii];
    P.lat = lat[ii];
    P.r = rad[ii];
    P.lon_rad = P.lon * kDegT;
    sincos(P.lat * kDegT, &P.sinphi, &P.cosphi);
    sh.point[threadIdx.x] = P;
    TessXyz X;
    geocentric(P.lon_rad, P.sinphi, P.cosphi, 1.0, X.up);
#pragma unroll
    for (int c = 0; c < 3; ++c) X.x[c] = P.r * X.up[c];
    double acc = 0.0;
    int ovf = 0;
    const int64_t c0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t c1 = c0 + chunk_len < n_src ? c0 + chunk_len : n_src;
    for (int64_t t0 = c0; t0 < c1; t0 += kTessTile) {
        const int cnt = (int)(c1 - t0 < kTessTile ? c1 - t0 : kTessTile);
        __syncthreads();
        const double *src = reinterpret_cast<const double *>(fars + t0);
        double *dst = reinterpret_cast<double *>(sh.tile);
        for (int q = threadIdx.x; q < cnt * kFarDoubles; q += blockDim.x) dst[q] = src[q];
        __syncthreads();
        if (__any(ovf)) continue;
        unsigned mask = 0;
        for (int p = 0; p < cnt; ++p) {
            const TessFar &F = sh.tile[p];
            const double dx = X.x[0] - F.c[0], dy = X.x[1] - F.c[1], dz = X.x[2] - F.c[2];
            const double d2 = fma(dx, dx, fma(dy, dy, dz * dz));
            // (a point at infinity is neither: its terms are 1 / inf)
            const bool far = d2 >= F.far2 && d2 < 1e300, near = d2 < F.near2;
            if (__any(far)) {
                const double v = tess_glq_far<kPot>(X, F);
                acc += far ? v : 0.0;
            }
            if (!far && !near) {
                const TessRoot &R = roots[t0 + p];
                int n_lon, n_lat, n_rad;
                if (tess_divided<kRadial>(P, R, ratio, n_lon, n_lat, n_rad))
                    mask |= 1u << p;
                else
                    acc += tess_glq_root<kPot>(P, R);
            } else if (near) {
                mask |= 1u << p;
            }
        }
        // lanes past the last point repeat it: nothing to divide for them
        if (__any(mask != 0))
            tess_divide<kPot, kRadial>(sh, valid ? mask : 0u, roots + t0, ratio,
                                       cheb ? cheb + t0 * kChebN : nullptr, acc, ovf);
    }
    if (valid) partial[(int64_t)blockIdx.y * n_obs + i] = acc;
    if (ovf) atomicMax(overflow, ovf);
}

// Sets *flag if a point lies strictly inside a tesseroid
// (_tesseroid_utils.py check_points_outside_tesseroids; the longitude is
// given in [-180, 180) and in [0, 360)).  One point per lane, tesseroids read
// as wave-uniform scalars.
__global__ __launch_bounds__(256) void tess_inside_kernel(
    const double *__restrict__ lon180, const double *__restrict__ lon360,
    const double *__restrict__ lat, const double *__restrict__ rad, int n_obs,
    const double *__restrict__ tess, int64_t n_src, int64_t chunk_len, int *__restrict__ flag) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int ii = i < n_obs ? i : n_obs - 1;
    const double a = lon180[ii], b = lon360[ii], y = lat[ii], r = rad[ii];
    const int64_t c0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t c1 = c0 + chunk_len < n_src ? c0 + chunk_len : n_src;
    bool inside = false;
    for (int64_t p = c0; p < c1; ++p) {
        const double *t = tess + 6 * p;
        const bool in_lon = (t[0] < a && a < t[1]) || (t[0] < b && b < t[1]);
        inside = inside || (in_lon && t[2] < y && y < t[3] && t[4] < r && r < t[5]);
    }
    if (inside) atomicOr(flag, 1);
}

// out[i] = scale * sum over chunks in order of partial[c][i].
template <int P>
__global__ __launch_bounds__(dev::SumShape<P>::threads) void reduce_tess_kernel(
    const double *__restrict__ partial, int64_t chunks, int64_t n_obs, double scale,
    double *__restrict__ out) {
    int64_t i;
    double sum;
    if (dev::chunk_sum<P>(partial, chunks, n_obs, i, sum)) out[i] = scale * sum;
}

template <int P>
int launch_reduce(const double *partial, int64_t chunks, int64_t n_obs, double scale, double *out,
                  hipStream_t stream) {
    using S = dev::SumShape<P>;
    hipLaunchKernelGGL((reduce_tess_kernel<P>), dim3((unsigned)((n_obs + S::outputs - 1) / S::outputs)),
                       dim3(S::threads), 0, stream, partial, chunks, n_obs, scale, out);
    HMX_LAUNCHED("reduce_tess_kernel");
    return HMX_OK;
}

// Workspace: the chunk partials, then (256-byte aligned) one TessRoot and one
// TessFar per tesseroid.
inline size_t tess_partial_bytes(int64_t chunks, int64_t n_obs) {
    return ((size_t)chunks * (size_t)n_obs * sizeof(double) + 255) / 256 * 256;
}
inline size_t tess_workspace_bytes(int64_t chunks, int64_t n_obs, int64_t n_tess) {
    return tess_partial_bytes(chunks, n_obs) + (size_t)n_tess * (sizeof(TessRoot) + sizeof(TessFar));
}

__global__ void fill_zero_tess_kernel(double *__restrict__ out, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = 0.0;
}

}  // namespace
}  // namespace hmx

extern "C" {

int hmx_tesseroid_workspace_bytes(int64_t n_obs, int64_t n_tesseroids, size_t *bytes) {
    hmx::clear_error();
    if (!bytes) return hmx::fail(HMX_ERR_ARG, "bytes is NULL");
    if (n_obs < 0 || n_tesseroids < 0) return hmx::fail(HMX_ERR_ARG, "negative size");
    const int cu = hmx::device_cu_count();
    if (cu < 0) return cu;
    *bytes = hmx::tess_workspace_bytes(hmx::prism_chunks(n_obs, n_tesseroids, cu), n_obs,
                                       n_tesseroids);
    return HMX_OK;
}

int hmx_tesseroid_gravity(const double *longitude, const double *latitude, const double *radius,
                          int64_t n_obs, const double *tesseroids, const double *density_nodes,
                          const double *density_cheb, int64_t n_tesseroids, uint32_t field,
                          int radial_discretization, double *out, int *overflow, void *workspace,
                          size_t workspace_bytes, void *stream) {
    using namespace hmx;
    clear_error();
    if (n_obs < 0 || n_tesseroids < 0) return fail(HMX_ERR_ARG, "negative size");
    if (n_obs > INT32_MAX || n_tesseroids > INT32_MAX)
        return fail(HMX_ERR_ARG, "more than 2^31-1 points or tesseroids");
    if (field != HMX_POTENTIAL && field != HMX_G_Z)
        return fail(HMX_ERR_ARG, "tesseroids support only potential and g_z (mask 0x%x)", field);
    if (n_obs == 0) return HMX_OK;
    if (!longitude || !latitude || !radius || !out || !overflow)
        return fail(HMX_ERR_ARG, "NULL array");
    hipStream_t s = (hipStream_t)stream;
    if (n_tesseroids == 0) {
        hipLaunchKernelGGL(fill_zero_tess_kernel, dim3((unsigned)((n_obs + 255) / 256)),
                           dim3(256), 0, s, out, n_obs);
        HMX_LAUNCHED("fill_zero_tess_kernel");
        return HMX_OK;
    }
    if (!tesseroids || !density_nodes) return fail(HMX_ERR_ARG, "NULL tesseroid array");
    const int cu = device_cu_count();
    if (cu < 0) return cu;
    const int64_t chunks = prism_chunks(n_obs, n_tesseroids, cu);
    const size_t need = tess_workspace_bytes(chunks, n_obs, n_tesseroids);
    if (!workspace || workspace_bytes < need)
        return fail(HMX_ERR_ARG, "workspace too small: %zu < %zu bytes", workspace_bytes, need);
    double *partial = static_cast<double *>(workspace);
    TessRoot *roots = reinterpret_cast<TessRoot *>(static_cast<char *>(workspace) +
                                                   tess_partial_bytes(chunks, n_obs));
    TessFar *fars = reinterpret_cast<TessFar *>(roots + n_tesseroids);
    const bool pot = field == HMX_POTENTIAL;
    // distance-size ratios of tesseroid_gravity.py:32
    const double ratio = pot ? 1.0 : 2.5;
    hipLaunchKernelGGL(tess_root_kernel, dim3((unsigned)((n_tesseroids + 255) / 256)), dim3(256),
                       0, s, tesseroids, density_nodes, n_tesseroids, ratio, radial_discretization,
                       roots, fars);
    HMX_LAUNCHED("tess_root_kernel");
    const int64_t chunk_len = (n_tesseroids + chunks - 1) / chunks;
    dim3 grid((unsigned)((n_obs + kObsPerBlock - 1) / kObsPerBlock), (unsigned)chunks);
#define HMX_TESS(P, R)                                                                           \
    hipLaunchKernelGGL((tesseroid_kernel<P, R>), grid, dim3(kObsPerBlock), 0, s, longitude,     \
                       latitude, radius, (int)n_obs, roots, fars, n_tesseroids, chunk_len,      \
                       ratio,                                                                   \
                       density_cheb, partial, overflow)
    if (pot && radial_discretization) HMX_TESS(true, true);
    else if (pot) HMX_TESS(true, false);
    else if (radial_discretization) HMX_TESS(false, true);
    else HMX_TESS(false, false);
#undef HMX_TESS
    HMX_LAUNCHED("tesseroid_kernel");
    // g_z points down: the reference flips the sign of the upward kernel
    // and converts to mGal (tesseroid_gravity.py:207-211).
    const double scale = pot ? 1.0 : -1e5;
    return dev::sum_parts(chunks, n_obs, 16) == 1
               ? launch_reduce<1>(partial, chunks, n_obs, scale, out, s)
               : launch_reduce<16>(partial, chunks, n_obs, scale, out, s);
}

int hmx_tesseroid_points_inside(const double *longitude_180, const double *longitude_360,
                                const double *latitude, const double *radius, int64_t n_obs,
                                const double *tesseroids, int64_t n_tesseroids, int *flag,
                                void *stream) {
    using namespace hmx;
    clear_error();
    if (n_obs < 0 || n_tesseroids < 0) return fail(HMX_ERR_ARG, "negative size");
    if (n_obs > INT32_MAX || n_tesseroids > INT32_MAX)
        return fail(HMX_ERR_ARG, "more than 2^31-1 points or tesseroids");
    if (n_obs == 0 || n_tesseroids == 0) return HMX_OK;
    if (!longitude_180 || !longitude_360 || !latitude || !radius || !tesseroids || !flag)
        return fail(HMX_ERR_ARG, "NULL array");
    const int cu = device_cu_count();
    if (cu < 0) return cu;
    const int64_t chunks = forward_chunks(n_obs, n_tesseroids, cu);
    dim3 grid((unsigned)((n_obs + 255) / 256), (unsigned)chunks);
    hipLaunchKernelGGL(tess_inside_kernel, grid, dim3(256), 0, (hipStream_t)stream, longitude_180,
                       longitude_360, latitude, radius, (int)n_obs, tesseroids, n_tesseroids,
                       (n_tesseroids + chunks - 1) / chunks, flag);
    HMX_LAUNCHED("tess_inside_kernel");
    return HMX_OK;
}

}  // extern "C"
