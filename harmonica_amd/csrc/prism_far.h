// Far form of the prism g_u kernel: the vertical attraction of a prism whose
// horizontal half-diagonal h is small next to its distance.
//
// The sum over the 8 vertices that gu_sum evaluates is
//   S = int int [1/r_B - 1/r_T] dx dy   over the prism's rectangle,
// with r_T, r_B the distances to the top and bottom faces (the integral over
// z is exact, so tall prisms need no other treatment).  With (x, y, z) the
// face centre seen from the point, s = x^2 + y^2, and a point of the face
// displaced by d = (dx, dy), s becomes s + delta, delta = 2 (x dx + y dy) +
// d^2, and Taylor's formula in delta averaged over the rectangle gives
//   <1/r> = (1/r) [1 + sum_m C_m(x^2, y^2) u^m],  u = 1 / r^2,
//   C_m = sum_{i + j = m} c_ij,
//   c_ij = (-1)^m binom(2m, m) 4^(j-m) binom(m, 2j) <(x dx + y dy)^(2j) d^(2(i-j))>
// where 2i is the order of a term in the size of the rectangle (only even
// orders survive the average) and 0 <= j <= i.  Orders up to 2I need
// C_1 .. C_2I.  The C_m are the same for both faces: a face then costs one
// reciprocal square root and 2I + 2 multiply-adds.
//
// Truncation: the omitted order 2I + 2 is the average of |d|^(2I+2) P(cos)
// / r^(2I+2), at most (h/r)^(2I+2) / (2I + 3) (a rectangle shrunk to a
// line; 0.6 of that for a square).  far_ratio2 takes the distance from which
// this is below 4e-15 of 1/r (measured against 40-digit quadrature of
// squares and thin rectangles at that distance: 3e-16 to 3.6e-15, see the
// tests).  gu_sum's own error there is larger: its terms are of size r, so
// it is off by a few 2^-53 r where the face integral is below 4 h^2 / r.
#pragma once

#include "prism_device.h"

namespace hmx {
namespace dev {

// Largest I, and up to which I the constants c_ijk are staged as such.
constexpr int kFarMax = 6;
constexpr int kFarPlain = 3;
constexpr int far_base(int i) {  // index of c_i00
    int n = 0;
    for (int t = 1; t < i; ++t) n += (t + 1) * (t + 2) / 2;
    return n;
}
constexpr int far_index(int i, int j, int k) { return far_base(i) + j * (j + 1) / 2 + k; }
constexpr int kFarConsts = far_base(kFarPlain + 1);
static_assert(kFarConsts == 19, "c_ijk up to i = 3");

constexpr double far_binom(int n, int k) {
    double b = 1.0;
    for (int t = 0; t < k; ++t) b = b * (n - t) / (t + 1);
    return b;
}

// Factor of X^k Y^(j-k) sum_p binom(i-j, p) mu_i[k+p] in c_ij.
constexpr double far_factor(int i, int j, int k) {
    const int m = i + j;
    double f = far_binom(2 * m, m) * far_binom(m, 2 * j) * far_binom(2 * j, 2 * k);
    for (int t = 0; t < m - j; ++t) f *= 0.25;
    return m % 2 ? -f : f;
}

// The constants of order 2i of a rectangle with squared half-sides A (along
// x) and B (along y): mu_i[q] = <dx^2q dy^(2i-2q)> = A^q B^(i-q) / ((2q + 1)
// (2i - 2q + 1)), summed with binomial weights by repeated pairwise addition.
template <int I>
__device__ __forceinline__ void far_order_consts(double A, double B, double *c) {
    double D[I + 1];
    double pa[I + 1], pb[I + 1];
    pa[0] = pb[0] = 1.0;
#pragma unroll
    for (int q = 1; q <= I; ++q) {
        pa[q] = pa[q - 1] * A;
        pb[q] = pb[q - 1] * B;
    }
#pragma unroll
    for (int q = 0; q <= I; ++q)
        D[q] = pa[q] * pb[I - q] * (1.0 / ((2 * q + 1) * (2 * I - 2 * q + 1)));
#pragma unroll
    for (int j = I; j >= 0; --j) {
#pragma unroll
        for (int k = 0; k <= j; ++k) c[far_index(I, j, k)] = far_factor(I, j, k) * D[k];
#pragma unroll
        for (int q = 0; q < j; ++q) D[q] = D[q] + D[q + 1];
    }
}

// The same averages in polar angles, d = |d| (cos th, sin th) and (x, y) =
// s^(1/2) (cos ph, sin ph): with cos^2j a = sum_q w_jq cos 2qa,
//   <(x dx + y dy)^(2j) d^(2(i-j))> = s^j sum_(q <= j) w_jq m_iq cos 2q ph,
//   m_iq = <d^2i cos 2q th>
// (the sines average to 0 over a rectangle), so the i + 1 moments m_iq of an
// order take the place of its (i + 1)(i + 2)/2 constants, and what remains of
// c_ij is a number far_polar(i, j, q).  Orders above 2 kFarPlain are formed
// so: 27 numbers per prism in LDS up to order 12, where the c_ijk are 83 (35
// KB of LDS, and registers that do not hold an order's 28), for about 40 more
// operations a pair at order 10.  48 models of up to 200,000 prisms of
// different rectangles: 119.5 ms with c_ijk up to order 10, 121.4 with the
// moments up to order 10, 111.4 with the moments up to order 12, 112.5 with
// c_ijk up to order 8 or 10 and the moments beyond (the arithmetic is then
// less, the LDS traffic more); with the c_ijk of order 12 it spills (214 ms).
constexpr int far_moment(int i, int q) { return (i - 1) * (i + 2) / 2 + q; }
constexpr int kFarMoments = far_moment(kFarMax + 1, 0);
static_assert(far_moment(1, 0) == 0 && far_moment(2, 0) == 2 && kFarMoments == 27, "m_iq");

constexpr double far_polar(int i, int j, int q) {
    const int m = i + j;
    double f = far_binom(2 * m, m) * far_binom(m, 2 * j) * far_binom(2 * j, j - q);
    for (int t = 0; t < m; ++t) f *= 0.25;
    return (q ? 2.0 : 1.0) * (m % 2 ? -f : f);
}

// Coefficient of dx^2p dy^(2(i-p)) in d^2i cos 2q th.
constexpr double far_angular(int i, int q, int p) {
    double f = 0.0;
    for (int k = 0; k <= q; ++k)
        if (p >= k && p - k <= i - q) {
            const double b = far_binom(2 * q, 2 * k) * far_binom(i - q, p - k);
            f += (q - k) % 2 ? -b : b;
        }
    return f;
}

// The moments of order 2I of a rectangle (A, B as in far_order_consts).
template <int I>
__device__ __forceinline__ void far_order_moments(double A, double B, double *m) {
    double pa[I + 1], pb[I + 1], mu[I + 1];
    pa[0] = pb[0] = 1.0;
#pragma unroll
    for (int q = 1; q <= I; ++q) {
        pa[q] = pa[q - 1] * A;
        pb[q] = pb[q - 1] * B;
    }
#pragma unroll
    for (int p = 0; p <= I; ++p)
        mu[p] = pa[p] * pb[I - p] * (1.0 / ((2 * p + 1) * (2 * (I - p) + 1)));
#pragma unroll
    for (int q = 0; q <= I; ++q) {
        double v = 0.0;
#pragma unroll
        for (int p = 0; p <= I; ++p) v = fma(far_angular(I, q, p), mu[p], v);
        m[far_moment(I, q)] = v;
    }
}

// far_polar(i, j, q) in scalar registers, set where it is used (83 of them
// hoisted out of the loop over prisms would not fit the registers).
template <int i, int j, int q>
__device__ __forceinline__ double polar_const() {
    constexpr unsigned long long bits = __builtin_bit_cast(unsigned long long, far_polar(i, j, q));
    constexpr int low = (int)(bits & 0xffffffffull);
    int hi, lo = 0;
    asm volatile("s_mov_b32 %0, %1" : "=s"(hi) : "i"((int)(bits >> 32)));
    if constexpr (low != 0) asm volatile("s_mov_b32 %0, %1" : "=s"(lo) : "i"(low));
    return __hiloint2double(hi, lo);
}

// Adds the terms (i, j .. i, q) to C_(i+j), with h = m_iq s^j cos 2q ph.
template <int I, int i, int q, int j>
__device__ __forceinline__ void polar_terms(double s, double h, double (&C)[2 * I + 1]) {
    // the first term to reach C_m: i = ceil(m / 2), q = 0
    constexpr bool first = q == 0 && i == (i + j + 1) / 2;
    const double f = polar_const<i, j, q>();
    C[i + j] = first ? f * h : fma(f, h, C[i + j]);
    if constexpr (j < i) polar_terms<I, i, q, j + 1>(s, h * s, C);
}

template <int I, int i, int q, class Consts>
__device__ __forceinline__ void polar_order(double s, const double (&T)[I + 1], const Consts &c,
                                            double (&C)[2 * I + 1]) {
    const double m = c.moment(far_moment(i, q));
    polar_terms<I, i, q, q>(s, q ? m * T[q] : m, C);
    if constexpr (q < i)
        polar_order<I, i, q + 1>(s, T, c, C);
    else if constexpr (i < I)
        polar_order<I, i + 1, 0>(s, T, c, C);
}

// C_1 .. C_2I from the moments.
template <int I, class Consts>
__device__ __forceinline__ void far_coefs_polar(double X, double Y, const Consts &c,
                                                double (&C)[2 * I + 1]) {
    const double s = X + Y, t1 = X - Y, t2 = 2.0 * t1, s2 = s * s;
    double T[I + 1];  // s^q cos 2q ph
    T[0] = 1.0;
    T[1] = t1;
#pragma unroll
    for (int q = 2; q <= I; ++q) T[q] = fma(t2, T[q - 1], q == 2 ? -s2 : -s2 * T[q - 2]);
    polar_order<I, 1, 0>(s, T, c, C);
}

// C_1 .. C_2I at X = x^2, Y = y^2; c(index) gives a constant.
template <int I, class Consts>
__device__ __forceinline__ void far_coefs(double X, double Y, const Consts &c,
                                          double (&C)[2 * I + 1]) {
    if constexpr (I > kFarPlain) {
        far_coefs_polar<I>(X, Y, c, C);
        return;
    }
    double mono[I + 1][I + 1];  // X^k Y^(j-k)
    mono[0][0] = 1.0;
#pragma unroll
    for (int j = 1; j <= I; ++j) {
        mono[j][0] = j == 1 ? Y : mono[j - 1][0] * Y;
#pragma unroll
        for (int k = 1; k <= j; ++k) mono[j][k] = j == 1 ? X : mono[j - 1][k - 1] * X;
    }
    // order by order, so that few constants are in registers at a time
#pragma unroll
    for (int i = 1; i <= I; ++i) {
        C[2 * i] = C[2 * i - 1] = 0.0;
#pragma unroll
        for (int j = 0; j <= i; ++j) {
            // the first order to reach C_m is i = ceil(m / 2), with j = m - i
            const bool first = i == (i + j + 1) / 2;
#pragma unroll
            for (int k = 0; k <= j; ++k) {
                const double ck = c(far_index(i, j, k));
                if (j == 0)
                    C[i] = first ? ck : C[i] + ck;
                else if (first && k == 0)
                    C[i + j] = ck * mono[j][k];
                else
                    C[i + j] = fma(ck, mono[j][k], C[i + j]);
            }
        }
    }
}

// <1/r> over the face at height z, s = x^2 + y^2.
template <int I>
__device__ __forceinline__ double far_face(double s, double z, const double (&C)[2 * I + 1]) {
    const double inv = dm::rsqrt_pos(fma(z, z, s));
    const double u = inv * inv;
    double p = C[2 * I];
#pragma unroll
    for (int m = 2 * I - 1; m >= 1; --m) p = fma(p, u, C[m]);
    return fma(inv, p * u, inv);
}

// <1/r> and its derivative -d<1/r>/dz / z = <1/r^3> (the sums over m with C_m
// and (2m + 1) C_m: Horner's scheme for the polynomial and its derivative).
template <int I>
__device__ __forceinline__ void far_face_top(double s, double z, const double (&C)[2 * I + 1],
                                             double &f, double &f3) {
    const double inv = dm::rsqrt_pos(fma(z, z, s));
    const double u = inv * inv;
    double p = C[2 * I], d = C[2 * I];
#pragma unroll
    for (int m = 2 * I - 1; m >= 1; --m) {
        p = fma(p, u, C[m]);
        d = fma(d, u, p);
    }
    // p = sum C_m u^(m-1), d = its derivative's scheme: sum m C_m u^(m-1)
    const double inv3 = inv * u;
    f = fma(inv, p * u, inv);
    f3 = fma(inv3, u * fma(2.0, d, p), inv3);
}

// Square of the distance, in units of the half-diagonal h of the rectangle,
// from which order 2I suffices: (1 / ((2I + 3) 4e-15))^(1 / (2I + 2)) =
// 181, 48, 21.8, 12.9, 8.8 for I = 2, 3, 4, 5, 6.
__device__ __forceinline__ constexpr double far_ratio2(int I) {
    return I == 2   ? 181.0 * 181.0
           : I == 3 ? 48.0 * 48.0
           : I == 4 ? 21.8 * 21.8
           : I == 5 ? 12.9 * 12.9
                    : 8.8 * 8.8;
}

// The squared half-diagonal that decides on the far form, NaN (never far) for a
// prism without area, whose far form is 0 times a sum that is not finite at the
// points of its axis, and for sizes whose powers could leave the range of
// doubles: with 1e-10 < h < 1e10 and distances below 1e14 the largest, (h r)^12
// and r^-25, stay below 1e290.
__device__ __forceinline__ double far_half2(double A, double B) {
#pragma clang fp contract(off)
    const double h2 = A + B;
    return h2 > 1e-20 && h2 < 1e20 ? h2 : __builtin_nan("");
}

// A staged far prism: the rectangle's centre from the workgroup's origin, top,
// bottom, weight times area, far_half2.  The centre is formed from bounds
// already shifted to the origin, so its rounding is relative to its distance
// from the workgroup's points and not to the coordinates' size.
struct alignas(16) FarPrism {
    double x, y, t, b, w, h2;
};

// Constants in LDS (kept per prism: stride kFarStride) or, for a tile of
// equal rectangles, in scalar registers.
// The c_ijk, then the moments, each 16-byte aligned.
constexpr int kFarMomentsAt = (kFarConsts + 1) / 2 * 2;
constexpr int kFarStride = (kFarMomentsAt + kFarMoments + 1) / 2 * 2;
struct FarLds {
    const double *c;
    __device__ __forceinline__ double operator()(int k) const { return c[k]; }
    __device__ __forceinline__ double moment(int k) const { return c[kFarMomentsAt + k]; }
};
__device__ __forceinline__ double wave_uniform(double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}
__device__ __forceinline__ uint64_t wave_uniform(unsigned long long v) {
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (uint64_t)hi << 32 | lo;
}
template <int I>
struct FarScalar {
    double c[far_base(I + 1)];
    __device__ __forceinline__ explicit FarScalar(const double *lds) {
#pragma unroll
        for (int k = 0; k < far_base(I + 1); ++k) c[k] = wave_uniform(lds[k]);
    }
    __device__ __forceinline__ double operator()(int k) const { return c[k]; }
};

// weight * S of the staged prism at (x, y, u), x and y relative to the
// workgroup's origin.
template <int I, class Consts>
__device__ __forceinline__ double far_gz(const FarPrism &rec, const Consts &c, double px, double py,
                                         double pu) {
    const double x = rec.x - px, y = rec.y - py;
    const double X = x * x, Y = y * y, s = X + Y;
    double C[2 * I + 1];
    far_coefs<I>(X, Y, c, C);
    return rec.w * (far_face<I>(s, rec.b - pu, C) - far_face<I>(s, rec.t - pu, C));
}

// Bounding box of the points of a wave (x and y relative to the origin), and
// the squared distance of its farthest corner from the origin.
struct FarBox {
    double x0, x1, y0, y1, u0, u1, reach2;
};

// Whether the coordinates relative to the origin are good enough for a prism
// at squared distance d2 of points up to reach2 (squared) from the origin.
// Point and prism round to about 2^-53 of their distance R from it, 2 R / r
// roundings of the distance r between them; the closed form, which takes their
// difference from the coordinates as given, is off by 4 to 16 (r/h)^2
// roundings.  So points of a workgroup may be spread widely (2 R / r <= 4
// (r/h)^2: R up to 1360 h at the shortest r, 8.8 h), but one that lies a
// continent away, or at a placeholder's 1e20 m, does not spoil the others.
__device__ __forceinline__ bool far_resolved(double d2, double h2, double reach2) {
#pragma clang fp contract(off)
    return d2 * d2 * d2 >= 0.25 * reach2 * (h2 * h2);
}

// Whether far_resolved can fail at the distances of the far form, 8.8 h and
// more.  Asked once per wave and prism: in all lanes' own tests far_resolved
// cost 1 to 4% of calls with many near prisms.
__device__ __forceinline__ bool far_unsure(double h2, double reach2) {
#pragma clang fp contract(off)
    return !(reach2 <= 1.85e6 * h2);
}

// The same rule as a larger h2: order 2I and lower ones by it start where
// far_resolved holds.  For kernels that have no registers for a test beside the
// distance's: the six tensor fields' and ten fields' close pairs took 13% longer
// with one.  By FP32 logarithm and exponential, 1e-4 on the far side.
__device__ __forceinline__ float far_reach(double reach2) {  // log2(R^2 / 4)
#pragma clang fp contract(off)
    return __builtin_amdgcn_logf((float)reach2) - 2.0f;
}
template <int I>
__device__ __forceinline__ double far_sure_half2(double h2, float reach) {
#pragma clang fp contract(off)
    const float log_h2 = __builtin_amdgcn_logf((float)h2);
    const float log_r2 = fmaf(2.0f, log_h2, reach) * (1.0f / 3.0f);
    const double least = (double)__builtin_amdgcn_exp2f(log_r2) * (1.0001 / far_ratio2(I));
    return h2 < least ? least : h2;
}

// A lane's value, the same for all lanes (lane uniform in the wave).
__device__ __forceinline__ double lane_value(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Smallest squared distance from the box to the nearer face centre of a
// staged prism; NaN (never far) if the prism or the whole box is NaN.  (No
// contraction here and below: kernels that share the work of a pair have to
// come to the same decision.)
__device__ __forceinline__ double far_distance2(const FarBox &b, const FarPrism &p) {
#pragma clang fp contract(off)
    // fmax drops a NaN operand: keep it with the sum of the differences
    const double nan_guard = ((p.x - b.x0) + (p.y - b.y0) + (p.t - b.u0) + (p.b - b.u0)) * 0.0;
    const double dx = fmax(fmax(b.x0 - p.x, p.x - b.x1), 0.0);
    const double dy = fmax(fmax(b.y0 - p.y, p.y - b.y1), 0.0);
    const double dt = fmax(fmax(b.u0 - p.t, p.t - b.u1), 0.0);
    const double db = fmax(fmax(b.u0 - p.b, p.b - b.u1), 0.0);
    const double d = fmin(dt, db);
    return fma(dx, dx, fma(dy, dy, d * d)) + nan_guard;
}

// Whether order 2I serves a prism at squared distance d2 (see far_half2 on the
// upper bound).
template <int I>
__device__ __forceinline__ bool far_enough(double d2, double h2) {
#pragma clang fp contract(off)
    return d2 >= far_ratio2(I) * h2 && d2 < 1e28;
}

// Prisms staged per pass of the g_u kernels, at most one per lane of a wave,
// so that a wave sorts a tile into the forms with one comparison and one
// ballot; with 32 a workgroup's LDS (27 KB) lets registers, not LDS, set the
// waves per SIMD.
constexpr int kGzTile = 32;
constexpr int kGzWaves = 4;
constexpr int kGzThreads = 64 * kGzWaves;
constexpr int kGzList = 256;

// One staged prism of the closed form: bounds and weight.
struct alignas(16) GzPrism {
    double w, e, s, n, b, t, grho, pad;
};

// Prisms given as (m, 6) rows [W, E, S, N, B, T] and densities, for gz_stage.
struct GzExplicit {
    const double *prisms, *density;
    __device__ bool get(int64_t p, double (&b)[6], double &rho) const {
#pragma unroll
        for (int c = 0; c < 6; ++c) b[c] = prisms[6 * p + c];
        rho = density[p];
        return false;
    }
};

// LDS of a g_u workgroup, one point per lane.
struct GzShared {
    GzPrism tile[kGzTile];
    FarPrism far[kGzTile];
    // constants per prism, if the rectangles differ; the last entry holds
    // those of the workgroup's first prism
    alignas(16) double consts[(kGzTile + 1) * kFarStride];
    FarBox box[kGzWaves];
    double A, B;        // squared half-sides of the last entry
    unsigned live;      // prisms of the tile that are not left out
    unsigned different; // 0: every live prism has the last entry's rectangle
    // closed-form pairs of a wave and their values (gz_close)
    uint16_t list[kGzWaves][kGzList];
    double value[kGzWaves][64];
    dm::Tables tables;
};

__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    return v;
}

// A lane's point: as given, and relative to the workgroup's origin (xo, yo).
struct GzPoint {
    double e, n, u, x, y, xo, yo;
};

// Bounding box of the wave's points into box[wave] (read after the next
// barrier).
__device__ __forceinline__ void point_box(const GzPoint &pt, FarBox *box) {
#pragma clang fp contract(off)
    FarBox b{wave_min(pt.x), wave_max(pt.x), wave_min(pt.y),
             wave_max(pt.y), wave_min(pt.u), wave_max(pt.u), 0.0};
    b.reach2 = fmax(b.x0 * b.x0, b.x1 * b.x1) + fmax(b.y0 * b.y0, b.y1 * b.y1);
    if ((threadIdx.x & 63) == 0) box[threadIdx.x >> 6] = b;
}

// All constants of a rectangle, in three parts of similar cost.
__device__ __forceinline__ void far_consts(double A, double B, int part, double *c) {
    if (part == 0) {
        far_order_consts<1>(A, B, c);
        far_order_consts<2>(A, B, c);
        far_order_consts<3>(A, B, c);
    } else if (part == 1) {
        far_order_moments<1>(A, B, c + kFarMomentsAt);
        far_order_moments<2>(A, B, c + kFarMomentsAt);
        far_order_moments<3>(A, B, c + kFarMomentsAt);
        far_order_moments<4>(A, B, c + kFarMomentsAt);
    } else {
        far_order_moments<5>(A, B, c + kFarMomentsAt);
        far_order_moments<6>(A, B, c + kFarMomentsAt);
    }
}

// Squared half-sides of a prism's rectangle.
__device__ __forceinline__ void half_sides2(const double (&b)[6], double &A, double &B) {
#pragma clang fp contract(off)
    const double width = b[1] - b[0], length = b[3] - b[2];
    A = 0.25 * width * width;
    B = 0.25 * length * length;
}

// The last entry of constants from prism p (the first of the workgroup's chunk).
template <class Src>
__device__ __forceinline__ void gz_table(const Src &src, int64_t p, GzShared &sh) {
    if (threadIdx.x < 3) {
        double b[6], rho, A, B;
        src.get(p, b, rho);
        half_sides2(b, A, B);
        far_consts(A, B, threadIdx.x, sh.consts + kGzTile * kFarStride);
        if (threadIdx.x == 0) {
            sh.A = A;
            sh.B = B;
        }
    }
}

// The staged record of a prism (weight: of the far form, times the area).
__device__ __forceinline__ FarPrism far_prism(const double (&b)[6], double xo, double yo,
                                              double weight) {
#pragma clang fp contract(off)
    double A, B;
    half_sides2(b, A, B);
    const double area = (b[1] - b[0]) * (b[3] - b[2]);
    return FarPrism{0.5 * ((b[0] - xo) + (b[1] - xo)), 0.5 * ((b[2] - yo) + (b[3] - yo)),
                    b[5],                              b[4],
                    weight * area,                     far_half2(A, B)};
}

// Whether squared half-sides are equal enough to share constants: to 2^-36, as
// the sides of equal cells of some metres round at coordinates of some 1e6 m.
// The constants scale corrections of up to (h/r)^2 / 3, so sharing them is off
// by up to that part of 2^-36: 6e-14 of <1/r> at the shortest distance, 8.8
// half-diagonals, 1e-14 at 21.8 (order 8), 2e-15 at 48 (order 6).  The closed
// form is off by up to 16 (r/h)^2 2^-53 = 1.4e-13 at 8.8.  (The two constants of
// order 2 from each prism itself leave 1e-15, but cost g_zz of 20,011 bodies
// 10%, a layer of 100 x 100 cells 3%.)
__device__ __forceinline__ bool far_alike(double A, double B, double A0, double B0) {
    return fabs(A - A0) <= 0x1p-36 * A0 && fabs(B - B0) <= 0x1p-36 * B0;
}

// Stages prisms [t0, t0 + cnt), cnt <= kGzTile.  Src::get(p, bounds, rho)
// returns whether the prism is left out.  Holds every barrier it needs before
// and after.  Grids of equal cells, by far the most common layers, use the
// last entry's constants; a tile with other rectangles gets its own, prism by
// prism.
template <class Src>
__device__ __forceinline__ void gz_stage(const Src &src, int64_t t0, int cnt, double xo, double yo,
                                         GzShared &sh) {
    __syncthreads();
    if (threadIdx.x < 64) {
        const int q = threadIdx.x;
        double b[6] = {}, rho = 0.0;
        bool skip = true;
        if (q < cnt) skip = src.get(t0 + q, b, rho);
        double A, B;
        half_sides2(b, A, B);
        if (q < cnt) {
            sh.tile[q] = GzPrism{b[0], b[1], b[2], b[3], b[4], b[5], kG * rho, 0.0};
            sh.far[q] = far_prism(b, xo, yo, kG * rho);
        }
        const bool same = far_alike(A, B, sh.A, sh.B);
        const uint64_t live = __ballot(!skip), different = __ballot(!skip && !same);
        if (q == 0) {
            sh.live = (unsigned)live;
            sh.different = different ? 1u : 0u;
        }
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(sh.different)) {
        // one part per half wave
        static_assert(kGzTile == 32 && kGzThreads >= 96, "room for three parts");
        const int q = threadIdx.x & 31, part = threadIdx.x >> 5;
        if (q < cnt && part < 3) {
            double A, B;
            const GzPrism &t = sh.tile[q];
            const double b[6] = {t.w, t.e, t.s, t.n, 0.0, 0.0};
            half_sides2(b, A, B);
            far_consts(A, B, part, sh.consts + q * kFarStride);
        }
        __syncthreads();
    }
}

// Squared distance of the lane's own point from the nearer face centre.
__device__ __forceinline__ double lane_distance2(const FarPrism &p, double px, double py,
                                                 double pu) {
    const double x = p.x - px, y = p.y - py, t = p.t - pu, z = p.b - pu;
    return fma(x, x, fma(y, y, fmin(t * t, z * z)));
}

// Calls f(p) for the set bits p of a wave-uniform mask, in order.
template <class Mask, class F>
__device__ __forceinline__ void for_bits(Mask mask, const F &f) {
    while (mask) {
        const int p = sizeof(Mask) == 8 ? __builtin_ctzll(mask) : __builtin_ctz((unsigned)mask);
        mask &= mask - 1;
        f(p);
    }
}

// Orders a wave's own LDS writes before its reads (the wave's LDS operations
// complete in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The constants of prism p of the tile (different: 0 or 1).
__device__ __forceinline__ const double *gz_consts(const double *consts, int p,
                                                   unsigned different) {
    return consts + (kGzTile + (p - kGzTile) * (int)different) * kFarStride;
}

// Adds the closed form of the pairs in `mask` (bit p: prism p of the tile at
// the lane's point).  The wave's pairs are listed by lane and prism and
// evaluated 64 at a time, one pair per lane whoever's it is, and each lane
// adds the values of its own pairs in order.  Always the general closed
// form: listed pairs lie between the prism's planes too often for 64 of them
// to need the lean one.
__device__ __forceinline__ void gz_close(GzShared &sh, unsigned mask, const GzPoint &pt,
                                         double &acc) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint16_t *list = sh.list[wave];
    double *value = sh.value[wave];
    while (any_lane(mask != 0)) {
        const int count = __popc(mask);
        int incl = count;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o);
            if (lane >= o) incl += v;
        }
        const int total = __builtin_amdgcn_readlane(incl, 63);
        const int n = total < kGzList ? total : kGzList;
        // the lane's entries [at, end); pairs past the list's end wait for the
        // next round
        const int at = incl - count < kGzList ? incl - count : kGzList;
        int end = at;
        while (mask && end < kGzList) {
            list[end++] = (uint16_t)((unsigned)__builtin_ctz(mask) | lane << 5);
            mask &= mask - 1;
        }
        wave_sync();
        for (int b = 0; b < n; b += 64) {
            const unsigned pair = list[b + lane < n ? b + lane : b];
            const int from = pair >> 5;
            const double e = __shfl(pt.e, from), nn = __shfl(pt.n, from), u = __shfl(pt.u, from);
            const GzPrism sp = sh.tile[pair & 31u];
            value[lane] = sp.grho * gu_sum<false, true>(sp.e - e, sp.w - e, sp.n - nn, sp.s - nn,
                                                        sp.t - u, sp.b - u, sh.tables, nullptr);
            wave_sync();
            for (int k = at > b ? at : b; k < end && k < b + 64; ++k) acc += value[k - b];
            wave_sync();
        }
    }
}

// Close lanes from which a wave evaluates the lean closed form for all its
// lanes rather than list its pairs (about 300 against 400 issue slots).  Lanes
// that need the general form go to the list either way, and no longer take the
// wave's other lanes along.
constexpr int kGzInline = 40;

// Adds the prisms of `near`, which the bounding box does not show to be far
// from all of the wave's points.  Each lane takes order 2 kFarMax where its own
// distance allows and the closed form elsewhere, so the form of a pair does
// not depend on the points that share its wave (bar the orders of the far
// form, which agree to 4e-15) and neither, to rounding, does the result on
// their order.
__device__ __forceinline__ void gz_near(GzShared &sh, unsigned near, unsigned unsure,
                                        unsigned different, const GzPoint &pt, double &acc) {
    // the lane's pairs that its offset from the origin does not resolve
    unsigned mask = 0, coarse = 0;
    for_bits(near & unsure, [&](int p) {
        const double d2 = lane_distance2(sh.far[p], pt.x, pt.y, pt.u);
        double px = pt.x, py = pt.y;  // their squares only here, not held in registers
        asm volatile("" : "+v"(px), "+v"(py));
        const bool fine = far_resolved(d2, sh.far[p].h2, fma(px, px, py * py));
        coarse |= fine ? 0u : 1u << p;
    });
    for_bits(near, [&](int p) {
        const FarPrism rec = sh.far[p];
        const double d2 = lane_distance2(rec, pt.x, pt.y, pt.u);
        const bool close = !far_enough<kFarMax>(d2, rec.h2) || ((coarse >> p) & 1u);
        if (any_lane(!close)) {
            const double v =
                far_gz<kFarMax>(rec, FarLds{gz_consts(sh.consts, p, different)}, pt.x, pt.y, pt.u);
            acc += close ? 0.0 : v;
        }
        const GzPrism sp = sh.tile[p];
        const bool lean = close && !needs_general<0x8u>(pt.e, pt.n, pt.u, sp.w, sp.e, sp.s, sp.n,
                                                        sp.b, sp.t);
        if (__popcll(__ballot(lean)) >= kGzInline) {
            const double v = sp.grho * gu_sum<false, false>(sp.e - pt.e, sp.w - pt.e, sp.n - pt.n,
                                                            sp.s - pt.n, sp.t - pt.u, sp.b - pt.u,
                                                            sh.tables, nullptr);
            acc += lean ? v : 0.0;
            mask |= close && !lean ? 1u << p : 0u;
        } else {
            mask |= close ? 1u << p : 0u;
        }
    });
    gz_close(sh, mask, pt, acc);
}

// One order of the far form, its constants in scalar registers where the
// tile's rectangles are equal (up to order 6: 19 constants).
template <int I>
__device__ __forceinline__ void gz_far(const GzShared &sh, unsigned different, unsigned mask,
                                       const GzPoint &pt, double &acc) {
    if (!mask) return;
    if constexpr (I <= kFarPlain) {
        if (!different) {
            const FarScalar<I> c(sh.consts + kGzTile * kFarStride);
            for_bits(mask, [&](int p) { acc += far_gz<I>(sh.far[p], c, pt.x, pt.y, pt.u); });
            return;
        }
    }
    for_bits(mask, [&](int p) {
        acc += far_gz<I>(sh.far[p], FarLds{gz_consts(sh.consts, p, different)}, pt.x, pt.y, pt.u);
    });
}

// Whether no prism like the chunk's first one is unsure for the wave (uniform;
// after the first gz_stage).  Per prism of every tile this cost 1% of a model of
// 1,000,000 prisms.
__device__ __forceinline__ bool gz_sure(const GzShared &sh) {
    return !any_lane(far_unsure(0.999 * (sh.A + sh.B), sh.box[threadIdx.x >> 6].reach2));
}

// Adds the g_u of the staged tile at the wave's points (sure: gz_sure).  The forms are chosen
// per prism and wave from the distance between the prism's face centres and
// the bounding box of the wave's points: the lowest order that serves all of
// them, uniform in the wave; then the prisms nearer than that, lane by lane.
__device__ __forceinline__ void gz_tile(int cnt, bool sure, const GzPoint &pt, double &acc,
                                        GzShared &sh) {
    const int q = threadIdx.x & 63;
    const unsigned live = __builtin_amdgcn_readfirstlane(sh.live);
    const unsigned different = __builtin_amdgcn_readfirstlane(sh.different);
    const FarPrism mine = sh.far[q < cnt ? q : 0];
    const FarBox &box = sh.box[threadIdx.x >> 6];
    double d2 = far_distance2(box, mine);
    unsigned unsure = 0;
    if (different || !sure) {
        unsure = (unsigned)__ballot(far_unsure(mine.h2, box.reach2));
        if (unsure && !far_resolved(d2, mine.h2, box.reach2)) d2 = -1.0;
    }
    unsigned rest = live;
    auto take = [&](bool far) {
        const unsigned m = (unsigned)__ballot(far) & rest;
        rest &= ~m;
        return m;
    };
    const unsigned m2 = take(far_enough<2>(d2, mine.h2)), m3 = take(far_enough<3>(d2, mine.h2));
    const unsigned m4 = take(far_enough<4>(d2, mine.h2)), m5 = take(far_enough<5>(d2, mine.h2));
    const unsigned m6 = take(far_enough<6>(d2, mine.h2));
    gz_far<2>(sh, different, m2, pt, acc);
    gz_far<3>(sh, different, m3, pt, acc);
    gz_far<4>(sh, different, m4, pt, acc);
    gz_far<5>(sh, different, m5, pt, acc);
    gz_far<6>(sh, different, m6, pt, acc);
    if (rest) gz_near(sh, rest, unsure, different, pt, acc);
}

}  // namespace dev
}  // namespace hmx
