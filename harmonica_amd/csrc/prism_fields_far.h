// Far form of any set of prism fields (potential, accelerations, tensor), by
// the expansion of prism_far.h.
//
// The z-integral of 1/r is ln(z + r), so the potential is the face average of
// l_T - l_B, l = ln(z + r); with q = |z| and lambda = ln(q + r), l = lambda
// for z >= 0 and ln(x^2 + y^2) - lambda for z < 0, so for a point above the
// top or below the bottom V = sg (lambda_T - lambda_B), sg the sign of z (the
// logarithm of x^2 + y^2 cancels; points between the two, whichever of them
// is higher, take the closed form).  g_u is the average of phi_B - phi_T, phi = 1/r, and the other fields
// are derivatives of these two.  With f^(m) the m-th derivative with respect
// to s = x^2 + y^2, the average of f over the rectangle is sum_m K_m f^(m), K_m
// the polynomials C_m of prism_far.h without phi's factor, and
//   d<f>/dx   = 2x (sum_m K_m f^(m+1) + sum_m K'_m f^(m)),   K' = dK/dX, X = x^2,
//   d2<f>/dx2 = d<f>/dx / x + 4X (sum_m K_m f^(m+2) + 2 sum_m K'_m f^(m+1)
//               + sum_m K''_m f^(m)),
// likewise along y and for the mixed derivative, and d<phi>/dz = 2z sum_m K_m
// phi^(m+1): the same sums serve several fields, and the derivatives of K
// need no constants of their own.  phi^(m) = L_m u^m / r, L_m = (-1)^m (2m -
// 1)!!/2^m; lambda^(m) = L_m g_m with g_1 = -u t, g_2 = -u^2 t (1 + t) / 3, t =
// r/(r + q), and from s lambda' = (1 - q phi) / 2, differentiated m times,
//   g_(m+1) = (2m g_m + q u^m / r) / ((2m + 1) s).
// The two faces are subtracted first, and that recurrence then runs on the
// differences alone.  It amplifies rounding by r^2/s a step, on terms smaller
// by (h/r)^2 a step: by h^2/s together, so points closer than 2 h to the
// prism's vertical axis (straight above it) take the closed form too.  g_nn
// follows from Laplace's equation where g_ee and g_uu are selected.
//
// The truncation of a second derivative is up to about 60 times that of the
// average (2e-13 of the field at the shortest distance of order 4, measured;
// 5e-14 at order 6); the closed form, of terms of order one for a field of
// order (h/r)^2, is off by 3e-12 and 3e-13 there.
//
// Two kernels share a call: the far form in one (three or four waves per SIMD,
// 97% of the issue cycles busy; in one kernel with the closed forms' 230
// registers it had two, and 40% of them were idle), the close pairs in the
// other, which adds to the first one's partial sums.  Both take the same
// decisions from the same records.  Ten fields as above: 29.3 -> 14.4 ms;
// magnetic field of 90,000 prisms at 13,130 points: 16.1 -> 11.2 ms; g_zz of
// 20,011 bodies at 2999 points, the pair kernels: 459 -> 396 us.
#pragma once

#include "prism_far.h"

namespace hmx {
namespace dev {

// What a field set needs of the expansion.
template <unsigned M>
struct FarNeeds {
    using F = FieldSet<M>;
    static constexpr bool nn_direct = F::nn && !(F::ee && F::uu);
    static constexpr bool lambda1 = F::ge || F::gn || F::ee || nn_direct;  // first derivatives
    static constexpr bool lambda2 = F::ee || nn_direct || F::en;           // second
    static constexpr bool lambda = F::pot || lambda1 || lambda2;
    static constexpr bool phi1 = F::uu || F::eu || F::nu;
    static constexpr bool phi = F::gu || phi1;
    static constexpr bool kx = F::ge || F::ee || F::en || F::eu;
    static constexpr bool ky = F::gn || nn_direct || F::en || F::nu;
    // logarithms along horizontal edges without a coefficient (on_edge_line)
    static constexpr bool edges = F::eu || F::nu;
    // Highest order 2I.  317 x 290 cells, ten fields at 13,320 points: up to
    // order 6 19.4 ms (close pairs 6.5), up to order 8 14.4 ms (1.9).
    static constexpr int orders = lambda ? 4 : 5;
    static constexpr int consts = far_base(orders + 1);
    static constexpr int stride = (consts + 1) / 2 * 2;
};

// c_ijk of prism_far.h without phi's factor, in place of far_order_consts.
constexpr double far_plain(int i, int j, int k) {
    const int m = i + j;
    double f = far_binom(m, 2 * j) * far_binom(2 * j, 2 * k);
    for (int t = 0; t < j; ++t) f *= 4.0;
    for (int t = 2; t <= m; ++t) f /= t;
    return f;
}

template <int I>
__device__ __forceinline__ void far_order_plain(double A, double B, double *c) {
    double scaled[far_base(I + 1)];
    far_order_consts<I>(A, B, scaled);
#pragma unroll
    for (int j = 0; j <= I; ++j)
#pragma unroll
        for (int k = 0; k <= j; ++k)
            c[far_index(I, j, k)] =
                scaled[far_index(I, j, k)] * (far_plain(I, j, k) / far_factor(I, j, k));
}

// All constants of a rectangle, one order per part (0 .. orders - 1).
template <unsigned M>
__device__ __forceinline__ void far_plain_consts(double A, double B, int part, double *c) {
    if (part == 0) far_order_plain<1>(A, B, c);
    if (part == 1) far_order_plain<2>(A, B, c);
    if (part == 2) far_order_plain<3>(A, B, c);
    if constexpr (FarNeeds<M>::orders >= 4)
        if (part == 3) far_order_plain<4>(A, B, c);
    if constexpr (FarNeeds<M>::orders >= 5)
        if (part == 4) far_order_plain<5>(A, B, c);
}

// K (dx = dy = 0) or its derivative d^(dx+dy) K / dX^dx dY^dy at orders up to 2I:
// out[m] for m >= 2 (dx + dy) (smaller ones are 0), and K_0 = 1.
template <int I, int DX, int DY, class Consts>
__device__ __forceinline__ void far_poly(const double (&mono)[I + 1][I + 1], const Consts &c,
                                         double (&out)[2 * I + 1]) {
    constexpr int D = DX + DY;
    auto falling = [](int n, int d) { return d == 0 ? 1 : d == 1 ? n : n * (n - 1); };
#pragma unroll
    for (int m = D ? 2 * D : 1; m <= 2 * I; ++m) {
        double v = 0.0;
        bool first = true;
#pragma unroll
        for (int j = D; j <= I; ++j) {
            const int i = m - j;
            if (i < 1 || i > I || j > i) continue;
#pragma unroll
            for (int k = DX; k <= j - DY; ++k) {
                const double ck = c(far_index(i, j, k));
                const int f = falling(k, DX) * falling(j - k, DY);
                if (j == D) {  // a constant term
                    v = first ? f * ck : fma((double)f, ck, v);
                } else {
                    const double x = f * mono[j - D][k - DX];
                    v = first ? ck * x : fma(ck, x, v);
                }
                first = false;
            }
        }
        out[m] = v;
    }
    out[0] = D ? 0.0 : 1.0;
}

// 1 / d for finite d > 0 (two Newton steps in one third-order correction).
__device__ __forceinline__ double far_rcp(double d) {
    const double y = __builtin_amdgcn_rcp(d);
    const double e = fma(-d, y, 1.0);
    return fma(y * e, 1.0 + e, y);
}

// The fields of FieldSet<M> of a prism of unit weight, per area, from order 2I
// (x, y: the rectangle's centre from the point; zt, zb: top and bottom).
template <int I, unsigned M, class Consts>
__device__ __forceinline__ void far_fields(double x, double y, double zt, double zb,
                                           const Consts &c, double (&vs)[FieldSet<M>::count],
                                           const dm::Tables &tab) {
    using F = FieldSet<M>;
    using Q = FarNeeds<M>;
    constexpr int N = 2 * I;                       // K_0 .. K_N
    constexpr int NV = Q::lambda2 ? N + 2 : (Q::lambda1 ? N + 1 : N);  // lambda derivatives
    constexpr int NZ = Q::lambda ? NV - 1 : N + 1;  // z times phi derivatives
    constexpr int NW = Q::phi1 ? N + 1 : N;         // phi derivatives
    constexpr int NU = NZ > NW ? NZ : NW;
    const double X = x * x, Y = y * y, s = X + Y;
    const double sg = zb >= 0.0 ? 1.0 : -1.0;
    // differences of the faces' derivatives over L_m: phi bottom - top and z phi
    // bottom - top, lambda top - bottom
    double dw[NU + 1], dz[NU + 1], dv[NV + 1], len[2];
#pragma unroll
    for (int face = 0; face < 2; ++face) {  // bottom, then top
        const double z = face ? zt : zb;
        const double r2 = fma(z, z, s), inv = dm::rsqrt_pos(r2), u = inv * inv;
        double w = inv;
#pragma unroll
        for (int m = 0; m <= NU; ++m) {
            if (m) w *= u;
            if (Q::phi && m <= NW) dw[m] = face ? dw[m] - w : w;
            if ((Q::lambda || F::uu) && m >= 1 && m <= NZ)
                dz[m] = face ? fma(-z, w, dz[m]) : z * w;
        }
        if constexpr (Q::lambda) {
            const double q = fabs(z), t = far_rcp(fma(q, inv, 1.0)), ut = u * t;
            if constexpr (F::pot) len[face] = fma(r2, inv, q);
            dv[1] = face ? dv[1] - ut : ut;
            const double g2 = u * fma(ut, t, ut) * (1.0 / 3.0);
            dv[2] = face ? dv[2] - g2 : g2;
        }
    }
    if constexpr (Q::lambda) {
        const double is = sg * far_rcp(s);  // q phi top - bottom = -sg dz
#pragma unroll
        for (int m = 2; m < NV; ++m)
            dv[m + 1] = (is * (1.0 / (2 * m + 1))) * fma(2.0 * m * sg, dv[m], -dz[m]);
    }
    double L = 1.0;
#pragma unroll
    for (int m = 1; m <= (NV > NU ? NV : NU); ++m) {
        L *= -0.5 * (2 * m - 1);
        if (Q::phi && m <= NW) dw[m] *= L;
        if (F::uu && m <= N + 1) dz[m] *= L;
        if (Q::lambda && m <= NV) dv[m] *= L;
    }
    double mono[I + 1][I + 1];  // X^k Y^(j-k)
    mono[0][0] = 1.0;
#pragma unroll
    for (int j = 1; j <= I; ++j) {
        mono[j][0] = j == 1 ? Y : mono[j - 1][0] * Y;
#pragma unroll
        for (int k = 1; k <= j; ++k) mono[j][k] = j == 1 ? X : mono[j - 1][k - 1] * X;
    }
    // sum_m P_m d[m + shift] for m = from .. N
    auto dot = [&](const double(&P)[N + 1], const double *d, int shift, int from) {
        double v = P[N] * d[N + shift];
#pragma unroll
        for (int m = N - 1; m >= from; --m) v = fma(P[m], d[m + shift], v);
        return v;
    };
    double K[N + 1], P[N + 1];
    far_poly<I, 0, 0>(mono, c, K);
    if constexpr (F::gu) vs[F::slot(3)] = dot(K, dw, 0, 1) + dw[0];
    if constexpr (F::uu) vs[F::slot(6)] = -2.0 * (dot(K, dz, 1, 1) + dz[1]);
    if constexpr (F::pot) {
        const double l = dm::log_pos(dm::div(len[1], len[0]), tab);
        vs[F::slot(0)] = sg * (l + dot(K, dv, 0, 1));
    }
    double w1 = 0.0, v1 = 0.0, v2 = 0.0;
    if constexpr (F::eu || F::nu) w1 = dot(K, dw, 1, 1) + dw[1];
    if constexpr (Q::lambda1) v1 = dot(K, dv, 1, 1) + dv[1];
    if constexpr (Q::lambda2) v2 = dot(K, dv, 2, 1) + dv[2];
    double ex = 0.0, ny = 0.0, v1x = 0.0;
    if constexpr (Q::kx) {
        far_poly<I, 1, 0>(mono, c, P);
        if constexpr (F::eu) vs[F::slot(8)] = -2.0 * x * (w1 + dot(P, dw, 0, 2));
        if constexpr (F::ge || F::ee) ex = 2.0 * sg * (v1 + dot(P, dv, 0, 2));
        if constexpr (F::ge) vs[F::slot(1)] = -x * ex;
        if constexpr (F::ee || F::en) v1x = dot(P, dv, 1, 2);
    }
    if constexpr (F::ee) {
        far_poly<I, 2, 0>(mono, c, P);
        vs[F::slot(4)] = fma(4.0 * sg * X, v2 + fma(2.0, v1x, dot(P, dv, 0, 4)), ex);
    }
    if constexpr (Q::ky) {
        far_poly<I, 0, 1>(mono, c, P);
        if constexpr (F::nu) vs[F::slot(9)] = -2.0 * y * (w1 + dot(P, dw, 0, 2));
        if constexpr (F::gn || Q::nn_direct) ny = 2.0 * sg * (v1 + dot(P, dv, 0, 2));
        if constexpr (F::gn) vs[F::slot(2)] = -y * ny;
        double v1y = 0.0;
        if constexpr (Q::nn_direct || F::en) v1y = dot(P, dv, 1, 2);
        if constexpr (Q::nn_direct) {
            far_poly<I, 0, 2>(mono, c, P);
            vs[F::slot(5)] = fma(4.0 * sg * Y, v2 + fma(2.0, v1y, dot(P, dv, 0, 4)), ny);
        }
        if constexpr (F::en) {
            far_poly<I, 1, 1>(mono, c, P);
            vs[F::slot(7)] = 4.0 * sg * (x * y) * (v2 + ((v1x + v1y) + dot(P, dv, 0, 4)));
        }
    }
    if constexpr (F::nn && !Q::nn_direct) vs[F::slot(5)] = -(vs[F::slot(4)] + vs[F::slot(6)]);
}

// The staged record of a prism per unit weight; one with its bottom above its
// top as the prism between them, of the opposite sign (point above or below
// both is asked by these heights).
__device__ __forceinline__ FarPrism field_prism(const double (&b)[6], const GzPoint &pt) {
    FarPrism p = far_prism(b, pt.xo, pt.yo, 1.0);
    if (p.t < p.b) p = FarPrism{p.x, p.y, p.b, p.t, -p.w, p.h2};
    return p;
}

// Points level with a prism's top or bottom: where such a point lies on the line
// of a horizontal edge, the logarithm along the edge, of ln(x + r) for x < 0,
// has the argument 0 and counts as 0 (the convention of the closed form,
// prism_device.h), in g_ez along northing and in g_nz along easting.  By that,
// and not by the field's limit, which the far form gives, field sets with these
// two leave level points to the closed form.

// Whether the far form of the highest order serves the lane's own point (h2:
// far_sure_half2).
template <unsigned M>
__device__ __forceinline__ bool field_lane_far(const FarPrism &p, double h2, const GzPoint &pt) {
#pragma clang fp contract(off)
    const double x = p.x - pt.x, y = p.y - pt.y, t = p.t - pt.u, z = p.b - pt.u;
    const double s = fma(x, x, y * y), d2 = s + fmin(t * t, z * z);
    const bool far = far_enough<FarNeeds<M>::orders>(d2, h2);
    if constexpr (FarNeeds<M>::lambda) {
        const bool outside = FarNeeds<M>::edges ? t < 0.0 || z > 0.0 : t <= 0.0 || z >= 0.0;
        return far && s >= 4.0 * h2 && outside;
    }
    return FarNeeds<M>::edges ? far && t != 0.0 && z != 0.0 : far;
}

// Whether order 2I serves every point in the box.
template <int I, unsigned M>
__device__ __forceinline__ bool field_box_far(double d2, double h2, const FarPrism &p,
                                              const FarBox &b) {
#pragma clang fp contract(off)
    if constexpr (FarNeeds<M>::lambda) {
        const double dx = fmax(fmax(b.x0 - p.x, p.x - b.x1), 0.0);
        const double dy = fmax(fmax(b.y0 - p.y, p.y - b.y1), 0.0);
        const bool outside = FarNeeds<M>::edges ? p.t < b.u0 || p.b > b.u1
                                                : p.t <= b.u0 || p.b >= b.u1;
        if (!(fma(dx, dx, dy * dy) >= 4.0 * h2 && outside)) return false;
    } else if constexpr (FarNeeds<M>::edges) {
        const bool level = (b.u0 <= p.t && p.t <= b.u1) || (b.u0 <= p.b && p.b <= b.u1);
        if (level) return false;
    }
    return far_enough<I>(d2, h2);
}

// What a call sums: Op::fields the field set, Op::weights per prism, Op::values
// sums per point and
//   Op::combine(weight, vs, out)  the sums' terms from the fields of unit weight,
//   Op::closed<kGeneral>(e, n, u, b, weight, acc, flags, tab)  the closed form.
template <class Op>
struct FieldFarShared {
    using Q = FarNeeds<Op::fields>;
    FarPrism far[kGzTile];  // w: the rectangle's area
    double weight[kGzTile][Op::weights];
    // constants per prism, if the rectangles differ; the last entry holds
    // those of the workgroup's first prism
    alignas(16) double consts[(kGzTile + 1) * Q::stride];
    FarBox box[kGzWaves];
    double A, B;
    unsigned live, different;
    dm::Tables tables;
};

// The lane's point i (the last one past the end), the origin at the first
// point of the workgroup, and the wave's box.
__device__ __forceinline__ GzPoint field_point(const double *__restrict__ oe,
                                               const double *__restrict__ on,
                                               const double *__restrict__ ou, int64_t base,
                                               int64_t n_obs, FarBox *box) {
    const int64_t i = base + threadIdx.x, ii = i < n_obs ? i : n_obs - 1;
    GzPoint pt{oe[ii], on[ii], ou[ii], 0.0, 0.0, oe[base], on[base]};
    pt.x = pt.e - pt.xo;
    pt.y = pt.n - pt.yo;
    point_box(pt, box);
    return pt;
}

// One order of the far form for the prisms in `mask`.
template <int I, class Op>
__device__ __forceinline__ void field_far(const FieldFarShared<Op> &sh, unsigned different,
                                          unsigned mask, const GzPoint &pt,
                                          double (&acc)[Op::values]) {
    using Q = FarNeeds<Op::fields>;
    auto pair = [&](int p, const auto &c) {
        const FarPrism rec = sh.far[p];
        double vs[FieldSet<Op::fields>::count], out[Op::values];
        far_fields<I, Op::fields>(rec.x - pt.x, rec.y - pt.y, rec.t - pt.u, rec.b - pt.u, c, vs,
                                  sh.tables);
        Op::combine(sh.weight[p], vs, out);
#pragma unroll
        for (int s = 0; s < Op::values; ++s) acc[s] = fma(rec.w, out[s], acc[s]);
    };
    if (!mask) return;
    if constexpr (I <= 3) {
        if (!different) {
            const FarScalar<I> c(sh.consts + kGzTile * Q::stride);
            for_bits(mask, [&](int p) { pair(p, c); });
            return;
        }
    }
    for_bits(mask, [&](int p) {
        pair(p, FarLds{sh.consts + (kGzTile + (p - kGzTile) * (int)different) * Q::stride});
    });
}

// The far pairs of 256 points (from `base`) and the prisms [c0, c1), added to acc.
template <class Op, class Src>
__device__ __forceinline__ void field_far_chunk(const Src &src, const double *__restrict__ oe,
                                                const double *__restrict__ on,
                                                const double *__restrict__ ou, int64_t base,
                                                int64_t n_obs, int64_t c0, int64_t c1,
                                                double (&acc)[Op::values],
                                                FieldFarShared<Op> &sh) {
    constexpr unsigned M = Op::fields;
    using Q = FarNeeds<M>;
    if constexpr (FieldSet<M>::pot) dm::load_tables(&sh.tables);
    const GzPoint pt = field_point(oe, on, ou, base, n_obs, sh.box);
    if (threadIdx.x < Q::orders && c0 < c1) {
        double b[6], weight[Op::weights], A, B;
        src.get(c0, b, weight);
        half_sides2(b, A, B);
        far_plain_consts<M>(A, B, threadIdx.x, sh.consts + kGzTile * Q::stride);
        if (threadIdx.x == 0) {
            sh.A = A;
            sh.B = B;
        }
    }
    for (int64_t t0 = c0; t0 < c1; t0 += kGzTile) {
        const int cnt = (int)(c1 - t0 < kGzTile ? c1 - t0 : kGzTile);
        __syncthreads();
        if (threadIdx.x < 64) {
            const int q = threadIdx.x;
            double b[6] = {}, weight[Op::weights] = {}, A, B;
            bool skip = true;
            if (q < cnt) skip = src.get(t0 + q, b, weight);
            half_sides2(b, A, B);
            if (q < cnt) {
                sh.far[q] = field_prism(b, pt);
#pragma unroll
                for (int k = 0; k < Op::weights; ++k) sh.weight[q][k] = weight[k];
            }
            const bool same = far_alike(A, B, sh.A, sh.B);
            const uint64_t live = __ballot(!skip), other = __ballot(!skip && !same);
            if (q == 0) {
                sh.live = (unsigned)live;
                sh.different = other ? 1u : 0u;
            }
        }
        __syncthreads();
        const unsigned live = __builtin_amdgcn_readfirstlane(sh.live);
        const unsigned different = __builtin_amdgcn_readfirstlane(sh.different);
        if (different) {
            static_assert(kGzTile == 32 && kGzThreads >= 160, "one order per half wave");
            const int q = threadIdx.x & 31, part = threadIdx.x >> 5;
            if (q < cnt && part < Q::orders) {
                double b[6], weight[Op::weights], A, B;
                src.get(t0 + q, b, weight);
                half_sides2(b, A, B);
                far_plain_consts<M>(A, B, part, sh.consts + q * Q::stride);
            }
            __syncthreads();
        }
        const int q = threadIdx.x & 63;
        const FarPrism mine = sh.far[q < cnt ? q : 0];
        const FarBox &box = sh.box[threadIdx.x >> 6];
        const double d2 = far_distance2(box, mine);
        const double h2 = far_sure_half2<Q::orders>(mine.h2, far_reach(box.reach2));
        unsigned rest = live;
        auto take = [&](bool far) {
            const unsigned m = (unsigned)__ballot(far) & rest;
            rest &= ~m;
            return m;
        };
        const unsigned m2 = take(field_box_far<2, M>(d2, h2, mine, box));
        const unsigned m3 = take(field_box_far<3, M>(d2, h2, mine, box));
        field_far<2>(sh, different, m2, pt, acc);
        field_far<3>(sh, different, m3, pt, acc);
        if constexpr (Q::orders >= 4)
            field_far<4>(sh, different, take(field_box_far<4, M>(d2, h2, mine, box)), pt, acc);
        if constexpr (Q::orders >= 5)
            field_far<5>(sh, different, take(field_box_far<5, M>(d2, h2, mine, box)), pt, acc);
        // prisms that are far from some of the wave's points only
        for_bits(rest, [&](int p) {
            const bool far = field_lane_far<M>(sh.far[p], lane_value(h2, p), pt);
            if (!any_lane(far)) return;
            double v[Op::values] = {};
            field_far<Q::orders>(sh, different, 1u << p, pt, v);
#pragma unroll
            for (int s = 0; s < Op::values; ++s) acc[s] += far ? v[s] : 0.0;
        });
    }
}

// LDS of one wave of the close kernel: the prisms near its points.
template <class Op>
struct FieldCloseWave {
    double bounds[64][6];
    double weight[64][Op::weights];
    FarPrism far[64];
    uint16_t list[kGzList];
    double value[64];
};
template <class Op>
struct FieldCloseShared {
    FieldCloseWave<Op> wave[kGzWaves];
    FarBox box[kGzWaves];
    dm::Tables tables;
};

// The closed form of the pairs in `mask` (bit p: the wave's prism p at the
// lane's point), as gz_close.
template <class Op>
__device__ __forceinline__ void field_close(FieldCloseWave<Op> &sh, const dm::Tables &tables,
                                            uint64_t mask, const GzPoint &pt,
                                            double (&acc)[Op::values], uint32_t &flags) {
    const int lane = threadIdx.x & 63;
    while (any_lane(mask != 0)) {
        const int count = __popcll(mask);
        int incl = count;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o);
            if (lane >= o) incl += v;
        }
        const int total = __builtin_amdgcn_readlane(incl, 63);
        const int n = total < kGzList ? total : kGzList;
        const int at = incl - count < kGzList ? incl - count : kGzList;
        int end = at;
        while (mask && end < kGzList) {
            sh.list[end++] = (uint16_t)((unsigned)__builtin_ctzll(mask) | lane << 6);
            mask &= mask - 1;
        }
        wave_sync();
        for (int b = 0; b < n; b += 64) {
            const unsigned pair = sh.list[b + lane < n ? b + lane : b];
            const int from = pair >> 6, p = pair & 63u;
            const double e = __shfl(pt.e, from), nn = __shfl(pt.n, from), u = __shfl(pt.u, from);
            double out[Op::values] = {};
            Op::template closed<true>(e, nn, u, sh.bounds[p], sh.weight[p], out, flags, tables);
#pragma unroll
            for (int s = 0; s < Op::values; ++s) {
                sh.value[lane] = out[s];
                wave_sync();
                double sum = 0.0;
                for (int k = at > b ? at : b; k < end && k < b + 64; ++k) sum += sh.value[k - b];
                acc[s] += sum;
                wave_sync();
            }
        }
    }
}

// Lanes from which a wave evaluates the lean closed form for all of them (as
// kGzInline; the general form of a field set costs more beside the lean one,
// and each field of a listed pair is added by itself).  Six tensor fields of
// 147 x 133 cells of 903 m at 8008 points 870 m above the highest, this
// kernel: 965 us with any lane that needs the general form sending all of the
// wave's to the list, 707 with only such lanes listed and a limit of 40, 545
// with 24, 530 with 16 or 10; ten fields of 317 x 290 cells, the call: 14.0,
// 13.9, 13.6, 13.7 and 13.8 ms.
constexpr int kFieldInline = 24;

// The close pairs of 256 points and the prisms [c0, c1), added to acc.  Each
// wave by itself: a lane reads a prism (the next one while this tile is
// worked on), and only tiles with a prism near the wave's points go to LDS;
// with the workgroup's barriers per tile the waves waited for each other most
// of the time (magnetic field of 90,000 prisms at 13,130 points, up to order
// 6: 5.0 -> 3.0 ms).  Returns whether the wave had any.
template <class Op, class Src>
__device__ __forceinline__ bool field_close_chunk(const Src &src, const double *__restrict__ oe,
                                                  const double *__restrict__ on,
                                                  const double *__restrict__ ou, int64_t base,
                                                  int64_t n_obs, int64_t c0, int64_t c1,
                                                  double (&acc)[Op::values], uint32_t &flags,
                                                  FieldCloseShared<Op> &shared) {
    constexpr unsigned M = Op::fields;
    using Q = FarNeeds<M>;
    dm::load_tables(&shared.tables);
    const GzPoint pt = field_point(oe, on, ou, base, n_obs, shared.box);
    __syncthreads();
    const int q = threadIdx.x & 63;
    const FarBox box = shared.box[threadIdx.x >> 6];
    const float reach = far_reach(box.reach2);
    FieldCloseWave<Op> &sh = shared.wave[threadIdx.x >> 6];
    bool any = false, skip = true;
    double b[6] = {}, weight[Op::weights] = {};
    if (c0 + q < c1) skip = src.get(c0 + q, b, weight);
    for (int64_t t0 = c0; t0 < c1; t0 += 64) {
        FarPrism rec = field_prism(b, pt);
        rec.h2 = far_sure_half2<Q::orders>(rec.h2, reach);
        const uint64_t near = __ballot(
            !skip && !field_box_far<Q::orders, M>(far_distance2(box, rec), rec.h2, rec, box));
        if (near) {
            sh.far[q] = rec;
#pragma unroll
            for (int k = 0; k < 6; ++k) sh.bounds[q][k] = b[k];
#pragma unroll
            for (int k = 0; k < Op::weights; ++k) sh.weight[q][k] = weight[k];
        }
        skip = true;
        if (t0 + 64 + q < c1) skip = src.get(t0 + 64 + q, b, weight);
        if (!near) continue;
        any = true;
        wave_sync();
        uint64_t mask = 0;
        for_bits(near, [&](int p) {
            const bool close = !field_lane_far<M>(sh.far[p], sh.far[p].h2, pt);
            const double *t = sh.bounds[p];
            const bool lean = close && !needs_general<M>(pt.e, pt.n, pt.u, t[0], t[1], t[2], t[3],
                                                         t[4], t[5]);
            if (__popcll(__ballot(lean)) >= kFieldInline) {
                double out[Op::values] = {};
                uint32_t none = 0;
                Op::template closed<false>(pt.e, pt.n, pt.u, t, sh.weight[p], out, none,
                                           shared.tables);
#pragma unroll
                for (int s = 0; s < Op::values; ++s) acc[s] += lean ? out[s] : 0.0;
                mask |= close && !lean ? 1ull << p : 0ull;
            } else {
                mask |= close ? 1ull << p : 0ull;
            }
        });
        field_close<Op>(sh, shared.tables, mask, pt, acc, flags);
        wave_sync();
    }
    return any;
}

// LDS of a workgroup that evaluates every pair by the closed form.
template <class Op>
struct FieldClosedShared {
    double bounds[64][6];
    double weight[64][Op::weights];
    unsigned long long live;
    dm::Tables tables;
};

// All pairs of 256 points and the prisms [c0, c1) by the closed form, added to
// acc: per wave first the prisms that no lane needs the general form for, then
// the others, in two loops, which keep the forms' registers apart.
template <class Op, class Src>
__device__ __forceinline__ void field_closed_chunk(const Src &src, const double *__restrict__ oe,
                                                   const double *__restrict__ on,
                                                   const double *__restrict__ ou, int64_t base,
                                                   int64_t n_obs, int64_t c0, int64_t c1,
                                                   double (&acc)[Op::values], uint32_t &flags,
                                                   FieldClosedShared<Op> &sh) {
    dm::load_tables(&sh.tables);
    const int64_t i = base + threadIdx.x, ii = i < n_obs ? i : n_obs - 1;
    const double e = oe[ii], n = on[ii], u = ou[ii];
    for (int64_t t0 = c0; t0 < c1; t0 += 64) {
        __syncthreads();
        if (threadIdx.x < 64) {
            const int q = threadIdx.x;
            double b[6], weight[Op::weights];
            bool skip = true;
            if (t0 + q < c1) {
                skip = src.get(t0 + q, b, weight);
#pragma unroll
                for (int k = 0; k < 6; ++k) sh.bounds[q][k] = b[k];
#pragma unroll
                for (int k = 0; k < Op::weights; ++k) sh.weight[q][k] = weight[k];
            }
            const uint64_t live = __ballot(!skip);
            if (q == 0) sh.live = live;
        }
        __syncthreads();
        const uint64_t live = wave_uniform(sh.live);
        uint64_t general = 0;
        for_bits(live, [&](int p) {
            const double *t = sh.bounds[p];
            if (any_lane(needs_general<Op::fields>(e, n, u, t[0], t[1], t[2], t[3], t[4], t[5]))) {
                general |= 1ull << p;
                return;
            }
            Op::template closed<false>(e, n, u, t, sh.weight[p], acc, flags, sh.tables);
        });
        for_bits(general, [&](int p) {
            Op::template closed<true>(e, n, u, sh.bounds[p], sh.weight[p], acc, flags, sh.tables);
        });
    }
}

}  // namespace dev
}  // namespace hmx
