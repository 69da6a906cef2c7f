// FP64 device math for the pairwise kernels: square root, reciprocal square
// root, quotient, natural logarithm and arctangents.  They drop the
// special-case handling the kernels never need (infinities, negative
// arguments) and use the hardware v_rsq_f64 / v_rcp_f64 estimates (relative
// error below 2^-24) with Newton-type refinement; their accuracy against
// mpmath is checked by tests/test_gpu_devmath.py through hmx_devmath_eval.
//
// On gfx950 an FP64 VALU instruction takes 4 cycles per wave, v_rsq_f64 and
// v_rcp_f64 about 16, and 32-bit integer instructions about 2, so the
// routines favour fused multiply-adds and integer bit manipulation over
// extra reciprocals and 64-bit selects.
//
// Methods (all from the literature, constants generated by
// gen_devmath_tables.py):
//  * sqrt: one Goldschmidt step from the reciprocal-square-root estimate and
//    one residual correction (Markstein's formulation);
//  * quotient: one Newton-Raphson step on the reciprocal estimate, then one
//    residual correction of the quotient;
//  * log: table-driven logarithm of P. T. P. Tang (ACM TOMS 16(4), 1990):
//    a = 2^e m, m in [0.5, 1), c_j ~ 1/F_j with F_j = (1 + j/128)/2 <= m,
//    ln a = e ln2 - ln c_j + log1p(m c_j - 1), -ln c_j stored as lead +
//    trail so that e ln2_hi + lead is exact; log1p on [0, 2^-7) by a
//    degree-6 minimax polynomial;
//  * atan(num / den), 0 <= num <= den: c_j = j/32 nearest to the ratio,
//    atan(t) = atan(c_j) + atan((t - c_j) / (1 + t c_j)) (|delta| <= 1/64,
//    odd minimax polynomial of degree 7); atan2 and the ratio form add the
//    octant.
#pragma once

#include <hip/hip_runtime.h>

#include "devmath_tables.h"

namespace hmx {
namespace dm {

struct alignas(32) LogEntry {
    double c, lead, trail, pad;
};

// Tables copied to LDS by every workgroup that uses log_pos / the arctangents.
struct alignas(32) Tables {
    LogEntry log_tab[128];
    double2 atan_tab[33];
};

// Cooperative copy of the constant tables into LDS; the caller must
// __syncthreads() before use.
__device__ __forceinline__ void load_tables(Tables *t) {
    for (int i = threadIdx.x; i < 128; i += blockDim.x)
        t->log_tab[i] = LogEntry{kLogTable[i][0], kLogTable[i][1], kLogTable[i][2], 0.0};
    for (int i = threadIdx.x; i < 33; i += blockDim.x)
        t->atan_tab[i] = make_double2(kAtanTable[i][0], kAtanTable[i][1]);
}

// sqrt(s) for finite s > 0.  The estimate y ~ 1/sqrt(s) has a relative
// error e < 2^-24; one Goldschmidt step gives g ~ sqrt(s) with error
// 1.5 e^2 < 2^-47, and the residual correction g + (s - g^2) y / 2 brings
// it to about one ulp (the error of y only scales the correction).
__device__ __forceinline__ double sqrt_pos(double s) {
    const double y = __builtin_amdgcn_rsq(s);
    const double h = 0.5 * y;
    double g = s * y;
    const double r = fma(-g, h, 0.5);
    g = fma(g, r, g);
    const double d = fma(-g, g, s);
    return fma(d, h, g);
}

// sqrt(s) for finite s >= 0 (exact 0 for 0).
__device__ __forceinline__ double sqrt_nn(double s) {
    const double g = sqrt_pos(s);
    return s == 0.0 ? 0.0 : g;
}

// 1 / sqrt(s) for finite s > 0: the estimate y has the residual
// e = 1 - s y^2 (|e| < 2^-22), and 1/sqrt(s) = y (1 - e)^(-1/2)
// = y + y e (1/2 + 3/8 e) up to 5/16 e^3 < 2^-67: five FP64 operations in a
// chain of four after the estimate (nine and seven with a Goldschmidt step
// followed by a Newton step, which is bound by the same two roundings, of
// s y and of the sum).  The pairwise 1/r kernels are bound by FP64 issue,
// and this is the largest part of a pair: 300,007 point masses at 65,536
// points, g_z, 12.76 -> 10.56 ms; 30,011 sources on a 401 x 367 grid, 3.14 ->
// 2.58 ms, with the same error against 64-bit sums (2.1e-15).
__device__ __forceinline__ double rsqrt_pos(double s) {
    const double y = __builtin_amdgcn_rsq(s);
    const double e = fma(-(s * y), y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// n / d for finite nonzero d (within about one ulp): y ~ 1/d to 2^-47
// after one Newton step, q = n y, and the residual n - d q (one fma)
// corrects q.
__device__ __forceinline__ double div(double n, double d) {
    double y = __builtin_amdgcn_rcp(d);
    const double e = fma(-d, y, 1.0);
    y = fma(y, e, y);
    const double q = n * y;
    const double rem = fma(-d, q, n);
    return fma(rem, y, q);
}

// ln(a) for finite normal a > 0 (any input reads the table in bounds).
__device__ __forceinline__ double log_pos(double a, const Tables &T) {
    const double m = __builtin_amdgcn_frexp_mant(a);  // a = 2^e m, m in [0.5, 1)
    const double ed = (double)__builtin_amdgcn_frexp_exp(a);
    // j = the top 7 fraction bits of a, which are those of m
    const unsigned j = ((unsigned)__double2hiint(a) >> 13) & 127u;
    const LogEntry t = T.log_tab[j];
    const double r = fma(m, t.c, -1.0);  // in [0, 2^-7) up to rounding
    double p = fma(r, kLogPoly[4], kLogPoly[3]);
    p = fma(r, p, kLogPoly[2]);
    p = fma(r, p, kLogPoly[1]);
    p = fma(r, p, kLogPoly[0]);
    const double hi = fma(ed, kLn2Hi, t.lead);  // exact
    const double lo = fma(ed, kLn2Lo, t.trail);
    return hi + (fma(r * r, p, r) + lo);
}

// atan(num / den) in [0, pi/4] for 0 <= num <= den, den > 0.
__device__ __forceinline__ double atan_unit(double num, double den, const Tables &T) {
    // Nearest j to 32 num / den from the rough quotient (0 <= j <= 32; the
    // bound also keeps a NaN's table index in range): adding 1.5 * 2^52
    // rounds to an integer held in the low word.
    const double u = fma(num * __builtin_amdgcn_rcp(den), 32.0, 0x1.8p52);
    const unsigned j = min((unsigned)__double2loint(u), 32u);
    const double c = fma(u, 0.03125, -0x1.8p47);  // j / 32, exact
    const double delta = div(fma(-c, den, num), fma(c, num, den));
    const double d2 = delta * delta;
    double q = fma(d2, kAtanPoly[2], kAtanPoly[1]);
    q = fma(d2, q, kAtanPoly[0]);
    const double2 at = T.atan_tab[j];
    return at.x + fma(delta * d2, q, delta + at.y);
}

// Principal value of atan(a / b); +-pi/2 by the sign of a when b == 0; 0
// when a == 0.
__device__ __forceinline__ double atan_ratio(double a, double b, const Tables &T) {
    const double aa = fabs(a), bb = fabs(b);
    const bool inv = aa > bb;
    double res = atan_unit(fmin(aa, bb), fmax(aa, bb), T);
    res = inv ? (kHalfPiHi - res) + kHalfPiLo : res;
    const bool neg = (a < 0.0) != (b < 0.0);
    res = neg ? -res : res;
    return a == 0.0 ? 0.0 : res;
}

// atan2(a, b) in [-pi, pi] for finite a, b (the sign of the result is the
// sign bit of a, so atan2(-0, b < 0) = -pi as in IEEE 754).  kZeroSafe:
// atan2(+-0, 0) = +-0; without it the caller guarantees (a, b) != (0, 0).
// The quadrant adds k pi/2 (k = 0, 1, 2) to +-atan_unit, which gives a
// value in [0, pi] before the sign.
template <bool kZeroSafe = true>
__device__ __forceinline__ double atan2_full(double a, double b, const Tables &T) {
    const double aa = fabs(a), bb = fabs(b);
    const double hi = fmax(aa, bb);
    const double res = atan_unit(fmin(aa, bb), kZeroSafe ? fmax(hi, 0x1p-1022) : hi, T);
    const bool inv = aa > bb, negb = b < 0.0;
    // inv, b >= 0: pi/2 - t;  inv, b < 0: pi/2 + t;  b < 0: pi - t;  else t
    const double kd = (double)(inv ? 1 : (negb ? 2 : 0));
    const double t = inv != negb ? -res : res;
    return copysign(fma(kd, kHalfPiLo, fma(kd, kHalfPiHi, t)), a);
}

// v with its sign flipped where `sign` is 0x80000000 (0 leaves it): one
// integer xor on the high word.
__device__ __forceinline__ double flip_sign(double v, unsigned sign) {
    return __hiloint2double((int)((unsigned)__double2hiint(v) ^ sign), __double2loint(v));
}

// 0x80000000 where `neg`, else 0.
__device__ __forceinline__ unsigned sign_mask(bool neg) { return neg ? 0x80000000u : 0u; }

}  // namespace dm
}  // namespace hmx
