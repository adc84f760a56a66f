// i2_math.hpp -- FP64 square root, logarithm and two-argument arctangent
// for the quadrature hot loop.
//
// The library versions cost about 16 (sqrt), 92 (log) and 99 (atan2) VALU
// instructions on gfx950; the inner integral needs three of each of the
// first two and one atan2 per quadrature point, so they dominate the kernel.
// These versions drop the range handling the hot loop never needs, are
// branch-free on the normal path, and stay within about 2 ulp (checked on the
// host against 120-bit references).
//
// Methods (textbook):
//   sqrt:  s > 0 normal: y ~ 1/sqrt(s) from the hardware estimate, one
//          Goldschmidt step g = s y, h = y/2, r = 1/2 - g h, then
//          g + (s - g^2) h (one correction; within 1 ulp, not always
//          correctly rounded).
//   log:   x = 2^k m with m in [1/2, 1) (frexp); j = rint(512 m) - 256 picks
//          c_j = 1/2 + j/512 from a 257-entry table of invc_j = 1/c_j (rounded)
//          and T_j = -log(invc_j) (hi + lo); r = m invc_j - 1 by one fma,
//          |r| <= 2^-9; log1p(r) by its Taylor series to r^6; log x =
//          (k ln2_hi + T_hi) + (k ln2_lo + T_lo + log1p r).  c_256 = 1 and
//          c_0 = 1/2 exactly, so there is no cancellation near x = 1.  No division.
//   atan2: reduce to t = min(|x|,|y|)/max(|x|,|y|) in [0, 1]; the nearest
//          centre c = k/32 (from a reciprocal estimate) and a 33-entry table of
//          atan(k/32) (hi + lo) give atan t = atan c + atan u with
//          u = (n - c d)/(d + c n) for t = n/d, |u| <= 2^-6; atan u by its
//          Taylor series to u^9/9; then the octant and quadrant identities.
//   1/x and a/b (rcp_pos, div_pos): hardware reciprocal estimate refined by
//          Newton steps with fma residuals; used where the operand is a
//          product of distances, far inside [2^-1000, 2^1000].
// Non-finite, zero, negative and subnormal arguments take the library path
// (log, atan2).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#ifndef I2_HD
#define I2_HD __host__ __device__
#endif

namespace i2m {

constexpr double LN2_HI = 0.69314718036912382;         // ln 2 to 32 significant bits
constexpr double LN2_LO = 1.9082149292705877e-10;      // ln 2 - LN2_HI
constexpr double PI_HI = 3.1415926535897931, PI_LO = 1.2246467991473532e-16;
constexpr double PIO2_HI = 1.5707963267948966, PIO2_LO = 6.123233995736766e-17;

// library calls for arguments outside the fast paths, kept out of line
static I2_HD __noinline__ double log_slow(double x) { return ::log(x); }
static I2_HD __noinline__ double atan2_slow(double y, double x) { return ::atan2(y, x); }

// estimate of 1/sqrt(s): the hardware instruction on the device, the library on the host
__device__ __forceinline__ double rsq_estimate(double s) { return __builtin_amdgcn_rsq(s); }
__host__ inline double rsq_estimate(double s) { return 1.0 / ::sqrt(s); }

// estimate of 1/x: the hardware instruction on the device; on the host a
// single-precision reciprocal of the mantissa, so that host checks exercise
// the refinement from a low-precision start
__device__ __forceinline__ double rcp_estimate(double x) { return __builtin_amdgcn_rcp(x); }
__host__ inline double rcp_estimate(double x) {
    int k;
    const double m = ::frexp(x, &k);
    return ::ldexp((double)(1.0f / (float)m), -k);
}

// 1/x for |x| in [2^-1000, 2^1000]: estimate (relative error below 2^-24 on
// gfx950, measured by the device math test), then two Newton steps
// y += y (1 - x y), each with the residual exact in one fma: 2^-24 -> 2^-48
// -> rounding
I2_HD __forceinline__ double rcp_pos(double x) {
    double y = rcp_estimate(x);
    double e = fma(-x, y, 1.0);
    y = fma(y, e, y);
    e = fma(-x, y, 1.0);
    return fma(y, e, y);
}

// The same from one cubic step y += y (e + e^2), e = 1 - x y: 2^-24 -> 2^-72,
// then rounding.  One instruction less than two Newton steps; used by the
// inner integral, where it runs once per point and panel.
I2_HD __forceinline__ double rcp_cubic(double x) {
    const double y = rcp_estimate(x);
    const double e = fma(-x, y, 1.0);
    return fma(y, fma(e, e, e), y);
}

// a / b for |b| in [2^-1000, 2^1000]: one Newton step on 1/b (relative error
// eps ~ 2^-48), the quotient q = a y, and one residual correction
// q + (a - b q) y, whose relative error is eps^2 plus rounding
I2_HD __forceinline__ double div_pos(double a, double b) {
    double y = rcp_estimate(b);
    y = fma(y, fma(-b, y, 1.0), y);
    const double q = a * y;
    return fma(fma(-b, q, a), y, q);
}

// sqrt of a positive normal number (squared distances of the hot loop)
I2_HD __forceinline__ double sqrt_pos(double s) {
    const double y = rsq_estimate(s);
    double g = s * y, h = 0.5 * y;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    const double d = fma(-g, g, s);
    return fma(d, h, g);
}

// The same from one cubic step: with y ~ 1/sqrt(s), g = s y and e = 1 - g y,
// sqrt(s) = g (1 - e)^(-1/2) = g + g e (1/2 + 3 e/8 + ...), truncated below
// 2^-70 and within 1 ulp (g's own rounding enters by half through e).  Five
// instructions after the estimate instead of seven; used by the inner integral.
I2_HD __forceinline__ double sqrt_cubic(double s) {
    const double y = rsq_estimate(s);
    const double g = s * y;
    const double e = fma(-g, y, 1.0);
    return fma(g * e, fma(e, 0.375, 0.5), g);
}

// sqrt(s) as sqrt_cubic and 1/sqrt(s) from the same estimate (y + y e (1/2 + 3 e/8))
I2_HD __forceinline__ double sqrt_rsqrt(double s, double* inv) {
    const double y = rsq_estimate(s);
    const double g = s * y;
    const double e = fma(-g, y, 1.0);
    const double c = fma(e, 0.375, 0.5);
    *inv = fma(y * e, c, y);
    return fma(g * e, c, g);
}

// a * b + c for a Horner step whose addend c is a constant.  On the device
// this is one three-operand v_fma_f64: left to itself the compiler keeps such
// constants in VGPRs and emits a copy into the accumulator before each
// two-operand v_fmac_f64.
I2_HD __forceinline__ double fma_k(double a, double b, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
    double d;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
    return d;
#else
    return fma(a, b, c);
#endif
}

// Reduction tables (gen_math_tables.py), held as arrays so that an entry's
// address is a shift of its index: log entries j = 0..256 for the centres
// c_j = 1/2 + j/512, atan entries k = 0..32 for atan(k/32).
struct LogEntry { double invc, thi, tlo; };
struct AtanEntry { double hi, lo; };
constexpr int LOGTAB_N = 257;
constexpr int ATANTAB_N = 33;
struct MathTable {
    double invc[LOGTAB_N], thi[LOGTAB_N], tlo[LOGTAB_N];
    AtanEntry atan[ATANTAB_N];
};
constexpr LogEntry h_logent[LOGTAB_N] = {
#include "i2_logtab.inc"
};
constexpr AtanEntry h_atanent[ATANTAB_N] = {
#include "i2_atantab.inc"
};
constexpr MathTable make_mathtab() {
    MathTable t{};
    for (int k = 0; k < LOGTAB_N; ++k) { t.invc[k] = h_logent[k].invc; t.thi[k] = h_logent[k].thi; t.tlo[k] = h_logent[k].tlo; }
    for (int k = 0; k < ATANTAB_N; ++k) t.atan[k] = h_atanent[k];
    return t;
}
static constexpr MathTable h_mathtab = make_mathtab();
static __constant__ LogEntry c_logent[LOGTAB_N] = {
#include "i2_logtab.inc"
};
static __constant__ AtanEntry c_atanent[ATANTAB_N] = {
#include "i2_atantab.inc"
};
// copies the tables into `s` (LDS) with the threads of the block; the caller synchronises
__device__ __forceinline__ void fill_mathtab(MathTable& s) {
    for (int k = threadIdx.x; k < LOGTAB_N; k += blockDim.x) {
        s.invc[k] = c_logent[k].invc; s.thi[k] = c_logent[k].thi; s.tlo[k] = c_logent[k].tlo;
    }
    for (int k = threadIdx.x; k < ATANTAB_N; k += blockDim.x) s.atan[k] = c_atanent[k];
}

// log of a positive normal number with the reduction table `tab` (LDS on the device)
// true for positive normal numbers (one class test on the device)
I2_HD __forceinline__ bool pos_normal(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_class(x, 0x100);   // bit 8: positive normal
#else
    return x >= 2.2250738585072014e-308 && x <= 1.7976931348623157e308;
#endif
}

// The table log for any x: log x for positive normal x, a meaningless value
// otherwise.  Every argument reads inside the table, since the index comes
// from the bits of x.  Callers check pos_normal(x) and redo the other lanes
// with log_slow.
I2_HD __forceinline__ double log_tab_any(double x, const MathTable* __restrict__ tab) {
    int k;
    const double m = frexp(x, &k);                 // x = m 2^k, m in [1/2, 1) for normal x
    // nearest centre c_j = 1/2 + j/512 (ties upward): with f the fraction bits
    // of a normal x (m = (1 + f)/2), j = floor(256 f + 1/2), from the top 9
    // fraction bits b = floor(512 f) as (b + 1) >> 1, in [0, 256] for any bits
    uint64_t bits;
    memcpy(&bits, &x, sizeof bits);
    const int j = (int)((((uint32_t)(bits >> 43) & 0x1ffu) + 1u) >> 1);
    const double r = fma(m, tab->invc[j], -1.0);   // |r| <= 2^-9
    // log1p(r) = r - r^2/2 + r^3/3 - r^4/4 + r^5/5 - r^6/6 (truncation below 2^-56 relative),
    // as r + r^2 (-1/2 + (r/3)(1 - 3r/4 + 3r^2/5 - r^3/2)): the constants 1/3 and
    // -1/6 would share their low word, which the compiler then copies into
    // place on every call
    const double q = fma(r, fma(r, fma_k(r, -0.5, 0.6), -0.75), 1.0);
    const double p = fma(r * r, fma(r * (1.0 / 3.0), q, -0.5), r);
    // k ln2_hi + T_hi is exact: k ln2_hi has 53 bits, and for k = 1 and
    // c_j < sqrt(1/2) the two terms cancel by Sterbenz' lemma
    const double dk = (double)k;
    return fma(dk, LN2_HI, tab->thi[j]) + (fma(dk, LN2_LO, tab->tlo[j]) + p);
}

// log of an argument that is not positive normal: -inf at 0, NaN below,
// infinity and NaN themselves, subnormals scaled into the table's range.  Inline,
// so that the quadrature kernels make no calls (a call reserves the callee's
// registers and a stack frame in every kernel that contains it).
I2_HD __forceinline__ double log_rare(double x, const MathTable* __restrict__ tab) {
    const double t = log_tab_any(x * 0x1p54, tab) - 54.0 * 0.69314718055994530942;
    const double big = x + x;                                  // infinity or NaN
    return x > 0.0 ? (x <= 1.7976931348623157e308 ? t : big) : (x == 0.0 ? -HUGE_VAL : (x - x) / 0.0);
}

I2_HD __forceinline__ double log_tab(double x, const MathTable* __restrict__ tab) {
    if (!pos_normal(x)) return log_slow(x);
    return log_tab_any(x, tab);
}

// true where atan2_any is atan2: |x| + |y| in [2^-999, 2^999] (so neither
// argument is infinite or NaN and the quotient's reduction stays normal)
I2_HD __forceinline__ bool atan2_in_range(double y, double x) {
    const double sum = fabs(x) + fabs(y);
    return sum >= 0x1p-999 && sum <= 0x1p999;
}

// The table atan2 for any (y, x): atan2(y, x) where atan2_in_range(y, x),
// a meaningless value otherwise (the table index is clamped before its
// conversion, so that NaN and infinite quotients read entry 32).  Callers
// redo the other lanes with atan2_slow.
I2_HD __forceinline__ double atan2_any(double y, double x, const MathTable* __restrict__ tab) {
    const double ax = fabs(x), ay = fabs(y);
    const bool swap = ay > ax;
    const double n = fmin(ax, ay);
    const double d = fmax(ax, ay);                   // t = n/d in [0, 1], d >= 2^-1000
    // centre c = k/32 nearest to t, from the reciprocal estimate (relative error
    // far below 2^-10): k in [0, 32] and |t - c| <= 2^-6 (1 + 2^-10); 32 t + 1/2
    // lies in [1/2, 32.5] for in-range arguments, where the fmin changes no k
    const int k = (int)fmin(fma(n * rcp_estimate(d), 32.0, 0.5), 32.0);
    const double c = (double)k * (1.0 / 32.0);
    const double u = div_pos(fma(-c, d, n), fma(c, n, d));   // atan t = atan c + atan u
    const double w = u * u;
    // atan u = u - u^3/3 + u^5/5 - u^7/7 + u^9/9 (truncation below 2^-60 relative)
    double p = fma_k(w, 1.0 / 9.0, -1.0 / 7.0);
    p = fma_k(p, w, 1.0 / 5.0);
    p = fma_k(p, w, -1.0 / 3.0);
    const double au = fma(u * w, p, u);
    const AtanEntry b = tab->atan[k];
    double r = b.hi + (au + b.lo);                   // atan t, t in [0, 1]
    if (swap) r = PIO2_HI - r + PIO2_LO;             // atan(1/t) = pi/2 - atan t
    if (x < 0.0) r = PI_HI - r + PI_LO;              // second and third quadrants
    // r >= 0 here, and atan2 takes the sign of y (for y = -0 as well): one
    // bit operation instead of compares and a branch
    return copysign(r, y);
}

// atanh(z)/z for z^2 = s in [0, 1/16] (relative error below 2^-54.9) and
// atan(u)/u for u^2 = v in [0, 0.003] (below 2^-62): 1 + s q(s), q interpolating
// (f - 1)/s at the Chebyshev nodes of the interval (gen_math_tables.py).  DISTANT:
// the same on s in [0, 1/144] (below 2^-55.6) and v in [0, 3.7e-5] (below 2^-67)
template <bool DISTANT>
I2_HD __forceinline__ double atanh_over(double s) {
    if (DISTANT) {
        double q = fma_k(s, 0.09225773056807902, 0.11110289065026226);
        q = fma_k(q, s, 0.14285716327371326);
        q = fma_k(q, s, 0.19999999998226609);
        q = fma_k(q, s, 0.3333333333333358);
        return fma(q, s, 1.0);
    }
    double q = fma_k(s, 0.07395269887839463, 0.06506094123632396);
    q = fma_k(q, s, 0.07700982152842295);
    q = fma_k(q, s, 0.09090651861920544);
    q = fma_k(q, s, 0.11111115233521718);
    q = fma_k(q, s, 0.1428571425336631);
    q = fma_k(q, s, 0.2000000000009649);
    q = fma_k(q, s, 0.33333333333333287);
    return fma(q, s, 1.0);
}
template <bool DISTANT>
I2_HD __forceinline__ double atan_over(double v) {
    if (DISTANT) {
        const double q = fma_k(fma_k(v, -0.14285097640048655, 0.19999999991444123), v, -0.33333333333333315);
        return fma(q, v, 1.0);
    }
    double q = fma_k(v, -0.09033459667472876, 0.11110960509214748);
    q = fma_k(q, v, -0.14285714124452448);
    q = fma_k(q, v, 0.19999999999939544);
    q = fma_k(q, v, -0.3333333333333333);
    return fma(q, v, 1.0);
}

// cos(2 pi u) for u in [0, 1]: the nearest quarter turn exactly, then cos(2 pi r)
// = 1 + r^2 c(r^2) or sin(2 pi r) = r s(r^2) for |r| <= 1/8, c and s interpolants
// as above (relative error below 2^-55 and 2^-54.5)
I2_HD __forceinline__ double cos_turns(double u) {
    const double k = rint(4.0 * u);
    const double r = fma(k, -0.25, u), v = r * r;
    double c = fma_k(v, -1.6990343940660637, 7.903206911569678);
    c = fma_k(c, v, -26.426253275854723);
    c = fma_k(c, v, 60.24464135270201);
    c = fma_k(c, v, -85.4568172066438);
    c = fma_k(c, v, 64.93939402266824);
    c = fma_k(c, v, -19.739208802178716);
    c = fma(c, v, 1.0);
    double s = fma_k(v, 3.7808689593022957, -15.093804209987114);
    s = fma_k(s, v, 42.058685020160894);
    s = fma_k(s, v, -76.70585970427454);
    s = fma_k(s, v, 81.60524927594804);
    s = fma_k(s, v, -41.341702240399634);
    s = fma_k(s, v, 6.283185307179586);
    s *= -r;                                   // cos(pi/2 + x) = -sin x
    const int q = (int)k;
    const double t = (q & 1) ? s : c;
    return (q & 2) ? -t : t;
}

// atan2 outside atan2_in_range: (0, 0) by the signs, magnitudes near the ends
// of the exponent range scaled into the table path's, NaN for infinite and
// NaN arguments (no panel has them without NaN elsewhere)
I2_HD __forceinline__ double atan2_rare(double y, double x, const MathTable* __restrict__ tab) {
    const double sum = fabs(x) + fabs(y), k = sum < 1.0 ? 0x1p600 : 0x1p-600;
    double h = atan2_any(y * k, x * k, tab);
    if (sum == 0.0) h = copysign(copysign(1.0, x) < 0.0 ? PI_HI : 0.0, y);
    if (!(sum <= 1.7976931348623157e308)) h = sum - sum;
    return h;
}

I2_HD __forceinline__ double atan2_fast(double y, double x, const MathTable* __restrict__ tab) {
    // zero, tiny, huge, infinite and NaN arguments take the library path
    if (!atan2_in_range(y, x)) return atan2_slow(y, x);
    return atan2_any(y, x, tab);
}

}  // namespace i2m
