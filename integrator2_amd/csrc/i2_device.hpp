// i2_device.hpp -- gfx950 device math of the panel-pair integrator (FP64).
//
// Formulas follow andreyypopov/integrator2 src/evaluators/evaluatorJ3DK.cu
// (cited per function); the layout is MI355X-first: per-panel invariants
// (edge tangents, normal, area) live in a 192-byte Panel record built once
// per mesh, per-pair invariants of the singular parts are built once per task
// and kept in registers, and only the per-point work runs inside the
// quadrature loops.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <math.h>

// Device math is also compiled for the host so that the C ABI can expose
// host-side evaluations of the same formulas for checking.
#define I2_HD __host__ __device__
// Hot FP64 kernels: cap the unified VGPR+AGPR budget at 256 so that two
// wavefronts fit per SIMD; the quadrature loop's latency (LDS table loads,
// transcendental chains) needs the second wavefront to hide it.
#define I2_TWO_WAVES __attribute__((amdgpu_waves_per_eu(2)))
// The disjoint sweep fits three (168 registers, a few spills outside its
// quadrature loop): two measured the same time, four 15 % more (spills in it).
#define I2_THREE_WAVES __attribute__((amdgpu_waves_per_eu(3)))

#include "i2_math.hpp"

namespace i2d {

// ------------------------------------------------------------ constants
// src/common/constants.h:13-24
constexpr double DOUBLE_MIN = 2e-6;
constexpr double EPS_ZERO = 1e-6;
constexpr double EPS_ZERO2 = 1e-10;
constexpr double EPS_PSI_THETA2 = 1e-6 * 1e-6;
constexpr double PI = 3.14159265358979323846;
constexpr double TWO_PI = 6.28318530717958647692;
constexpr double RECIP_4PI = 0.079577471545947667884;
constexpr double LOG2 = 0.69314718055994530942;

constexpr int MAX_POINTS = 16;   // largest rule has 13 points

// Quadrature rule passed by value as a kernel argument (lands in SGPRs):
// barycentric (L1, L2, L3 = 1 - L1 - L2) and weights, per
// src/NumericalIntegrator3d.cu:197-216.
struct Rule {
    double L1[MAX_POINTS], L2[MAX_POINTS], L3[MAX_POINTS], w[MAX_POINTS];
    double reach;   // largest sum_k |L_k - 1/3| over the points outside the triangle, at least 1 (see panel_ball)
    double pow2p;   // 2^order, the Runge factor (src/evaluators/evaluator3d.cu:101-106)
    int n;
    int order;
    // Index of the rule's centroid point (L1 = L2 = 1/3 up to the literals'
    // rounding), or -1.  The centroid of a triangle is also the centroid of its
    // central level-1 child, so a pass over levels 0 and 1 evaluates it once.
    int centroid;
    int pad;        // zero: no padding bytes (rules are compared with memcmp)
};

// The centroid index of a rule with n points given as barycentric (L1, L2).
inline int rule_centroid(const double* L1, const double* L2, int n) {
    for (int k = 0; k < n; ++k)
        if (fabs(L1[k] - 1.0 / 3.0) <= 1e-14 && fabs(L2[k] - 1.0 / 3.0) <= 1e-14) return k;
    return -1;
}

// How far a rule's points reach from a triangle's centroid, relative to its
// vertices: 1 where every point lies in the triangle (|p - c| is convex), else
// the bound |p - c| <= sum_k |L_k - 1/3| |v_k - c|.  At least 1, so that the
// ball of a panel also holds the points of its sub-panels.
inline double rule_reach(const double* L1, const double* L2, const double* L3, int n) {
    double reach = 1.0;
    for (int k = 0; k < n; ++k) {
        const double s = fabs(L1[k] - 1.0 / 3.0) + fabs(L2[k] - 1.0 / 3.0) + fabs(L3[k] - 1.0 / 3.0);
        if (!(L1[k] >= 0.0 && L2[k] >= 0.0 && L3[k] >= 0.0)) reach = s > reach || s != s ? s : reach;
    }
    return reach;
}

// ------------------------------------------------------------ vectors
// Generic over the scalar so that the per-task geometry and closed forms can
// also run in forward-mode dual numbers (the adjoint); d3 and q4 are the FP64
// types of the forward kernels.  val() is the value used by branch tests.
I2_HD __forceinline__ double val(double x) { return x; }

template <class T> struct v3t { T x, y, z; };
using d3 = v3t<double>;
template <class T> I2_HD __forceinline__ v3t<T> operator+(v3t<T> a, v3t<T> b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
template <class T> I2_HD __forceinline__ v3t<T> operator-(v3t<T> a, v3t<T> b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
template <class T> I2_HD __forceinline__ v3t<T> operator-(v3t<T> a) { return {-a.x, -a.y, -a.z}; }
template <class S, class T> I2_HD __forceinline__ v3t<T> operator*(S s, v3t<T> a) { return {a.x * s, a.y * s, a.z * s}; }
template <class T> I2_HD __forceinline__ T dot(v3t<T> a, v3t<T> b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
template <class T> I2_HD __forceinline__ v3t<T> cross(v3t<T> a, v3t<T> b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
template <class T> I2_HD __forceinline__ T vlen(v3t<T> a) { return sqrt(dot(a, a)); }
template <class T> I2_HD __forceinline__ v3t<T> unit(v3t<T> a) { const T inv = T(1.0) / vlen(a); return {a.x * inv, a.y * inv, a.z * inv}; }
template <class T> I2_HD __forceinline__ v3t<T> divs(v3t<T> a, T s) { return {a.x / s, a.y / s, a.z / s}; }

// (Psi, Theta) accumulator
template <class T> struct q4t { T x, y, z, w; };
using q4 = q4t<double>;
I2_HD __forceinline__ q4 q4zero() { return {0.0, 0.0, 0.0, 0.0}; }
template <class T> I2_HD __forceinline__ q4t<T> operator+(q4t<T> a, q4t<T> b) { return {a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w}; }
template <class T> I2_HD __forceinline__ q4t<T> operator-(q4t<T> a, q4t<T> b) { return {a.x - b.x, a.y - b.y, a.z - b.z, a.w - b.w}; }
template <class S, class T> I2_HD __forceinline__ q4t<T> operator*(S s, q4t<T> a) { return {a.x * s, a.y * s, a.z * s, a.w * s}; }

// Per-panel record: vertices A, B, C (reference vertex order), the edge
// tangents of the inner integral (taua = (C-B)/|C-B|, taub = (A-C)/|A-C|,
// tauc = (B-A)/|B-A|, evaluatorJ3DK.cu:286-288), unit normal and area
// (src/Mesh3d.cu:23-32, 62-71) and the vertex indices.
struct alignas(16) Panel {
    d3 a, b, c;
    d3 ta, tb, tc;
    d3 n;
    double area;
    int v0, v1, v2, pad;
};
static_assert(sizeof(Panel) == 192, "Panel record is 192 bytes");

// ------------------------------------------------------------ helpers of cuda_math
// src/common/cuda_math.cuh:31-49
I2_HD __forceinline__ double sign_db(double x) {
    if (fabs(x) < DOUBLE_MIN) return 0.0;
    return (x > DOUBLE_MIN) ? 1.0 : -1.0;
}
I2_HD __forceinline__ double arg_db(double x) { return (x > DOUBLE_MIN) ? 0.0 : PI; }
// src/common/cuda_math.cu:14-27
template <class T> I2_HD __forceinline__ T angle(v3t<T> a, v3t<T> b) {
    const T den = sqrt(dot(a, a) * dot(b, b));
    if (val(den) < EPS_ZERO) return T(0.0);
    const T r = dot(a, b) / den;
    if (val(r) >= 1.0) return T(0.0);
    if (val(r) <= -1.0) return T(PI);
    return acos(r);
}

// ------------------------------------------------------------ inner integral
// evaluatorJ3DK.cu:266-313.  (Psi, Theta) of panel J at point p, with
// Theta n_J + Psi x n_J = integral over K_J of (p - r)/|p - r|^3.
I2_HD __forceinline__ q4 theta_psi(d3 p, const d3& A, const d3& B, const d3& C, const d3& ta, const d3& tb, const d3& tc) {
    d3 ova = p - A, ovb = p - B, ovc = p - C;
    const double lva = vlen(ova), lvb = vlen(ovb), lvc = vlen(ovc);
    ova = divs(ova, lva); ovb = divs(ovb, lvb); ovc = divs(ovc, lvc);
    const double rac = dot(ova, tc), rbc = dot(ovb, tc), rba = dot(ovb, ta),
                 rca = dot(ovc, ta), rcb = dot(ovc, tb), rab = dot(ova, tb);
    // the degenerate branches (point on an edge line) keep the ratio of distances
    const double n1 = (fabs(rbc + 1.0) < 0.5 * EPS_PSI_THETA2) ? lvb : lva * (1.0 + rac);
    const double d1 = (fabs(rbc + 1.0) < 0.5 * EPS_PSI_THETA2) ? lva : lvb * (1.0 + rbc);
    const double n2 = (fabs(rca + 1.0) < 0.5 * EPS_PSI_THETA2) ? lvc : lvb * (1.0 + rba);
    const double d2 = (fabs(rca + 1.0) < 0.5 * EPS_PSI_THETA2) ? lvb : lvc * (1.0 + rca);
    const double n3 = (fabs(rab + 1.0) < 0.5 * EPS_PSI_THETA2) ? lva : lvc * (1.0 + rcb);
    const double d3_ = (fabs(rab + 1.0) < 0.5 * EPS_PSI_THETA2) ? lvc : lva * (1.0 + rab);
    const double t1 = log(n1 / d1), t2 = log(n2 / d2), t3 = log(n3 / d3_);
    q4 r;
    r.x = t1 * tc.x + t2 * ta.x + t3 * tb.x;
    r.y = t1 * tc.y + t2 * ta.y + t3 * tb.y;
    r.z = t1 * tc.z + t2 * ta.z + t3 * tb.z;
    r.w = 2.0 * atan2(dot(cross(ova, ovb), ovc), 1.0 + dot(ova, ovb) + dot(ovb, ovc) + dot(ovc, ova));
    return r;
}

// The kernels' form of the inner integral.  Psi_j(p) is the sum over K_j's
// edges of tau_e times the line integral of 1/|p - r| along the edge, and with
// l the distances of p to the edge's ends, S their sum and L the edge length
// that integral is t = ln((S + L)/(S - L)) = 2 atanh(L/S): the reference's
// log of (l + d.tau) ratios, without dot products and without their
// cancellation near the edge's extension (S - L cancels near the edge itself
// only).  Theta = 2 atan2(y, x) with both arguments scaled by la lb lc > 0 (Van
// Oosterom and Strackee, IEEE Trans. Biomed. Eng. 30 (1983) 125-126): y =
// da.((B - A) x (C - A)), x = la lb lc + da.db lc + db.dc la + dc.da lb.  Away
// from the edges, P = S^2 - L^2 = 2 (la lb + da.db) gives 2 x = P_c lc + P_a la
// + P_b lb - 4 la lb lc, and every term comes from the three distances and
// per-panel constants.
//
// The tangents are constant over K_i, so the quadrature sums the three t and
// Theta/2 and multiplies by the tangents once per sum (psi_of_terms).
// K_j for the inner integral: vertices, edge tangents (as in the Panel
// record), edge lengths La = |C - B|, Lb = |A - C|, Lc = |B - A| and
// N2 = (B - A) x (C - A) (twice the area times the unit normal)
struct JGeom { d3 a, b, c, ta, tb, tc; double La, Lb, Lc; d3 N2; };
I2_HD __forceinline__ JGeom make_jgeom(d3 a, d3 b, d3 c, d3 ta, d3 tb, d3 tc) {
    // 0 * tau: a panel with a zero edge (NaN tangent) stays NaN in every term
    return {a, b, c, ta, tb, tc, vlen(c - b) + 0.0 * ta.x, vlen(a - c) + 0.0 * tb.x, vlen(b - a) + 0.0 * tc.x,
            cross(b - a, c - a)};
}
// e = S - L without cancellation, 2 |u x v|^2 / ((lu lv - u.v) n) with n = S +
// L, from (S - L)(S + L) = 2 (lu lv + u.v) and (lu lv + u.v)(lu lv - u.v) =
// |u x v|^2.  True in the reference's degenerate branch, a point on the edge's
// line, which takes lv/lu in place of n/e (evaluatorJ3DK.cu:294-307).
I2_HD __forceinline__ bool edge_gap(d3 u, d3 v, double lu, double lv, double L, double n, double& e) {
    const d3 c = cross(u, v);
    const double c2 = dot(c, c);
    e = 2.0 * c2 / (fma(lu, lv, -dot(u, v)) * n);
    return c2 < EPS_PSI_THETA2 * (L * L) * (lv * lv);
}
// atan2(y, x) for any arguments: the table path, then the lanes outside its range
I2_HD __forceinline__ double atan2_terms(double y, double x, const i2m::MathTable* __restrict__ lt) {
    double h = i2m::atan2_any(y, x, lt);
    if (__builtin_expect(!i2m::atan2_in_range(y, x), 0)) h = i2m::atan2_rare(y, x, lt);
    return h;
}
// Terms of one point: line integrals t along A->B, B->C, C->A (the edges of
// tau_c, tau_a, tau_b) and Theta/2.  For any point; `lt` holds the reduction
// tables of log and atan2.  One rare branch: an edge closer than about L/30
// (S - L below S/1024), and atan2 arguments outside the table path's range.
I2_HD __forceinline__ q4 theta_terms(d3 p, const JGeom& J, const i2m::MathTable* __restrict__ lt) {
    const d3 da = p - J.a, db = p - J.b, dc = p - J.c;
    const double la = i2m::sqrt_cubic(dot(da, da)), lb = i2m::sqrt_cubic(dot(db, db)), lc = i2m::sqrt_cubic(dot(dc, dc));
    const double S1 = la + lb, S2 = lb + lc, S3 = lc + la;
    double n1 = S1 + J.Lc, n2 = S2 + J.La, n3 = S3 + J.Lb;
    double e1 = S1 - J.Lc, e2 = S2 - J.La, e3 = S3 - J.Lb;
    const double s = 0x1p-10;
    if (__builtin_expect(fmin(fmin(fma(-s, S1, e1), fma(-s, S2, e2)), fma(-s, S3, e3)) < 0.0, 0)) {
        if (e1 < s * S1 && edge_gap(da, db, la, lb, J.Lc, n1, e1)) { n1 = lb; e1 = la; }
        if (e2 < s * S2 && edge_gap(db, dc, lb, lc, J.La, n2, e2)) { n2 = lc; e2 = lb; }
        if (e3 < s * S3 && edge_gap(dc, da, lc, la, J.Lb, n3, e3)) { n3 = la; e3 = lc; }
    }
    const double e12 = e1 * e2;
    const double inv = i2m::rcp_cubic(e12 * e3);
    const double i12 = inv * e3;
    // x from the dot products: beside an edge x and y both vanish, and P there
    // has the rounding of S^2, several times that of da.db
    const double y = dot(da, J.N2);
    const double x = la * lb * lc + dot(da, db) * lc + dot(db, dc) * la + dot(dc, da) * lb;
    // a ratio is positive and normal unless it is NaN, which the table path
    // keeps: no range test is needed
    const double t1 = i2m::log_tab_any(n1 * (i12 * e2), lt);
    const double t2 = i2m::log_tab_any(n2 * (i12 * e1), lt);
    const double t3 = i2m::log_tab_any(n3 * (inv * e12), lt);
    const double h = atan2_terms(y, x, lt);
    return {t1, t2, t3, h};
}
// The same for a point of a control panel K_i at least twice K_j's longest edge
// away from all of K_j (z = L/S <= 1/4 per edge; the solid angle is at most
// (sqrt 3/4)/4, so that |tan(Theta/2)| <= 0.0542): polynomials instead of
// tables, one reciprocal of S1 S2 S3 2x, no branch.  DISTANT: at least six
// longest edges (z <= 1/12, |tan(Theta/2)| <= 0.00602), with shorter
// polynomials.  The line integrals come without their factor 2 L (far_scale).
//
// The point is p = m + b0 U + b1 V, with m the centroid of K_i, U = A_i - C_i,
// V = B_i - C_i and (b0, b1) its first two barycentric coordinates less 1/3
// (FarFrame, FarPoint).  m itself, rounded, would shift all of the panel's points
// by some 2^-53 |m| together: with m = C_i + (U + V)/3 kept in two parts, m - a is
// (C_i - a) + (U + V)/3 and only differences of coordinates enter (pairs of a
// mesh 500 radii from the origin: median error 2.2e-14 instead of 8.3e-14).
//
// A squared distance to a vertex is then |m - a|^2 + 2 b0 U.(m - a) + 2 b1
// V.(m - a) + |b0 U + b1 V|^2: three instructions with the last term, common to
// all vertices, in `pp`; and da.N2 is affine in (b0, b1).  It loses no more than
// the plain difference because K_i's points lie nearer to m than to K_j
// (panel_far).  From S1 S2 S3 = la^2 (lb + lc) + lb^2 (lc + la) + lc^2 (la + lb) +
// 2 la lb lc, 2 x = S1 S2 S3 - (L_c^2 lc + L_a^2 la + L_b^2 lb).
//
// 94 FP64 instructions, DISTANT 83; from vertex differences and the three P it
// was 110, theta_terms takes 184, and the reference's formula as the kernels
// evaluated it before that (six dot products, table logs and atan2) 212.  Rows
// of 5,120 panels, where 81 % of the wavefronts are distant and 6 % general:
// 7.31 -> 6.77 ms.
struct FarFrame { d3 o, g, U, V; double uu, uv, vv; };   // m = o + g
I2_HD __forceinline__ FarFrame far_frame(d3 a, d3 b, d3 c) {
    const d3 U = a - c, V = b - c;
    return {c, (1.0 / 3.0) * (U + V), U, V, dot(U, U), 2.0 * dot(U, V), dot(V, V)};
}
// m - x
I2_HD __forceinline__ d3 from_vertex(const FarFrame& F, d3 x) { return (F.o - x) + F.g; }
// A quadrature point in that frame, with the products the kernels need of it
struct alignas(16) FarPoint { double b0, b1, b00, b01, b11, w; };
I2_HD __forceinline__ FarPoint far_point(double b0, double b1, double w) { return {b0, b1, b0 * b0, b0 * b1, b1 * b1, w}; }
I2_HD __forceinline__ double far_pp(const FarFrame& F, const FarPoint& Q) { return fma(Q.b11, F.vv, fma(Q.b01, F.uv, Q.b00 * F.uu)); }
// K_j in a control panel's frame: the vertices' distance polynomials, 2 da.N2
// and the squared edge lengths
struct FarGeom { double ka, ua, va, kb, ub, vb, kc, uc, vc, ky, uy, vy, q1, q2, q3; };
I2_HD __forceinline__ FarGeom far_geom(const FarFrame& F, const JGeom& J) {
    const d3 a = from_vertex(F, J.a), b = from_vertex(F, J.b), c = from_vertex(F, J.c), N = 2.0 * J.N2;
    return {dot(a, a), 2.0 * dot(F.U, a), 2.0 * dot(F.V, a), dot(b, b), 2.0 * dot(F.U, b), 2.0 * dot(F.V, b),
            dot(c, c), 2.0 * dot(F.U, c), 2.0 * dot(F.V, c), dot(a, N), dot(F.U, N), dot(F.V, N),
            J.Lc * J.Lc, J.La * J.La, J.Lb * J.Lb};
}
// from the three distances
template <bool DISTANT>
I2_HD __forceinline__ q4 theta_terms_of(double la, double lb, double lc, double b0, double b1, const FarGeom& G) {
    const double y = fma(b0, G.uy, fma(b1, G.vy, G.ky));           // 2 y
    const double S1 = la + lb, S2 = lb + lc, S3 = lc + la;
    const double s12 = S1 * S2, s123 = s12 * S3;
    const double x = fma(-G.q3, lb, fma(-G.q2, la, fma(-G.q1, lc, s123)));   // 2 x
    const double inv = i2m::rcp_cubic(s123 * x);
    const double i = inv * x, i3 = i * S3;
    const double r1 = i3 * S2, r2 = i3 * S1, r3 = i * s12, u = y * (inv * s123);
    return {r1 * i2m::atanh_over<DISTANT>(G.q1 * (r1 * r1)), r2 * i2m::atanh_over<DISTANT>(G.q2 * (r2 * r2)),
            r3 * i2m::atanh_over<DISTANT>(G.q3 * (r3 * r3)), u * i2m::atan_over<DISTANT>(u * u)};
}
// one vertex's distance polynomial
struct VertexPoly { double k, u, v; };
I2_HD __forceinline__ VertexPoly vertex_poly(const FarFrame& F, d3 x) {
    const d3 a = from_vertex(F, x);
    return {dot(a, a), 2.0 * dot(F.U, a), 2.0 * dot(F.V, a)};
}
I2_HD __forceinline__ double vertex_distance(const VertexPoly& x, double b0, double b1, double pp) {
    return i2m::sqrt_cubic(fma(b0, x.u, fma(b1, x.v, x.k + pp)));
}
template <bool DISTANT>
I2_HD __forceinline__ q4 theta_terms_far(double b0, double b1, double pp, const FarGeom& G) {
    return theta_terms_of<DISTANT>(vertex_distance({G.ka, G.ua, G.va}, b0, b1, pp), vertex_distance({G.kb, G.ub, G.vb}, b0, b1, pp),
                                   vertex_distance({G.kc, G.uc, G.vc}, b0, b1, pp), b0, b1, G);
}
// sums of theta_terms_far to sums of theta_terms
I2_HD __forceinline__ q4 far_scale(q4 T, const JGeom& J) { return {2.0 * J.Lc * T.x, 2.0 * J.La * T.y, 2.0 * J.Lb * T.z, T.w}; }
// (Psi, Theta) of a sum of terms
I2_HD __forceinline__ q4 psi_of_terms(q4 T, const JGeom& J) {
    return {T.x * J.tc.x + T.y * J.ta.x + T.z * J.tb.x, T.x * J.tc.y + T.y * J.ta.y + T.z * J.tb.y,
            T.x * J.tc.z + T.y * J.ta.z + T.z * J.tb.z, 2.0 * T.w};
}
I2_HD __forceinline__ q4 theta_psi_fast(d3 p, const JGeom& J, const i2m::MathTable* __restrict__ lt) {
    return psi_of_terms(theta_terms(p, J, lt), J);
}

// Bounding ball of a control panel's quadrature points on every refinement
// level: centroid, and the radius of its vertices times the rule's reach
struct Ball { d3 c; double r; };
I2_HD __forceinline__ Ball panel_ball(d3 a, d3 b, d3 c, double reach) {
    const d3 m = (1.0 / 3.0) * (a + b + c);
    const d3 u = a - m, v = b - m, w = c - m;
    return {m, reach * sqrt(fmax(fmax(dot(u, u), dot(v, v)), dot(w, w)))};
}
// How far K_j is from the control panel in ball B: 1 where theta_terms_far holds
// for every quadrature point, 2 where its DISTANT form does, else 0.  K_j lies
// within 2/3 of its longest edge M of its centroid (a vertex is 2/3 of a
// median away), so every distance to it is at least k M if the centroids are
// B.r + (k + 2/3) M apart, and at least 2 B.r if they are 3 B.r + 2/3 M apart
// (1 + 2^-20 covers the rounding of this test).  The scale test keeps
// S1 S2 S3 2x in range.  NaN panels are not far.
I2_HD __forceinline__ int panel_far(const Ball& B, const JGeom& J) {
    const d3 d = (1.0 / 3.0) * (J.a + J.b + J.c) - B.c;
    const double M = fmax(fmax(J.La, J.Lb), J.Lc), d2 = dot(d, d), far = 2.0 * fmax(M, B.r), distant = fmax(6.0 * M, 2.0 * B.r);
    const double base = fma(M, 2.0 / 3.0, B.r), n1 = (base + far) * (1.0 + 0x1p-20), n2 = (base + distant) * (1.0 + 0x1p-20);
    const bool scale = M >= 0x1p-150 && d2 <= 0x1p300;
    return !(scale && d2 >= n1 * n1) ? 0 : (d2 >= n2 * n2 ? 2 : 1);
}
// The form a wavefront takes for its pairs: the least that holds for all of
// them (0 general, 1 far, 2 distant).
__device__ __forceinline__ int wave_form(bool valid, const Ball& B, const JGeom& J) {
    const int f = valid ? panel_far(B, J) : 2;
    return __ballot(f == 0) != 0ull ? 0 : (__ballot(f == 1) != 0ull ? 1 : 2);
}

// ------------------------------------------------------------ singular parts
// Edge-sharing pair: vertices of K_j rotated so that JA is off the shared
// edge (evaluatorJ3DK.cu:797-847), plus the tangents and 1/|JC-JB| that
// evaluatorJ3DK.cu:338-343 recompute per point.
template <class T> struct EdgeCtxT { v3t<T> JB, JC, taua, taub, tauc; T ilvc; };
using EdgeCtx = EdgeCtxT<double>;
template <class T> I2_HD __forceinline__ EdgeCtxT<T> edge_ctx(v3t<T> JA, v3t<T> JB, v3t<T> JC) {
    EdgeCtxT<T> c;
    c.JB = JB; c.JC = JC;
    c.taua = unit(JA - JC);
    c.taub = unit(JB - JA);
    v3t<T> tc = JC - JB;
    c.ilvc = T(1.0) / vlen(tc);
    c.tauc = c.ilvc * tc;
    return c;
}
// evaluatorJ3DK.cu:315-350
I2_HD __forceinline__ q4 sing_edge(d3 p, const EdgeCtx& c) {
    d3 va = p - c.JB, vb = p - c.JC;
    const double lva = vlen(va), lvb = vlen(vb);
    va = divs(va, lva); vb = divs(vb, lvb);
    const double l1 = log((lvb * dot(c.tauc, c.tauc - vb)) / (lva * dot(c.tauc, c.tauc - va)));
    const double l2 = log(lva * dot(c.taub, c.taub + va) * c.ilvc);
    const double l3 = log(lvb * dot(c.taua, c.taua - vb) * c.ilvc);
    q4 r;
    r.x = l1 * c.tauc.x - l2 * c.taub.x - l3 * c.taua.x;
    r.y = l1 * c.tauc.y - l2 * c.taub.y - l3 * c.taua.y;
    r.z = l1 * c.tauc.z - l2 * c.taub.z - l3 * c.taua.z;
    r.w = 2.0 * (atan2(dot(cross(va, c.taub), c.tauc), dot(c.taub - c.tauc, c.taub + va)) -
                 atan2(dot(cross(vb, c.taua), c.tauc), dot(c.taua - c.tauc, c.taua - vb)));
    return r;
}

// l - t.v and l + t.v for a unit tangent t and l = |v|, recomputed as
// |v x t|^2 / (l -+ t.v) where they fall below 1e-4 l (cancellation near the
// line through the vertex along t).
I2_HD __forceinline__ double l_minus_tv(double l, d3 v, d3 t, double tv) {
    const d3 c = cross(v, t);
    return dot(c, c) / (l + tv);
}

// The singular parts below without unit vectors, as theta_psi_fast: with
// v = p - vertex and l = |v|, the reference's l (1 -+ t.(v/l)) is l -+ t.v
// (|t| = 1), recomputed without cancellation when small, and the arguments of
// each atan2 are both scaled by l > 0.  Logs and atan2 from i2_math.hpp.
I2_HD __forceinline__ q4 sing_edge_fast(d3 p, const EdgeCtx& c, const i2m::MathTable* __restrict__ lt) {
    const d3 va = p - c.JB, vb = p - c.JC;
    const double lva = i2m::sqrt_pos(dot(va, va)), lvb = i2m::sqrt_pos(dot(vb, vb));
    const double ca = dot(c.tauc, va), cb = dot(c.tauc, vb), ba = dot(c.taub, va), ab = dot(c.taua, vb);
    double N = lvb - cb, D = lva - ca, P2 = lva + ba, P3 = lvb - ab;
    const double s = 1e-4;
    if (__builtin_expect(fmin(fmin(N, P3) - s * lvb, fmin(D, P2) - s * lva) < 0.0, 0)) {
        if (N < s * lvb) N = l_minus_tv(lvb, vb, c.tauc, cb);
        if (D < s * lva) D = l_minus_tv(lva, va, c.tauc, ca);
        if (P2 < s * lva) P2 = l_minus_tv(lva, va, c.taub, -ba);
        if (P3 < s * lvb) P3 = l_minus_tv(lvb, vb, c.taua, ab);
    }
    const double a1 = N * i2m::rcp_pos(D), a2 = P2 * c.ilvc, a3 = P3 * c.ilvc;
    const double y1 = dot(cross(va, c.taub), c.tauc), x1 = dot(c.taub - c.tauc, lva * c.taub + va);
    const double y2 = dot(cross(vb, c.taua), c.tauc), x2 = dot(c.taua - c.tauc, lvb * c.taua - vb);
    // branch-free table paths, the rare lanes outside their ranges redone
    const bool o1 = i2m::pos_normal(a1), o2 = i2m::pos_normal(a2), o3 = i2m::pos_normal(a3);
    const bool o4 = i2m::atan2_in_range(y1, x1), o5 = i2m::atan2_in_range(y2, x2);
    double l1 = i2m::log_tab_any(a1, lt);
    double l2 = i2m::log_tab_any(a2, lt);
    double l3 = i2m::log_tab_any(a3, lt);
    double g1 = i2m::atan2_any(y1, x1, lt);
    double g2 = i2m::atan2_any(y2, x2, lt);
    if (__builtin_expect(!(o1 & o2 & o3 & o4 & o5), 0)) {
        if (!o1) l1 = i2m::log_rare(a1, lt);
        if (!o2) l2 = i2m::log_rare(a2, lt);
        if (!o3) l3 = i2m::log_rare(a3, lt);
        if (!o4) g1 = i2m::atan2_rare(y1, x1, lt);
        if (!o5) g2 = i2m::atan2_rare(y2, x2, lt);
    }
    q4 r;
    r.x = l1 * c.tauc.x - l2 * c.taub.x - l3 * c.taua.x;
    r.y = l1 * c.tauc.y - l2 * c.taub.y - l3 * c.taua.y;
    r.z = l1 * c.tauc.z - l2 * c.taub.z - l3 * c.taua.z;
    r.w = 2.0 * (g1 - g2);
    return r;
}

// Vertex-sharing pair: JA is the shared vertex; e and the two delta angles
// follow evaluatorJ3DK.cu:376-399 (two sign flips of e).
template <class T> struct VertexCtxT { v3t<T> JA, taua, taub, e; T invAri; };
using VertexCtx = VertexCtxT<double>;
template <class T>
I2_HD __forceinline__ v3t<T> vertex_e(v3t<T> nI, v3t<T> nJ, v3t<T> taua, v3t<T> taub, T* dA, T* dB) {
    v3t<T> e = cross(nI, nJ);
    if (val(dot(e, e)) < EPS_ZERO2) e = taub;
    else e = unit(e);
    T dx = atan2(dot(cross(taua, e), nJ), -dot(e, taua));
    T dy = atan2(dot(cross(e, taub), nJ), dot(e, taub));
    if ((PI - fabs(val(dx)) < EPS_ZERO) || (PI - fabs(val(dy)) < EPS_ZERO)) {
        e = -e;
        dx = atan2(dot(cross(taua, e), nJ), -dot(e, taua));
        dy = atan2(dot(cross(e, taub), nJ), dot(e, taub));
    }
    if ((val(dx) * val(dy) < 0) && (fabs(val(dx) - val(dy)) > PI)) {
        e = -e;
        dx = atan2(dot(cross(taua, e), nJ), -dot(e, taua));
        dy = atan2(dot(cross(e, taub), nJ), dot(e, taub));
    }
    *dA = dx; *dB = dy;
    return e;
}
template <class T>
I2_HD __forceinline__ VertexCtxT<T> vertex_ctx(v3t<T> JA, v3t<T> JB, v3t<T> JC, v3t<T> nI, v3t<T> nJ, T areaI) {
    VertexCtxT<T> c;
    c.JA = JA;
    c.taua = unit(JA - JC);
    c.taub = unit(JB - JA);
    T dA, dB;
    c.e = vertex_e(nI, nJ, c.taua, c.taub, &dA, &dB);
    c.invAri = T(1.0) / sqrt(areaI);   // rsqrt(measures[i]), evaluatorJ3DK.cu:401
    return c;
}
// evaluatorJ3DK.cu:352-407
I2_HD __forceinline__ q4 sing_vertex(d3 p, const VertexCtx& c) {
    d3 ovc = p - c.JA;
    const double lvc = vlen(ovc);
    ovc = divs(ovc, lvc);
    const double la = log((lvc * (1.0 + dot(c.taua, ovc))) * c.invAri);
    const double lb = log((lvc * (1.0 - dot(c.taub, ovc))) * c.invAri);
    q4 r;
    r.x = -(la * c.taua.x + lb * c.taub.x);
    r.y = -(la * c.taua.y + lb * c.taub.y);
    r.z = -(la * c.taua.z + lb * c.taub.z);
    r.w = 2.0 * (atan2(dot(cross(ovc, c.taua), c.e), dot(c.e - ovc, c.e - c.taua)) +
                 atan2(dot(cross(ovc, c.taub), c.e), dot(c.e - ovc, c.e + c.taub)));
    return r;
}

I2_HD __forceinline__ q4 sing_vertex_fast(d3 p, const VertexCtx& c, const i2m::MathTable* __restrict__ lt) {
    const d3 d = p - c.JA;
    const double l = i2m::sqrt_pos(dot(d, d));
    const double sa = dot(c.taua, d), sb = dot(c.taub, d);
    double na = l + sa, nb = l - sb;
    const double s = 1e-4;
    if (__builtin_expect(fmin(na, nb) < s * l, 0)) {
        if (na < s * l) na = l_minus_tv(l, d, c.taua, -sa);
        if (nb < s * l) nb = l_minus_tv(l, d, c.taub, sb);
    }
    const double a1 = na * c.invAri, a2 = nb * c.invAri;
    const d3 le = l * c.e;
    const double y1 = dot(cross(d, c.taua), c.e), x1 = dot(le - d, c.e - c.taua);
    const double y2 = dot(cross(d, c.taub), c.e), x2 = dot(le - d, c.e + c.taub);
    // branch-free table paths, the rare lanes outside their ranges redone
    const bool o1 = i2m::pos_normal(a1), o2 = i2m::pos_normal(a2);
    const bool o3 = i2m::atan2_in_range(y1, x1), o4 = i2m::atan2_in_range(y2, x2);
    double la = i2m::log_tab_any(a1, lt);
    double lb = i2m::log_tab_any(a2, lt);
    double g1 = i2m::atan2_any(y1, x1, lt);
    double g2 = i2m::atan2_any(y2, x2, lt);
    if (__builtin_expect(!(o1 & o2 & o3 & o4), 0)) {
        if (!o1) la = i2m::log_rare(a1, lt);
        if (!o2) lb = i2m::log_rare(a2, lt);
        if (!o3) g1 = i2m::atan2_rare(y1, x1, lt);
        if (!o4) g2 = i2m::atan2_rare(y2, x2, lt);
    }
    q4 r;
    r.x = -(la * c.taua.x + lb * c.taub.x);
    r.y = -(la * c.taua.y + lb * c.taub.y);
    r.z = -(la * c.taua.z + lb * c.taub.z);
    r.w = 2.0 * (g1 + g2);
    return r;
}

// ------------------------------------------------------------ topology of a pair
I2_HD __forceinline__ int vid(const Panel& P, int k) { return k == 0 ? P.v0 : (k == 1 ? P.v1 : P.v2); }
// a, b or c by a run-time index, as selects between values: passed by value,
// because a conditional between members of a record selects an address, and
// the whole record then lives in scratch memory
I2_HD __forceinline__ d3 pick(d3 a, d3 b, d3 c, int k) {
    return {k == 0 ? +a.x : (k == 1 ? +b.x : +c.x), k == 0 ? +a.y : (k == 1 ? +b.y : +c.y), k == 0 ? +a.z : (k == 1 ? +b.z : +c.z)};
}
I2_HD __forceinline__ d3 vtx(const Panel& P, int k) { return pick(P.a, P.b, P.c, k); }
// number of shared vertex indices (src/Mesh3d.cu:111-122)
I2_HD __forceinline__ int shared_count(const Panel& I, const Panel& J) {
    int c = 0;
    if (I.v0 == J.v0 || I.v0 == J.v1 || I.v0 == J.v2) ++c;
    if (I.v1 == J.v0 || I.v1 == J.v1 || I.v1 == J.v2) ++c;
    if (I.v2 == J.v0 || I.v2 == J.v1 || I.v2 == J.v2) ++c;
    return c;
}
// evaluatorJ3DK.cu:782-795: position of the shared vertex (last match wins)
I2_HD __forceinline__ void shifts_vertex(const Panel& I, const Panel& J, int* s1, int* s2) {
    int a = 0, b = 0;
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j)
            if (vid(I, i) == vid(J, j)) { a = i; b = j; }
    *s1 = a; *s2 = b;
}
// evaluatorJ3DK.cu:797-825: position of the vertex off the shared edge
I2_HD __forceinline__ void shifts_edge(const Panel& I, const Panel& J, int* s1, int* s2) {
    int mi = 0, mj = 0;   // bit masks of matched positions
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j)
            if (vid(I, i) == vid(J, j)) { mi |= 1 << i; mj |= 1 << j; }
    *s1 = (mi & 1) == 0 ? 0 : ((mi & 2) == 0 ? 1 : 2);
    *s2 = (mj & 1) == 0 ? 0 : ((mj & 2) == 0 ? 1 : 2);
}

// ------------------------------------------------------------ analytic singular integrals
// evaluatorJ3DK.cu:418-421
template <class T> I2_HD __forceinline__ T phi_f(T sA, T cA, T sG, T cG, T sXi, T cosLambda) {
    return 2.0 * atan2(sXi * sA * sG, 1.0 - cA + cG + cosLambda);
}
// evaluatorJ3DK.cu:438-461 -> (q_Theta, q_Psi)
template <class T>
I2_HD inline void q_theta_psi(T sA, T cA, T sB, T cB, T sG, T cG, T sNu, T cNu, T sXi, T cXi, T cosMu, T cosLambda, T* qT, T* qP) {
    const T phi1 = phi_f(sA, cA, sG, cG, sXi, cosLambda);
    const T phi2 = phi_f(sA, -cA, sG, -cG, sXi, cosLambda);
    const T iS = 1.0 / (sA * (1.0 - cosMu * cosMu));
    *qT = phi1 + sG * sNu * iS * ((cB * sG - cXi * sB * cG) * phi2 +
                                  sXi * sB * (0.5 * (1.0 + cosMu) * log((1.0 + cB) / (1.0 - cNu)) +
                                              0.5 * (1.0 - cosMu) * log((1.0 - cB) / (1.0 + cNu)) +
                                              log((1.0 + cosLambda) / (1.0 - cG))));
    *qP = 1.5 - iS * (sB * (cNu + cosMu * cosLambda) * log(1.0 + cosLambda) +
                      sNu * (cB + cosMu * cG) * log(1.0 - cG) +
                      sB * (1.0 - cosMu) * (cNu - cosLambda) * log(sB / sNu) +
                      sNu * sB * (sB * cG - cXi * sG * cB) * log((1.0 - cNu) / (1.0 + cB)) +
                      phi2 * sXi * sG * sNu * sB);
}
// evaluatorJ3DK.cu:474-481 (coplanar case; q_Theta takes its documented value 0)
template <class T> I2_HD inline void q_theta_psi_zero(T sB, T cB, T sNu, T cNu, T sinAlpha, T* qT, T* qP) {
    *qT = T(0.0);
    *qP = 1.5 - (cNu * sB * log(1.0 + cNu) + sNu * cB * log(1.0 - cB) + sinAlpha - sB + sNu + sB * cNu * log(sB / sNu)) / sinAlpha;
}

// evaluatorJ3DK.cu:603-672: closed-form integral over K_i of the edge-sharing singular part.
// (IA, IB, IC) and (JA, JB, JC) are rotated so that IA and JA are off the shared edge.
template <class T>
I2_HD inline q4t<T> integrate_sing_edge(v3t<T> IA, v3t<T> IB, v3t<T> IC, v3t<T> JA, v3t<T> JB, v3t<T> JC, v3t<T> nI,
                                        v3t<T> nJ, T areaI) {
    const v3t<T> taua = unit(JA - JC), taub = unit(JB - JA), tauc = unit(JC - JB);
    const T alpha = angle(IA - IC, IB - IC);
    const T beta = angle(IC - IB, IA - IB);
    const T gamma = angle(JC - JB, JA - JB);
    const T delta = angle(JB - JC, JA - JC);
    const T nu = PI - alpha - beta;
    const T xi = atan2(dot(cross(nI, nJ), tauc), dot(nI, nJ));
    T sA, cA, sB, cB, sG, cG, sD, cD, sX, cX;
    sincos(alpha, &sA, &cA); sincos(beta, &sB, &cB); sincos(gamma, &sG, &cG);
    sincos(delta, &sD, &cD); sincos(xi, &sX, &cX);
    const T sNu = sA * cB + cA * sB;
    const T cNu = sA * sB - cA * cB;
    const T cosSigma = -(cA * cD + cX * sA * sD);
    const T cosMu = -(cB * cG + cX * sB * sG);
    const T cosLambda = -(cA * cG - cX * sA * sG);
    const T cosTheta = -(cB * cD - cX * sB * sD);
    const T qab = sNu * log(tan(0.5 * alpha) * tan(0.5 * nu)) / sB +
                       sNu * log(tan(0.5 * beta) * tan(0.5 * nu)) / sA +
                       log(tan(0.5 * alpha) * tan(0.5 * beta));
    T qAT, qAP, qBT, qBP;
    if ((fabs(val(xi)) < EPS_ZERO) && (fabs(val(beta) - val(gamma)) < EPS_ZERO)) q_theta_psi_zero(sB, cB, sNu, cNu, sA, &qAT, &qAP);
    else q_theta_psi(sA, cA, sB, cB, sG, cG, sNu, cNu, sX, cX, cosMu, cosLambda, &qAT, &qAP);
    if ((fabs(val(xi)) < EPS_ZERO) && (fabs(val(alpha) - val(delta)) < EPS_ZERO)) q_theta_psi_zero(sA, cA, sNu, cNu, sB, &qBT, &qBP);
    else q_theta_psi(sB, cB, sA, cA, sD, cD, sNu, cNu, sX, cX, cosSigma, cosTheta, &qBT, &qBP);
    q4t<T> r;
    const v3t<T> v = areaI * (qAP * taub + qBP * taua - qab * tauc);
    r.x = v.x; r.y = v.y; r.z = v.z;
    r.w = areaI * (qAT + qBT);
    return r;
}

// evaluatorJ3DK.cu:511-601 -> (q^Theta, q^Psi) for vertex-sharing pairs
template <class T>
I2_HD inline void q_theta_psi_cont(T sXi, T cXi, T mu, T sMu, T cMu, T logSinMu, T logSinNu, T psi, T sPsi, T cPsi, T nu,
                                   T sNu, T cNu, T kappa, T sinKappa, T sinNuPsi, T sinMuPsi, T delta, T sD, T cD,
                                   T cosLambda, T cosTheta, T cosEta, T cosSigma, T cosChi, T* qT, T* qP) {
    const T logOneCosTheta = log(1.0 + cosTheta);
    const T logOneCosLambda = log(1.0 + cosLambda);
    const T Lambda1 = logOneCosLambda - logOneCosTheta + logSinNu - logSinMu;
    const T Lambda2 = log(tan(0.5 * nu) * tan(0.5 * mu));
    T s05D, c05D;
    sincos(0.5 * delta, &s05D, &c05D);
    const T tan05Delta = s05D / c05D;
    T sMP, cMP, sNP, cNP;
    sincos(0.5 * (mu - psi), &sMP, &cMP);
    sincos(0.5 * (nu + psi), &sNP, &cNP);
    const T Amu = atan2(tan05Delta * cMP * sXi, tan05Delta * cMP * cXi + sMP);
    const T Anu = atan2(tan05Delta * sNP * sXi, tan05Delta * sNP * cXi + cNP);
    T sT, cT, sT2, cT2;
    sincos(0.5 * (mu - psi) - 0.5 * (nu + psi), &sT, &cT);
    sincos(0.5 * kappa, &sT2, &cT2);
    const T W = atan2(sD * sT2 * sXi, cT2 + sD * cT * cXi + cD * sT);
    sincos(delta - psi, &sT, &cT);
    const T D = 1.0 / (sT * sT + sD * sPsi * (1.0 - cXi) * (cT + cosSigma));
    const T G = cPsi * (sD * cosSigma * cXi + cD * cosChi - sD * sD / sPsi);
    const T gent = 2.0 * (Anu * sMu * sinNuPsi - Amu * sNu * sinMuPsi -
                               D * sMu * sNu * sD * (W * cosEta + 0.5 * sPsi * sXi * (Lambda1 - Lambda2 * cosSigma))) /
                        (sPsi * sinKappa);
    const T gens = 0.5 * (3.0 - LOG2) +
                        (sMu * sNu / sinKappa) * ((logOneCosLambda - logOneCosTheta) * cPsi / sPsi +
                                                  D * (Lambda1 * sD * cosEta / sPsi + Lambda2 * cosChi -
                                                       2.0 * W * sD * sXi - G * (logSinNu - logSinMu))) -
                        (cMu * sNu * (logOneCosLambda - logSinMu) + sMu * cNu * (logOneCosTheta - logSinNu)) / sinKappa -
                        0.5 * (logSinMu + logSinNu - log(sinKappa));
    const double mulPsi = sign_db(val(sXi * sPsi));
    const double mulDelta = sign_db(val(sXi * sD));
    if ((fabs(val(sXi)) < EPS_ZERO) && (1.0 - fabs(val(cosSigma)) < 0.5 * EPS_ZERO2) && (fabs(val(sPsi)) > EPS_ZERO)) {
        const double ara = arg_db(val(sin(0.5 * (nu + psi)) * cosSigma));
        const double arb = arg_db(val(cos(0.5 * (mu - psi)) * cosSigma));
        *qT = 2.0 * mulPsi * cosSigma * cXi / (sinKappa * sPsi) * (sMu * sinNuPsi * ara - sNu * sinMuPsi * arb);
        *qP = 0.5 * (1.0 - LOG2) - 0.5 * log((1.0 - cosSigma * cMu) * (1.0 + cosSigma * cNu) / sinKappa) +
              cosSigma * (sMu - sNu + 0.5 * sin(mu - nu) * Lambda2) / sinKappa;
        return;
    }
    if ((fabs(val(sXi)) < EPS_ZERO) && (fabs(val(sPsi)) > EPS_ZERO)) {
        const double are = arg_db(val(sin(0.5 * (nu + mu)) + sin(0.5 * (mu - nu) - psi + delta * cXi)));
        const double arc = arg_db(val(1.0 / tan(0.5 * (nu + psi)) + tan(0.5 * delta) * cXi));
        const double ard = arg_db(val(tan(0.5 * (mu - psi)) + tan(0.5 * delta) * cXi));
        *qT = 2.0 * mulDelta * (sD * sMu * sNu / cosChi * cXi * are + sMu * sinNuPsi * arc - sNu * sinMuPsi * ard) / (sinKappa * sPsi);
        *qP = gens;
        return;
    }
    if (fabs(val(sin(psi))) < EPS_ZERO) {
        if (fabs(val(delta)) > EPS_ZERO) {
            *qT = 2.0 * (sMu * sNu * (W * cD * cXi - 0.5 * (Lambda1 - Lambda2 * cosSigma) * sXi) / sD +
                         (Anu + mulDelta * arg_db(val(sin(0.5 * (nu + psi))))) * sMu * cNu +
                         (Amu + mulDelta * arg_db(val(cos(0.5 * (mu - psi))))) * cMu * sNu) / sinKappa;
            *qP = 0.5 * (3.0 - LOG2) - 0.5 * (log((1.0 + cosLambda) * (1.0 + cosTheta) / sinKappa) - sin(mu - nu) / sinKappa * Lambda1) -
                  sMu * sNu * ((Lambda1 * cD - Lambda2 * cPsi) * cXi + 2.0 * W * sXi) / (sinKappa * sD);
        } else {
            *qT = T(2.0 * arg_db(val(cPsi)));
            *qP = 0.5 * (1.0 - LOG2) - 0.5 * log((1.0 - cPsi * cMu) * (1.0 + cPsi * cNu) / sinKappa) +
                  (0.5 * sin(mu - nu) * Lambda1 + cPsi * (sMu - sNu)) / sinKappa;
        }
        return;
    }
    *qT = gent;
    *qP = gens;
}

// evaluatorJ3DK.cu:674-780: closed-form integral over K_i of the vertex-sharing
// singular part.  IA and JA are the shared vertex.
template <class T>
I2_HD inline q4t<T> integrate_sing_vertex(v3t<T> IA, v3t<T> IB, v3t<T> IC, v3t<T> JA, v3t<T> JB, v3t<T> JC, v3t<T> nI,
                                          v3t<T> nJ, T areaI) {
    const v3t<T> taua = unit(JA - JC), taub = unit(JB - JA);
    T dA, dB;
    const v3t<T> e = vertex_e(nI, nJ, taua, taub, &dA, &dB);
    const T xi = atan2(dot(cross(nI, nJ), e), dot(nI, nJ));
    T sDA, cDA, sDB, cDB, sX, cX;
    sincos(dA, &sDA, &cDA); sincos(dB, &sDB, &cDB); sincos(xi, &sX, &cX);
    const v3t<T> s = IC - IB;
    const T nu = angle(IA - IB, IC - IB);
    const T mu = angle(IB - IC, IA - IC);
    const T kappa = angle(IB - IA, IC - IA);
    T sMu, cMu, sNu, cNu;
    sincos(mu, &sMu, &cMu); sincos(nu, &sNu, &cNu);
    const T logSinNu = log(sNu), logSinMu = log(sMu);
    const T sinKappa = sin(kappa);
    const T psi = atan2(dot(cross(e, s), nI), dot(e, s));
    T sPsi, cPsi, sNP, cNP, sMP, cMP;
    sincos(psi, &sPsi, &cPsi);
    sincos(nu + psi, &sNP, &cNP);
    sincos(mu - psi, &sMP, &cMP);
    T qAT, qAP, qBT, qBP;
    {
        const T cosSigma = sDA * sPsi * cX + cDA * cPsi;
        const T cosChi = sDA * cPsi * cX - cDA * sPsi;
        const T cosEta = cDA * sPsi * cX - sDA * cPsi;
        const T cosTheta = sDA * sNP * cX + cDA * cNP;
        const T cosLambda = sDA * sMP * cX - cDA * cMP;
        q_theta_psi_cont(sX, cX, mu, sMu, cMu, logSinMu, logSinNu, psi, sPsi, cPsi, nu, sNu, cNu, kappa, sinKappa,
                         sNP, sMP, dA, sDA, cDA, cosLambda, cosTheta, cosEta, cosSigma, cosChi, &qAT, &qAP);
    }
    {
        const T cosSigma = sDB * sPsi * cX + cDB * cPsi;
        const T cosChi = sDB * cPsi * cX - cDB * sPsi;
        const T cosEta = cDB * sPsi * cX - sDB * cPsi;
        const T cosTheta = sDB * sNP * cX + cDB * cNP;
        const T cosLambda = sDB * sMP * cX - cDB * cMP;
        q_theta_psi_cont(sX, cX, mu, sMu, cMu, logSinMu, logSinNu, psi, sPsi, cPsi, nu, sNu, cNu, kappa, sinKappa,
                         sNP, sMP, dB, sDB, cDB, cosLambda, cosTheta, cosEta, cosSigma, cosChi, &qBT, &qBP);
    }
    q4t<T> r;
    const v3t<T> v = areaI * (qAP * taua + qBP * taub);
    r.x = v.x; r.y = v.y; r.z = v.z;
    r.w = (fabs(val(xi)) < EPS_ZERO) ? T(0.0) : (areaI * (qAT - qBT));
    return r;
}

// ------------------------------------------------------------ finalize
// evaluatorJ3DK.cu:224-241 (vertex-sharing, with the 2*pi*p wrap of Theta)
// wrap count p of Theta' = Theta + 2 p (2 pi S_i) into [-2 pi S_i, 2 pi S_i]
I2_HD __forceinline__ int wrap_count(double theta, double areaI) {
    int p = 0;
    const double refTheta = TWO_PI * areaI;
    if (theta > refTheta) p = -((int)trunc((theta - refTheta) / (2.0 * refTheta)) + 1);
    else if (theta < -refTheta) p = ((int)trunc((-refTheta - theta) / (2.0 * refTheta)) + 1);
    return p;
}
template <class T> I2_HD __forceinline__ v3t<T> finalize_vertex_p(q4t<T> I, v3t<T> nJ, T areaI, int p) {
    const T refTheta = TWO_PI * areaI;
    const v3t<T> psi = {I.x, I.y, I.z};
    return RECIP_4PI * ((I.w + 2.0 * p * refTheta) * nJ + cross(psi, nJ));
}
I2_HD __forceinline__ d3 finalize_vertex(q4 I, d3 nJ, double areaI) {
    return finalize_vertex_p(I, nJ, areaI, wrap_count(I.w, areaI));
}
// evaluatorJ3DK.cu:254-264
template <class T> I2_HD __forceinline__ v3t<T> finalize_plain(q4t<T> I, v3t<T> nJ) {
    const v3t<T> psi = {I.x, I.y, I.z};
    return RECIP_4PI * (I.w * nJ + cross(psi, nJ));
}

// ------------------------------------------------------------ Runge rule
// src/common/cuda_math.cuh:270-300 and src/evaluators/evaluator3d.cu:83-92
I2_HD __forceinline__ double runge_criterion(q4 cur, q4 prev, double pow2p) {
    const q4 num = cur - prev;
    const q4 den = pow2p * prev - cur;
    const double x = (fabs(num.x) < DOUBLE_MIN && fabs(den.x) < DOUBLE_MIN) ? 0.0 : num.x / den.x;
    const double y = (fabs(num.y) < DOUBLE_MIN && fabs(den.y) < DOUBLE_MIN) ? 0.0 : num.y / den.y;
    const double z = (fabs(num.z) < DOUBLE_MIN && fabs(den.z) < DOUBLE_MIN) ? 0.0 : num.z / den.z;
    const double w = (fabs(num.w) < EPS_ZERO2 && fabs(den.w) < EPS_ZERO2) ? 0.0 : num.w / den.w;
    return fabs(x) + fabs(y) + fabs(z) + fabs(w);
}

// ------------------------------------------------------------ sub-panels
// A sub-panel of refinement level L is reached from the original panel by L
// midpoint splits (src/NumericalIntegrator3d.cu:54-72): children
// {m_AB, B, m_BC}, {m_BC, C, m_CA}, {m_CA, A, m_AB}, {m_BC, m_CA, m_AB}.
// `path` holds the child digits, most significant split first.
I2_HD __forceinline__ void sub_panel(d3& a, d3& b, d3& c, int level, uint32_t path) {
    for (int l = level - 1; l >= 0; --l) {
        const int ch = (path >> (2 * l)) & 3;
        const d3 mBC = 0.5 * (b + c), mCA = 0.5 * (c + a), mAB = 0.5 * (a + b);
        if (ch == 0) { a = mAB; c = mBC; }
        else if (ch == 1) { a = mBC; b = c; c = mCA; }
        else if (ch == 2) { b = a; a = mCA; c = mAB; }
        else { a = mBC; b = mCA; c = mAB; }
    }
}

// Barycentric coordinates on the original panel of the point with coordinates
// b on sub-panel `path`: the splits undone from the last to the first (child 0
// {m_AB, B, m_BC} takes (x, y, z) to (x/2, (1 + y)/2, z/2), and so on).
I2_HD __forceinline__ d3 sub_point(d3 b, int level, uint32_t path) {
    for (int l = 0; l < level; ++l, path >>= 2) {
        const int ch = path & 3;
        const double x = 0.5 * b.x, y = fma(0.5, b.y, 0.5), z = 0.5 * b.z;
        b.x = ch == 0 ? x : (ch == 1 ? z : (ch == 2 ? y : 0.5 - x));
        b.y = ch == 0 ? y : (ch == 1 ? x : (ch == 2 ? z : 1.0 - y));
        b.z = ch == 0 ? z : (ch == 1 ? y : (ch == 2 ? x : 0.5 - z));
    }
    return b;
}

// Point q of the n 4^level points of a rule on a panel's sub-panels, in order:
// the rule's point q - n s of sub-panel s = q / n.  The quotient by one
// multiplication with ceil(2^32 / n), exact for n <= 16 and q <= 2^28 (level
// 12).  For n = 1 that factor does not fit 32 bits; 0 stands for it, and s = q.
I2_HD __forceinline__ uint32_t split_factor(uint32_t n) { return n > 1 ? (uint32_t)((0x100000000ull + n - 1) / n) : 0u; }
I2_HD __forceinline__ uint32_t split_point(uint32_t q, uint32_t factor) {
    return factor != 0u ? (uint32_t)(((uint64_t)q * factor) >> 32) : q;
}

// A rule's point on a sub-panel, barycentric on the original panel, with its
// weight: 32-byte records that the kernels keep in LDS for levels 0 and 1
// (the rule's points on the panel, then on its four level-1 children).
struct alignas(32) BaryPoint { double b0, b1, b2, w; };
// vertices of level-1 child `ch` in those coordinates (sub_panel's children)
I2_HD __forceinline__ void child_bary(int ch, d3& ba, d3& bb, d3& bc) {
    const d3 A = {1.0, 0.0, 0.0}, B = {0.0, 1.0, 0.0}, C = {0.0, 0.0, 1.0};
    const d3 mAB = {0.5, 0.5, 0.0}, mBC = {0.0, 0.5, 0.5}, mCA = {0.5, 0.0, 0.5};
    if (ch == 0) { ba = mAB; bb = B; bc = mBC; }
    else if (ch == 1) { ba = mBC; bb = C; bc = mCA; }
    else if (ch == 2) { ba = mCA; bb = A; bc = mAB; }
    else { ba = mBC; bb = mCA; bc = mAB; }
}
// record t of the 5 npts of a rule given as barycentric arrays and weights
I2_HD __forceinline__ BaryPoint bary_point(const double* L1, const double* L2, const double* L3, const double* w, int npts, int t) {
    const int sub = t / npts, k = t - sub * npts;
    d3 ba = {1.0, 0.0, 0.0}, bb = {0.0, 1.0, 0.0}, bc = {0.0, 0.0, 1.0};
    if (sub > 0) child_bary(sub - 1, ba, bb, bc);
    d3 b = L1[k] * ba;
    b = b + L2[k] * bb;
    b = b + L3[k] * bc;
    return {b.x, b.y, b.z, w[k]};
}
I2_HD __forceinline__ d3 at_bary(const BaryPoint& Q, d3 a, d3 b, d3 c) {
    d3 p = Q.b0 * a;
    p = p + Q.b1 * b;
    return p + Q.b2 * c;
}

// A disjoint pair's far terms (without far_scale) summed with the weights over
// points k0, k0 + step, ... of the sub-panels sub, sub + G, ... of `level`, in
// barycentric coordinates of K_i less 1/3.  R: the rule's arrays, n points.
template <bool DISTANT, class R>
__device__ __forceinline__ q4 quad_far(const R& rule, int n, int level, int sub, int G, int k0, int step, const FarFrame& F,
                                       const FarGeom& J) {
    q4 acc = q4zero();
    const double h = 1.0 / 3.0;
    for (uint32_t c = sub; c < (1u << (2 * level)); c += G) {
        d3 a = {1.0 - h, -h, 0.0}, b = {-h, 1.0 - h, 0.0}, o = {-h, -h, 0.0};
        sub_panel(a, b, o, level, c);
        for (int k = k0; k < n; k += step) {
            const double l1 = rule.L1[k], l2 = rule.L2[k], l3 = rule.L3[k], w = rule.w[k];
            const FarPoint Q = far_point(l1 * a.x + l2 * b.x + l3 * o.x, l1 * a.y + l2 * b.y + l3 * o.y, w);
            const q4 t = theta_terms_far<DISTANT>(Q.b0, Q.b1, far_pp(F, Q), J);
            acc = {fma(w, t.x, acc.x), fma(w, t.y, acc.y), fma(w, t.z, acc.z), fma(w, t.w, acc.w)};
        }
    }
    return acc;
}

}  // namespace i2d
