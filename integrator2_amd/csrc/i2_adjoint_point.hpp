// i2_adjoint_point.hpp -- reverse mode of the per-point functions of the
// quadrature loops, derived by hand: the inner integral thetaPsi
// (theta_terms_rev and theta_terms_far_rev in the kernels; theta_psi_fast_rev,
// with the tangents as free parameters, which no kernel runs, for the host) and the two singular parts (evaluatorJ3DK.cu:315-350, 352-407).
//
// Each function recomputes the forward intermediates of one point, returns the
// forward value f, and adds gb . df/dx to the cotangents of the point p and of
// the function's parameters (triangle vertices and tangents, or the singular
// context).  Parameters are treated as free variables; the per-task chain from
// the parameters to the vertex coordinates is applied once per task.
#pragma once
#include "i2_device.hpp"

namespace i2d {

I2_HD __forceinline__ void axpy(d3& y, double a, d3 x) { y.x += a * x.x; y.y += a * x.y; y.z += a * x.z; }

I2_HD __forceinline__ double l_plus_dtau(double l, d3 d, d3 t) {
    const d3 c = cross(d, t);
    return dot(c, c) / (l - dot(d, t));
}
// Rare branch of the six l + d.tau terms: terms below 1e-4 l recomputed
// without cancellation, then the reference's degenerate branch (a point on an
// edge line of K_j keeps the ratio of distances, evaluatorJ3DK.cu:294-307).
I2_HD __forceinline__ void fix_terms(const JGeom& J, d3 da, d3 db, d3 dc, double la, double lb, double lc,
                                     double& n1, double& e1, double& n2, double& e2, double& n3, double& e3,
                                     bool& f1, bool& f2, bool& f3) {
    const double s = 1e-4;
    if (n1 < s * la) n1 = l_plus_dtau(la, da, J.tc);
    if (e1 < s * lb) e1 = l_plus_dtau(lb, db, J.tc);
    if (n2 < s * lb) n2 = l_plus_dtau(lb, db, J.ta);
    if (e2 < s * lc) e2 = l_plus_dtau(lc, dc, J.ta);
    if (n3 < s * lc) n3 = l_plus_dtau(lc, dc, J.tb);
    if (e3 < s * la) e3 = l_plus_dtau(la, da, J.tb);
    const double h = 0.5 * EPS_PSI_THETA2;
    f1 = fabs(e1) < h * lb; f2 = fabs(e2) < h * lc; f3 = fabs(e3) < h * la;
    if (f1) { n1 = lb; e1 = la; }
    if (f2) { n2 = lc; e2 = lb; }
    if (f3) { n3 = la; e3 = lc; }
}
// one test per distance for the rare branch (the per-term tests are repeated
// inside it rather than kept live through the common path)
I2_HD __forceinline__ bool terms_need_fix(double la, double lb, double lc, double n1, double e1, double n2, double e2,
                                          double n3, double e3) {
    const double s = 1e-4;
    return fmin(fmin(fmin(n1, e3) - s * la, fmin(e1, n2) - s * lb), fmin(e2, n3) - s * lc) < 0.0;
}
// cotangents of the parameters of thetaPsi over K_j: vertices and edge tangents
struct TPBar { d3 a, b, c, ta, tb, tc; };

I2_HD __forceinline__ q4 theta_psi_fast_rev(d3 p, const JGeom& J, const i2m::MathTable* __restrict__ lt, q4 gb, d3* pbar,
                                            TPBar& g) {
    // ---- forward, from the l + d.tau of the reference formula
    const d3 da = p - J.a, db = p - J.b, dc = p - J.c;
    const double qa = dot(da, da), qb = dot(db, db), qc = dot(dc, dc);
    const double la = i2m::sqrt_pos(qa), lb = i2m::sqrt_pos(qb), lc = i2m::sqrt_pos(qc);
    const double s1 = dot(da, J.tc), s2 = dot(db, J.ta), s3 = dot(dc, J.tb);
    double n1 = la + s1, e1 = lb + dot(db, J.tc);
    double n2 = lb + s2, e2 = lc + dot(dc, J.ta);
    double n3 = lc + s3, e3 = la + dot(da, J.tb);
    bool f1 = false, f2 = false, f3 = false;
    if (__builtin_expect(terms_need_fix(la, lb, lc, n1, e1, n2, e2, n3, e3), 0))
        fix_terms(J, da, db, dc, la, lb, lc, n1, e1, n2, e2, n3, e3, f1, f2, f3);
    const double e12 = e1 * e2;
    const double inv = i2m::rcp_pos(e12 * e3);
    const double a1 = n1 * (e2 * e3) * inv, a2 = n2 * (e1 * e3) * inv, a3 = n3 * e12 * inv;
    // the solid angle from da, db, dc directly: with the tangents and vertices
    // as free parameters of this function, x and y then depend on da, db, dc only
    const double pab = dot(da, db), pbc = dot(db, dc), pca = dot(dc, da);
    const double y = dot(cross(da, db), dc);
    const double x = la * lb * lc + pab * lc + pbc * la + pca * lb;
    // branch-free table paths, the rare lanes outside their ranges redone
    const bool o1 = i2m::pos_normal(a1), o2 = i2m::pos_normal(a2), o3 = i2m::pos_normal(a3);
    const bool o4 = i2m::atan2_in_range(y, x);
    double t1 = i2m::log_tab_any(a1, lt);
    double t2 = i2m::log_tab_any(a2, lt);
    double t3 = i2m::log_tab_any(a3, lt);
    double th = i2m::atan2_any(y, x, lt);
    if (__builtin_expect(!(o1 & o2 & o3 & o4), 0)) {
        if (!o1) t1 = i2m::log_rare(a1, lt);
        if (!o2) t2 = i2m::log_rare(a2, lt);
        if (!o3) t3 = i2m::log_rare(a3, lt);
        if (!o4) th = i2m::atan2_rare(y, x, lt);
    }
    q4 r;
    r.x = t1 * J.tc.x + t2 * J.ta.x + t3 * J.tb.x;
    r.y = t1 * J.tc.y + t2 * J.ta.y + t3 * J.tb.y;
    r.z = t1 * J.tc.z + t2 * J.ta.z + t3 * J.tb.z;
    r.w = 2.0 * th;
    // ---- reverse
    const d3 gP = {gb.x, gb.y, gb.z};
    const double tb1 = dot(gP, J.tc), tb2 = dot(gP, J.ta), tb3 = dot(gP, J.tb);
    axpy(g.tc, t1, gP); axpy(g.ta, t2, gP); axpy(g.tb, t3, gP);
    // t_k = log n_k - log e_k: reciprocals from two refined reciprocals
    const double invn = i2m::rcp_pos(n1 * n2 * n3);
    const double rn1 = n2 * n3 * invn, rn2 = n1 * n3 * invn, rn3 = n1 * n2 * invn;
    const double re1 = e2 * e3 * inv, re2 = e1 * e3 * inv, re3 = e12 * inv;
    const double nb1 = tb1 * rn1, eb1 = -tb1 * re1;
    const double nb2 = tb2 * rn2, eb2 = -tb2 * re2;
    const double nb3 = tb3 * rn3, eb3 = -tb3 * re3;
    double lab = 0.0, lbb = 0.0, lcb = 0.0;
    d3 dab = {0.0, 0.0, 0.0}, dbb = dab, dcb = dab;
    if (!f1) { lab += nb1; axpy(dab, nb1, J.tc); axpy(g.tc, nb1, da); lbb += eb1; axpy(dbb, eb1, J.tc); axpy(g.tc, eb1, db); }
    else { lbb += nb1; lab += eb1; }
    if (!f2) { lbb += nb2; axpy(dbb, nb2, J.ta); axpy(g.ta, nb2, db); lcb += eb2; axpy(dcb, eb2, J.ta); axpy(g.ta, eb2, dc); }
    else { lcb += nb2; lbb += eb2; }
    if (!f3) { lcb += nb3; axpy(dcb, nb3, J.tb); axpy(g.tb, nb3, dc); lab += eb3; axpy(dab, eb3, J.tb); axpy(g.tb, eb3, da); }
    else { lab += nb3; lcb += eb3; }
    // Theta = 2 atan2(y, x)
    // (the derivative of y = da.(db x dc) in da, db, dc: the cross products)
    const double r2 = i2m::rcp_pos(x * x + y * y);
    const double yb = 2.0 * gb.w * x * r2, xb = -2.0 * gb.w * y * r2;
    axpy(dab, yb, cross(db, dc)); axpy(dbb, yb, cross(dc, da)); axpy(dcb, yb, cross(da, db));
    lab += xb * (lb * lc + pbc);
    lbb += xb * (la * lc + pca);
    lcb += xb * (la * lb + pab);
    axpy(dab, xb * lc, db); axpy(dab, xb * lb, dc);
    axpy(dbb, xb * lc, da); axpy(dbb, xb * la, dc);
    axpy(dcb, xb * la, db); axpy(dcb, xb * lb, da);
    // l = |d|
    const double il = i2m::rcp_pos(la * lb * lc);
    axpy(dab, lab * (lb * lc * il), da);
    axpy(dbb, lbb * (la * lc * il), db);
    axpy(dcb, lcb * (la * lb * il), dc);
    *pbar = dab + dbb + dcb;
    g.a = g.a - dab; g.b = g.b - dbb; g.c = g.c - dcb;
    return r;
}

// Reverse mode of the terms of the inner integral (theta_terms): with P = (S -
// L)(S + L) per edge,
//   t = ln((S + L)/(S - L)):  dt = (2 S dL - 2 L dS)/P,
//   Theta/2 = h = atan2(Y, X), X = 2 x = P_c lc + P_a la + P_b lb - 4 la lb lc
//   and Y = 2 da.N2:  X^2 + Y^2 = P_c P_a P_b (for unit vectors |1 + a.b + b.c +
//   c.a|^2 + (a.(b x c))^2 = 2 (1 + a.b)(1 + b.c)(1 + c.a)),
// so one reciprocal of the three P serves every derivative.  Parameters are
// the distances through p and the vertices, the edge lengths and N2.
//
// Cotangents summed over a pair's points.  a, b, c: sums of (dL/dl)/l d per
// vertex, whose negatives belong to the vertices; y: sum of 2 dL/dY, times N2
// another share of vertex a; n: dL/dN2; Lc, La, Lb: half of dL/dL; T: the
// weighted terms themselves.
struct TermsBar { d3 a, b, c, n; double y, Lc, La, Lb; q4 T; };
I2_HD __forceinline__ TermsBar terms_bar_zero() {
    const d3 z = {0.0, 0.0, 0.0};
    return {z, z, z, z, 0.0, 0.0, 0.0, 0.0, q4zero()};
}
// One point of weight w, with the cotangents ct of the weighted terms; returns
// the point's cotangent.
I2_HD __forceinline__ d3 theta_terms_rev(d3 p, const JGeom& J, const i2m::MathTable* __restrict__ lt, double w, const q4& ct,
                                         TermsBar& g) {
    const d3 da = p - J.a, db = p - J.b, dc = p - J.c;
    double ila, ilb, ilc;
    const double la = i2m::sqrt_rsqrt(dot(da, da), &ila), lb = i2m::sqrt_rsqrt(dot(db, db), &ilb),
                 lc = i2m::sqrt_rsqrt(dot(dc, dc), &ilc);
    const double S1 = la + lb, S2 = lb + lc, S3 = lc + la;
    const double c1 = w * ct.x, c2 = w * ct.y, c3 = w * ct.z, ch = w * ct.w;
    const double Y = 2.0 * dot(da, J.N2);
    double xa = 0.0, xb = 0.0, xc = 0.0;           // dL/dl of terms in the degenerate branch
    double m1 = c1, m2 = c2, m3 = c3;
    const double n1 = S1 + J.Lc, n2 = S2 + J.La, n3 = S3 + J.Lb;
    double e1 = S1 - J.Lc, e2 = S2 - J.La, e3 = S3 - J.Lb;
    double r1 = 0.0, r2 = 0.0, r3 = 0.0;            // ratios of terms in the degenerate branch
    const double s = 0x1p-10;
    if (__builtin_expect(fmin(fmin(fma(-s, S1, e1), fma(-s, S2, e2)), fma(-s, S3, e3)) < 0.0, 0)) {
        if (e1 < s * S1) {
            if (edge_gap(da, db, la, lb, J.Lc, n1, e1)) { r1 = lb / la; xb += c1 / lb; xa -= c1 / la; m1 = 0.0; }
        }
        if (e2 < s * S2) {
            if (edge_gap(db, dc, lb, lc, J.La, n2, e2)) { r2 = lc / lb; xc += c2 / lc; xb -= c2 / lb; m2 = 0.0; }
        }
        if (e3 < s * S3) {
            if (edge_gap(dc, da, lc, la, J.Lb, n3, e3)) { r3 = la / lc; xa += c3 / la; xc -= c3 / lc; m3 = 0.0; }
        }
    }
    const double P1 = n1 * e1, P2 = n2 * e2, P3 = n3 * e3;
    const double P12 = P1 * P2;
    const double R = i2m::rcp_cubic(P12 * P3);
    const double R3 = R * P3;
    const double iP1 = R3 * P2, iP2 = R3 * P1, iP3 = R * P12;
    const double a1 = r1 != 0.0 ? r1 : n1 * n1 * iP1, a2 = r2 != 0.0 ? r2 : n2 * n2 * iP2, a3 = r3 != 0.0 ? r3 : n3 * n3 * iP3;
    const double X = 2.0 * (la * lb * lc + dot(da, db) * lc + dot(db, dc) * la + dot(dc, da) * lb);
    const double t1 = i2m::log_tab_any(a1, lt), t2 = i2m::log_tab_any(a2, lt), t3 = i2m::log_tab_any(a3, lt);
    const double h = atan2_terms(Y, X, lt);
    g.T = {fma(w, t1, g.T.x), fma(w, t2, g.T.y), fma(w, t3, g.T.z), fma(w, h, g.T.w)};
    // ---- reverse; dX/dl_a = P_a + 2 l_a (l_b + l_c)
    m1 *= iP1; m2 *= iP2; m3 *= iP3;
    const double Rh = R * ch;
    const double xb_ = -(Y * Rh), yb = 2.0 * (X * Rh);          // dL/dX and 2 dL/dY
    g.Lc = fma(S1, m1, fma(-J.Lc, xb_ * lc, g.Lc));
    g.La = fma(S2, m2, fma(-J.La, xb_ * la, g.La));
    g.Lb = fma(S3, m3, fma(-J.Lb, xb_ * lb, g.Lb));
    const double E1 = 2.0 * J.Lc * m1, E2 = 2.0 * J.La * m2, E3 = 2.0 * J.Lb * m3;
    const double sa = (fma(xb_, fma(la + la, S2, P2), xa) - (E1 + E3)) * ila,
                 sb = (fma(xb_, fma(lb + lb, S3, P3), xb) - (E1 + E2)) * ilb,
                 sc = (fma(xb_, fma(lc + lc, S1, P1), xc) - (E2 + E3)) * ilc;
    axpy(g.a, sa, da); axpy(g.b, sb, db); axpy(g.c, sc, dc);
    axpy(g.n, yb, da);
    g.y += yb;
    d3 pb = yb * J.N2;
    axpy(pb, sa, da); axpy(pb, sb, db); axpy(pb, sc, dc);
    return pb;
}
// The same for theta_terms_far.  With da = (m - a) + b0 U + b1 V every vector
// sum over the points follows from sums of scalars: of sa = (dL/dl_a)/l_a, sb,
// sc and y = 2 dL/dY, alone and times b0 and b1, and of s = sa + sb + sc times
// b0^2, b0 b1 and b1^2.  Twenty-two sums and no vector per point: 156 FP64
// instructions (DISTANT; 170 at 2 longest edges), where summing the vectors
// took 217 and theta_terms_rev takes 310.
struct FarBar { double a, b, c, y, a0, b0, c0, y0, a1, b1, c1, y1, s00, s01, s11, Lc, La, Lb; q4 T; };
I2_HD __forceinline__ FarBar far_bar_zero() {
    return {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, q4zero()};
}
template <bool DISTANT>
I2_HD __forceinline__ void theta_terms_far_rev(const FarPoint& Q, const FarFrame& F, const FarGeom& G, const JGeom& J, const q4& ct,
                                               FarBar& g) {
    const double pp = far_pp(F, Q);
    double ila, ilb, ilc;
    const double la = i2m::sqrt_rsqrt(fma(Q.b0, G.ua, fma(Q.b1, G.va, G.ka + pp)), &ila),
                 lb = i2m::sqrt_rsqrt(fma(Q.b0, G.ub, fma(Q.b1, G.vb, G.kb + pp)), &ilb),
                 lc = i2m::sqrt_rsqrt(fma(Q.b0, G.uc, fma(Q.b1, G.vc, G.kc + pp)), &ilc);
    const double Y = fma(Q.b0, G.uy, fma(Q.b1, G.vy, G.ky));
    const double S1 = la + lb, S2 = lb + lc, S3 = lc + la;
    const double s12 = S1 * S2, s123 = s12 * S3;
    const double X = fma(-G.q3, lb, fma(-G.q2, la, fma(-G.q1, lc, s123)));
    const double inv = i2m::rcp_cubic(s123 * X);
    const double i = inv * X, iX = inv * s123, i3 = i * S3;
    const double r1 = i3 * S2, r2 = i3 * S1, r3 = i * s12, u = Y * iX, v = u * u;
    const double w = Q.w;
    g.T = {fma(w, r1 * i2m::atanh_over<DISTANT>(G.q1 * (r1 * r1)), g.T.x), fma(w, r2 * i2m::atanh_over<DISTANT>(G.q2 * (r2 * r2)), g.T.y),
           fma(w, r3 * i2m::atanh_over<DISTANT>(G.q3 * (r3 * r3)), g.T.z), fma(w, u * i2m::atan_over<DISTANT>(v), g.T.w)};
    // ---- reverse
    const double P1 = fma(S1, S1, -G.q1), P2 = fma(S2, S2, -G.q2), P3 = fma(S3, S3, -G.q3), P12 = P1 * P2;
    // 1/(P1 P2 P3) = 1/(X^2 + Y^2) = (1/X)^2/(1 + v), v <= 3.7e-5 where DISTANT
    const double R = DISTANT ? (iX * iX) * fma(fma(1.0 - v, v, -1.0), v, 1.0) : i2m::rcp_cubic(P12 * P3);
    const double R3 = R * P3;
    const double m1 = (w * ct.x) * (R3 * P2), m2 = (w * ct.y) * (R3 * P1), m3 = (w * ct.z) * (R * P12);
    const double Rh = R * (w * ct.w);
    const double xb = -(Y * Rh), yb = 2.0 * (X * Rh);           // dL/dX and 2 dL/dY
    g.Lc = fma(S1, m1, fma(-J.Lc, xb * lc, g.Lc));
    g.La = fma(S2, m2, fma(-J.La, xb * la, g.La));
    g.Lb = fma(S3, m3, fma(-J.Lb, xb * lb, g.Lb));
    const double E1 = 2.0 * J.Lc * m1, E2 = 2.0 * J.La * m2, E3 = 2.0 * J.Lb * m3;
    const double sa = fma(xb, fma(la + la, S2, P2), -(E1 + E3)) * ila, sb = fma(xb, fma(lb + lb, S3, P3), -(E1 + E2)) * ilb,
                 sc = fma(xb, fma(lc + lc, S1, P1), -(E2 + E3)) * ilc;
    g.a += sa; g.b += sb; g.c += sc; g.y += yb;
    g.a0 = fma(Q.b0, sa, g.a0); g.b0 = fma(Q.b0, sb, g.b0); g.c0 = fma(Q.b0, sc, g.c0); g.y0 = fma(Q.b0, yb, g.y0);
    g.a1 = fma(Q.b1, sa, g.a1); g.b1 = fma(Q.b1, sb, g.b1); g.c1 = fma(Q.b1, sc, g.c1); g.y1 = fma(Q.b1, yb, g.y1);
    const double t = sa + sb + sc;
    g.s00 = fma(Q.b00, t, g.s00); g.s01 = fma(Q.b01, t, g.s01); g.s11 = fma(Q.b11, t, g.s11);
}
// The vector sums: g as theta_terms_rev leaves it, and added to X0 and X1 the
// points' cotangents times their first two barycentric coordinates.
I2_HD __forceinline__ void far_bar_expand(const FarBar& f, const FarFrame& F, const JGeom& J, TermsBar& g, d3& X0, d3& X1) {
    const d3 a = from_vertex(F, J.a), b = from_vertex(F, J.b), c = from_vertex(F, J.c);
    g.a = f.a * a; axpy(g.a, f.a0, F.U); axpy(g.a, f.a1, F.V);
    g.b = f.b * b; axpy(g.b, f.b0, F.U); axpy(g.b, f.b1, F.V);
    g.c = f.c * c; axpy(g.c, f.c0, F.U); axpy(g.c, f.c1, F.V);
    g.n = f.y * a; axpy(g.n, f.y0, F.U); axpy(g.n, f.y1, F.V);
    g.y = f.y; g.Lc = f.Lc; g.La = f.La; g.Lb = f.Lb;
    g.T = far_scale(f.T, J);
    d3 Xs = g.a + g.b + g.c;
    axpy(Xs, f.y, J.N2);
    auto along = [&](d3& X, double sa, double sb, double sc, double sy, double su, double sv) {
        axpy(X, 1.0 / 3.0, Xs);
        axpy(X, sy, J.N2); axpy(X, sa, a); axpy(X, sb, b); axpy(X, sc, c); axpy(X, su, F.U); axpy(X, sv, F.V);
    };
    along(X0, f.a0, f.b0, f.c0, f.y0, f.s00, f.s01);
    along(X1, f.a1, f.b1, f.c1, f.y1, f.s01, f.s11);
}
// Cotangents of K_j's vertices from a pair's sums: ct as in theta_terms_rev,
// nb the cotangent of the unit normal and gP that of the quadrature sum of
// Psi = T.x tau_c + T.y tau_a + T.z tau_b (ct.x = gP.tau_c, ...).
I2_HD __forceinline__ void terms_chain(const JGeom& J, const q4& ct, const TermsBar& g, d3 gP, d3 nb, double iLa, double iLb,
                                       double iLc, double iN, d3 n, d3& Ab, d3& Bb, d3& Cb) {
    Ab = -g.a; Bb = -g.b; Cb = -g.c;
    axpy(Ab, -g.y, J.N2);
    // an edge e = L tau: dL/de = (T gP - (T gP.tau) tau)/L + dL/dL tau
    auto edge = [&](double T, double c, double Lh, double iL, d3 tau) {
        const double k = T * iL;
        d3 e = k * gP;
        axpy(e, fma(2.0, Lh, -(k * c)), tau);
        return e;
    };
    const d3 ec = edge(g.T.x, ct.x, g.Lc, iLc, J.tc), ea = edge(g.T.y, ct.y, g.La, iLa, J.ta),
             eb = edge(g.T.z, ct.z, g.Lb, iLb, J.tb);
    Bb = Bb + ec - ea; Ab = Ab - ec + eb; Cb = Cb + ea - eb;
    // N2 = (B - A) x (C - A), n = N2/|N2|
    d3 N = iN * nb;
    axpy(N, -dot(N, n), n);
    N = N + g.n;
    const d3 gu = cross(J.c - J.a, N), gv = cross(N, J.b - J.a);
    Bb = Bb + gu; Cb = Cb + gv; Ab = Ab - gu - gv;
}

// d(u / |u|) backwards: cotangent of u from that of the unit vector
I2_HD __forceinline__ d3 unit_rev(d3 u, d3 ub) {
    const double l = sqrt(dot(u, u));
    const d3 t = (1.0 / l) * u;
    return (1.0 / l) * (ub - dot(ub, t) * t);
}

// cotangents of the edge-sharing context
// (ilvc, and VertexBar's invAri: times that constant, d/d log)
struct EdgeBar { d3 JB, JC, taua, taub, tauc; double ilvc; };

// log and atan2 from the tables; reciprocals of quantities that are not small
// differences by rcp_pos.  The unit vectors and the differences 1 -+ t.(v/l)
// keep sing_edge's and sing_vertex's operations: their rounding is what these
// derivatives amplify.
I2_HD __forceinline__ double log_terms(double x, const i2m::MathTable* __restrict__ lt) {
    double t = i2m::log_tab_any(x, lt);
    if (__builtin_expect(!i2m::pos_normal(x), 0)) t = i2m::log_rare(x, lt);
    return t;
}
I2_HD __forceinline__ q4 sing_edge_rev(d3 p, const EdgeCtx& c, const i2m::MathTable* __restrict__ lt, q4 gb, d3* pbar, EdgeBar& g) {
    // ---- forward, as sing_edge
    const d3 pa = p - c.JB, pb = p - c.JC;
    const double lva = vlen(pa), lvb = vlen(pb);
    const d3 va = divs(pa, lva), vb = divs(pb, lvb);
    const double P1 = dot(c.tauc, c.tauc - vb), Q1 = dot(c.tauc, c.tauc - va);
    const double P2 = dot(c.taub, c.taub + va), P3 = dot(c.taua, c.taua - vb);
    const double l1 = log_terms((lvb * P1) / (lva * Q1), lt);
    const double l2 = log_terms(lva * P2 * c.ilvc, lt);
    const double l3 = log_terms(lvb * P3 * c.ilvc, lt);
    q4 r;
    r.x = l1 * c.tauc.x - l2 * c.taub.x - l3 * c.taua.x;
    r.y = l1 * c.tauc.y - l2 * c.taub.y - l3 * c.taua.y;
    r.z = l1 * c.tauc.z - l2 * c.taub.z - l3 * c.taua.z;
    const double y1 = dot(cross(va, c.taub), c.tauc), x1 = dot(c.taub - c.tauc, c.taub + va);
    const double y2 = dot(cross(vb, c.taua), c.tauc), x2 = dot(c.taua - c.tauc, c.taua - vb);
    r.w = 2.0 * (atan2_terms(y1, x1, lt) - atan2_terms(y2, x2, lt));
    // ---- reverse
    const double ila = i2m::rcp_pos(lva), ilb = i2m::rcp_pos(lvb);
    const d3 gP = {gb.x, gb.y, gb.z};
    const double l1b = dot(gP, c.tauc), l2b = -dot(gP, c.taub), l3b = -dot(gP, c.taua);
    axpy(g.tauc, l1, gP); axpy(g.taub, -l2, gP); axpy(g.taua, -l3, gP);
    const double lvab = (l2b - l1b) * ila, lvbb = (l1b + l3b) * ilb;
    const double P1b = l1b / P1, Q1b = -l1b / Q1, P2b = l2b / P2, P3b = l3b / P3;
    g.ilvc += l2b + l3b;
    d3 vab = {0.0, 0.0, 0.0}, vbb = vab;
    axpy(g.tauc, P1b, 2.0 * c.tauc - vb); axpy(vbb, -P1b, c.tauc);
    axpy(g.tauc, Q1b, 2.0 * c.tauc - va); axpy(vab, -Q1b, c.tauc);
    axpy(g.taub, P2b, 2.0 * c.taub + va); axpy(vab, P2b, c.taub);
    axpy(g.taua, P3b, 2.0 * c.taua - vb); axpy(vbb, -P3b, c.taua);
    const double th1b = 2.0 * gb.w, th2b = -2.0 * gb.w;
    const double q1 = i2m::rcp_pos(x1 * x1 + y1 * y1), q2 = i2m::rcp_pos(x2 * x2 + y2 * y2);
    const double y1b = th1b * x1 * q1, x1b = -th1b * y1 * q1;
    const double y2b = th2b * x2 * q2, x2b = -th2b * y2 * q2;
    axpy(vab, y1b, cross(c.taub, c.tauc)); axpy(g.taub, y1b, cross(c.tauc, va)); axpy(g.tauc, y1b, cross(va, c.taub));
    axpy(g.taub, x1b, (c.taub + va) + (c.taub - c.tauc)); axpy(g.tauc, -x1b, c.taub + va); axpy(vab, x1b, c.taub - c.tauc);
    axpy(vbb, y2b, cross(c.taua, c.tauc)); axpy(g.taua, y2b, cross(c.tauc, vb)); axpy(g.tauc, y2b, cross(vb, c.taua));
    axpy(g.taua, x2b, (c.taua - vb) + (c.taua - c.tauc)); axpy(g.tauc, -x2b, c.taua - vb); axpy(vbb, -x2b, c.taua - c.tauc);
    // va = pa / |pa|, vb = pb / |pb|
    d3 pab = ila * (vab - dot(vab, va) * va);
    d3 pbb = ilb * (vbb - dot(vbb, vb) * vb);
    axpy(pab, lvab, va);
    axpy(pbb, lvbb, vb);
    *pbar = pab + pbb;
    g.JB = g.JB - pab;
    g.JC = g.JC - pbb;
    return r;
}

// cotangents of the vertex-sharing context
struct VertexBar { d3 JA, taua, taub, e; double invAri; };

I2_HD __forceinline__ q4 sing_vertex_rev(d3 p, const VertexCtx& c, const i2m::MathTable* __restrict__ lt, q4 gb, d3* pbar, VertexBar& g) {
    // ---- forward, as sing_vertex
    const d3 pc = p - c.JA;
    const double lvc = vlen(pc);
    const d3 o = divs(pc, lvc);
    const double A1 = 1.0 + dot(c.taua, o), B1 = 1.0 - dot(c.taub, o);
    const double la = log_terms((lvc * A1) * c.invAri, lt);
    const double lb = log_terms((lvc * B1) * c.invAri, lt);
    q4 r;
    r.x = -(la * c.taua.x + lb * c.taub.x);
    r.y = -(la * c.taua.y + lb * c.taub.y);
    r.z = -(la * c.taua.z + lb * c.taub.z);
    const double y1 = dot(cross(o, c.taua), c.e), x1 = dot(c.e - o, c.e - c.taua);
    const double y2 = dot(cross(o, c.taub), c.e), x2 = dot(c.e - o, c.e + c.taub);
    r.w = 2.0 * (atan2_terms(y1, x1, lt) + atan2_terms(y2, x2, lt));
    // ---- reverse
    const double ilc = i2m::rcp_pos(lvc);
    const d3 gP = {gb.x, gb.y, gb.z};
    const double lab = -dot(gP, c.taua), lbb = -dot(gP, c.taub);
    axpy(g.taua, -la, gP); axpy(g.taub, -lb, gP);
    const double lvcb = (lab + lbb) * ilc;
    g.invAri += lab + lbb;
    const double A1b = lab / A1, B1b = lbb / B1;
    d3 ob = {0.0, 0.0, 0.0};
    axpy(g.taua, A1b, o); axpy(ob, A1b, c.taua);
    axpy(g.taub, -B1b, o); axpy(ob, -B1b, c.taub);
    const double thb = 2.0 * gb.w;
    const double q1 = i2m::rcp_pos(x1 * x1 + y1 * y1), q2 = i2m::rcp_pos(x2 * x2 + y2 * y2);
    const double y1b = thb * x1 * q1, x1b = -thb * y1 * q1;
    const double y2b = thb * x2 * q2, x2b = -thb * y2 * q2;
    axpy(ob, y1b, cross(c.taua, c.e)); axpy(g.taua, y1b, cross(c.e, o)); axpy(g.e, y1b, cross(o, c.taua));
    axpy(g.e, x1b, (c.e - c.taua) + (c.e - o)); axpy(ob, -x1b, c.e - c.taua); axpy(g.taua, -x1b, c.e - o);
    axpy(ob, y2b, cross(c.taub, c.e)); axpy(g.taub, y2b, cross(c.e, o)); axpy(g.e, y2b, cross(o, c.taub));
    axpy(g.e, x2b, (c.e + c.taub) + (c.e - o)); axpy(ob, -x2b, c.e + c.taub); axpy(g.taub, x2b, c.e - o);
    d3 pcb = ilc * (ob - dot(ob, o) * o);
    axpy(pcb, lvcb, o);
    *pbar = pcb;
    g.JA = g.JA - pcb;
    return r;
}

}  // namespace i2d
