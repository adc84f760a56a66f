// i2_adjoint.hip -- hand-written adjoint: dL/d(vertex coordinates) of the
// scalar loss
//
//   L = sum over all ordered pairs (i, j) of  w_ij Theta_ij + v_ij . J_ij
//
// with Theta_ij the Theta channel of the pair's reported integrals, J_ij its
// result, and w_ij ~ N(0,1), v_ij ~ N(0,1)^3 drawn counter-based from (seed,
// pair id i*nT + j), so that no weight is stored.  The refinement tree of
// every pair (its reported level, from the forward pass's convergence
// iteration and K), the 2 pi p wrap of vertex-sharing pairs and every branch
// of the formulas are those of the forward pass (piecewise-constant choices
// are not differentiated).  Nothing of the forward pass is stored beyond the
// per-pair convergence iteration: every quadrature point is recomputed.
//
//   k_adj_disjoint  disjoint pairs.  An item is a wavefront of 64 control
//                   panels i (one per lane) and a tile of panels j that it
//                   walks in step, so K_j is uniform: the cotangents of K_i
//                   stay in registers for the whole tile and those of K_j are
//                   summed over the wavefront into the slot of (wavefront, j).
//                   Pairs at reported level >= 2 are marked per lane.
//   k_adj_deep      the marked pairs, from a list, 16 or 64 lanes each over
//                   their 13 * 4^L points, to a record per pair.
//   k_adj_deep_sum  those records, added to their item's slots in a fixed order.
//   k_adj_singular  vertex- and edge-sharing pairs: 16 lanes per pair, or a
//                   wavefront per pair above reported level 2; reverse mode
//                   over the points; the cotangents of the per-pair quantities
//                   go to a record per pair.
//   k_adj_singular_dual  the per-pair chain of every record: forward-mode
//                   dual numbers along the 18 vertex coordinates of the pair
//                   (one per lane, 3.5 pairs per wavefront) through the
//                   per-pair geometry, singular-part contexts and the
//                   closed-form singular integrals, one slot per coordinate.
//   k_adj_panel_sum, k_adj_gather, k_adj_loss_part, k_adj_loss  dL/dX per
//                   vertex coordinate and L per mesh, summed from the slots in
//                   a fixed order.
//
// No sum depends on the order in which workgroups finish: every partial has a
// slot of its own and the gathers add the slots in an order fixed by the mesh
// alone, so two runs give the same bits (the reference's gathers are FP64
// atomics, src/NumericalIntegrator3d.cu:168-171).
#include "i2_adjoint.hpp"
#include "i2_adjoint_point.hpp"
#include "i2_dual.hpp"

#include <algorithm>
#include <cstring>

namespace i2 {
using namespace i2d;

// ------------------------------------------------------------ loss weights
I2_HD __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
// N(0,1) by Box-Muller from two 53-bit uniforms in (0, 1) of the splitmix64
// hash of (seed, pair id, stream); streams 0 (w) and 1..3 (v).  Table log and
// polynomial cosine: four draws of the libraries' functions were an eighth of
// k_adj_disjoint's instructions.  The bound keeps the root's estimate finite where u1
// rounds to 1.
I2_HD __forceinline__ double normal_draw(uint64_t seed, uint64_t pid, uint64_t stream, const i2m::MathTable* __restrict__ lt) {
    const uint64_t base = mix64(seed ^ mix64(pid * 4ull + stream));
    const double u1 = ((double)(mix64(base ^ 0x1ull) >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    const double u2 = ((double)(mix64(base ^ 0x2ull) >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    return i2m::sqrt_pos(fmax(-2.0 * i2m::log_tab_any(u1, lt), 0x1p-900)) * i2m::cos_turns(u2);
}

struct Weights { double w; d3 v; };
__device__ __forceinline__ Weights weights(uint64_t seed, int i, int j, int nT, const i2m::MathTable* __restrict__ lt) {
    const uint64_t pid = (uint64_t)i * (uint64_t)nT + (uint64_t)j;
    return {normal_draw(seed, pid, 0, lt), {normal_draw(seed, pid, 1, lt), normal_draw(seed, pid, 2, lt), normal_draw(seed, pid, 3, lt)}};
}
// cotangent of a pair's (Psi, Theta): dL/dPsi = n_j x v / (4 pi), dL/dTheta = w + v . n_j / (4 pi)
__device__ __forceinline__ q4 task_cotangent(const Weights& W, d3 nJ) {
    const d3 a = RECIP_4PI * cross(nJ, W.v);
    return {a.x, a.y, a.z, W.w + RECIP_4PI * dot(W.v, nJ)};
}

// ------------------------------------------------------------ helpers
__device__ __forceinline__ int64_t uniform64a(int64_t x) {
    const int lo = __builtin_amdgcn_readfirstlane((int)(x & 0xffffffff));
    const int hi = __builtin_amdgcn_readfirstlane((int)(x >> 32));
    return ((int64_t)hi << 32) | (uint32_t)lo;
}
__device__ __forceinline__ int find_base_a(const int64_t* base, int n, int64_t x) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (base[mid] <= x) lo = mid; else hi = mid - 1;
    }
    return lo;
}
__device__ __forceinline__ int64_t rank_disjoint(const AdjMesh& M, int i, int j) {
    int64_t below = 0;
    for (int64_t q = M.nbr_start[i]; q < M.nbr_start[i + 1]; ++q) {
        if (M.nbr[q] < j) ++below; else break;
    }
    return M.row_start[i] + (j - i - 1) - below;
}
__device__ __forceinline__ int64_t task_disjoint(const AdjMesh& M, int i, int j) {
    return (i < j) ? rank_disjoint(M, i, j) : M.npairs[I2_NOT_NEIGHBORS] + rank_disjoint(M, j, i);
}
__device__ __forceinline__ int reported_level(const AdjArgs& A, int c, int K) {
    if (A.fixed) return A.last_level;
    if (A.quirk && c >= 1 && ((K - c) & 1)) return c - 1;
    return c;
}
// A wavefront-uniform double or panel, moved to scalar registers
__device__ __forceinline__ double uniform_d(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffll));
    const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ d3 uniform_d3(d3 v) { return {uniform_d(v.x), uniform_d(v.y), uniform_d(v.z)}; }
__device__ __forceinline__ Panel uniform_panel(const Panel& P) {
    Panel U;
    U.a = uniform_d3(P.a); U.b = uniform_d3(P.b); U.c = uniform_d3(P.c);
    U.ta = uniform_d3(P.ta); U.tb = uniform_d3(P.tb); U.tc = uniform_d3(P.tc);
    U.n = uniform_d3(P.n); U.area = uniform_d(P.area);
    U.v0 = __builtin_amdgcn_readfirstlane(P.v0); U.v1 = __builtin_amdgcn_readfirstlane(P.v1);
    U.v2 = __builtin_amdgcn_readfirstlane(P.v2); U.pad = 0;
    return U;
}
__device__ __forceinline__ JGeom uniform_jgeom(const JGeom& J) {
    return {J.a, J.b, J.c, J.ta, J.tb, J.tc, uniform_d(J.La), uniform_d(J.Lb), uniform_d(J.Lc), uniform_d3(J.N2)};
}
// v, of which the compiler doesn't know that it is v
__device__ __forceinline__ d3 opaque(d3 v) {
    asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z));
    return v;
}
__device__ __forceinline__ double wsum(double x) {
    for (int m = 1; m < 64; m <<= 1) x += __shfl_xor(x, m);
    return x;
}
__device__ __forceinline__ void store3(double* dst, d3 v) { dst[0] = v.x; dst[1] = v.y; dst[2] = v.z; }
__device__ __forceinline__ void add_to3(double* dst, d3 v) { dst[0] += v.x; dst[1] += v.y; dst[2] += v.z; }
__device__ __forceinline__ double dot4(q4 a, q4 b) { return a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w; }

struct RuleSh {
    double L1[MAX_POINTS], L2[MAX_POINTS], L3[MAX_POINTS], w[MAX_POINTS];
    i2m::MathTable lt;
};
__device__ __forceinline__ void load_rule_sh(RuleSh& s, const Rule& R) {
    for (int k = threadIdx.x; k < MAX_POINTS; k += blockDim.x) {
        s.L1[k] = R.L1[k]; s.L2[k] = R.L2[k]; s.L3[k] = R.L3[k]; s.w[k] = R.w[k];
    }
    i2m::fill_mathtab(s.lt);
}

// Vertex cotangents of a panel from those of its tangents and normal
// (ta = unit(C - B), tb = unit(A - C), tc = unit(B - A), n = unit((B - A) x (C - A)))
// and of its area (S = |(B - A) x (C - A)| / 2).
__device__ __forceinline__ void panel_chain(const Panel& P, d3 tab, d3 tbb, d3 tcb, d3 nb, double Sb, d3& Ab, d3& Bb, d3& Cb) {
    const d3 ua = unit_rev(P.c - P.b, tab);
    Cb = Cb + ua; Bb = Bb - ua;
    const d3 ub = unit_rev(P.a - P.c, tbb);
    Ab = Ab + ub; Cb = Cb - ub;
    const d3 uc = unit_rev(P.b - P.a, tcb);
    Bb = Bb + uc; Ab = Ab - uc;
    const d3 u = P.b - P.a, v = P.c - P.a;
    const d3 cr = cross(u, v);
    d3 crb = unit_rev(cr, nb);
    axpy(crb, 0.5 * Sb, P.n);
    const d3 gu = cross(v, crb), gv = cross(crb, u);
    Bb = Bb + gu; Cb = Cb + gv; Ab = Ab - gu - gv;
}

__device__ __forceinline__ void load_bary(BaryPoint* P, FarPoint* F, const RuleSh& R, int npts) {
    for (int t = threadIdx.x; t < 5 * npts; t += blockDim.x) {
        const BaryPoint Q = bary_point(R.L1, R.L2, R.L3, R.w, npts, t);
        P[t] = Q;
        F[t] = far_point(Q.b0 - 1.0 / 3.0, Q.b1 - 1.0 / 3.0, Q.w);
    }
}

// Sums of nine values over the wavefront, in a fixed order: pairs of registers
// exchange halves and then rows, so that one register ends with four values'
// sums, one per row of 16 lanes, and each row is summed by rotations.  57
// instructions and no LDS instead of nine six-step butterflies through LDS.
__device__ __forceinline__ double swap_add(double a, double b, bool half) {
    const uint64_t x = __double_as_longlong(a), y = __double_as_longlong(b);
    uint64_t p, q;
    if (half) {
        const auto l = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
        p = ((uint64_t)h[0] << 32) | l[0]; q = ((uint64_t)h[1] << 32) | l[1];
    } else {
        const auto l = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
        p = ((uint64_t)h[0] << 32) | l[0]; q = ((uint64_t)h[1] << 32) | l[1];
    }
    return __longlong_as_double((long long)p) + __longlong_as_double((long long)q);
}
template <int N> __device__ __forceinline__ double ror_add(double v) {
    const uint64_t x = __double_as_longlong(v);
    const unsigned l = __builtin_amdgcn_mov_dpp((int)(unsigned)x, 0x120 + N, 0xf, 0xf, false);
    const unsigned h = __builtin_amdgcn_mov_dpp((int)(unsigned)(x >> 32), 0x120 + N, 0xf, 0xf, false);
    return v + __longlong_as_double((long long)(((uint64_t)h << 32) | l));
}
__device__ __forceinline__ double row_sum16(double v) { return ror_add<1>(ror_add<2>(ror_add<4>(ror_add<8>(v)))); }
// four sums in one register: row 0 a, row 1 b, row 2 c, row 3 d
__device__ __forceinline__ double sum_rows4(double a, double b, double c, double d) {
    return row_sum16(swap_add(swap_add(a, c, true), swap_add(b, d, true), false));
}
__device__ __forceinline__ double sum_all(double v) { return row_sum16(swap_add(swap_add(v, v, true), swap_add(v, v, true), false)); }
// the nine cotangents of K_j's vertices, summed over the wavefront into its slot
__device__ __forceinline__ void store_sum9(double* slot, int lane, d3 a, d3 b, d3 c) {
    const double s0 = sum_rows4(a.x, a.y, a.z, b.x), s1 = sum_rows4(b.y, b.z, c.x, c.y), s2 = sum_all(c.z);
    const int row = lane >> 4;
    if ((lane & 15) == 0) { slot[row] = s0; slot[4 + row] = s1; }
    if (lane == 0) slot[8] = s2;
}

// ------------------------------------------------------------ disjoint sweep
constexpr int ADJ_BLOCK = 256;
// panels j per disjoint item at most (one bit of a lane's mask each)
constexpr int ADJ_TILE = 32;

// Reverse mode over the points k0 <= k < k1 of one pair: the general form, and
// the far one's scalar sums.
__device__ __forceinline__ void points_rev(const RuleSh& R, const BaryPoint* pts, int k0, int k1, const Panel& I, const JGeom& JG,
                                           const q4& ct, TermsBar& g, d3& X0, d3& X1) {
    for (int k = k0; k < k1; ++k) {
        const BaryPoint Q = pts[k];
        const d3 p = at_bary(Q, I.a, I.b, I.c);
        const d3 pb = theta_terms_rev(p, JG, &R.lt, Q.w, ct, g);
        axpy(X0, Q.b0, pb); axpy(X1, Q.b1, pb);
    }
}
template <bool DISTANT>
__device__ __forceinline__ void points_far_rev(const FarPoint* pts, int npts, bool act0, bool act1, const FarFrame& F,
                                               const FarGeom& G, const JGeom& JG, const q4& ct, FarBar& f) {
    // the pairs at reported level 0, then those at level 1
    if (act0) for (int k = 0; k < npts; ++k) theta_terms_far_rev<DISTANT>(pts[k], F, G, JG, ct, f);
    if (act1) for (int k = npts; k < 5 * npts; ++k) theta_terms_far_rev<DISTANT>(pts[k], F, G, JG, ct, f);
}

// One wavefront per workgroup: an item is a wavefront of 64 control panels i
// and a tile of panels j.
__global__ __launch_bounds__(64) I2_TWO_WAVES void k_adj_disjoint(AdjArgs A) {
    __shared__ RuleSh R;
    __shared__ BaryPoint pts[5 * MAX_POINTS];
    __shared__ FarPoint fpts[5 * MAX_POINTS];
    __shared__ long long item_sh;
    load_rule_sh(R, A.rule);
    __syncthreads();
    const int lane = threadIdx.x;
    const int npts = A.rule.n;
    load_bary(pts, fpts, R, npts);
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) {
            const unsigned long long pos = atomicAdd(&A.counters[0], 1ull);
            item_sh = pos < (unsigned long long)A.disjoint_items ? (long long)pos : -1ll;
        }
        __syncthreads();
        const int64_t item = uniform64a(item_sh);
        if (item < 0) break;
        const int m = __builtin_amdgcn_readfirstlane(find_base_a(A.item_base, A.nmeshes, item));
        const AdjMesh& M = A.meshes[m];
        const int64_t rr = item - A.item_base[m];
        const int JT = M.jt;
        const int jtiles = M.jtiles;
        const int iw = (int)(rr / jtiles), jt = (int)(rr % jtiles);
        const int i = iw * 64 + lane;
        const bool ivalid = i < M.nT;
        const Panel I = M.panels[ivalid ? i : 0];
        const Ball ball = panel_ball(I.a, I.b, I.c, A.rule.reach);
        const int K = M.K[I2_NOT_NEIGHBORS];
        // cotangents of K_i through its points: of vertices a and b, and of the points' sum
        d3 X0 = {0.0, 0.0, 0.0}, X1 = X0, Xs = X0;
        double Sb = 0.0, loss = 0.0;
        uint32_t deep = 0u;                           // bit j - j0: (i, j) is at reported level >= 2
        const int j0 = jt * JT, j1 = min(M.nT, j0 + JT);
        // two bits per j, read before the points' loop so that the loads overlap:
        // reported level 0 or 1, 2: that of k_adj_deep, 3: not a pair
        uint64_t levels = ~0ull;
        {
            const int ii = ivalid ? i : 0;
            // pairs (i, j > i) stand in row i's order, without the neighbours
            const int64_t n0 = M.nbr_start[ii], n1 = M.nbr_start[ii + 1], row = M.row_start[ii];
            int64_t q = n0;
            while (q < n1 && M.nbr[q] < j0) ++q;
            int next = q < n1 ? M.nbr[q] : INT32_MAX;
            const int8_t* conv = M.conv[I2_NOT_NEIGHBORS];
            for (int j = j0; j < j1; ++j) {
                int64_t z = row + (j - ii - 1) - (q - n0);
                bool nb = next == j;
                if (nb) { ++q; next = q < n1 ? M.nbr[q] : INT32_MAX; }
                if (__ballot(ii > j) != 0ull) {         // pairs (j < i): row j's order, the same list for all lanes
                    int below = 0;
                    bool nbj = false;
                    for (int64_t r = M.nbr_start[j]; r < M.nbr_start[j + 1]; ++r) {
                        const int x = M.nbr[r];
                        below += x < ii;
                        nbj |= x == ii;
                    }
                    if (ii > j) { z = M.npairs[I2_NOT_NEIGHBORS] + M.row_start[j] + (ii - j - 1) - below; nb = nbj; }
                }
                if (ivalid && j != ii && !nb) {
                    const int lev = reported_level(A, conv[z], K);
                    levels &= ~((uint64_t)(3 - min(lev, 2)) << (2 * (j - j0)));
                }
            }
        }
        double* const kjw = M.kj + (int64_t)iw * M.nT * 9;   // this wavefront's K_j slots
        for (int j = j0; j < j1; ++j) {
            const Panel J = uniform_panel(M.panels[j]);   // j is uniform: K_j lives in scalar registers
            const int lev = (int)(levels >> (2 * (j - j0))) & 3;
            const bool valid = lev < 2;
            if (lev == 2) deep |= 1u << (j - j0);
            if (__ballot(valid) == 0ull) continue;   // the slot keeps the zeros of k_adj_zero
            Weights W = {0.0, {0.0, 0.0, 0.0}};
            if (valid) W = weights(A.seed, i, j, M.nT, &R.lt);
            const q4 gb = task_cotangent(W, J.n);
            const JGeom JG = uniform_jgeom(make_jgeom(J.a, J.b, J.c, J.ta, J.tb, J.tc));
            const d3 gP = {gb.x, gb.y, gb.z};
            const double fa = lev == 1 ? 0.25 * I.area : I.area;
            const q4 ct = {fa * dot(gP, J.tc), fa * dot(gP, J.ta), fa * dot(gP, J.tb), 2.0 * fa * gb.w};
            const int form = wave_form(valid, ball, JG);
            TermsBar g = terms_bar_zero();
            if (form == 0) {
                for (int lv = 0; lv < 2; ++lv) {      // the pairs at reported level 0, then those at level 1
                    const bool act = valid && lev == lv;
                    if (__ballot(act) == 0ull) continue;
                    if (!act) continue;
                    points_rev(R, pts, lv == 0 ? 0 : npts, lv == 0 ? npts : 5 * npts, I, JG, ct, g, X0, X1);
                }
            } else {
                FarBar f = far_bar_zero();
                {
                    const FarFrame F = far_frame(I.a, I.b, I.c);
                    const FarGeom G = far_geom(F, JG);
                    if (form == 1) points_far_rev<false>(fpts, npts, valid && lev == 0, valid && lev == 1, F, G, JG, ct, f);
                    else points_far_rev<true>(fpts, npts, valid && lev == 0, valid && lev == 1, F, G, JG, ct, f);
                }
                // the frame again, not held across the points: 24 registers (96
                // spilled with it, 70 without; 5,120 panels 10.64 -> 10.51 ms)
                far_bar_expand(f, far_frame(I.a, I.b, opaque(I.c)), JG, g, X0, X1);
            }
            d3 nb = {0.0, 0.0, 0.0};
            if (valid) {
                const q4 F = psi_of_terms(g.T, JG);
                const q4 Iv = fa * F;
                Sb += dot4(gb, F) * (fa / I.area);
                const d3 psi = {Iv.x, Iv.y, Iv.z};
                nb = RECIP_4PI * (Iv.w * W.v + cross(W.v, psi));
                const d3 Jr = finalize_plain(Iv, J.n);
                loss += W.w * Iv.w + dot(W.v, Jr);
                Xs = Xs + g.a + g.b + g.c;
                axpy(Xs, g.y, JG.N2);
            }
            // K_j: each lane's chain to the vertices, summed over the wavefront into its slot
            d3 Ab, Bb, Cb;
            terms_chain(JG, ct, g, fa * gP, nb, i2m::rcp_cubic(JG.La), i2m::rcp_cubic(JG.Lb), i2m::rcp_cubic(JG.Lc),
                        i2m::rcp_cubic(2.0 * J.area), J.n, Ab, Bb, Cb);
            store_sum9(kjw + 9 * (int64_t)j, lane, Ab, Bb, Cb);
        }
        if (__ballot(deep != 0u) != 0ull) {         // the item's marked pairs, lanes in order
            const int cnt = __popc(deep);
            int run = cnt;
            for (int d = 1; d < 64; d <<= 1) {
                const int v = __shfl_up(run, d);
                if (lane >= d) run += v;
            }
            const int n = __builtin_amdgcn_readlane(run, 63);
            unsigned long long base = 0ull;
            if (lane == 0) base = atomicAdd(&A.counters[2], (unsigned long long)n);
            base = (unsigned long long)uniform64a((int64_t)base);
            DeepItem* d = A.deep_items;
            A.deep_mask[item * 64 + lane] = deep;
            if (lane == 0) d[atomicAdd(&A.counters[1], 1ull)] = {item, (int64_t)base, n};
            if (base + n <= (unsigned long long)A.deep_cap) {
                int64_t at = (int64_t)base + run - cnt;
                for (uint32_t r = deep; r != 0u; r &= r - 1u) {
                    const int b = (int)__builtin_ctz(r);
                    const int level = reported_level(A, M.conv[I2_NOT_NEIGHBORS][task_disjoint(M, i, j0 + b)], K);
                    A.deep_pairs[at++] = {item, (int16_t)(lane * ADJ_TILE + b), (int16_t)level};
                }
            } else {                                // the list's last entries, which hold no item
                for (int64_t q = (int64_t)base + lane; q < A.deep_cap; q += 64) A.deep_pairs[q] = {-1, 0, 0};
            }
        }
        if (ivalid) {
            d3 X2 = Xs - X0 - X1;
            if (Sb != 0.0 || dot(X0, X0) + dot(X1, X1) + dot(X2, X2) != 0.0) {
                const d3 zero = {0.0, 0.0, 0.0};
                panel_chain(I, zero, zero, zero, zero, Sb, X0, X1, X2);
            }
            double* kslot = M.ki + ((int64_t)jt * M.nT + i) * 9;
            store3(kslot, X0); store3(kslot + 3, X1); store3(kslot + 6, X2);
        }
        loss = wsum(loss);
        if (lane == 0) A.item_loss[item] = loss;
    }
}

// The disjoint pairs at reported level >= 2, as k_adj_disjoint listed them: a
// wavefront takes its pair if it is above level 2 (832 points in 13 rounds), and
// every fourth one the pairs at level 2 among its four, 16 lanes each (208
// points are 13 rounds of 16 lanes, and what is done once per pair serves four
// pairs per instruction), and leaves a pair's cotangents in its record.  k_adj_deep_sum
// adds an item's records to the item's slots, lanes and then each lane's j in
// order, so the order in which items are listed does not matter.  Pairs beyond
// the list's end are done there as well, in the same way, one after another.
//
// With an item as the unit of work the longest item (over a hundred pairs on a
// thin torus) set the time, at 20 % of the issue slots: 1.15 ms on two tori of
// 3,072 panels against 0.80 as a list, and 0.41 against 0.13 ms on 5,120 panels.
constexpr int DEEP_NK = 11;             // per pair: X0, X1, X2 (9), Sb, loss
constexpr int DEEP_REC = DEEP_NK + 9;   // and the cotangents of K_j's vertices
__device__ __forceinline__ double quad_lane(double v, int q) {
    const uint64_t x = __double_as_longlong(v);
    const int lo = (int)(unsigned)x, hi = (int)(unsigned)(x >> 32);
    unsigned l, h;
    if (q == 0) { l = __builtin_amdgcn_mov_dpp(lo, 0x00, 0xf, 0xf, false); h = __builtin_amdgcn_mov_dpp(hi, 0x00, 0xf, 0xf, false); }
    else if (q == 1) { l = __builtin_amdgcn_mov_dpp(lo, 0x55, 0xf, 0xf, false); h = __builtin_amdgcn_mov_dpp(hi, 0x55, 0xf, 0xf, false); }
    else if (q == 2) { l = __builtin_amdgcn_mov_dpp(lo, 0xaa, 0xf, 0xf, false); h = __builtin_amdgcn_mov_dpp(hi, 0xaa, 0xf, 0xf, false); }
    else { l = __builtin_amdgcn_mov_dpp(lo, 0xff, 0xf, 0xf, false); h = __builtin_amdgcn_mov_dpp(hi, 0xff, 0xf, 0xf, false); }
    return __longlong_as_double((long long)(((uint64_t)h << 32) | l));
}
// One pair by G lanes: 16 (a row of the wavefront) or 64.
template <int G> __device__ __forceinline__ double group_sum(double v) { return G == 16 ? row_sum16(v) : sum_all(v); }
template <int G> __device__ __forceinline__ void group_sum3(d3& v) { v = {group_sum<G>(v.x), group_sum<G>(v.y), group_sum<G>(v.z)}; }
template <int G>
__device__ __forceinline__ void deep_pair(const AdjArgs& A, const RuleSh& R, const AdjMesh& M, int i, int j, int level, int s,
                                          double* rec) {
    const Panel I = M.panels[i];
    const Panel J = M.panels[j];
    // one of the pair's four draws per lane of a quad
    const double draw = normal_draw(A.seed, (uint64_t)i * (uint64_t)M.nT + (uint64_t)j, (uint64_t)(s & 3), &R.lt);
    const Weights W = {quad_lane(draw, 0), {quad_lane(draw, 1), quad_lane(draw, 2), quad_lane(draw, 3)}};
    const q4 gb = task_cotangent(W, J.n);
    const JGeom JG = make_jgeom(J.a, J.b, J.c, J.ta, J.tb, J.tc);
    const int npts = A.rule.n;
    double fa = I.area;
    for (int l = 0; l < level; ++l) fa *= 0.25;
    const d3 gP = {gb.x, gb.y, gb.z};
    const q4 ct = {fa * dot(gP, J.tc), fa * dot(gP, J.ta), fa * dot(gP, J.tb), 2.0 * fa * gb.w};
    TermsBar g = terms_bar_zero();
    d3 X0 = {0.0, 0.0, 0.0}, X1 = X0;
    const uint32_t total = (uint32_t)npts << (2 * level);
    const uint32_t factor = split_factor(npts);
    // the pair's own form, whatever pairs share its wavefront (the list's order
    // changes from run to run)
    if (panel_far(panel_ball(I.a, I.b, I.c, A.rule.reach), JG) != 0) {
        const FarFrame Fr = far_frame(I.a, I.b, I.c);
        const FarGeom FG = far_geom(Fr, JG);
        FarBar f = far_bar_zero();
        for (uint32_t q = s; q < total; q += G) {
            const uint32_t sub = split_point(q, factor), k = q - sub * npts;
            const d3 beta = sub_point(d3{R.L1[k], R.L2[k], R.L3[k]}, level, sub);
            theta_terms_far_rev<false>(far_point(beta.x - 1.0 / 3.0, beta.y - 1.0 / 3.0, R.w[k]), Fr, FG, JG, ct, f);
        }
        double* v = reinterpret_cast<double*>(&f);
#pragma unroll
        for (int k = 0; k < (int)(sizeof(FarBar) / sizeof(double)); ++k) v[k] = group_sum<G>(v[k]);
        // the frame again, as in k_adj_disjoint (1,280 panels at fixed level 2: 8.45 -> 7.66 ms)
        far_bar_expand(f, far_frame(I.a, I.b, opaque(I.c)), JG, g, X0, X1);
    } else {
        for (uint32_t q = s; q < total; q += G) {
            const uint32_t sub = split_point(q, factor), k = q - sub * npts;
            const d3 beta = sub_point(d3{R.L1[k], R.L2[k], R.L3[k]}, level, sub);
            const d3 p = beta.x * I.a + beta.y * I.b + beta.z * I.c;
            const d3 pb = theta_terms_rev(p, JG, &R.lt, R.w[k], ct, g);
            axpy(X0, beta.x, pb); axpy(X1, beta.y, pb);
        }
        group_sum3<G>(g.a); group_sum3<G>(g.b); group_sum3<G>(g.c); group_sum3<G>(g.n); group_sum3<G>(X0); group_sum3<G>(X1);
        g.T = {group_sum<G>(g.T.x), group_sum<G>(g.T.y), group_sum<G>(g.T.z), group_sum<G>(g.T.w)};
        g.y = group_sum<G>(g.y); g.La = group_sum<G>(g.La); g.Lb = group_sum<G>(g.Lb); g.Lc = group_sum<G>(g.Lc);
    }
    const q4 F = psi_of_terms(g.T, JG);
    const q4 Iv = fa * F;
    const d3 psi = {Iv.x, Iv.y, Iv.z};
    const d3 nb = RECIP_4PI * (Iv.w * W.v + cross(W.v, psi));
    const d3 Jr = finalize_plain(Iv, J.n);
    d3 X2 = g.a + g.b + g.c;
    axpy(X2, g.y, JG.N2);
    X2 = X2 - X0 - X1;
    d3 Ab, Bb, Cb;
    terms_chain(JG, ct, g, fa * gP, nb, i2m::rcp_cubic(JG.La), i2m::rcp_cubic(JG.Lb), i2m::rcp_cubic(JG.Lc),
                i2m::rcp_cubic(2.0 * J.area), J.n, Ab, Bb, Cb);
    if (s == 0) {
        store3(rec, X0); store3(rec + 3, X1); store3(rec + 6, X2);
        rec[9] = dot4(gb, F) * (fa / I.area);
        rec[10] = W.w * Iv.w + dot(W.v, Jr);
        store3(rec + 11, Ab); store3(rec + 14, Bb); store3(rec + 17, Cb);
    }
}

// the tile's first j and wavefront of control panels of an item of mesh M
__device__ __forceinline__ void item_at(const AdjArgs& A, const AdjMesh& M, int m, int64_t item, int* iw, int* jt) {
    const int64_t rr = item - A.item_base[m];
    *iw = (int)(rr / M.jtiles);
    *jt = (int)(rr % M.jtiles);
}
__global__ __launch_bounds__(256) I2_TWO_WAVES void k_adj_deep(AdjArgs A) {
    __shared__ RuleSh R;
    const int64_t n = min((int64_t)A.counters[2], A.deep_cap);
    // one quarter of the grid for each of four consecutive pairs: a workgroup's
    // wavefronts then have the same kind of work, and the first quarter, which
    // takes the pairs at level 2, covers all XCDs
    const int quarter = gridDim.x / 4, r = blockIdx.x / quarter;
    int64_t four = 16 * (int64_t)(blockIdx.x % quarter);
    if (four >= n) return;
    load_rule_sh(R, A.rule);
    __syncthreads();
    const int lane = threadIdx.x & 63, row = lane >> 4;
    for (four += 4 * (threadIdx.x >> 6); four < n; four += 16 * (int64_t)quarter) {
        // four pairs, one per row; this wavefront's own is number r
        const int64_t q = four + row;
        const DeepPair e = A.deep_pairs[min(q, n - 1)];
        const bool here = q < n && e.item >= 0;   // an item that did not fit has no entries
        const int level = here ? e.level : 0;
        if (__ballot(r == 0 ? level != 0 : level > 2) == 0ull) continue;
        const int64_t item = here ? e.item : 0;
        const int m = find_base_a(A.item_base, A.nmeshes, item);
        const AdjMesh& M = A.meshes[m];
        int iw, jt;
        item_at(A, M, m, item, &iw, &jt);
        const int i = iw * 64 + e.at / ADJ_TILE, j = jt * M.jt + e.at % ADJ_TILE;
        if (r == 0 && here && level == 2) deep_pair<16>(A, R, M, i, j, level, lane & 15, A.deep_rec + q * DEEP_REC);
        const int from = 16 * r, wl = __builtin_amdgcn_readlane(level, from);
        if (wl > 2)
            deep_pair<64>(A, R, A.meshes[__builtin_amdgcn_readlane(m, from)], __builtin_amdgcn_readlane(i, from),
                          __builtin_amdgcn_readlane(j, from), wl, lane, A.deep_rec + (four + r) * DEEP_REC);
    }
}

// One wavefront per listed item: lane l adds the records of its pairs (panel
// i) to K_i's slot, lane b those of panel j0 + b to K_j's.
__global__ __launch_bounds__(64) I2_TWO_WAVES void k_adj_deep_sum(AdjArgs A) {
    __shared__ RuleSh R;
    __shared__ double rec[4][DEEP_REC];
    __shared__ uint16_t list[64 * ADJ_TILE];   // an unlisted item's pairs
    __shared__ uint32_t masks[64];
    __shared__ int starts[64];
    const int64_t nitems = (int64_t)A.counters[1];
    const int lane = threadIdx.x;
    bool loaded = false;
    for (int64_t x = blockIdx.x; x < nitems; x += gridDim.x) {
        const DeepItem D = A.deep_items[x];
        const int m = __builtin_amdgcn_readfirstlane(find_base_a(A.item_base, A.nmeshes, D.item));
        const AdjMesh& M = A.meshes[m];
        int iw, jt;
        item_at(A, M, m, D.item, &iw, &jt);
        const int j0 = jt * M.jt;
        const uint32_t mask = A.deep_mask[D.item * 64 + lane];
        const int cnt = __popc(mask);
        int at = cnt;
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(at, d);
            if (lane >= d) at += v;
        }
        at -= cnt;
        __syncthreads();
        masks[lane] = mask;
        starts[lane] = at;
        __syncthreads();
        double ki[DEEP_NK] = {}, kj[9] = {};
        if (D.base + D.n <= A.deep_cap) {
            const double* rec0 = A.deep_rec + D.base * DEEP_REC;
            for (int q = 0; q < cnt; ++q)
                for (int c = 0; c < DEEP_NK; ++c) ki[c] += rec0[(int64_t)(at + q) * DEEP_REC + c];
            for (uint64_t some = __ballot(mask != 0u); some != 0ull; some &= some - 1ull) {
                const int l = (int)__builtin_ctzll(some);
                const uint32_t lm = masks[l];
                if (lane < ADJ_TILE && ((lm >> lane) & 1u)) {
                    const double* r = rec0 + (int64_t)(starts[l] + __popc(lm & ((1u << lane) - 1u))) * DEEP_REC + DEEP_NK;
                    for (int c = 0; c < 9; ++c) kj[c] += r[c];
                }
            }
        } else {
            if (!loaded) { load_rule_sh(R, A.rule); loaded = true; }
            const int K = M.K[I2_NOT_NEIGHBORS];
            int k = at;
            for (uint32_t r = mask; r != 0u; r &= r - 1u) list[k++] = (uint16_t)(lane * ADJ_TILE + __builtin_ctz(r));
            __syncthreads();
            for (int first = 0; first < D.n; first += 4) {
                const int row = lane >> 4, q = first + row;
                const int e = list[min(q, D.n - 1)];
                const int i = iw * 64 + e / ADJ_TILE, j = j0 + e % ADJ_TILE;
                const int level = q < D.n ? reported_level(A, M.conv[I2_NOT_NEIGHBORS][task_disjoint(M, i, j)], K) : 0;
                if (level == 2) deep_pair<16>(A, R, M, i, j, level, lane & 15, rec[row]);
                for (int r = 0; r < 4; ++r) {
                    const int wl = __builtin_amdgcn_readlane(level, 16 * r);
                    if (wl > 2)
                        deep_pair<64>(A, R, M, __builtin_amdgcn_readlane(i, 16 * r), __builtin_amdgcn_readlane(j, 16 * r), wl, lane, rec[r]);
                }
                __syncthreads();
                for (int r = 0; r < 4 && first + r < D.n; ++r) {
                    const int f = list[first + r];
                    if (lane == f / ADJ_TILE) for (int c = 0; c < DEEP_NK; ++c) ki[c] += rec[r][c];
                    if (lane == f % ADJ_TILE) for (int c = 0; c < 9; ++c) kj[c] += rec[r][DEEP_NK + c];
                }
                __syncthreads();
            }
        }
        if (mask != 0u) {
            const int i = iw * 64 + lane;
            d3 X0 = {ki[0], ki[1], ki[2]}, X1 = {ki[3], ki[4], ki[5]}, X2 = {ki[6], ki[7], ki[8]};
            const Panel I = M.panels[i];
            const d3 zero = {0.0, 0.0, 0.0};
            panel_chain(I, zero, zero, zero, zero, ki[9], X0, X1, X2);
            double* kslot = M.ki + ((int64_t)jt * M.nT + i) * 9;
            add_to3(kslot, X0); add_to3(kslot + 3, X1); add_to3(kslot + 6, X2);
        }
        const double loss = wsum(ki[10]);
        if (lane == 0) A.item_loss[D.item] += loss;
        // the j of the tile that hold a pair of the item (OR of the lanes' masks)
        uint32_t anyj = mask;
        for (int d = 1; d < 64; d <<= 1) anyj |= (uint32_t)__shfl_xor((int)anyj, d);
        if (lane < ADJ_TILE && ((anyj >> lane) & 1u)) {
            double* kslot = M.kj + ((int64_t)iw * M.nT + j0 + lane) * 9;
            for (int c = 0; c < 9; ++c) kslot[c] += kj[c];
        }
    }
}

// ------------------------------------------------------------ singular pairs
using i2ad::D3;
using i2ad::Dual;
using i2ad::Q4;

__device__ __forceinline__ D3 dual_vertex(d3 x, int slot, int my_slot, int axis) {
    D3 r = {Dual(x.x), Dual(x.y), Dual(x.z)};
    if (slot == my_slot) {
        if (axis == 0) r.x.d = 1.0; else if (axis == 1) r.y.d = 1.0; else r.z.d = 1.0;
    }
    return r;
}
__device__ __forceinline__ double dd(d3 bar, D3 x) { return bar.x * x.x.d + bar.y * x.y.d + bar.z * x.z.d; }
// a, b or c by a run-time index, as selects (an indexed local array would live in scratch memory)
template <class T>
__device__ __forceinline__ T pick3(int s, const T& a, const T& b, const T& c) { return s == 0 ? a : (s == 1 ? b : c); }

// One singular task by G lanes (16: a row of the wavefront, four tasks at a
// time; 64).  Two loops over the points, the inner integral's and then the
// singular part's, so that one set of sums and of geometry is live at a time:
// with both in one loop the kernel held 512 registers, one wavefront per SIMD.
// Points are found from their number alone (sub_point): vertices of sub-panels
// kept over the rule's points made it spill.
// What belongs to the whole pair (closed-form integral, normals, areas) follows
// in k_adj_singular_dual, which has the closed form's value beside its
// derivatives.
template <int TYPE, int G>
__device__ __forceinline__ void singular_task(const AdjArgs& A, const RuleSh& R, const AdjMesh& M, int64_t t, int i, int j,
                                              int level, int s) {
    const Panel I = M.panels[i];
    const int npts = A.rule.n;
    const uint32_t total = (uint32_t)npts << (2 * level);
    const uint32_t factor = split_factor(npts);
    double fa = I.area;
    for (int l = 0; l < level; ++l) fa *= 0.25;
    // one of the pair's four draws per lane of a quad
    const double draw = normal_draw(A.seed, (uint64_t)i * (uint64_t)M.nT + (uint64_t)j, (uint64_t)(s & 3), &R.lt);
    const Weights W = {quad_lane(draw, 0), {quad_lane(draw, 1), quad_lane(draw, 2), quad_lane(draw, 3)}};
    SingRec& r = A.sing_rec[t];
    q4 gb, F;
    d3 X0 = {0.0, 0.0, 0.0}, X1 = X0, X2;
    {
        const Panel J = M.panels[j];
        gb = task_cotangent(W, J.n);
        const JGeom JG = make_jgeom(J.a, J.b, J.c, J.ta, J.tb, J.tc);
        const d3 gP = {gb.x, gb.y, gb.z};
        const q4 ct = {fa * dot(gP, J.tc), fa * dot(gP, J.ta), fa * dot(gP, J.tb), 2.0 * fa * gb.w};
        TermsBar g = terms_bar_zero();
        for (uint32_t q = s; q < total; q += G) {
            const uint32_t sub = split_point(q, factor), k = q - sub * npts;
            const d3 beta = sub_point(d3{R.L1[k], R.L2[k], R.L3[k]}, level, sub);
            const d3 p = beta.x * I.a + beta.y * I.b + beta.z * I.c;
            const d3 pb = theta_terms_rev(p, JG, &R.lt, R.w[k], ct, g);
            axpy(X0, beta.x, pb); axpy(X1, beta.y, pb);
        }
        group_sum3<G>(g.a); group_sum3<G>(g.b); group_sum3<G>(g.c); group_sum3<G>(g.n); group_sum3<G>(X0); group_sum3<G>(X1);
        g.T = {group_sum<G>(g.T.x), group_sum<G>(g.T.y), group_sum<G>(g.T.z), group_sum<G>(g.T.w)};
        g.y = group_sum<G>(g.y); g.La = group_sum<G>(g.La); g.Lb = group_sum<G>(g.Lb); g.Lc = group_sum<G>(g.Lc);
        F = psi_of_terms(g.T, JG);
        X2 = g.a + g.b + g.c;
        axpy(X2, g.y, JG.N2);
        X2 = X2 - X0 - X1;
        d3 Ab, Bb, Cb;
        terms_chain(JG, ct, g, fa * gP, d3{0.0, 0.0, 0.0}, i2m::rcp_cubic(JG.La), i2m::rcp_cubic(JG.Lb), i2m::rcp_cubic(JG.Lc),
                    i2m::rcp_cubic(2.0 * J.area), J.n, Ab, Bb, Cb);
        if (s == 0) { r.g[0] = Ab; r.g[1] = Bb; r.g[2] = Cb; }
    }
    const Panel J = M.panels[j];
    int s1, s2;
    EdgeCtx ec;
    VertexCtx vc;
    if (TYPE == I2_ATTACHED_NEIGHBORS) {
        shifts_edge(I, J, &s1, &s2);
        ec = edge_ctx(vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3));
    } else {
        shifts_vertex(I, J, &s1, &s2);
        vc = vertex_ctx(vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3), I.n, J.n, I.area);
    }
    const d3 z3 = {0.0, 0.0, 0.0};
    EdgeBar ge = {z3, z3, z3, z3, z3, 0.0};
    VertexBar gv = {z3, z3, z3, z3, 0.0};
    q4 Fs = q4zero();
    d3 Y0 = z3, Y1 = z3;
    for (uint32_t q = s; q < total; q += G) {
        const uint32_t sub = split_point(q, factor), k = q - sub * npts;
        // these derivatives amplify the point's rounding: it comes from the
        // sub-panel's vertices, as in the quadrature
        d3 a = I.a, b = I.b, c = I.c;
        sub_panel(a, b, c, level, sub);
        d3 p = R.L1[k] * a;
        p = p + R.L2[k] * b;
        p = p + R.L3[k] * c;
        const d3 beta = sub_point(d3{R.L1[k], R.L2[k], R.L3[k]}, level, sub);
        const q4 gm = -(fa * R.w[k]) * gb;
        d3 ps;
        const q4 f = TYPE == I2_ATTACHED_NEIGHBORS ? sing_edge_rev(p, ec, &R.lt, gm, &ps, ge) : sing_vertex_rev(p, vc, &R.lt, gm, &ps, gv);
        Fs = Fs + R.w[k] * f;
        axpy(Y0, beta.x, ps); axpy(Y1, beta.y, ps);
    }
    group_sum3<G>(Y0); group_sum3<G>(Y1);
    Fs = {group_sum<G>(Fs.x), group_sum<G>(Fs.y), group_sum<G>(Fs.z), group_sum<G>(Fs.w)};
    d3 Y2;
    if (TYPE == I2_ATTACHED_NEIGHBORS) {
        group_sum3<G>(ge.JB); group_sum3<G>(ge.JC); group_sum3<G>(ge.taua); group_sum3<G>(ge.taub); group_sum3<G>(ge.tauc);
        ge.ilvc = group_sum<G>(ge.ilvc) / ec.ilvc;
        Y2 = -(ge.JB + ge.JC) - Y0 - Y1;      // the points' cotangents are minus the vertices'
    } else {
        group_sum3<G>(gv.JA); group_sum3<G>(gv.taua); group_sum3<G>(gv.taub); group_sum3<G>(gv.e);
        gv.invAri = group_sum<G>(gv.invAri) / vc.invAri;
        Y2 = -gv.JA - Y0 - Y1;
    }
    if (s == 0) {
        r.i = i; r.j = j; r.s1 = s1; r.s2 = s2;
        if (TYPE == I2_ATTACHED_NEIGHBORS) {
            r.cb[0] = ge.JB; r.cb[1] = ge.JC; r.cb[2] = ge.taua; r.cb[3] = ge.taub; r.cb[4] = ge.tauc;
            r.cs = ge.ilvc;
        } else {
            r.cb[0] = gv.JA; r.cb[1] = gv.taua; r.cb[2] = gv.taub; r.cb[3] = gv.e; r.cb[4] = z3;
            r.cs = gv.invAri;
        }
        r.X[0] = X0 + Y0; r.X[1] = X1 + Y1; r.X[2] = X2 + Y2;
        r.F = F - Fs;
        r.fa = fa;
        r.gb = gb;
        r.w = W.w;
        r.v = W.v;
    }
}

// Forward mode along coordinate d = 3 * slot + axis (slots 0..2 = K_i's,
// 3..5 = K_j's vertices) of a singular task's per-task chain: panel normals,
// area and tangents, the singular context and the closed-form singular
// integral, weighted by the cotangents the point loop left in the record and
// those of the pair's values, which the closed form's value completes.  Returns
// the task's whole dL/d(coordinate d), and in `loss` the task's term of L.
template <int TYPE>
__device__ __forceinline__ double singular_chain(const AdjMesh& M, const SingRec& r, int d, double* loss) {
    const Panel I = M.panels[r.i];
    const Panel J = M.panels[r.j];
    const int s1 = r.s1, s2 = r.s2;
    const int slot = d / 3, axis = d % 3;
    const D3 ia = dual_vertex(I.a, 0, slot, axis), ib = dual_vertex(I.b, 1, slot, axis), ic = dual_vertex(I.c, 2, slot, axis);
    const D3 ja = dual_vertex(J.a, 3, slot, axis), jb = dual_vertex(J.b, 4, slot, axis), jc = dual_vertex(J.c, 5, slot, axis);
    const D3 cri = cross(ib - ia, ic - ia), crj = cross(jb - ja, jc - ja);
    const D3 nI = unit(cri), nJ = unit(crj);
    const Dual SI = vlen(cri) * Dual(0.5);
    const D3 i0 = pick3(s1, ia, ib, ic), i1 = pick3((s1 + 1) % 3, ia, ib, ic), i2v = pick3((s1 + 2) % 3, ia, ib, ic);
    const D3 j0 = pick3(s2, ja, jb, jc), j1 = pick3((s2 + 1) % 3, ja, jb, jc), j2 = pick3((s2 + 2) % 3, ja, jb, jc);
    double dl = 0.0;
    const d3 gx = pick3(slot % 3, slot < 3 ? r.X[0] : r.g[0], slot < 3 ? r.X[1] : r.g[1], slot < 3 ? r.X[2] : r.g[2]);
    dl += (axis == 0 ? gx.x : (axis == 1 ? gx.y : gx.z));
    Q4 sd;
    if (TYPE == I2_ATTACHED_NEIGHBORS) {
        const EdgeCtxT<Dual> c = edge_ctx(j0, j1, j2);
        dl += dd(r.cb[0], c.JB) + dd(r.cb[1], c.JC) + dd(r.cb[2], c.taua) + dd(r.cb[3], c.taub) + dd(r.cb[4], c.tauc) +
              r.cs * c.ilvc.d;
        sd = integrate_sing_edge(i0, i1, i2v, j0, j1, j2, nI, nJ, SI);
    } else {
        const VertexCtxT<Dual> c = vertex_ctx(j0, j1, j2, nI, nJ, SI);
        dl += dd(r.cb[0], c.JA) + dd(r.cb[1], c.taua) + dd(r.cb[2], c.taub) + dd(r.cb[3], c.e) + r.cs * c.invAri.d;
        sd = integrate_sing_vertex(i0, i1, i2v, j0, j1, j2, nI, nJ, SI);
    }
    const q4 gb = r.gb;
    dl += gb.x * sd.x.d + gb.y * sd.y.d + gb.z * sd.z.d + gb.w * sd.w.d;
    const q4 Iv = r.fa * r.F + q4{sd.x.v, sd.y.v, sd.z.v, sd.w.v};
    const int pw = TYPE == I2_SIMPLE_NEIGHBORS ? wrap_count(Iv.w, I.area) : 0;
    const d3 Jr = TYPE == I2_SIMPLE_NEIGHBORS ? finalize_vertex_p(Iv, J.n, I.area, pw) : finalize_plain(Iv, J.n);
    const d3 psi = {Iv.x, Iv.y, Iv.z};
    const double thetaw = Iv.w + 2.0 * pw * (TWO_PI * I.area);
    const d3 nb = RECIP_4PI * (thetaw * r.v + cross(r.v, psi));
    const double Sb = dot4(gb, r.F) * (r.fa / I.area) + (TYPE == I2_SIMPLE_NEIGHBORS ? pw * dot(r.v, J.n) : 0.0);
    dl += dd(nb, nJ) + Sb * SI.d;
    *loss = r.w * Iv.w + dot(r.v, Jr);
    return dl;
}

// The singular tasks in three launches, by their reported level: STEP 0 takes
// those at levels 0 and 1, 16 lanes each (52 points of the 13-point rule in
// four rounds), and lists the others, the list's start for level 2 and its end
// for the rest; STEP 1 takes level 2, 16 lanes each (208 points in 13 rounds),
// STEP 2 the rest, a wavefront each (832 points in 13 rounds).  Every task has
// a record of its own, so the lists' order does not matter.
template <int STEP>
__global__ __launch_bounds__(ADJ_BLOCK) I2_TWO_WAVES void k_adj_singular(AdjArgs A) {
    __shared__ RuleSh R;
    constexpr int G = STEP == 2 ? 64 : 16;
    const int64_t groups = (int64_t)gridDim.x * (ADJ_BLOCK / G), g0 = (int64_t)blockIdx.x * (ADJ_BLOCK / G);
    const int64_t count = STEP == 0 ? A.singular_tasks : (int64_t)A.counters[2 + STEP];
    if (g0 >= count) return;
    load_rule_sh(R, A.rule);
    __syncthreads();
    const int s = threadIdx.x & (G - 1);
    for (int64_t e = g0 + threadIdx.x / G; e < count; e += groups) {
        const int64_t t = STEP == 0 ? e : A.sing_deep[STEP == 1 ? e : A.singular_tasks - 1 - e];
        const int b = find_base_a(A.sing_base, 2 * A.nmeshes, t);
        const int type = b / A.nmeshes == 0 ? I2_SIMPLE_NEIGHBORS : I2_ATTACHED_NEIGHBORS;
        const AdjMesh& M = A.meshes[b % A.nmeshes];
        const int64_t z = t - A.sing_base[b];
        const int64_t n = M.npairs[type];
        const int32_t* L = M.lists[type];
        const int64_t k = z < n ? z : z - n;
        int i = L[3 * k], j = L[3 * k + 1];
        if (z >= n) { const int x = i; i = j; j = x; }
        const int level = reported_level(A, M.conv[type][z], M.K[type]);
        if (STEP == 0 && level >= 2) {
            if (s == 0) {
                if (level == 2) A.sing_deep[atomicAdd(&A.counters[3], 1ull)] = t;
                else A.sing_deep[A.singular_tasks - 1 - (int64_t)atomicAdd(&A.counters[4], 1ull)] = t;
            }
            continue;
        }
        if (type == I2_ATTACHED_NEIGHBORS) singular_task<I2_ATTACHED_NEIGHBORS, G>(A, R, M, t, i, j, level, s);
        else singular_task<I2_SIMPLE_NEIGHBORS, G>(A, R, M, t, i, j, level, s);
    }
}

// The per-task chains of all singular tasks: 18 coordinates per task, one per
// lane (tasks are ordered by type, so wavefronts rarely mix the two types).
__global__ __launch_bounds__(ADJ_BLOCK) void k_adj_singular_dual(AdjArgs A) {
    const int64_t total = A.singular_tasks * 18;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (int64_t)gridDim.x * blockDim.x) {
        const int64_t t = g / 18;
        const int d = (int)(g - 18 * t);
        const int b = find_base_a(A.sing_base, 2 * A.nmeshes, t);
        const AdjMesh& M = A.meshes[b % A.nmeshes];
        const SingRec& r = A.sing_rec[t];
        double loss;
        A.sing_dl[g] = (b / A.nmeshes == 0) ? singular_chain<I2_SIMPLE_NEIGHBORS>(M, r, d, &loss)
                                            : singular_chain<I2_ATTACHED_NEIGHBORS>(M, r, d, &loss);
        if (d == 0) A.sing_rec[t].loss = loss;
    }
}

// The slots of each panel vertex coordinate: its tiles as the control panel,
// then its wavefronts of control panels as the influencing panel.  A workgroup
// takes 16 consecutive (panel, coordinate)s, 16 threads each: thread s adds
// slots s, s + 16, ..., and a fixed tree adds the threads.  The slots are read
// once and lines of 16 values at a time; one thread per coordinate left 325
// loads in series, 82 us for 320 panels.
__global__ __launch_bounds__(256) void k_adj_panel_sum(AdjArgs A) {
    __shared__ double part[16][17];
    const int64_t total = 9 * A.npanels;
    const int c = threadIdx.x & 15, s = threadIdx.x >> 4;
    for (int64_t q0 = 16 * (int64_t)blockIdx.x; q0 < total; q0 += 16 * (int64_t)gridDim.x) {
        const int64_t q = q0 + c;
        double acc = 0.0;
        if (q < total) {
            const int64_t gp = q / 9;
            const int comp = (int)(q - 9 * gp);
            const int m = find_base_a(A.pbase, A.nmeshes, gp);
            const AdjMesh& M = A.meshes[m];
            const int64_t p = gp - A.pbase[m];
            const int64_t stride = 9 * (int64_t)M.nT;
            const double* ki = M.ki + 9 * p + comp;
            for (int t = s; t < M.jtiles; t += 16) acc += ki[stride * t];
            const double* kj = M.kj + 9 * p + comp;
            for (int t = s; t < M.niw; t += 16) acc += kj[stride * t];
        }
        __syncthreads();
        part[s][c] = acc;
        __syncthreads();
        for (int h = 8; h > 0; h >>= 1) {
            if (s < h) part[s][c] += part[s + h][c];
            __syncthreads();
        }
        if (s == 0 && q < total) A.psum[q] = part[0][c];
    }
}

// Panel p's singular tasks: the sum of corner c's coordinates over entries r, r
// + 4, ... of its pairs with later panels (row p of the two lists: it is I of
// task (p, q) and J of (q, p)) and with earlier ones (the mesh's lists of those).
__device__ __forceinline__ d3 singular_corner(const AdjArgs& A, const AdjMesh& M, int m, int p, int c, int r) {
    d3 acc = {0.0, 0.0, 0.0};
    const int64_t b0 = A.sing_base[m], b1 = A.sing_base[A.nmeshes + m];
    const int64_t s0 = M.off[0][p], n0 = M.off[0][p + 1] - s0, a0 = M.off[1][p], n1 = n0 + M.off[1][p + 1] - a0;
    const int64_t e0 = M.back_start[p], n = n1 + M.back_start[p + 1] - e0;
    for (int64_t x = r; x < n; x += 4) {
        int64_t k = x < n0 ? 2 * (s0 + x) : (x < n1 ? 2 * (a0 + x - n0) + 1 : M.back[e0 + x - n1]);
        if (k < 0) continue;
        const int64_t t = ((k & 1) ? b1 : b0) + (k >> 1), u = t + ((k & 1) ? M.npairs[1] : M.npairs[0]);
        const int first = x < n1 ? c : 3 + c, second = x < n1 ? 3 + c : c;
        const double *v = A.sing_dl + 18 * t + 3 * first, *w = A.sing_dl + 18 * u + 3 * second;
        acc = acc + d3{v[0], v[1], v[2]} + d3{w[0], w[1], w[2]};
    }
    return acc;
}

// dL/dX, 32 lanes per vertex: four lanes take panel l, l + 8, ... at the vertex,
// with its panel sums and, each a quarter of them, its singular tasks'
// coordinates of that corner, and a butterfly adds the lanes.  The order
// depends on the mesh alone.  The lists are the mesh preparation's: lists made
// for the gather on the host and uploaded took 0.2 ms per call on 320 panels and
// 0.9 on 5,120.
__global__ __launch_bounds__(256) void k_adj_gather(AdjArgs A) {
    const int s = (threadIdx.x & 31) >> 2, r = threadIdx.x & 3;
    const int64_t groups = (int64_t)gridDim.x * (blockDim.x / 32);
    for (int64_t gv = (int64_t)blockIdx.x * (blockDim.x / 32) + (threadIdx.x >> 5); gv < A.nvtx; gv += groups) {
        const int m = find_base_a(A.vbase, A.nmeshes, gv);
        const AdjMesh& M = A.meshes[m];
        const int64_t v = gv - A.vbase[m], e0 = M.inc_start[v], e1 = M.inc_start[v + 1];
        d3 acc = {0.0, 0.0, 0.0};
        for (int64_t e = e0 + s; e < e1; e += 8) {
            const int p = M.inc[e];
            if (e > e0 && M.inc[e - 1] == p) continue;      // a panel with this vertex twice is listed twice
            for (int c = 0; c < 3; ++c) {
                if (M.tri[3 * (int64_t)p + c] != v) continue;
                const double* ps = A.psum + 9 * (A.pbase[m] + p) + 3 * c;
                if (r == 0) acc = acc + d3{ps[0], ps[1], ps[2]};
                acc = acc + singular_corner(A, M, m, p, c, r);
            }
        }
        for (int d = 1; d < 32; d <<= 1) {
            acc.x += __shfl_xor(acc.x, d); acc.y += __shfl_xor(acc.y, d); acc.z += __shfl_xor(acc.z, d);
        }
        if ((threadIdx.x & 31) == 0) { double* d = M.dX + 3 * v; d[0] = acc.x; d[1] = acc.y; d[2] = acc.z; }
    }
}

// L of each mesh in two passes.  k_adj_loss_part: LOSS_PARTS workgroups per
// mesh, each over a fixed contiguous share of the mesh's terms (its disjoint
// items, then its vertex-sharing tasks, then its edge-sharing tasks), each
// thread over a fixed strided subset, then a fixed reduction tree.
// k_adj_loss: the mesh's partials by a fixed tree.
constexpr int LOSS_PARTS = 64;
__device__ __forceinline__ double block_sum256(double v, double* part) {
    part[threadIdx.x] = v;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) part[threadIdx.x] += part[threadIdx.x + h];
        __syncthreads();
    }
    return part[0];
}
__global__ __launch_bounds__(256) void k_adj_loss_part(AdjArgs A) {
    __shared__ double part[256];
    const int m = blockIdx.x / LOSS_PARTS, b = blockIdx.x % LOSS_PARTS;
    const AdjMesh& M = A.meshes[m];
    const int64_t ni = A.item_base[m + 1] - A.item_base[m];
    const int64_t n0 = 2 * M.npairs[0], n1 = 2 * M.npairs[1];
    const int64_t n = ni + n0 + n1;
    const int64_t e0 = n * b / LOSS_PARTS, e1 = n * (b + 1) / LOSS_PARTS;
    double v = 0.0;
    for (int64_t e = e0 + threadIdx.x; e < e1; e += 256) {
        if (e < ni) v += A.item_loss[A.item_base[m] + e];
        else if (e < ni + n0) v += A.sing_rec[A.sing_base[m] + (e - ni)].loss;
        else v += A.sing_rec[A.sing_base[A.nmeshes + m] + (e - ni - n0)].loss;
    }
    const double t = block_sum256(v, part);
    if (threadIdx.x == 0) A.loss_part[blockIdx.x] = t;
}
__global__ __launch_bounds__(256) void k_adj_loss(AdjArgs A) {
    __shared__ double part[256];
    const int m = blockIdx.x;
    const double v = (int)threadIdx.x < LOSS_PARTS ? A.loss_part[m * LOSS_PARTS + threadIdx.x] : 0.0;
    const double t = block_sum256(v, part);
    if (threadIdx.x == 0) *A.meshes[m].loss = t;
}

__global__ void k_adj_zero(unsigned long long* c, int nc, double* kj, int64_t nkj) {
    if (blockIdx.x == 0 && (int)threadIdx.x < nc) c[threadIdx.x] = 0ull;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < nkj; q += (int64_t)gridDim.x * blockDim.x) kj[q] = 0.0;
}

// ------------------------------------------------------------ host side
int adjoint_launch(AdjState& S, hipStream_t st) {
    hipLaunchKernelGGL(k_adj_zero, dim3(4 * S.grid), dim3(256), 0, st, S.d_counters.p, N_ADJ_COUNTERS, S.d_kj.p, S.kj_total);
    I2_TRY(check_launch("k_adj_zero"));
    // two streams, as in the forward pass
    const bool two = S.args.singular_tasks > 0;
    if (two) {
        I2_TRY(S.side->fork(st));
    }
    hipLaunchKernelGGL(k_adj_disjoint, dim3(4 * S.grid), dim3(64), 0, st, S.args);
    I2_TRY(check_launch("k_adj_disjoint"));
    if (two) {
        const hipStream_t sst = S.side->stream;
        const int64_t blocks = std::min<int64_t>((S.args.singular_tasks + 15) / 16, 4 * (int64_t)S.grid);
        hipLaunchKernelGGL(k_adj_singular<0>, dim3((unsigned)blocks), dim3(ADJ_BLOCK), 0, sst, S.args);
        hipLaunchKernelGGL(k_adj_singular<1>, dim3((unsigned)blocks), dim3(ADJ_BLOCK), 0, sst, S.args);
        hipLaunchKernelGGL(k_adj_singular<2>, dim3((unsigned)std::min<int64_t>(4 * blocks, 4 * (int64_t)S.grid)), dim3(ADJ_BLOCK), 0, sst, S.args);
        I2_TRY(check_launch("k_adj_singular"));
        hipLaunchKernelGGL(k_adj_singular_dual, dim3(S.grid), dim3(ADJ_BLOCK), 0, sst, S.args);
        I2_TRY(check_launch("k_adj_singular_dual"));
    }
    hipLaunchKernelGGL(k_adj_deep, dim3(16 * S.grid), dim3(256), 0, st, S.args);
    I2_TRY(check_launch("k_adj_deep"));
    hipLaunchKernelGGL(k_adj_deep_sum, dim3(4 * S.grid), dim3(64), 0, st, S.args);
    I2_TRY(check_launch("k_adj_deep_sum"));
    if (two) I2_TRY(S.side->join(st));
    if (S.args.npanels > 0) {
        const int64_t blocks = std::min<int64_t>((9 * S.args.npanels + 15) / 16, 16 * (int64_t)S.grid);
        hipLaunchKernelGGL(k_adj_panel_sum, dim3((unsigned)blocks), dim3(256), 0, st, S.args);
        I2_TRY(check_launch("k_adj_panel_sum"));
    }
    if (S.args.nvtx > 0) {
        const int64_t blocks = std::min<int64_t>((S.args.nvtx + 7) / 8, 16 * (int64_t)S.grid);
        hipLaunchKernelGGL(k_adj_gather, dim3((unsigned)blocks), dim3(256), 0, st, S.args);
        I2_TRY(check_launch("k_adj_gather"));
    }
    hipLaunchKernelGGL(k_adj_loss_part, dim3(S.args.nmeshes * LOSS_PARTS), dim3(256), 0, st, S.args);
    I2_TRY(check_launch("k_adj_loss_part"));
    hipLaunchKernelGGL(k_adj_loss, dim3(S.args.nmeshes), dim3(256), 0, st, S.args);
    I2_TRY(check_launch("k_adj_loss"));
    return I2_OK;
}

// Panels j per disjoint item of a mesh.  2,048 wavefronts are in flight (two per
// SIMD), so a mesh wants some four rounds of items; smaller tiles cost a K_i
// slot and the chain of K_i each.  Measured, forward and gradient: 320 panels
// 4.1 ms with tiles of 32 (50 items), 1.76 ms with 1; 1,280 panels 6.1 ms with
// 32, 4.0 with 4, 3.8 with 2, 4.05 with 1; 5,120 panels 26.4-27.1 ms with 32 (6.25
// rounds), 25.0 with 16.  Above 16,384 panels the slots (nT^2/jt * 72 bytes) keep
// the tile at 32.  From the mesh's size alone, so that a mesh has the same sums
// in any batch.
static int adjoint_tile(int nT) {
    const int64_t niw = (nT + 63) / 64;
    int jt = nT > 16384 ? ADJ_TILE : ADJ_TILE / 2;
    while (jt > 1 && niw * ((nT + jt - 1) / jt) < 8192) jt /= 2;
    return jt;
}

// Builds the adjoint's descriptors for meshes D (panels, lists, convergence
// iterations and device K already set): the partial-cotangent slots, dX and
// loss (one block of 3 nV + 1 doubles per mesh), and the vertex gather's
// lists from each mesh's cells and vertex- and edge-sharing pair lists.
int adjoint_setup(AdjState& S, int device, std::vector<AdjMesh> D, const std::vector<const i2_mesh*>& meshes,
                  const i2_integrator* it, uint64_t seed, const int* K) {
    int cus = 0;
    I2_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    S.grid = std::max(1, cus) * 4;
    const int M = (int)D.size();
    if ((int)meshes.size() != M) { set_error("adjoint setup: %d descriptors for %d meshes", M, (int)meshes.size()); return I2_ERR_INVALID; }
    AdjArgs& A = S.args;
    S.nV.assign(M, 0);
    for (int m = 0; m < M; ++m) S.nV[m] = meshes[m]->nV;
    S.grad_off.assign(M + 1, 0);
    for (int m = 0; m < M; ++m) S.grad_off[m + 1] = S.grad_off[m] + 3 * S.nV[m] + 1;
    I2_TRY(S.d_grad.ensure(S.grad_off[M]));
    std::vector<int64_t> item_base(M + 1, 0), sing_base(2 * M + 1, 0), ki_off(M + 1, 0), kj_off(M + 1, 0), vbase(M + 1, 0),
        pbase(M + 1, 0);
    for (int m = 0; m < M; ++m) {
        const int64_t niw = (D[m].nT + 63) / 64;
        const int jt = adjoint_tile(D[m].nT);
        const int64_t jtiles = (D[m].nT + jt - 1) / jt;
        D[m].jt = jt;
        D[m].jtiles = (int)jtiles;
        D[m].niw = (int)niw;
        item_base[m + 1] = item_base[m] + niw * jtiles;
        ki_off[m + 1] = ki_off[m] + (int64_t)D[m].nT * jtiles * 9;
        kj_off[m + 1] = kj_off[m] + (int64_t)D[m].nT * D[m].niw * 9;
        vbase[m + 1] = vbase[m] + S.nV[m];
        pbase[m + 1] = pbase[m] + D[m].nT;
    }
    I2_TRY(S.d_ki.ensure(ki_off[M]));
    I2_TRY(S.d_kj.ensure(kj_off[M]));
    S.kj_total = kj_off[M];
    for (int m = 0; m < M; ++m) {
        D[m].dX = S.d_grad.p + S.grad_off[m];
        D[m].loss = S.d_grad.p + S.grad_off[m] + 3 * S.nV[m];
        D[m].ki = S.d_ki.p + ki_off[m];
        D[m].kj = S.d_kj.p + kj_off[m];
    }
    int64_t acc = 0;
    for (int kind = 0; kind < 2; ++kind)
        for (int m = 0; m < M; ++m) { sing_base[kind * M + m] = acc; acc += 2 * D[m].npairs[kind]; }
    sing_base[2 * M] = acc;

    for (int m = 0; m < M; ++m) {
        const i2_mesh& x = *meshes[m];
        if (!x.prepared) { set_error("adjoint setup: mesh %d is not prepared", m); return I2_ERR_STATE; }
        D[m].off[0] = x.d_off[0].p;
        D[m].off[1] = x.d_off[1].p;
        D[m].back_start = x.d_back_start.p;
        D[m].back = x.d_back.p;
        D[m].tri = x.d_tri.p;
        D[m].inc_start = x.d_inc_start.p;
        D[m].inc = x.d_inc.p;
    }
    // all tables in one upload
    const int64_t words = (int64_t)(sizeof(AdjMesh) * M + 7) / 8, kwords = K ? (3 * M + 1) / 2 : 0;
    std::vector<int64_t> table;
    for (const auto* v : {&pbase, &vbase, &item_base, &sing_base}) table.insert(table.end(), v->begin(), v->end());
    const int64_t at = (int64_t)table.size();
    table.resize(at + words + kwords);
    I2_TRY(S.d_base.ensure((int64_t)table.size()));
    if (K) {
        memcpy(table.data() + at + words, K, sizeof(int) * 3 * M);
        for (int m = 0; m < M; ++m) D[m].K = reinterpret_cast<const int*>(S.d_base.p + at + words) + 3 * m;
    }
    memcpy(table.data() + at, D.data(), sizeof(AdjMesh) * M);
    I2_HIP(hipMemcpy(S.d_base.p, table.data(), sizeof(int64_t) * table.size(), hipMemcpyHostToDevice));
    I2_TRY(S.d_psum.ensure(9 * pbase[M]));
    A.psum = S.d_psum.p;
    A.npanels = pbase[M];
    A.nvtx = vbase[M];
    A.pbase = S.d_base.p;
    A.vbase = A.pbase + M + 1;
    A.item_base = A.vbase + M + 1;
    A.sing_base = A.item_base + M + 1;
    A.meshes = reinterpret_cast<const AdjMesh*>(S.d_base.p + at);
    A.nmeshes = M;
    A.fixed = it->fixed;
    A.last_level = it->fixed ? it->fixed_level : it->max_level;
    A.quirk = it->quirk;
    A.rule = it->rule;
    A.seed = seed;
    A.disjoint_items = item_base[M];
    A.singular_tasks = sing_base[2 * M];
    if (A.singular_tasks > 0) I2_TRY(S.side->ensure());
    I2_TRY(S.d_sing_rec.ensure(A.singular_tasks));
    A.sing_rec = S.d_sing_rec.p;
    I2_TRY(S.d_sing_deep.ensure(A.singular_tasks));
    A.sing_deep = S.d_sing_deep.p;
    I2_TRY(S.d_sing_dl.ensure(18 * A.singular_tasks));
    A.sing_dl = S.d_sing_dl.p;
    I2_TRY(S.d_item_loss.ensure(A.disjoint_items));
    A.item_loss = S.d_item_loss.p;
    I2_TRY(S.d_loss_part.ensure((int64_t)LOSS_PARTS * M));
    A.loss_part = S.d_loss_part.p;
    I2_TRY(S.d_deep_mask.ensure(64 * A.disjoint_items));
    A.deep_mask = S.d_deep_mask.p;
    I2_TRY(S.d_deep_items.ensure(A.disjoint_items));
    A.deep_items = S.d_deep_items.p;
    // room for every pair of small meshes, 1/64 of the pairs of larger ones (0.6 %
    // are refined on 1,280 panels, 0.03 % on 5,120), at most 2^20 pairs (168 MB)
    int64_t pairs = 0;
    for (int m = 0; m < M; ++m) pairs += 2 * D[m].npairs[I2_NOT_NEIGHBORS];
    A.deep_cap = std::min<int64_t>(std::min(pairs, std::max<int64_t>(65536, pairs / 64)), (int64_t)1 << 20);
    I2_TRY(S.d_deep_pairs.ensure(A.deep_cap));
    I2_TRY(S.d_deep_rec.ensure(DEEP_REC * A.deep_cap));
    A.deep_pairs = S.d_deep_pairs.p;
    A.deep_rec = S.d_deep_rec.p;
    I2_TRY(S.d_counters.ensure(N_ADJ_COUNTERS));
    A.counters = S.d_counters.p;
    return I2_OK;
}

AdjMesh adjoint_mesh(const i2_mesh* mesh, const int8_t* const conv[3], const int* dK) {
    AdjMesh D{};
    D.panels = mesh->d_panels.p;
    D.row_start = mesh->d_row_start.p;
    D.nbr_start = mesh->d_nbr_start.p;
    D.nbr = mesh->d_nbr.p;
    D.lists[0] = mesh->d_simple.p;
    D.lists[1] = mesh->d_attached.p;
    for (int t = 0; t < 3; ++t) { D.npairs[t] = mesh->pairs[t]; D.conv[t] = conv[t]; }
    D.K = dK;
    D.nT = (int)mesh->nT;
    return D;
}

int adjoint_copy_out(const AdjState& S, int mesh, double* loss, double* dLdX) {
    const double* base = S.d_grad.p + S.grad_off[mesh];
    const int64_t nV = S.nV[mesh];
    // dL/dX and L stand one after the other: one copy
    std::vector<double> h((size_t)(3 * nV + 1));
    I2_HIP(hipMemcpy(h.data(), base, sizeof(double) * h.size(), hipMemcpyDeviceToHost));
    if (dLdX) memcpy(dLdX, h.data(), sizeof(double) * 3 * (size_t)nV);
    if (loss) *loss = h[(size_t)(3 * nV)];
    return I2_OK;
}

// Runs the adjoint of one mesh.
int adjoint_run(AdjState& S, hipStream_t st, double* loss, double* dLdX) {
    I2_HIP(hipEventRecord(S.e0, st));
    I2_TRY(adjoint_launch(S, st));
    I2_HIP(hipEventRecord(S.e1, st));
    I2_HIP(hipStreamSynchronize(st));
    float ms = 0.0f;
    I2_HIP(hipEventElapsedTime(&ms, S.e0, S.e1));
    S.ms = ms;
    return adjoint_copy_out(S, 0, loss, dLdX);
}

void adjoint_release(AdjState*& S) {
    if (!S) return;
    if (S->e0) (void)hipEventDestroy(S->e0);
    if (S->e1) (void)hipEventDestroy(S->e1);
    delete S;
    S = nullptr;
}

}  // namespace i2

using namespace i2;

extern "C" {

int i2_evaluator_loss_and_grad(i2_evaluator* ev, uint64_t seed, double* loss, double* dLdX) {
    if (!ev || !loss || !dLdX) { set_error("null argument"); return I2_ERR_INVALID; }
    if (!ev->ran || !ev->all_pairs) { set_error("run all pairs first: the loss is defined over every ordered pair"); return I2_ERR_STATE; }
    I2_TRY(results_current(ev));
    DeviceGuard g(ev->mesh->device);
    if (!g.ok) return I2_ERR_HIP;
    if (!ev->adj) {
        ev->adj = new AdjState;
        if (hipEventCreate(&ev->adj->e0) != hipSuccess || hipEventCreate(&ev->adj->e1) != hipSuccess) {
            (void)hipGetLastError();
            adjoint_release(ev->adj);
            set_error("event creation failed");
            return I2_ERR_HIP;
        }
        ev->adj->side = &ev->side;
    }
    const int8_t* conv[3];
    int K[3];
    for (int t = 0; t < 3; ++t) {
        K[t] = ev->type[t].K;
        if (ev->ran_path == 1) {
            const double4* ints;
            const double* res;
            engine_evaluator_outputs(ev, t, &ints, &res, &conv[t]);
        } else {
            conv[t] = ev->type[t].conv.p;
        }
    }
    AdjState& S = *ev->adj;
    I2_TRY(adjoint_setup(S, ev->mesh->device, {adjoint_mesh(ev->mesh, conv, nullptr)}, {ev->mesh}, ev->integ, seed, K));
    return adjoint_run(S, ev->stream, loss, dLdX);
}

int i2_evaluator_adjoint_ms(const i2_evaluator* ev, double* ms) {
    if (!ev || !ms) { set_error("null argument"); return I2_ERR_INVALID; }
    if (!ev->adj) { set_error("no adjoint run"); return I2_ERR_STATE; }
    *ms = ev->adj->ms;
    return I2_OK;
}

int i2_host_loss_weights(uint64_t seed, const int32_t* ij, int64_t n, int nT, double* out4) {
    if (!ij || !out4 || n < 0 || nT <= 0) { set_error("invalid argument"); return I2_ERR_INVALID; }
    for (int64_t q = 0; q < n; ++q) {
        const uint64_t pid = (uint64_t)ij[2 * q] * (uint64_t)nT + (uint64_t)ij[2 * q + 1];
        for (int s = 0; s < 4; ++s) out4[4 * q + s] = normal_draw(seed, pid, (uint64_t)s, &i2m::h_mathtab);
    }
    return I2_OK;
}

int i2_host_point_adjoint(int kind, const double* p3, const double* params, const double* gbar4, double* f4, double* pbar3,
                          double* parbar) {
    if (!p3 || !params || !gbar4 || !f4 || !pbar3 || !parbar) { set_error("null argument"); return I2_ERR_INVALID; }
    const d3 p = {p3[0], p3[1], p3[2]};
    const q4 gb = {gbar4[0], gbar4[1], gbar4[2], gbar4[3]};
    auto v = [&](int o) { return d3{params[o], params[o + 1], params[o + 2]}; };
    auto put = [&](int o, d3 x) { parbar[o] = x.x; parbar[o + 1] = x.y; parbar[o + 2] = x.z; };
    const d3 z3 = {0.0, 0.0, 0.0};
    d3 pb;
    q4 f;
    if (kind == 0) {
        const JGeom J = make_jgeom(v(0), v(3), v(6), v(9), v(12), v(15));
        TPBar g = {z3, z3, z3, z3, z3, z3};
        f = theta_psi_fast_rev(p, J, &i2m::h_mathtab, gb, &pb, g);
        put(0, g.a); put(3, g.b); put(6, g.c); put(9, g.ta); put(12, g.tb); put(15, g.tc);
    } else if (kind == 1) {
        const EdgeCtx c = {v(0), v(3), v(6), v(9), v(12), params[15]};
        EdgeBar g = {z3, z3, z3, z3, z3, 0.0};
        f = sing_edge_rev(p, c, &i2m::h_mathtab, gb, &pb, g);
        g.ilvc /= c.ilvc;
        put(0, g.JB); put(3, g.JC); put(6, g.taua); put(9, g.taub); put(12, g.tauc); parbar[15] = g.ilvc;
    } else if (kind == 2) {
        const VertexCtx c = {v(0), v(3), v(6), v(9), params[12]};
        VertexBar g = {z3, z3, z3, z3, 0.0};
        f = sing_vertex_rev(p, c, &i2m::h_mathtab, gb, &pb, g);
        g.invAri /= c.invAri;
        put(0, g.JA); put(3, g.taua); put(6, g.taub); put(9, g.e); parbar[12] = g.invAri;
    } else if (kind >= 3 && kind <= 5) {
        const d3 A = v(0), B = v(3), C = v(6), cr = cross(B - A, C - A);
        const JGeom J = make_jgeom(A, B, C, unit(C - B), unit(A - C), unit(B - A));
        TermsBar g = terms_bar_zero();
        if (kind == 3) {
            pb = theta_terms_rev(p, J, &i2m::h_mathtab, 1.0, gb, g);
        } else {   // p as a point of a control panel of K_j's size and shape
            const FarPoint Q = far_point(0.3, -0.2, 1.0);
            const d3 o = p - ((Q.b0 + 1.0 / 3.0) * A + (Q.b1 + 1.0 / 3.0) * B + (1.0 / 3.0 - Q.b0 - Q.b1) * C);
            const FarFrame F = far_frame(A + o, B + o, C + o);
            const FarGeom G = far_geom(F, J);
            FarBar fb = far_bar_zero();
            if (kind == 4) theta_terms_far_rev<false>(Q, F, G, J, gb, fb);
            else theta_terms_far_rev<true>(Q, F, G, J, gb, fb);
            d3 X0 = z3, X1 = z3;
            far_bar_expand(fb, F, J, g, X0, X1);
            pb = g.a + g.b + g.c;
            axpy(pb, g.y, J.N2);
        }
        f = g.T;
        g.T = q4zero();
        d3 ab, bb, cb;
        terms_chain(J, gb, g, z3, z3, 1.0 / J.La, 1.0 / J.Lb, 1.0 / J.Lc, 1.0 / vlen(cr), unit(cr), ab, bb, cb);
        put(0, ab); put(3, bb); put(6, cb);
    } else {
        set_error("unknown point function %d", kind);
        return I2_ERR_INVALID;
    }
    f4[0] = f.x; f4[1] = f.y; f4[2] = f.z; f4[3] = f.w;
    pbar3[0] = pb.x; pbar3[1] = pb.y; pbar3[2] = pb.z;
    return I2_OK;
}

}  // extern "C"
