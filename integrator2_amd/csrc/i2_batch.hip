// i2_batch.hip -- the batched persistent path: many meshes, all three
// neighbour types and every refinement level in one captured HIP graph of
// persistent kernels fed by device work queues.
//
// Semantics are those of EvaluatorJ3DK::numericalIntegration
// (src/evaluators/evaluatorJ3DK.cu:895-1012) applied per mesh and type: level
// 0, then iterations 1..maxLevel comparing consecutive levels by the Runge rule
// (src/evaluators/evaluator3d.cu:76-99).  A task's levels depend only on the
// task itself, so each task walks its own refinement levels; the only global
// quantity, the number of iterations K of a (mesh, type), is derived on the
// device from the levels the queues reached, and the reference's swapped
// result buffers (src/evaluators/evaluatorJ3DK.cu:976-990) are reproduced from
// each task's last two level values in the finalize kernel.
//
// Kernels (one graph):
//   k_sweep_disjoint  levels 0 and 1 of the disjoint pairs, enumerated implicitly:
//              an item is one control panel i and P consecutive panels j (i is
//              uniform, its panel record is read with scalar loads); lane
//              groups of LPP lanes share a pair and split its quadrature
//              points.  Persistent workgroups take runs of consecutive items,
//              the first by their number and the next from an atomic counter.
//   k_singular_closed, k_sweep_singular  closed forms, then levels 0 and 1, of the
//              vertex- and edge-sharing tasks from the meshes' lists, on a
//              second stream beside the disjoint pairs' kernels.
//   k_deep     refinement level L >= 2 of the tasks queued by level L-1: 16 or
//              64 lanes per task, fixed-order reduction.
//   k_levels / k_compute_K   K per (mesh, type) from queue membership.
//   per-pair outputs (value, J) are written by the task's last kernel for
//   K = maxLevel; k_finalize_pairs corrects the types whose K differs by an odd
//   number; k_finalize_rows   row sums for K's parity.
#include "i2_batch.hpp"
#include "i2_adjoint.hpp"

#include <algorithm>
#include <cstring>

namespace i2 {
using namespace i2d;

// ------------------------------------------------------------ device helpers
__device__ __forceinline__ int64_t uniform64(int64_t x) {
    const int lo = __builtin_amdgcn_readfirstlane((int)(x & 0xffffffff));
    const int hi = __builtin_amdgcn_readfirstlane((int)(x >> 32));
    return ((int64_t)hi << 32) | (uint32_t)lo;
}

// Task index of the ordered disjoint pair (i, j), i uniform over the workgroup,
// in [(i<j) list] ++ [reversed]: the pair's place in the row of its smaller
// panel, whose neighbours are no disjoint pairs.  Row i is the same for all
// lanes; with the general loop over 64-bit positions a pair took 130
// instructions for it.
__device__ __forceinline__ int64_t disjoint_task(const MeshDesc& M, int i, int j) {
    int below = 0;
    if (i < j) {
        for (int64_t q = M.nbr_start[i]; q < M.nbr_start[i + 1]; ++q) below += M.nbr[q] < j;
        return M.row_start[i] + (j - i - 1) - below;
    }
    const int64_t first = M.nbr_start[j];
    const int32_t* nbr = M.nbr + first;
    for (int n = (int)(M.nbr_start[j + 1] - first); below < n && nbr[below] < i; ++below) {}
    return M.npairs[I2_NOT_NEIGHBORS] + M.row_start[j] + (i - j - 1) - below;
}

__device__ __forceinline__ int find_base(const int64_t* base, int n, int64_t x) {
    int lo = 0, hi = n - 1;   // largest b < n with base[b] <= x
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (base[mid] <= x) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ JGeom jgeom(const Panel& P) { return make_jgeom(P.a, P.b, P.c, P.ta, P.tb, P.tc); }

template <int TYPE> struct Sing;
template <> struct Sing<I2_NOT_NEIGHBORS> {
    __device__ __forceinline__ void init(const Panel&, const Panel&) {}
    __device__ __forceinline__ q4 at(d3, const i2m::MathTable*) const { return q4zero(); }
};
template <> struct Sing<I2_ATTACHED_NEIGHBORS> {
    EdgeCtx c;
    __device__ __forceinline__ void init(const Panel& I, const Panel& J) {
        int s1, s2;
        shifts_edge(I, J, &s1, &s2);
        c = edge_ctx(vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3));
    }
    __device__ __forceinline__ q4 at(d3 p, const i2m::MathTable* lt) const { return sing_edge_fast(p, c, lt); }
};
template <> struct Sing<I2_SIMPLE_NEIGHBORS> {
    VertexCtx c;
    __device__ __forceinline__ void init(const Panel& I, const Panel& J) {
        int s1, s2;
        shifts_vertex(I, J, &s1, &s2);
        c = vertex_ctx(vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3), I.n, J.n, I.area);
    }
    __device__ __forceinline__ q4 at(d3 p, const i2m::MathTable* lt) const { return sing_vertex_fast(p, c, lt); }
};

// closed-form singular integral of a task (evaluatorJ3DK.cu:603-780)
__device__ __noinline__ q4 singular_integral(int type, const Panel& I, const Panel& J) {
    int s1, s2;
    if (type == I2_ATTACHED_NEIGHBORS) {
        shifts_edge(I, J, &s1, &s2);
        return integrate_sing_edge(vtx(I, s1), vtx(I, (s1 + 1) % 3), vtx(I, (s1 + 2) % 3),
                                   vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3), I.n, J.n, I.area);
    }
    shifts_vertex(I, J, &s1, &s2);
    return integrate_sing_vertex(vtx(I, s1), vtx(I, (s1 + 1) % 3), vtx(I, (s1 + 2) % 3),
                                 vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3), I.n, J.n, I.area);
}

// Rule held in LDS: (L1, L2, L3, w) per point, and the log reduction table
struct RuleLDS {
    double L1[MAX_POINTS], L2[MAX_POINTS], L3[MAX_POINTS], w[MAX_POINTS];
    i2m::MathTable lt;
};

__device__ __forceinline__ void load_rule(RuleLDS& s, const Rule& R) {
    for (int k = threadIdx.x; k < MAX_POINTS; k += blockDim.x) {
        s.L1[k] = R.L1[k]; s.L2[k] = R.L2[k]; s.L3[k] = R.L3[k]; s.w[k] = R.w[k];
    }
    i2m::fill_mathtab(s.lt);
}

// Partial quadrature sum_k w_k f(r_k) of one sub-panel over points k = s,
// s + step, ...  Disjoint pairs: the inner integral's terms, converted to (Psi,
// Theta) once per task by the caller.
template <int TYPE>
__device__ __forceinline__ q4 quad_part(const RuleLDS& R, int npts, int s, int step, d3 a, d3 b, d3 c, const JGeom& J,
                                        const Sing<TYPE>& sg) {
    q4 acc = q4zero();
    for (int k = s; k < npts; k += step) {
        d3 p = R.L1[k] * a;
        p = p + R.L2[k] * b;
        p = p + R.L3[k] * c;
        q4 f;
        if (TYPE == I2_NOT_NEIGHBORS) f = theta_terms(p, J, &R.lt);
        else f = theta_psi_fast(p, J, &R.lt) - sg.at(p, &R.lt);
        acc = acc + R.w[k] * f;
    }
    return acc;
}

// Quadrature points of a disjoint item's control panel K_i (uniform over the
// workgroup): the level-0 panel and its four level-1 children, in the order
// sweep_task sums them, computed once per item instead of once per pair.  Each
// point is a 32-byte record, two 128-bit LDS reads: |b0 U + b1 V|^2, (b0, b1)
// and the rule weight.
struct alignas(32) QPoint { double pp, b0, b1, w; };
// The panel's frame stands beside them: read where it is used (the index's empty
// statement keeps the reads there) it is not held in registers across the loops,
// which left 27 of them to spill, four so.  Rows of 5,120 panels 6.15 -> 6.09 ms.
struct PtsLDS {
    QPoint f[5 * MAX_POINTS];
    FarFrame F;
    __device__ __forceinline__ FarFrame frame() const {
        int again = 0;
        asm volatile("" : "+v"(again));
        return (&F)[again];
    }
};

// Levels 0 and 1 in one pass with a rule whose point 0 is the centroid: the
// centroid of K_i is also the centroid of its central level-1 child (child 4),
// so the integrand there is evaluated once, at child 4's point (the rule's
// literals put the two points 5e-16 edge lengths apart), and enters both sums.
__device__ __forceinline__ bool share_centroid(const BatchArgs& A) {
    return A.rule.centroid == 0 && !A.fixed && A.last_level >= 1;
}

__device__ __forceinline__ void load_points(PtsLDS& P, const Rule& R, const FarFrame& F) {
    const int npts = R.n;
    for (int t = threadIdx.x; t < 5 * npts; t += blockDim.x) {
        const BaryPoint Q = bary_point(R.L1, R.L2, R.L3, R.w, npts, t);
        const FarPoint x = far_point(Q.b0 - 1.0 / 3.0, Q.b1 - 1.0 / 3.0, Q.w);
        P.f[t] = {far_pp(F, x), x.b0, x.b1, x.w};
    }
    if (threadIdx.x == 0) P.F = F;
}

// The ways a wavefront evaluates the terms (forms of wave_form).  General: at
// the point itself.  Far: from the panel's own distance polynomials.  Shared:
// as far, with the distances of a tile's vertices computed once per vertex
// instead of once per panel corner.  sum() adds w times the terms of points k =
// k0, k0 + step, ... < k1 to acc, in that order.
struct GeneralTerms {
    const i2m::MathTable& lt;
    const PtsLDS& P;
    const JGeom& J;
    __device__ __forceinline__ q4 sum(int k0, int k1, int step, q4 acc) const {
        for (int k = k0; k < k1; k += step) {
            const QPoint Q = P.f[k];
            const FarFrame F = P.frame();
            const q4 t = theta_terms(F.o + (F.g + Q.b0 * F.U + Q.b1 * F.V), J, &lt);
            acc = {fma(Q.w, t.x, acc.x), fma(Q.w, t.y, acc.y), fma(Q.w, t.z, acc.z), fma(Q.w, t.w, acc.w)};
        }
        return acc;
    }
};
template <bool DISTANT>
struct FarTerms {
    const PtsLDS& P;
    const FarGeom& G;
    __device__ __forceinline__ q4 sum(int k0, int k1, int step, q4 acc) const {
        for (int k = k0; k < k1; k += step) {
            const QPoint Q = P.f[k];
            const q4 t = theta_terms_far<DISTANT>(Q.b0, Q.b1, Q.pp, G);
            acc = {fma(Q.w, t.x, acc.x), fma(Q.w, t.y, acc.y), fma(Q.w, t.z, acc.z), fma(Q.w, t.w, acc.w)};
        }
        return acc;
    }
};
// 64 consecutive panels of a mesh in a local order have some 45 to 66 vertices
// against 192 corners.  Four points at a time, lane v writes the distance of
// vertex v (and v + 64) to the wavefront's table in LDS, and each panel reads
// its three: 65 FP64 instructions per evaluation instead of 83, and three LDS
// reads.  One wavefront's LDS operations complete in order, so that the writes
// and the reads need no barrier, only wave_exchange.  Rows of 5,120 panels 6.75 -> 6.28
// ms, at 84 % of the issue slots instead of 94; the chip's clock follows the
// load (1.82 and 1.89 GHz), and two or three wavefronts per SIMD give the same.
constexpr int TILE_POINTS = 4;
// Orders a wavefront's LDS accesses before and after it, for the compiler as
// well: the fences are of one wavefront's scope and emit no instruction.
__device__ __forceinline__ void wave_exchange() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <bool DISTANT>
struct SharedTerms {
    const PtsLDS& P;
    const FarGeom& G;
    double* table;           // TILE_POINTS x TILE_VERTS
    VertexPoly v0, v1;       // this lane's vertices
    bool two;                // more than 64 of them (uniform)
    uint32_t corners;
    // N points from k on
    template <int N>
    __device__ __forceinline__ q4 points(int k, q4 acc) const {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int p = 0; p < N; ++p) {
            const QPoint Q = P.f[k + p];
            table[p * TILE_VERTS + lane] = vertex_distance(v0, Q.b0, Q.b1, Q.pp);
        }
        if (two && lane < TILE_VERTS - 64) {
#pragma unroll
            for (int p = 0; p < N; ++p) {
                const QPoint Q = P.f[k + p];
                table[p * TILE_VERTS + 64 + lane] = vertex_distance(v1, Q.b0, Q.b1, Q.pp);
            }
        }
        wave_exchange();
        const double *a = table + (corners & 255u), *b = table + ((corners >> 8) & 255u), *c = table + (corners >> 16);
#pragma unroll
        for (int p = 0; p < N; ++p) {
            const QPoint Q = P.f[k + p];
            const q4 t = theta_terms_of<DISTANT>(a[p * TILE_VERTS], b[p * TILE_VERTS], c[p * TILE_VERTS], Q.b0, Q.b1, G);
            acc = {fma(Q.w, t.x, acc.x), fma(Q.w, t.y, acc.y), fma(Q.w, t.z, acc.z), fma(Q.w, t.w, acc.w)};
        }
        wave_exchange();
        return acc;
    }
    __device__ __forceinline__ q4 sum(int k0, int k1, int, q4 acc) const {
        int k = k0;
        for (; k + TILE_POINTS <= k1; k += TILE_POINTS) acc = points<TILE_POINTS>(k, acc);
        for (; k < k1; ++k) acc = points<1>(k, acc);
        return acc;
    }
};
// Sums of the terms over level 0 (T0) and level 1 (T1) of a pair, lane s of LPP.
template <int LPP, class Terms>
__device__ __forceinline__ void sweep_terms(const Terms& E, int npts, bool share, bool need0, bool need1, int s, q4& T0, q4& T1) {
    int k0 = s, k1 = npts + s;
    if (share) {
        // point 0 of child 4 stands for point 0 of level 0 as well (lane 0 takes both)
        if (s == 0) {
            T0 = E.sum(4 * npts, 4 * npts + 1, 1, q4zero());
            T1 = T0;
            k0 = LPP;
        }
        // children 1 to 3 and child 4's other points around the shared one
        T0 = E.sum(k0, npts, LPP, T0);
        T1 = E.sum(k1, 4 * npts, LPP, T1);
        T1 = E.sum(4 * npts + k0, 5 * npts, LPP, T1);
        return;
    }
    if (need0) T0 = E.sum(k0, npts, LPP, T0);
    if (need1) T1 = E.sum(k1, 5 * npts, LPP, T1);
}

__device__ __forceinline__ q4 shfl_sum(q4 v, int G) {
    for (int m = 1; m < G; m <<= 1) {
        v.x += __shfl_xor(v.x, m);
        v.y += __shfl_xor(v.y, m);
        v.z += __shfl_xor(v.z, m);
        v.w += __shfl_xor(v.w, m);
    }
    return v;
}

// Result of one task step: finished at iteration c with I_c = cur and the
// value the reference's other buffer holds, prev (= I_{c-1}; = I_c when no
// comparison applies or the buffer swap is not reproduced).
struct StepOut {
    bool finished;
    bool pushed;
    int c;
    q4 cur, prev;
    bool unconv = false;   // finished at maxLevel with the Runge criterion above the tolerance
};

__device__ __forceinline__ void push_deep(const BatchArgs& A, int level, int type, int m, int i, int j, int64_t z, q4 prev) {
    const int qi = level * 3 + type;
    const unsigned long long slot = atomicAdd(&A.counters[1 + qi], 1ull);
    if (slot >= (unsigned long long)A.qcap[type]) {
        // counted: the host grows the queue and runs again.  No kernel finishes
        // the task in this run, but the adjoint of the same graph reads its
        // convergence iteration as a refinement level: it gets a valid one.
        int8_t* conv = A.meshes[m].conv[type];
        if (conv) conv[z] = 0;
        return;
    }
    QEntry e;
    e.m = m; e.i = i; e.j = j; e.pad = 0; e.z = z; e.pad2 = 0;
    e.prev = make_double4(prev.x, prev.y, prev.z, prev.w);
    A.queue[A.qoff[qi] + (int64_t)slot] = e;
}

// Writes a finished task: per-pair arrays, or its contribution to the row sums
// of both parities of K (returned in rp0/rp1 as (J, Theta)).
// Per-pair outputs are written for K = maxLevel (the fixed level in fixed
// mode), which is K whenever any task of the type reaches maxLevel: fin holds
// the value the buffer swap reports for that K, prev the other one, res its J.
// Where K turns out smaller by an odd number, the finalize kernels swap the two
// and recompute J.
template <int TYPE, int OUT>
__device__ __forceinline__ void finish_task(const BatchArgs& A, const MeshDesc& M, int64_t z, int i, int j, const StepOut& o,
                                            const Panel& I, const Panel& J, q4* rp0, q4* rp1) {
    q4 cur = o.cur, prev = o.prev;
    if (TYPE != I2_NOT_NEIGHBORS) {
        const double4 s4 = M.sing_val[TYPE][z];
        const q4 s = {s4.x, s4.y, s4.z, s4.w};
        cur = cur + s;
        prev = prev + s;
    }
    if (OUT == OUT_PER_PAIR) {
        const bool swap = A.quirk && o.c >= 1 && ((A.last_level - o.c) & 1);
        const q4 rep = swap ? prev : cur, other = swap ? cur : prev;
        M.fin[TYPE][z] = make_double4(rep.x, rep.y, rep.z, rep.w);
        M.prev[TYPE][z] = make_double4(other.x, other.y, other.z, other.w);
        M.conv[TYPE][z] = (int8_t)o.c;
        if (o.unconv && M.unconv[TYPE]) M.unconv[TYPE][i] = 1;
        // the panel records are re-read here so that no panel data stays live
        // across the quadrature loop
        const d3 nJ = M.panels[j].n;
        const d3 r = (TYPE == I2_SIMPLE_NEIGHBORS) ? finalize_vertex(rep, nJ, M.panels[i].area) : finalize_plain(rep, nJ);
        double* out = M.res[TYPE] + 3 * z;
        out[0] = r.x; out[1] = r.y; out[2] = r.z;
    } else {
        if (M.conv[TYPE]) M.conv[TYPE][z] = (int8_t)o.c;   // kept for the adjoint
        // K even selects I_c for even c, I_{c-1} for odd c; K odd the opposite
        const q4 v0 = ((o.c & 1) == 0) ? cur : prev;
        const q4 v1 = ((o.c & 1) == 1) ? cur : prev;
        const d3 r0 = (TYPE == I2_SIMPLE_NEIGHBORS) ? finalize_vertex(v0, J.n, I.area) : finalize_plain(v0, J.n);
        const d3 r1 = (TYPE == I2_SIMPLE_NEIGHBORS) ? finalize_vertex(v1, J.n, I.area) : finalize_plain(v1, J.n);
        *rp0 = {r0.x, r0.y, r0.z, v0.w};
        *rp1 = {r1.x, r1.y, r1.z, v1.w};
    }
}

__device__ __forceinline__ void add_row(const MeshDesc& M, int type, int i, q4 rp0, q4 rp1) {
    double* a0 = M.rowacc + (((size_t)type * 2 + 0) * M.nT + i) * 4;
    double* a1 = M.rowacc + (((size_t)type * 2 + 1) * M.nT + i) * 4;
    atomicAdd(a0 + 0, rp0.x); atomicAdd(a0 + 1, rp0.y); atomicAdd(a0 + 2, rp0.z); atomicAdd(a0 + 3, rp0.w);
    atomicAdd(a1 + 0, rp1.x); atomicAdd(a1 + 1, rp1.y); atomicAdd(a1 + 2, rp1.z); atomicAdd(a1 + 3, rp1.w);
}

// The Runge check of a task after its levels 0 and 1 (v0, v1).
template <int TYPE>
__device__ __forceinline__ StepOut sweep_check(const BatchArgs& A, int m, int i, int j, int64_t z, q4 v0, q4 v1) {
    StepOut o{false, false, 0, v0, v0};
    if (A.fixed) {
        if (A.last_level <= 1) { o.finished = true; o.c = A.last_level; o.cur = o.prev = (A.last_level == 0 ? v0 : v1); }
        else { push_deep(A, A.last_level, TYPE, m, i, j, z, v1); o.pushed = true; }
        return o;
    }
    if (A.last_level == 0) { o.finished = true; o.c = 0; o.cur = o.prev = v0; return o; }
    const double crit = runge_criterion(v1, v0, A.rule.pow2p);
    if (!(crit > A.tol) || A.last_level == 1) { o.finished = true; o.c = 1; o.cur = v1; o.prev = A.quirk ? v0 : v1; o.unconv = crit > A.tol; }
    else { push_deep(A, 2, TYPE, m, i, j, z, v1); o.pushed = true; }
    return o;
}

// A row's sums of the wavefront's lanes (or the whole smaller workgroup's), one
// set of atomics; the lanes' shares are cleared.
__device__ __forceinline__ void flush_row(const MeshDesc& M, int type, int i, q4& acc0, q4& acc1) {
    const int W = blockDim.x < 64 ? (int)blockDim.x : 64;
    acc0 = shfl_sum(acc0, W);
    acc1 = shfl_sum(acc1, W);
    if ((threadIdx.x & (W - 1)) == 0) add_row(M, type, i, acc0, acc1);
    acc0 = q4zero();
    acc1 = q4zero();
}

// The sums of a wavefront's pairs by the tile's shared distances; all 64 lanes
// take part.
template <bool DISTANT>
__device__ __forceinline__ void shared_sums(const BatchArgs& A, const PtsLDS& pts, const MeshDesc& M, int tile, uint32_t corners,
                                            double* table, const JGeom& JG, bool need0, bool need1, q4& T0,
                                            q4& T1) {
    const int32_t* list = M.tile_list + (int64_t)tile * TILE_LIST;
    const int lane = threadIdx.x & 63, n = list[0];
    const FarFrame F = pts.frame();
    auto vertex = [&](int k) {
        const double* x = M.xyz + 3 * (int64_t)list[1 + (k < n ? k : 0)];
        return vertex_poly(F, d3{x[0], x[1], x[2]});
    };
    const FarGeom G = far_geom(F, JG);
    const SharedTerms<DISTANT> E{pts, G, table, vertex(lane), vertex(lane + 64), n > 64, corners};
    sweep_terms<1>(E, A.rule.n, share_centroid(A), need0, need1, 0, T0, T1);
    T0 = far_scale(T0, JG);
    T1 = far_scale(T1, JG);
}

// Levels 0 and 1 of one disjoint task (lane group of LPP lanes), then the Runge
// check.  table: of the wavefront, whose pairs are with tile `tile` of the mesh
// (null: their panels are not one tile).
template <int LPP>
__device__ __forceinline__ StepOut sweep_task(const BatchArgs& A, const i2m::MathTable& lt, const MeshDesc& M, int m, int i, int j, int64_t z,
                                              bool valid, int s, const Panel& I, const Panel& J, const PtsLDS& pts, const Ball& ball,
                                              double* table, int tile) {
    const JGeom JG = jgeom(J);
    const int npts = A.rule.n;
    const bool need0 = !A.fixed || A.last_level == 0;
    const bool need1 = A.fixed ? A.last_level == 1 : A.last_level >= 1;
    q4 v0 = q4zero(), v1 = q4zero();
    // one loop per wavefront, in the form that holds for all its pairs
    const int form = wave_form(valid, ball, JG);
    q4 T0 = q4zero(), T1 = q4zero();
    if (LPP == 1 && form != 0 && table && M.tile_list[(int64_t)tile * TILE_LIST] > 0) {
        const uint32_t corners = M.corners[min(j, M.nT - 1)];
        if (form == 1) shared_sums<false>(A, pts, M, tile, corners, table, JG, need0, need1, T0, T1);
        else shared_sums<true>(A, pts, M, tile, corners, table, JG, need0, need1, T0, T1);
    } else if (valid) {
        if (form == 0) {
            sweep_terms<LPP>(GeneralTerms{lt, pts, JG}, npts, share_centroid(A), need0, need1, s, T0, T1);
        } else {
            const FarGeom G = far_geom(pts.frame(), JG);
            if (form == 1) sweep_terms<LPP>(FarTerms<false>{pts, G}, npts, share_centroid(A), need0, need1, s, T0, T1);
            else sweep_terms<LPP>(FarTerms<true>{pts, G}, npts, share_centroid(A), need0, need1, s, T0, T1);
            T0 = far_scale(T0, JG);
            T1 = far_scale(T1, JG);
        }
    }
    if (valid) {
        v0 = I.area * psi_of_terms(T0, JG);
        v1 = (0.25 * I.area) * psi_of_terms(T1, JG);
    }
    if (LPP > 1) {
        v0 = shfl_sum(v0, LPP);
        v1 = shfl_sum(v1, LPP);
    }
    if (!valid || s != 0) return StepOut{false, false, 0, v0, v0};
    return sweep_check<I2_NOT_NEIGHBORS>(A, m, i, j, z, v0, v1);
}

// Disjoint pairs, levels 0 and 1: item = (mesh, control panel i, P consecutive j),
// processed in rounds of blockDim/LPP pairs.  A workgroup claims A.sweep_chunk
// consecutive items at a time (the first by its number, without an atomic):
// claims of single items queue on one address, 129 against 92 us for 320
// panels at 4 lanes per pair and 3 % for 5,120 at one.  Consecutive items
// mostly share the control panel, whose points and row sums are then kept from
// one to the next.
template <int OUT, int LPP>
__global__ __launch_bounds__(256) I2_THREE_WAVES void k_sweep_disjoint(BatchArgs A) {
    __shared__ struct { PtsLDS pts; i2m::MathTable lt; } S;
    PtsLDS& pts = S.pts;
    __shared__ long long chunk_sh;
    extern __shared__ double wave_tables[];   // one table per wavefront, where each has a tile (tile_table_bytes)
    i2m::fill_mathtab(S.lt);
    const int P = A.pairs_per_item;
    double* const tables = LPP == 1 && P % 64 == 0 ? wave_tables : nullptr;
    const int per_round = blockDim.x / LPP;
    const int p0 = threadIdx.x / LPP, s = threadIdx.x % LPP;
    const int64_t chunks = (A.disjoint_items + A.sweep_chunk - 1) / A.sweep_chunk;
    for (int64_t chunk = blockIdx.x; chunk < chunks;) {
        const int64_t first = chunk * A.sweep_chunk, last = min(first + A.sweep_chunk, A.disjoint_items);
        int m = __builtin_amdgcn_readfirstlane(find_base(A.item_base, A.nmeshes, first));
        int i = -1, i_mesh = -1;
        q4 acc0 = q4zero(), acc1 = q4zero();   // this lane's share of row i's sums, for both parities of K
        for (int64_t item = first; item < last; ++item) {
            while (m + 1 < A.nmeshes && item >= A.item_base[m + 1]) ++m;
            const MeshDesc& M = A.meshes[m];
            const int64_t r = item - A.item_base[m];
            const int tiles = (M.nT + P - 1) / P;
            const int row = __builtin_amdgcn_readfirstlane((int)(r / tiles));
            const int tile = (int)(r - (int64_t)row * tiles);
            const Panel I = M.panels[row];
            if (row != i || m != i_mesh) {
                if (OUT == OUT_ROW_SUMS && i >= 0) flush_row(A.meshes[i_mesh], I2_NOT_NEIGHBORS, i, acc0, acc1);
                i = row;
                i_mesh = m;
                __syncthreads();
                load_points(pts, A.rule, far_frame(I.a, I.b, I.c));
                __syncthreads();
            }
            const Ball ball = panel_ball(I.a, I.b, I.c, A.rule.reach);
            for (int round = 0; round < P; round += per_round) {
                const int p = round + p0;
                const int j = tile * P + p;
                const bool in_range = p < P && j < M.nT;
                const Panel J = M.panels[in_range ? j : i];
                const bool valid = in_range && j != i && shared_count(I, J) == 0;
                // row sums alone need no place for the pair's own outputs
                const bool numbered = OUT == OUT_PER_PAIR || M.conv[I2_NOT_NEIGHBORS] != nullptr;
                const int64_t z = valid && numbered ? disjoint_task(M, i, j) : 0;
                const int tile64 = __builtin_amdgcn_readfirstlane((tile * P + p) >> 6);
                const StepOut o = sweep_task<LPP>(A, S.lt, M, m, i, j, z, valid, s, I, J, pts, ball,
                                                  tables && 64 * tile64 < M.nT ? tables + (threadIdx.x >> 6) * TILE_POINTS * TILE_VERTS : nullptr,
                                                  tile64);
                q4 rp0 = q4zero(), rp1 = q4zero();
                if (o.finished) finish_task<I2_NOT_NEIGHBORS, OUT>(A, M, z, i, j, o, I, J, &rp0, &rp1);
                if (OUT == OUT_ROW_SUMS) { acc0 = acc0 + rp0; acc1 = acc1 + rp1; }
            }
        }
        if (OUT == OUT_ROW_SUMS) flush_row(A.meshes[i_mesh], I2_NOT_NEIGHBORS, i, acc0, acc1);
        if (chunks <= (int64_t)gridDim.x) break;
        __syncthreads();
        if (threadIdx.x == 0) chunk_sh = (long long)gridDim.x + (long long)atomicAdd(&A.counters[0], 1ull);
        __syncthreads();
        chunk = uniform64(chunk_sh);
    }
}

// Vertex- and edge-sharing tasks, levels 0 and 1: G lanes per task, which
// split the 5 npts points of both levels.  What is done once per task (the
// singular part's context with its atan2, the panel records) is repeated by the
// group, some 1,000 instructions against 450 per point.  Bounds: with one
// lane per task the 65 points in series took 110-170 us whatever the mesh
// (320 panels: 59 wavefronts on 1,024 SIMDs).
template <int TYPE, int OUT, int G>
__device__ __forceinline__ void singular_sweep_task(const BatchArgs& A, const RuleLDS& R, const BaryPoint* pts, int m, int64_t z, int i,
                                                    int j, int s) {
    const MeshDesc& M = A.meshes[m];
    const Panel I = M.panels[i];
    const Panel J = M.panels[j];
    Sing<TYPE> sg;
    sg.init(I, J);
    const JGeom JG = jgeom(J);
    const int npts = A.rule.n;
    const bool need0 = !A.fixed || A.last_level == 0;
    const bool need1 = A.fixed ? A.last_level == 1 : A.last_level >= 1;
    const int k0 = need0 ? 0 : npts, k1 = need1 ? 5 * npts : npts;
    q4 v0 = q4zero(), v1 = q4zero();
    for (int k = k0 + s; k < k1; k += G) {
        const BaryPoint Q = pts[k];
        const d3 p = at_bary(Q, I.a, I.b, I.c);
        const q4 f = theta_psi_fast(p, JG, &R.lt) - sg.at(p, &R.lt);
        // not both with a weight of 0, which would carry one level's NaN into the other
        if (k < npts) v0 = v0 + Q.w * f;
        else v1 = v1 + Q.w * f;
    }
    v0 = I.area * shfl_sum(v0, G);
    v1 = (0.25 * I.area) * shfl_sum(v1, G);
    if (s != 0) return;
    const StepOut o = sweep_check<TYPE>(A, m, i, j, z, v0, v1);
    if (o.finished) {
        q4 rp0, rp1;
        finish_task<TYPE, OUT>(A, M, z, i, j, o, I, J, &rp0, &rp1);
        if (OUT == OUT_ROW_SUMS) add_row(M, TYPE, i, rp0, rp1);
    }
}
template <int OUT, int G>
__global__ __launch_bounds__(256) I2_TWO_WAVES void k_sweep_singular(BatchArgs A) {
    __shared__ RuleLDS R;
    __shared__ BaryPoint pts[5 * MAX_POINTS];
    load_rule(R, A.rule);
    __syncthreads();
    for (int t = threadIdx.x; t < 5 * A.rule.n; t += blockDim.x) pts[t] = bary_point(R.L1, R.L2, R.L3, R.w, A.rule.n, t);
    __syncthreads();
    const int s = threadIdx.x % G;
    const int64_t total = A.singular_items * 256, step = (int64_t)gridDim.x * (blockDim.x / G);
    for (int64_t g = (int64_t)blockIdx.x * (blockDim.x / G) + threadIdx.x / G; g < total; g += step) {
        const int b = find_base(A.sing_base, 2 * A.nmeshes, g >> 8);
        const int type = b / A.nmeshes == 0 ? I2_SIMPLE_NEIGHBORS : I2_ATTACHED_NEIGHBORS;
        const int m = b % A.nmeshes;
        const MeshDesc& M = A.meshes[m];
        const int64_t n = M.npairs[type];
        const int64_t z = (g >> 8) * 256 - A.sing_base[b] * 256 + (g & 255);
        if (z >= 2 * n) continue;
        const int64_t k = z < n ? z : z - n;
        int i = M.lists[type][3 * k], j = M.lists[type][3 * k + 1];
        if (z >= n) { const int t = i; i = j; j = t; }
        if (type == I2_SIMPLE_NEIGHBORS) singular_sweep_task<I2_SIMPLE_NEIGHBORS, OUT, G>(A, R, pts, m, z, i, j, s);
        else singular_sweep_task<I2_ATTACHED_NEIGHBORS, OUT, G>(A, R, pts, m, z, i, j, s);
    }
}

// Refinement level >= 2 of one queued task.
// G lanes, Q of them per sub-panel.  LEAN: the panels and the previous value are
// read again after the points instead of held across them (the index's empty
// statement keeps the compiler from joining the reads), which leaves 14-20
// registers to spill at three wavefronts per SIMD instead of 37-47.
template <int TYPE, int OUT, bool LEAN>
__device__ __forceinline__ void deep_task(const BatchArgs& A, const RuleLDS& R, int level, int G, int Q, int s,
                                          const QEntry* entry, bool valid) {
    const QEntry e = *entry;
    const MeshDesc& M = A.meshes[e.m];
    const Panel I = M.panels[e.i];
    const Panel J = M.panels[e.j];
    Sing<TYPE> sg;
    if (TYPE != I2_NOT_NEIGHBORS && valid) sg.init(I, J);
    const JGeom JG = jgeom(J);
    q4 acc = q4zero();
    if (valid) {
        double area = I.area;
        for (int l = 0; l < level; ++l) area *= 0.25;
        const uint32_t nsub = 1u << (2 * level);
        // A disjoint pair's form is its own, not its wavefront's: the queue's
        // order changes from run to run.  Refined pairs are near at tight
        // tolerances with the 13-point rule, but not at a fixed level or with
        // weaker rules: rows of 9,858 panels at fixed level 2 with 12 points
        // took 159 ms in the general form, 120 so.
        const int form = TYPE == I2_NOT_NEIGHBORS ? panel_far(panel_ball(I.a, I.b, I.c, A.rule.reach), JG) : 0;
        if (form != 0) {
            const FarFrame F = far_frame(I.a, I.b, I.c);
            const FarGeom FG = far_geom(F, JG);
            acc = area * far_scale(form == 1 ? quad_far<false>(R, A.rule.n, level, s / Q, G / Q, s % Q, Q, F, FG)
                                             : quad_far<true>(R, A.rule.n, level, s / Q, G / Q, s % Q, Q, F, FG), JG);
        } else {
            for (uint32_t c = s / Q; c < nsub; c += G / Q) {
                d3 a = I.a, b = I.b, cc = I.c;
                sub_panel(a, b, cc, level, c);
                acc = acc + area * quad_part<TYPE>(R, A.rule.n, s % Q, Q, a, b, cc, JG, sg);
            }
        }
    }
    acc = shfl_sum(acc, G);
    int again = 0;
    if (LEAN) asm volatile("" : "+v"(again));
    const Panel I1 = LEAN ? M.panels[e.i + again] : I, J1 = LEAN ? M.panels[e.j + again] : J;
    if (TYPE == I2_NOT_NEIGHBORS) acc = psi_of_terms(acc, LEAN ? jgeom(J1) : JG);
    if (!valid || s != 0) return;
    const double4 pv = LEAN ? entry[again].prev : e.prev;
    const q4 prev = {pv.x, pv.y, pv.z, pv.w};
    StepOut o{false, false, level, acc, acc};
    if (A.fixed) {
        o.finished = true;   // fixed mode queues tasks straight at the fixed level
    } else {
        const double crit = runge_criterion(acc, prev, A.rule.pow2p);
        if (!(crit > A.tol) || level == A.last_level) { o.finished = true; o.prev = A.quirk ? prev : acc; o.unconv = crit > A.tol; }
        else push_deep(A, level + 1, TYPE, e.m, e.i, e.j, e.z, acc);
    }
    if (o.finished) {
        q4 rp0, rp1;
        finish_task<TYPE, OUT>(A, M, e.z, e.i, e.j, o, I1, J1, &rp0, &rp1);
        if (OUT == OUT_ROW_SUMS) add_row(M, TYPE, e.i, rp0, rp1);
    }
}

// Refinement level L >= 2 of the queued tasks of the types in [t0, t1]: a
// wavefront per task from level 3 (a sub-panel per lane at level 3), at level 2
// 16 lanes per task, one sub-panel each, or a wavefront with four lanes per
// sub-panel where 16 lanes each would leave SIMDs empty (4 rounds of points
// instead of 13 in series, at 81 % of the lanes) and the rule has more than four
// points: with fewer there is no series to shorten, and a wavefront's tasks enter
// the next queue with one atomic, 26 ns each on its counter (320 panels' 3,780
// singular tasks with one point, all refined: 43 us with 16 lanes, 100 with 64).  A workgroup without a task
// ends before it loads the tables.  WAVES per SIMD: many disjoint tasks run with
// three (DEEP_THREE_WAVES), the others with two and nothing spilled.
template <int OUT, int T0, int T1, int WAVES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES))) void k_deep(BatchArgs A, int level) {
    __shared__ RuleLDS R;
    bool loaded = false;
    for (int type = T0; type <= T1; ++type) {
        const int qi = level * 3 + type;
        const unsigned long long cnt = min(A.counters[1 + qi], (unsigned long long)A.qcap[type]);
        const bool wide = level >= 3 || (cnt <= 8192 && A.rule.n > 4);
        const int G = wide ? 64 : 16, Q = level == 2 && wide ? 4 : 1;
        const int per_block = blockDim.x / G;
        if ((unsigned long long)blockIdx.x * per_block >= cnt) continue;   // uniform
        if (!loaded) {
            load_rule(R, A.rule);
            __syncthreads();
            loaded = true;
        }
        const int slot = threadIdx.x / G, s = threadIdx.x % G;
        const QEntry* q = A.queue + A.qoff[qi];
        for (unsigned long long base = (unsigned long long)blockIdx.x * per_block; base < cnt;
             base += (unsigned long long)gridDim.x * per_block) {
            const unsigned long long t = base + slot;
            const bool valid = t < cnt;
            const QEntry* e = q + (valid ? t : base);
            if (type == I2_NOT_NEIGHBORS) deep_task<I2_NOT_NEIGHBORS, OUT, WAVES == 3>(A, R, level, G, Q, s, e, valid);
            else if (type == I2_SIMPLE_NEIGHBORS) deep_task<I2_SIMPLE_NEIGHBORS, OUT, WAVES == 3>(A, R, level, G, Q, s, e, valid);
            else deep_task<I2_ATTACHED_NEIGHBORS, OUT, WAVES == 3>(A, R, level, G, Q, s, e, valid);
        }
    }
}

// Which meshes have tasks at each level >= 2: OR of mesh bits over the queues,
// reduced per wavefront, then per workgroup in LDS, before one atomic per
// workgroup and mask word (launched with one workgroup per CU: the atomics of
// all workgroups on one word are serialised).
__global__ __launch_bounds__(256) void k_levels(BatchArgs A) {
    __shared__ unsigned long long wg[MASK_WORDS];
    for (int L = 2; L <= A.last_level; ++L)
        for (int type = 0; type < 3; ++type) {
            const int qi = L * 3 + type;
            const unsigned long long cnt = min(A.counters[1 + qi], (unsigned long long)A.qcap[type]);
            if (cnt == 0) continue;   // uniform: the same counter for every thread
            const QEntry* q = A.queue + A.qoff[qi];
            if (threadIdx.x < MASK_WORDS) wg[threadIdx.x] = 0ull;
            __syncthreads();
            unsigned long long mask[MASK_WORDS];
            for (int w = 0; w < MASK_WORDS; ++w) mask[w] = 0ull;
            for (unsigned long long t = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; t < cnt;
                 t += (unsigned long long)gridDim.x * blockDim.x) {
                const int m = q[t].m;
                mask[m >> 6] |= 1ull << (m & 63);
            }
            for (int w = 0; w < MASK_WORDS; ++w) {
                unsigned long long v = mask[w];
                for (int o = 1; o < 64; o <<= 1) v |= __shfl_xor(v, o);
                if ((threadIdx.x & 63) == 0 && v) atomicOr(&wg[w], v);
            }
            __syncthreads();
            if (threadIdx.x < MASK_WORDS && wg[threadIdx.x]) atomicOr(&A.levelmask[qi * MASK_WORDS + threadIdx.x], wg[threadIdx.x]);
            __syncthreads();   // wg is cleared again for the next queue
        }
}

// K per (mesh, type): 0 when maxLevel = 0 (automatic) or no task; else the
// deepest level any of its tasks reached (at least 1).  Fixed mode: the level.
// With one mesh the queue counts say which levels were reached.
__global__ void k_compute_K(BatchArgs A) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= 3 * A.nmeshes) return;
    const int m = g / 3, type = g % 3;
    const bool any = A.meshes[m].npairs[type] > 0;
    int K = 0;
    if (A.fixed) K = A.last_level;
    else if (any && A.last_level >= 1) {
        K = 1;
        for (int L = 2; L <= A.last_level; ++L) {
            const bool reached = A.nmeshes == 1 ? A.counters[1 + L * 3 + type] != 0ull
                                                : (A.levelmask[(L * 3 + type) * MASK_WORDS + (m >> 6)] >> (m & 63)) & 1ull;
            if (reached) K = L;
        }
    }
    A.K[g] = K;
}

// Per-pair outputs were written for K = maxLevel.  Where the type's K differs
// from it by an odd number (the buffer swap reproduced), every task with
// c >= 1 reports the other level: fin and prev trade places and J is
// recomputed.  Otherwise nothing is left to do.
__device__ __forceinline__ bool needs_correction(const BatchArgs& A, int m, int type) {
    return A.quirk && ((A.K[3 * m + type] - A.last_level) & 1);
}
__device__ __forceinline__ void finalize_task(const BatchArgs& A, const MeshDesc& M, int m, int type, int64_t z, int i, int j) {
    if (M.conv[type][z] < 1) return;
    const double4 a = M.fin[type][z], b = M.prev[type][z];
    M.fin[type][z] = b;
    M.prev[type][z] = a;
    const q4 v = {b.x, b.y, b.z, b.w};
    const d3 nJ = M.panels[j].n;
    const d3 r = (type == I2_SIMPLE_NEIGHBORS) ? finalize_vertex(v, nJ, M.panels[i].area) : finalize_plain(v, nJ);
    double* o = M.res[type] + 3 * z;
    o[0] = r.x; o[1] = r.y; o[2] = r.z;
}

// The closed-form singular integral of every vertex- and edge-sharing task, one
// task per lane (the task's last kernel adds it to the level value; a refinement
// kernel would otherwise evaluate it on one lane of each lane group).
__global__ __launch_bounds__(256) void k_singular_closed(BatchArgs A) {
    const int64_t total = A.singular_items * 256;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (int64_t)gridDim.x * blockDim.x) {
        const int64_t item = g >> 8;
        const int b = find_base(A.sing_base, 2 * A.nmeshes, item);
        const int type = b / A.nmeshes == 0 ? I2_SIMPLE_NEIGHBORS : I2_ATTACHED_NEIGHBORS;
        const MeshDesc& M = A.meshes[b % A.nmeshes];
        const int64_t n = M.npairs[type];
        const int64_t z = (item - A.sing_base[b]) * 256 + (g & 255);
        if (z >= 2 * n) continue;
        const int64_t k = z < n ? z : z - n;
        int i = M.lists[type][3 * k], j = M.lists[type][3 * k + 1];
        if (z >= n) { const int t = i; i = j; j = t; }
        const q4 s = singular_integral(type, M.panels[i], M.panels[j]);
        M.sing_val[type][z] = make_double4(s.x, s.y, s.z, s.w);
    }
}

// All tasks whose type needs the correction.  Vertex- and edge-sharing tasks
// are enumerated as the singular sweep's; disjoint ones by rows i of the
// lexicographic pair list, one per workgroup pass: the lanes walk its pairs
// (i, j), j > i, and finalize (i, j) and its reversed task (j, i), with j from
// i's sorted neighbour list (no search).
__global__ __launch_bounds__(256) void k_finalize_pairs(BatchArgs A) {
    if (!A.quirk) return;
    const int64_t total = A.singular_items * 256;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (int64_t)gridDim.x * blockDim.x) {
        const int64_t item = g >> 8;
        const int b = find_base(A.sing_base, 2 * A.nmeshes, item);
        const int type = b / A.nmeshes == 0 ? I2_SIMPLE_NEIGHBORS : I2_ATTACHED_NEIGHBORS;
        const int m = b % A.nmeshes;
        if (!needs_correction(A, m, type)) continue;
        const MeshDesc& M = A.meshes[m];
        const int64_t n = M.npairs[type];
        const int64_t z = (item - A.sing_base[b]) * 256 + (g & 255);
        if (z >= 2 * n) continue;
        const int64_t k = z < n ? z : z - n;
        int i = M.lists[type][3 * k], j = M.lists[type][3 * k + 1];
        if (z >= n) { const int t = i; i = j; j = t; }
        finalize_task(A, M, m, type, z, i, j);
    }
    for (int64_t r = blockIdx.x; r < A.total_rows; r += gridDim.x) {
        const int m = find_base(A.row_base, A.nmeshes, r);
        if (!needs_correction(A, m, I2_NOT_NEIGHBORS)) {
            r += (A.row_base[m + 1] - 1 - r) / gridDim.x * gridDim.x;   // on to the next mesh
            continue;
        }
        const MeshDesc& M = A.meshes[m];
        const int ii = (int)(r - A.row_base[m]);
        const int64_t k0 = M.row_start[ii], cnt = M.row_start[ii + 1] - k0;
        const int64_t n = M.npairs[I2_NOT_NEIGHBORS];
        const int64_t q0 = M.nbr_start[ii], q1 = M.nbr_start[ii + 1];
        for (int64_t t = threadIdx.x; t < cnt; t += blockDim.x) {
            int64_t jj = ii + 1 + t;
            for (int64_t q = q0; q < q1; ++q) {
                if (M.nbr[q] <= jj) ++jj; else break;
            }
            finalize_task(A, M, m, I2_NOT_NEIGHBORS, k0 + t, ii, (int)jj);
            finalize_task(A, M, m, I2_NOT_NEIGHBORS, n + k0 + t, (int)jj, ii);
        }
    }
}

// Row sums for K's parity, summed over the three types: (sum_j J, sum_j
// Theta), the rows of all meshes.
__global__ void k_finalize_rows(BatchArgs A) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= A.total_rows) return;
    const int m = find_base(A.row_base, A.nmeshes, r);
    const MeshDesc& M = A.meshes[m];
    const int i = (int)(r - A.row_base[m]);
    double v[4] = {0, 0, 0, 0};
    for (int type = 0; type < 3; ++type) {
        const int par = A.K[3 * m + type] & 1;
        const double* acc = M.rowacc + (((size_t)type * 2 + par) * M.nT + i) * 4;
        for (int c = 0; c < 4; ++c) v[c] += acc[c];
    }
    for (int c = 0; c < 4; ++c) M.rowout[4 * (size_t)i + c] = v[c];
}

// The start of a run: counters, level masks and, per row of every mesh, the row
// sums or the unconverged flags (by a kernel: a memset recorded in a graph can
// give wrong results on later replays).
__global__ __launch_bounds__(256) void k_begin(BatchArgs A) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t q = t; q < N_COUNTERS; q += step) A.counters[q] = 0ull;
    for (int64_t q = t; q < MAX_LEVELS * 3 * MASK_WORDS; q += step) A.levelmask[q] = 0ull;
    for (int64_t r = t; r < A.total_rows; r += step) {
        const int m = find_base(A.row_base, A.nmeshes, r);
        const MeshDesc& M = A.meshes[m];
        const int64_t i = r - A.row_base[m];
        if (M.rowacc)
            for (int c = 0; c < 6; ++c) {
                double* a = M.rowacc + ((size_t)c * M.nT + i) * 4;
                a[0] = 0.0; a[1] = 0.0; a[2] = 0.0; a[3] = 0.0;
            }
        for (int type = 0; type < 3; ++type)
            if (M.unconv[type]) M.unconv[type][i] = 0;
    }
}

// ------------------------------------------------------------ host engine
int lanes_for_points_per_lane(int ppl) {
    switch (ppl) {
        case 1: return 16;   // 13 points over 16 lanes
        case 2: return 8;
        case 4: return 4;
        default: return 1;   // the whole rule in one lane
    }
}

// workgroup of the disjoint sweep: P pairs of LPP lanes, at most 256 lanes
static int sweep_block(int P, int lpp) { return std::min(256, P * lpp); }

// dynamic LDS: a table per wavefront if the wavefronts' pairs are tiles of 64
static size_t tile_table_bytes(int P, int lpp) {
    return lpp == 1 && P % 64 == 0 ? sizeof(double) * TILE_POINTS * TILE_VERTS * (size_t)(sweep_block(P, lpp) / 64) : 0;
}

template <int OUT, int LPP>
static int sweep_grid_for(int P, int* grid) {
    int dev = 0, cus = 0, per = 0;
    I2_HIP(hipGetDevice(&dev));
    I2_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    I2_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_sweep_disjoint<OUT, LPP>, sweep_block(P, LPP), tile_table_bytes(P, LPP)));
    *grid = std::max(1, cus * std::max(1, per));
    return I2_OK;
}

static int launch_sweep(const Engine& E, hipStream_t st) {
    const int lpp = lanes_for_points_per_lane(E.ppl);
    const dim3 blk(sweep_block(E.pairs_per_wg, lpp)), grd(E.sweep_grid);
#define I2_SWEEP(O, L) hipLaunchKernelGGL((k_sweep_disjoint<O, L>), grd, blk, tile_table_bytes(E.pairs_per_wg, L), st, E.args)
    if (E.out == OUT_PER_PAIR) {
        if (lpp == 1) I2_SWEEP(OUT_PER_PAIR, 1); else if (lpp == 4) I2_SWEEP(OUT_PER_PAIR, 4);
        else if (lpp == 8) I2_SWEEP(OUT_PER_PAIR, 8); else I2_SWEEP(OUT_PER_PAIR, 16);
    } else {
        if (lpp == 1) I2_SWEEP(OUT_ROW_SUMS, 1); else if (lpp == 4) I2_SWEEP(OUT_ROW_SUMS, 4);
        else if (lpp == 8) I2_SWEEP(OUT_ROW_SUMS, 8); else I2_SWEEP(OUT_ROW_SUMS, 16);
    }
#undef I2_SWEEP
    I2_TRY(check_launch("k_sweep_disjoint"));
    if (E.prof1) I2_HIP(hipEventRecord(E.prof1, st));
    return I2_OK;
}

static int launch_sweep_singular(const Engine& E, hipStream_t st) {
    if (E.args.singular_items > 0) {
        // 16 lanes per task until that is about two rounds of the wavefronts the
        // chip holds (two per SIMD), then 4
        const bool few = E.args.singular_items <= 64;
        const int64_t blocks = E.args.singular_items * (few ? 16 : 4);
        const dim3 grid((unsigned)std::min<int64_t>(blocks, E.deep_grid));
#define I2_SING(O, G) hipLaunchKernelGGL((k_sweep_singular<O, G>), grid, dim3(256), 0, st, E.args)
        if (E.out == OUT_PER_PAIR) { if (few) I2_SING(OUT_PER_PAIR, 16); else I2_SING(OUT_PER_PAIR, 4); }
        else { if (few) I2_SING(OUT_ROW_SUMS, 16); else I2_SING(OUT_ROW_SUMS, 4); }
#undef I2_SING
        I2_TRY(check_launch("k_sweep_singular"));
    }
    return I2_OK;
}

static int compute_grids(Engine& E) {
    const int lpp = lanes_for_points_per_lane(E.ppl);
    if (E.pairs_per_wg < 1 || E.pairs_per_wg > 4096 || (E.pairs_per_wg * lpp > 256 && (E.pairs_per_wg * lpp) % 256 != 0)) {
        set_error("pairs per workgroup %d not usable with %d lanes per pair", E.pairs_per_wg, lpp);
        return I2_ERR_INVALID;
    }
#define I2_GRID(O, L) sweep_grid_for<O, L>(E.pairs_per_wg, &E.sweep_grid)
    if (E.out == OUT_PER_PAIR) {
        if (lpp == 1) I2_TRY(I2_GRID(OUT_PER_PAIR, 1)); else if (lpp == 4) I2_TRY(I2_GRID(OUT_PER_PAIR, 4));
        else if (lpp == 8) I2_TRY(I2_GRID(OUT_PER_PAIR, 8)); else I2_TRY(I2_GRID(OUT_PER_PAIR, 16));
    } else {
        if (lpp == 1) I2_TRY(I2_GRID(OUT_ROW_SUMS, 1)); else if (lpp == 4) I2_TRY(I2_GRID(OUT_ROW_SUMS, 4));
        else if (lpp == 8) I2_TRY(I2_GRID(OUT_ROW_SUMS, 8)); else I2_TRY(I2_GRID(OUT_ROW_SUMS, 16));
    }
#undef I2_GRID
    int dev = 0, cus = 0;
    I2_HIP(hipGetDevice(&dev));
    I2_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    E.deep_grid = cus * 8;
    E.fin_grid = cus * 16;
    E.levels_grid = cus;
    return I2_OK;
}

// Ordered disjoint pairs of a run from which k_deep takes three wavefronts per
// SIMD.  Row sums, refinement to level 3 at 1e-8: 1,280 panels (1.6e6 pairs)
// 1.052 ms with two, 1.004 with three, a 5,120-panel ellipsoid's outputs 7.81 and
// 7.74; 320 panels (1e5 pairs), where each SIMD has a wavefront at most, 0.304 and
// 0.315.  12 workgroups per CU with three: fixed level 2 on 5,120 panels 37.3 ms
// with two, 37.1 so, 39.2 with 8 per CU, whose last round is a third full.
constexpr int64_t DEEP_THREE_WAVES = 1 << 20;

int batch_enqueue(Engine& E, hipStream_t st) {
    const BatchArgs& A = E.args;
    const unsigned row_blocks = (unsigned)std::max<int64_t>(1, std::min<int64_t>((A.total_rows + 255) / 256, E.fin_grid));
    hipLaunchKernelGGL(k_begin, dim3(row_blocks), dim3(256), 0, st, A);
    I2_TRY(check_launch("k_begin"));
    // The singular pairs' kernels and the disjoint pairs' share nothing but their
    // inputs and go on two streams: on few panels each is latency, and on many
    // the refinement kernels of the one fill the other's tails.  The sweep goes
    // first, so that its persistent workgroups start together: rows of 5,120
    // panels 6.26 ms in one stream, 6.30 with the singular kernels first, 5.87.
    // A profiled run, which times the disjoint sweep, keeps them apart.
    const bool many = E.ordered[I2_NOT_NEIGHBORS] >= DEEP_THREE_WAVES;
    auto deep = [&](int L, bool singular, hipStream_t on) -> int {
        const dim3 grid(singular || !many ? E.deep_grid : E.deep_grid / 2 * 3);   // whole rounds of resident workgroups
#define I2_DEEP(O, T0, T1, W) hipLaunchKernelGGL((k_deep<O, T0, T1, W>), grid, dim3(256), 0, on, A, L)
        if (E.out == OUT_PER_PAIR) {
            if (singular) I2_DEEP(OUT_PER_PAIR, 0, 1, 2); else if (many) I2_DEEP(OUT_PER_PAIR, 2, 2, 3); else I2_DEEP(OUT_PER_PAIR, 2, 2, 2);
        } else {
            if (singular) I2_DEEP(OUT_ROW_SUMS, 0, 1, 2); else if (many) I2_DEEP(OUT_ROW_SUMS, 2, 2, 3); else I2_DEEP(OUT_ROW_SUMS, 2, 2, 2);
        }
#undef I2_DEEP
        return check_launch("k_deep");
    };
    const int first_deep = A.fixed ? std::max(2, A.last_level) : 2;   // fixed mode queues tasks at its level only
    const bool two = A.singular_items > 0 && !E.prof0;
    if (two) I2_TRY(E.side->fork(st));
    const hipStream_t sst = two ? E.side->stream : st;
    if (E.prof0) I2_HIP(hipEventRecord(E.prof0, st));
    I2_TRY(launch_sweep(E, st));
    if (A.singular_items > 0) {
        hipLaunchKernelGGL(k_singular_closed, dim3(E.deep_grid), dim3(256), 0, sst, A);
        I2_TRY(check_launch("k_singular_closed"));
        I2_TRY(launch_sweep_singular(E, sst));
        for (int L = first_deep; L <= A.last_level; ++L) I2_TRY(deep(L, true, sst));
    }
    for (int L = first_deep; L <= A.last_level; ++L) I2_TRY(deep(L, false, st));
    if (two) I2_TRY(E.side->join(st));
    if (A.last_level >= 2 && A.nmeshes > 1) {
        hipLaunchKernelGGL(k_levels, dim3(E.levels_grid), dim3(256), 0, st, A);
        I2_TRY(check_launch("k_levels"));
    }
    hipLaunchKernelGGL(k_compute_K, dim3((3 * A.nmeshes + 255) / 256), dim3(256), 0, st, A);
    I2_TRY(check_launch("k_compute_K"));
    if (E.out == OUT_PER_PAIR) {
        if (A.quirk) {
            const int64_t most = std::max<int64_t>({A.total_rows, A.singular_items, 1});
            hipLaunchKernelGGL(k_finalize_pairs, dim3((unsigned)std::min<int64_t>(most, E.fin_grid)), dim3(256), 0, st, A);
            I2_TRY(check_launch("k_finalize_pairs"));
        }
    } else {
        hipLaunchKernelGGL(k_finalize_rows, dim3((unsigned)((A.total_rows + 255) / 256)), dim3(256), 0, st, A);
        I2_TRY(check_launch("k_finalize_rows"));
    }
    return I2_OK;
}

// Launch shape for a caller who has set none: one lane per pair, or four while
// that leaves most SIMDs without a wavefront (1,024 SIMDs).  Row sums by shape,
// one / four lanes: 80 panels (160 wavefronts) 220 / 196 us, 320 panels (1,600)
// 295 / 312, 1,280 panels 840 / 1,090; eight and sixteen lanes are slower than
// four on all three.  Where there are many wavefronts, two share a control
// panel's points: 6,144 panels of a torus 8.14 -> 8.01 ms, 5,120 of a sphere
// 5.46 -> 5.40, with 3,000 (141,000 wavefronts) equal.
void engine_auto_shape(Engine& E) {
    int64_t waves = 0;
    for (const MeshDesc& D : E.h_meshes) waves += (int64_t)D.nT * ((D.nT + 63) / 64);
    E.ppl = waves >= 512 ? 13 : 4;
    E.pairs_per_wg = waves >= 65536 ? 128 : 64 / lanes_for_points_per_lane(E.ppl);
}

int engine_setup(Engine& E, const i2_integrator& it) {
    const int M = (int)E.h_meshes.size();
    if (M < 1 || M > MAX_BATCH_MESHES) { set_error("a batch holds 1..%d meshes", MAX_BATCH_MESHES); return I2_ERR_RANGE; }
    BatchArgs& A = E.args;
    A.nmeshes = M;
    A.fixed = it.fixed;
    A.last_level = it.fixed ? it.fixed_level : it.max_level;
    A.quirk = it.quirk;
    A.tol = it.tol;
    A.rule = it.rule;
    A.pairs_per_item = E.pairs_per_wg;
    if (A.last_level >= MAX_LEVELS) { set_error("refinement level above %d", MAX_LEVELS - 1); return I2_ERR_RANGE; }
    I2_TRY(compute_grids(E));
    const int P = E.pairs_per_wg;
    // sweep items (disjoint per mesh; singular per (type, mesh), 256 tasks each)
    E.h_item_base.assign(M + 1, 0);
    E.h_sing_base.assign(2 * M + 1, 0);
    E.nT.resize(M);
    int64_t acc = 0;
    for (int m = 0; m < M; ++m) {
        const MeshDesc& D = E.h_meshes[m];
        E.h_item_base[m] = acc;
        acc += (int64_t)D.nT * ((D.nT + P - 1) / P);
    }
    E.h_item_base[M] = acc;
    A.disjoint_items = acc;
    // items per claim: some 32 claims per workgroup, at most 64 items each;
    // without claims where every workgroup has a few items at most
    A.sweep_chunk = acc <= 4 * (int64_t)E.sweep_grid ? std::max<int64_t>(1, (acc + E.sweep_grid - 1) / E.sweep_grid)
                                                     : std::max<int64_t>(1, std::min<int64_t>(64, acc / (32 * (int64_t)E.sweep_grid)));
    acc = 0;
    for (int kind = 0; kind < 2; ++kind)
        for (int m = 0; m < M; ++m) {
            E.h_sing_base[kind * M + m] = acc;
            acc += (2 * E.h_meshes[m].npairs[kind] + 255) / 256;
        }
    E.h_sing_base[2 * M] = acc;
    A.singular_items = acc;
    if (acc > 0) I2_TRY(E.side->ensure());   // before any capture
    int64_t pb = 0;
    E.ordered[0] = E.ordered[1] = E.ordered[2] = 0;
    for (int m = 0; m < M; ++m) {
        E.nT[m] = E.h_meshes[m].nT;
        for (int t = 0; t < 3; ++t) {
            pb += 2 * E.h_meshes[m].npairs[t];
            E.ordered[t] += 2 * E.h_meshes[m].npairs[t];
        }
    }
    E.total_tasks = pb;
    E.h_row_base.assign(M + 1, 0);
    for (int m = 0; m < M; ++m) E.h_row_base[m + 1] = E.h_row_base[m] + E.h_meshes[m].nT;
    A.total_rows = E.h_row_base[M];
    // queue segments: levels 2..last, capacity per type (grown after an
    // overflow, which costs a second run).  Most vertex- and edge-sharing tasks
    // are refined at tight tolerances and there are few of them: room for all
    // up to 4 M (256 MB per level), where an eighth overflowed on the first run
    // of every mesh above some 7,000 panels.
    for (int t = 0; t < 3; ++t)
        if (A.qcap[t] <= 0) {
            const int64_t least = t == I2_NOT_NEIGHBORS ? 65536 : (int64_t)4 << 20;
            A.qcap[t] = std::max<int64_t>(1, std::min<int64_t>(E.ordered[t], std::max<int64_t>(least, E.ordered[t] / 8)));
        }
    E.h_qoff.assign(MAX_LEVELS * 3, 0);
    int64_t qtot = 0;
    for (int L = 2; L <= A.last_level; ++L)
        for (int t = 0; t < 3; ++t) { E.h_qoff[L * 3 + t] = qtot; qtot += A.qcap[t]; }
    I2_TRY(E.d_queue.ensure(std::max<int64_t>(1, qtot)));
    I2_TRY(E.d_counters.ensure(N_COUNTERS + (3 * M + 1) / 2));
    I2_TRY(E.d_levelmask.ensure(MAX_LEVELS * 3 * MASK_WORDS));
    // all tables in one upload (six took 70 us of every run on a mesh that moves)
    E.h_tables.clear();
    auto table = [&](const std::vector<int64_t>& v) {
        const size_t at = E.h_tables.size();
        E.h_tables.insert(E.h_tables.end(), v.begin(), v.end());
        return at;
    };
    const size_t qoff = table(E.h_qoff), items = table(E.h_item_base), sing = table(E.h_sing_base), rows = table(E.h_row_base), meshes = E.h_tables.size();
    static_assert(sizeof(MeshDesc) % sizeof(int64_t) == 0, "descriptors behind the tables");
    E.h_tables.resize(meshes + M * sizeof(MeshDesc) / sizeof(int64_t));
    memcpy(E.h_tables.data() + meshes, E.h_meshes.data(), M * sizeof(MeshDesc));
    I2_TRY(E.d_tables.ensure((int64_t)E.h_tables.size()));
    const int64_t* d = E.d_tables.p;
    I2_HIP(hipMemcpy(E.d_tables.p, E.h_tables.data(), sizeof(int64_t) * E.h_tables.size(), hipMemcpyHostToDevice));
    A.meshes = reinterpret_cast<const MeshDesc*>(d + meshes);
    A.item_base = d + items;
    A.sing_base = d + sing;
    A.row_base = d + rows;
    A.qoff = d + qoff;
    A.counters = E.d_counters.p;
    A.queue = E.d_queue.p;
    A.levelmask = E.d_levelmask.p;
    A.K = reinterpret_cast<int*>(E.d_counters.p + N_COUNTERS);   // behind the counters: one copy brings both to the host
    return I2_OK;
}

int engine_check_queues(Engine& E, hipStream_t st, bool* overflow, std::vector<unsigned long long>* counts, std::vector<int>* K) {
    const size_t nK = 3 * E.h_meshes.size(), bytes = sizeof(unsigned long long) * N_COUNTERS + sizeof(int) * nK;
    if (!E.h_sync) {
        const size_t most = sizeof(unsigned long long) * N_COUNTERS + sizeof(int) * 3 * MAX_BATCH_MESHES;
        I2_HIP(hipHostMalloc((void**)&E.h_sync, most, hipHostMallocDefault));
    }
    I2_HIP(hipMemcpyAsync(E.h_sync, E.d_counters.p, bytes, hipMemcpyDeviceToHost, st));
    I2_HIP(hipStreamSynchronize(st));
    const unsigned long long* c = E.h_sync;
    *overflow = false;
    int64_t need[3] = {0, 0, 0};
    for (int L = 2; L <= E.args.last_level; ++L)
        for (int t = 0; t < 3; ++t) need[t] = std::max<int64_t>(need[t], (int64_t)c[1 + L * 3 + t]);
    for (int t = 0; t < 3; ++t)
        if (need[t] > E.args.qcap[t]) { *overflow = true; E.args.qcap[t] = need[t] + need[t] / 4 + 1; }
    counts->assign(c, c + N_COUNTERS);
    const int* k = reinterpret_cast<const int*>(c + N_COUNTERS);
    K->assign(k, k + nK);
    return I2_OK;
}

}  // namespace i2

// ------------------------------------------------------------ i2_batch objects
struct i2_batch {
    int device = 0;
    hipStream_t stream = nullptr;
    std::vector<const i2_mesh*> meshes;
    std::vector<uint64_t> generations;   // each mesh's generation when the graph was built
    i2_integrator cfg{};
    bool have_cfg = false;
    int out = i2::OUT_PER_PAIR;
    int P = 64, ppl = 13;
    bool tuned = false;                  // the caller set the launch shape
    i2::Engine E;
    bool dirty = true;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    // owned outputs per mesh
    struct Out {
        i2::DBuf<double4> fin[3], prev[3];
        i2::DBuf<int8_t> conv[3];
        i2::DBuf<double> res[3];
        i2::DBuf<unsigned long long> unconv;   // per type and control panel: unconverged at maxLevel (bytes)
        i2::DBuf<double4> sing_val[2];         // closed-form singular integrals per singular task
        i2::DBuf<double> rowacc, rowout;
    };
    i2::SideStream own_side;
    i2::SideStream* side = &own_side;          // the evaluator's, for its engine
    std::vector<Out> outs;
    i2::DBuf<int32_t> tile_lists;              // MeshDesc::tile_list of all meshes
    i2::DBuf<uint32_t> corners;
    std::vector<int> K;
    std::vector<unsigned long long> counts;
    bool ran = false;
    bool profile = false;
    double sweep_ms = 0.0;
    // adjoint in the same graph (forward + loss gradient)
    bool adjoint = false;
    uint64_t adj_seed = 1;
    i2::AdjState* adj = nullptr;
};

namespace i2 {

static MeshDesc desc_of(const i2_mesh* m) {
    MeshDesc D{};
    D.panels = m->d_panels.p;
    D.row_start = m->d_row_start.p;
    D.nbr_start = m->d_nbr_start.p;
    D.nbr = m->d_nbr.p;
    D.lists[0] = m->d_simple.p;
    D.lists[1] = m->d_attached.p;
    for (int t = 0; t < 3; ++t) D.npairs[t] = m->pairs[t];
    D.nT = (int)m->nT;
    return D;
}

static void drop_graph(i2_batch* b) {
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->exec = nullptr;
    b->graph = nullptr;
}

// true if every mesh is prepared and still the one the graph was built for
// (a later i2_mesh_set_data or i2_mesh_prepare may have reallocated its arrays
// and changed its pair counts)
static bool batch_current(const i2_batch* b) {
    if (b->generations.size() != b->meshes.size()) return false;
    for (size_t m = 0; m < b->meshes.size(); ++m)
        if (!b->meshes[m]->prepared || b->meshes[m]->generation != b->generations[m]) return false;
    return true;
}

// The vertex list of a tile of 64 panels, a wavefront each: corners in order
// (all panels' first corners, then the second and third), each vertex at its
// first corner.
__global__ __launch_bounds__(64) void k_tile_vertices(int nT, const int32_t* __restrict__ tri, int32_t* __restrict__ lists,
                                                      uint32_t* __restrict__ corners) {
    __shared__ int32_t id[192], rank[192];
    const int lane = threadIdx.x, j = 64 * blockIdx.x + lane;
    const bool in = j < nT;
    for (int c = 0; c < 3; ++c) id[64 * c + lane] = in ? tri[3 * (int64_t)j + c] : -1 - lane - 64 * c;
    __syncthreads();
    int32_t* list = lists + (int64_t)blockIdx.x * TILE_LIST;
    int first[3], n = 0;
    for (int c = 0; c < 3; ++c) {
        const int own = 64 * c + lane, x = id[own];
        int f = own;
        for (int k = own - 1; k >= 0; --k) if (id[k] == x) f = k;
        first[c] = f;
        const unsigned long long fresh = __ballot(in && f == own);
        if (in && f == own) {
            const int r = n + __popcll(fresh & ((1ull << lane) - 1ull));
            rank[own] = r;
            if (r < TILE_VERTS) list[1 + r] = x;
        }
        n += __popcll(fresh);
    }
    __syncthreads();
    if (lane == 0) list[0] = n <= TILE_VERTS ? n : 0;
    if (in) corners[j] = (uint32_t)rank[first[0]] | (uint32_t)rank[first[1]] << 8 | (uint32_t)rank[first[2]] << 16;
}

static int batch_prepare(i2_batch* b) {
    Engine& E = b->E;
    b->generations.clear();
    E.out = b->out;
    E.pairs_per_wg = b->P;
    E.ppl = b->ppl;
    const int M = (int)b->meshes.size();
    b->outs.resize(M);
    E.h_meshes.resize(M);
    for (int m = 0; m < M; ++m) {
        const i2_mesh* mesh = b->meshes[m];
        if (!mesh->prepared) { set_error("mesh %d is not prepared", m); return I2_ERR_STATE; }
        if (mesh->device != b->device) { set_error("mesh %d lives on device %d, batch on %d", m, mesh->device, b->device); return I2_ERR_INVALID; }
        MeshDesc D = desc_of(mesh);
        auto& o = b->outs[m];
        for (int t = 0; t < 2; ++t) {
            I2_TRY(o.sing_val[t].ensure(2 * mesh->pairs[t]));
            D.sing_val[t] = o.sing_val[t].p;
        }
        if (b->out == OUT_PER_PAIR) {
            for (int t = 0; t < 3; ++t) {
                const int64_t n = 2 * mesh->pairs[t];
                I2_TRY(o.fin[t].ensure(n)); I2_TRY(o.prev[t].ensure(n)); I2_TRY(o.conv[t].ensure(n)); I2_TRY(o.res[t].ensure(3 * n));
                D.fin[t] = o.fin[t].p; D.prev[t] = o.prev[t].p; D.conv[t] = o.conv[t].p; D.res[t] = o.res[t].p;
            }
            I2_TRY(o.unconv.ensure((3 * mesh->nT + 7) / 8));
            if (!b->cfg.fixed)
                for (int t = 0; t < 3; ++t) D.unconv[t] = reinterpret_cast<uint8_t*>(o.unconv.p) + t * mesh->nT;
        } else {
            I2_TRY(o.rowacc.ensure(24 * mesh->nT));
            I2_TRY(o.rowout.ensure(4 * mesh->nT));
            D.rowacc = o.rowacc.p;
            D.rowout = o.rowout.p;
            if (b->adjoint)
                for (int t = 0; t < 3; ++t) {
                    I2_TRY(o.conv[t].ensure(2 * mesh->pairs[t]));
                    D.conv[t] = o.conv[t].p;
                }
        }
        E.h_meshes[m] = D;
    }
    E.side = b->side;
    if (!b->tuned) engine_auto_shape(E);
    int64_t tiles = 0, panels = 0;
    for (const i2_mesh* mesh : b->meshes) { tiles += (mesh->nT + 63) / 64; panels += mesh->nT; }
    I2_TRY(b->tile_lists.ensure(TILE_LIST * tiles));
    I2_TRY(b->corners.ensure(panels));
    tiles = panels = 0;
    for (int m = 0; m < M; ++m) {
        const i2_mesh* mesh = b->meshes[m];
        const int64_t n = (mesh->nT + 63) / 64;
        MeshDesc& D = E.h_meshes[m];
        int32_t* lists = b->tile_lists.p + TILE_LIST * tiles;
        uint32_t* corners = b->corners.p + panels;
        hipLaunchKernelGGL(k_tile_vertices, dim3((unsigned)n), dim3(64), 0, b->stream, D.nT, mesh->d_tri.p, lists, corners);
        I2_TRY(check_launch("k_tile_vertices"));
        D.xyz = mesh->d_xyz.p;
        D.tile_list = lists;
        D.corners = corners;
        tiles += n;
        panels += mesh->nT;
    }
    I2_TRY(engine_setup(E, b->cfg));
    for (const i2_mesh* mesh : b->meshes) b->generations.push_back(mesh->generation);
    if (!b->adjoint) return I2_OK;
    if (!b->adj) {
        b->adj = new AdjState;
        if (hipEventCreate(&b->adj->e0) != hipSuccess || hipEventCreate(&b->adj->e1) != hipSuccess) {
            (void)hipGetLastError();
            set_error("event creation failed");
            return I2_ERR_HIP;
        }
    }
    b->adj->side = b->side;
    std::vector<AdjMesh> AD(M);
    for (int m = 0; m < M; ++m) AD[m] = adjoint_mesh(b->meshes[m], E.h_meshes[m].conv, E.args.K + 3 * m);
    return adjoint_setup(*b->adj, b->device, AD, b->meshes, &b->cfg, b->adj_seed);
}

static int batch_enqueue_all(i2_batch* b) {
    Engine& E = b->E;
    I2_TRY(batch_enqueue(E, b->stream));
    if (b->adjoint) I2_TRY(adjoint_launch(*b->adj, b->stream));
    return I2_OK;
}

// The engine without its profiling events while this lives
struct WithoutEvents {
    Engine& E;
    hipEvent_t p0, p1;
    explicit WithoutEvents(Engine& e) : E(e), p0(e.prof0), p1(e.prof1) { E.prof0 = E.prof1 = nullptr; }
    ~WithoutEvents() { E.prof0 = p0; E.prof1 = p1; }
};
static int batch_capture(i2_batch* b) {
    drop_graph(b);
    WithoutEvents plain(b->E);
    I2_HIP(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    const int st = batch_enqueue_all(b);
    hipGraph_t g = nullptr;
    const hipError_t ec = hipStreamEndCapture(b->stream, &g);
    if (st != I2_OK) { if (g) (void)hipGraphDestroy(g); return st; }
    if (ec != hipSuccess) { set_error("graph capture failed: %s", hipGetErrorString(ec)); return I2_ERR_HIP; }
    b->graph = g;
    I2_HIP(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
    return I2_OK;
}

static int batch_run(i2_batch* b, double* ms) {
    DeviceGuard g(b->device);
    if (!g.ok) return I2_ERR_HIP;
    if (b->meshes.empty()) { set_error("batch has no meshes"); return I2_ERR_STATE; }
    if (!b->have_cfg) { set_error("batch not configured (i2_batch_configure)"); return I2_ERR_STATE; }
    if (!batch_current(b)) { b->dirty = true; b->ran = false; }
    for (int attempt = 0; attempt < 4; ++attempt) {
        // The first run after a change launches its kernels directly, the next one
        // captures them: a mesh that changes with every run never pays for a
        // capture (preparation and run of 320 panels 517 -> 476 us).
        if (b->dirty) {
            I2_TRY(batch_prepare(b));
            drop_graph(b);
            b->dirty = false;
        } else if (!b->exec && !b->profile) {
            I2_TRY(batch_capture(b));
        }
        I2_HIP(hipEventRecord(b->e0, b->stream));
        if (b->profile) {
            // same kernels, launched directly so that events can bracket the sweep
            if (!b->E.prof0) I2_HIP(hipEventCreate(&b->E.prof0));
            if (!b->E.prof1) I2_HIP(hipEventCreate(&b->E.prof1));
            I2_TRY(batch_enqueue_all(b));
        } else if (b->exec) {
            I2_HIP(hipGraphLaunch(b->exec, b->stream));
        } else {
            WithoutEvents plain(b->E);
            I2_TRY(batch_enqueue_all(b));
        }
        I2_HIP(hipEventRecord(b->e1, b->stream));
        bool overflow = false;
        I2_TRY(engine_check_queues(b->E, b->stream, &overflow, &b->counts, &b->K));
        if (!overflow) {
            float f = 0.f;
            I2_HIP(hipEventElapsedTime(&f, b->e0, b->e1));
            if (ms) *ms = f;
            if (b->profile) {
                float g = 0.f;
                I2_HIP(hipEventElapsedTime(&g, b->E.prof0, b->E.prof1));
                b->sweep_ms = g;
            }
            b->ran = true;
            return I2_OK;
        }
        b->dirty = true;   // queues were grown: rebuild and run again
    }
    set_error("refinement queues kept overflowing");
    return I2_ERR_RANGE;
}

// The evaluator's fast path: one mesh, per-pair outputs into its type buffers.
int engine_run_evaluator(i2_evaluator* ev) {
    const i2_mesh* m = ev->mesh;
    i2_batch* b = ev->fast;
    if (!b) {
        b = new i2_batch;
        b->device = m->device;
        b->stream = ev->stream;
        b->side = &ev->side;
        if (hipEventCreate(&b->e0) != hipSuccess || hipEventCreate(&b->e1) != hipSuccess) {
            (void)hipGetLastError();
            delete b;
            set_error("event creation failed");
            return I2_ERR_HIP;
        }
        ev->fast = b;
    }
    if (b->meshes.size() != 1 || b->meshes[0] != m) { b->meshes.assign(1, m); b->dirty = true; }
    const i2_integrator& it = *ev->integ;
    if (!b->have_cfg || memcmp(&b->cfg.rule, &it.rule, sizeof(Rule)) != 0 || b->cfg.fixed != it.fixed ||
        b->cfg.fixed_level != it.fixed_level || b->cfg.max_level != it.max_level || b->cfg.tol != it.tol || b->cfg.quirk != it.quirk) {
        b->cfg = it;
        b->have_cfg = true;
        b->dirty = true;
    }
    if (b->P != ev->fast_P || b->ppl != ev->fast_ppl || b->tuned != ev->fast_tuned) {
        b->P = ev->fast_P;
        b->ppl = ev->fast_ppl;
        b->tuned = ev->fast_tuned;
        b->dirty = true;
    }
    b->out = OUT_PER_PAIR;
    b->profile = ev->profile;
    double ms = 0.0;
    I2_TRY(batch_run(b, &ms));
    ev->fast_sweep_ms = b->profile ? b->sweep_ms : 0.0;
    for (int t = 0; t < 3; ++t) {
        TypeState& ts = ev->type[t];
        ts.n = 2 * m->pairs[t];
        ts.implicit = (t == I2_NOT_NEIGHBORS);
        ts.K = b->K[t];
        ts.final_buf = 0;
        ts.ms = ms;
        ts.refined_tasks = 0;
    }
    return I2_OK;
}

void engine_evaluator_outputs(const i2_evaluator* ev, int type, const double4** ints, const double** res, const int8_t** conv) {
    const i2_batch* b = ev->fast;
    *ints = b->outs[0].fin[type].p;
    *res = b->outs[0].res[type].p;
    *conv = b->outs[0].conv[type].p;
}

const uint8_t* engine_evaluator_unconverged(const i2_evaluator* ev, int type) {
    const i2_batch* b = ev->fast;
    return reinterpret_cast<const uint8_t*>(b->outs[0].unconv.p) + type * ev->mesh->nT;
}

void engine_release_evaluator(i2_evaluator* ev) {
    i2_batch* b = ev->fast;
    if (!b) return;
    drop_graph(b);
    if (b->E.prof0) (void)hipEventDestroy(b->E.prof0);
    if (b->E.prof1) (void)hipEventDestroy(b->E.prof1);
    if (b->E.h_sync) (void)hipHostFree(b->E.h_sync);
    if (b->e0) (void)hipEventDestroy(b->e0);
    if (b->e1) (void)hipEventDestroy(b->e1);
    b->stream = nullptr;   // owned by the evaluator
    delete b;
    ev->fast = nullptr;
}

}  // namespace i2

using namespace i2;

extern "C" {

int i2_batch_create(i2_batch** out, int device) {
    if (!out) { set_error("null pointer"); return I2_ERR_INVALID; }
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) { (void)hipGetLastError(); set_error("no HIP device available"); return I2_ERR_HIP; }
    if (device < 0 || device >= count) { set_error("device %d out of range", device); return I2_ERR_INVALID; }
    DeviceGuard g(device);
    if (!g.ok) return I2_ERR_HIP;
    i2_batch* b = new i2_batch;
    b->device = device;
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess || hipEventCreate(&b->e0) != hipSuccess ||
        hipEventCreate(&b->e1) != hipSuccess) {
        (void)hipGetLastError();
        set_error("stream/event creation failed");
        i2_batch_destroy(b);
        return I2_ERR_HIP;
    }
    *out = b;
    return I2_OK;
}

void i2_batch_destroy(i2_batch* b) {
    if (!b) return;
    {
        DeviceGuard g(b->device);
        if (b->stream) (void)hipStreamSynchronize(b->stream);
        drop_graph(b);
        b->outs.clear();
        adjoint_release(b->adj);
        if (b->E.prof0) (void)hipEventDestroy(b->E.prof0);
        if (b->E.prof1) (void)hipEventDestroy(b->E.prof1);
        if (b->E.h_sync) (void)hipHostFree(b->E.h_sync);
        if (b->e0) (void)hipEventDestroy(b->e0);
        if (b->e1) (void)hipEventDestroy(b->e1);
        if (b->stream) (void)hipStreamDestroy(b->stream);
    }
    delete b;
}

int i2_batch_add_mesh(i2_batch* b, const i2_mesh* m, int* index) {
    if (!b || !m) { set_error("null argument"); return I2_ERR_INVALID; }
    if (!m->prepared) { set_error("mesh not prepared"); return I2_ERR_STATE; }
    if ((int)b->meshes.size() >= MAX_BATCH_MESHES) { set_error("batch is full (%d meshes)", MAX_BATCH_MESHES); return I2_ERR_RANGE; }
    b->meshes.push_back(m);
    if (index) *index = (int)b->meshes.size() - 1;
    b->dirty = true;
    b->ran = false;
    return I2_OK;
}

int i2_batch_clear(i2_batch* b) {
    if (!b) { set_error("null batch"); return I2_ERR_INVALID; }
    b->meshes.clear();
    b->dirty = true;
    b->ran = false;
    return I2_OK;
}

int i2_batch_configure(i2_batch* b, const i2_integrator* it, int outputMode) {
    if (!b || !it) { set_error("null argument"); return I2_ERR_INVALID; }
    if (outputMode != OUT_PER_PAIR && outputMode != OUT_ROW_SUMS) { set_error("bad output mode %d", outputMode); return I2_ERR_INVALID; }
    b->cfg = *it;
    b->have_cfg = true;
    b->out = outputMode;
    b->dirty = true;
    b->ran = false;
    return I2_OK;
}

int i2_batch_set_tuning(i2_batch* b, int pairsPerWorkgroup, int pointsPerLane) {
    if (!b) { set_error("null batch"); return I2_ERR_INVALID; }
    if (pairsPerWorkgroup < 1 || pairsPerWorkgroup > 4096 || (pairsPerWorkgroup & (pairsPerWorkgroup - 1)) != 0) {
        set_error("pairs per workgroup must be a power of two in [1, 4096]");
        return I2_ERR_INVALID;
    }
    if (pointsPerLane != 1 && pointsPerLane != 2 && pointsPerLane != 4 && pointsPerLane != 13) { set_error("points per lane must be 1, 2, 4 or 13"); return I2_ERR_INVALID; }
    b->P = pairsPerWorkgroup;
    b->ppl = pointsPerLane;
    b->tuned = true;
    b->dirty = true;
    return I2_OK;
}

int i2_batch_run(i2_batch* b, double* ms) {
    if (!b) { set_error("null batch"); return I2_ERR_INVALID; }
    return batch_run(b, ms);
}

int i2_batch_enable_adjoint(i2_batch* b, int enable, uint64_t seed) {
    if (!b) { set_error("null batch"); return I2_ERR_INVALID; }
    b->adjoint = enable != 0;
    b->adj_seed = seed;
    b->dirty = true;
    b->ran = false;
    return I2_OK;
}

int i2_batch_get_loss_and_grad(const i2_batch* b, int mesh, double* loss, double* dLdX) {
    if (!b || mesh < 0 || mesh >= (int)b->meshes.size() || !loss || !dLdX) { set_error("invalid argument"); return I2_ERR_INVALID; }
    if (b->ran && !batch_current(b)) { set_error("a mesh was changed or prepared again after the last run: run the batch again"); return I2_ERR_STATE; }
    if (!b->ran || !b->adjoint || !b->adj) { set_error("no adjoint results: enable the adjoint and run the batch"); return I2_ERR_STATE; }
    DeviceGuard g(b->device);
    if (!g.ok) return I2_ERR_HIP;
    return adjoint_copy_out(*b->adj, mesh, loss, dLdX);
}

int i2_batch_autotune(i2_batch* b, int reps, int includeWholeRule, int* bestP, int* bestPPL, double* table_ms) {
    if (!b || reps < 1) { set_error("invalid argument"); return I2_ERR_INVALID; }
    if (b->profile) { set_error("autotuning times graph replays: turn profiling off first"); return I2_ERR_STATE; }
    static const int Ps[4] = {16, 32, 64, 128};
    static const int PPLs[4] = {1, 2, 4, 13};
    const int nppl = includeWholeRule ? 4 : 3;
    double best = 1e300;
    int bp = b->P, bl = b->ppl;
    std::vector<double> t((size_t)reps);
    for (int a = 0; a < 4; ++a)
        for (int l = 0; l < nppl; ++l) {
            I2_TRY(i2_batch_set_tuning(b, Ps[a], PPLs[l]));
            double ms = 0.0;
            I2_TRY(batch_run(b, &ms));   // sizes the queues
            I2_TRY(batch_run(b, &ms));   // the second run after a change captures the graph
            for (int r = 0; r < reps; ++r) I2_TRY(batch_run(b, &t[(size_t)r]));
            std::sort(t.begin(), t.end());
            const double med = t[(size_t)reps / 2];
            if (table_ms) table_ms[a * nppl + l] = med;
            if (med < best) { best = med; bp = Ps[a]; bl = PPLs[l]; }
        }
    I2_TRY(i2_batch_set_tuning(b, bp, bl));
    if (bestP) *bestP = bp;
    if (bestPPL) *bestPPL = bl;
    return I2_OK;
}

int i2_batch_get_pair_results(const i2_batch* b, int mesh, int type, double* integrals4, double* results3, int8_t* conv) {
    if (!b || mesh < 0 || mesh >= (int)b->meshes.size() || type < 0 || type > 2) { set_error("invalid argument"); return I2_ERR_INVALID; }
    if (b->ran && !batch_current(b)) { set_error("a mesh was changed or prepared again after the last run: run the batch again"); return I2_ERR_STATE; }
    if (!b->ran || b->out != OUT_PER_PAIR) { set_error("no per-pair results"); return I2_ERR_STATE; }
    DeviceGuard g(b->device);
    if (!g.ok) return I2_ERR_HIP;
    const auto& o = b->outs[mesh];
    const int64_t n = 2 * b->meshes[mesh]->pairs[type];
    if (n == 0) return I2_OK;
    if (integrals4) I2_HIP(hipMemcpy(integrals4, o.fin[type].p, sizeof(double4) * n, hipMemcpyDeviceToHost));
    if (results3) I2_HIP(hipMemcpy(results3, o.res[type].p, sizeof(double) * 3 * n, hipMemcpyDeviceToHost));
    if (conv) I2_HIP(hipMemcpy(conv, o.conv[type].p, (size_t)n, hipMemcpyDeviceToHost));
    return I2_OK;
}

int i2_batch_get_row_sums(const i2_batch* b, int mesh, double* rows4) {
    if (!b || !rows4 || mesh < 0 || mesh >= (int)b->meshes.size()) { set_error("invalid argument"); return I2_ERR_INVALID; }
    if (b->ran && !batch_current(b)) { set_error("a mesh was changed or prepared again after the last run: run the batch again"); return I2_ERR_STATE; }
    if (!b->ran || b->out != OUT_ROW_SUMS) { set_error("no row sums"); return I2_ERR_STATE; }
    DeviceGuard g(b->device);
    if (!g.ok) return I2_ERR_HIP;
    I2_HIP(hipMemcpy(rows4, b->outs[mesh].rowout.p, sizeof(double) * 4 * b->meshes[mesh]->nT, hipMemcpyDeviceToHost));
    return I2_OK;
}

int i2_batch_refinement_iterations(const i2_batch* b, int mesh, int type, int* K) {
    if (!b || !K || mesh < 0 || mesh >= (int)b->meshes.size() || type < 0 || type > 2) { set_error("invalid argument"); return I2_ERR_INVALID; }
    if (b->ran && !batch_current(b)) { set_error("a mesh was changed or prepared again after the last run: run the batch again"); return I2_ERR_STATE; }
    if (!b->ran) { set_error("batch has not run"); return I2_ERR_STATE; }
    *K = b->K[3 * mesh + type];
    return I2_OK;
}

int i2_batch_level_counts(const i2_batch* b, int64_t* counts) {
    if (!b || !counts) { set_error("invalid argument"); return I2_ERR_INVALID; }
    if (b->ran && !batch_current(b)) { set_error("a mesh was changed or prepared again after the last run: run the batch again"); return I2_ERR_STATE; }
    if (!b->ran) { set_error("batch has not run"); return I2_ERR_STATE; }
    for (int L = 0; L < MAX_LEVELS; ++L)
        for (int t = 0; t < 3; ++t) counts[3 * L + t] = (L >= 2) ? (int64_t)b->counts[1 + 3 * L + t] : 0;
    for (int t = 0; t < 3; ++t) {
        int64_t n = 0;
        for (const i2_mesh* m : b->meshes) n += 2 * m->pairs[t];
        counts[t] = n;
        counts[3 + t] = (b->cfg.fixed && b->cfg.fixed_level == 0) || (!b->cfg.fixed && b->cfg.max_level == 0) ? 0 : n;
    }
    return I2_OK;
}

int i2_batch_set_profiling(i2_batch* b, int enable) {
    if (!b) { set_error("null batch"); return I2_ERR_INVALID; }
    b->profile = enable != 0;
    return I2_OK;
}

int i2_batch_sweep_ms(const i2_batch* b, double* ms) {
    if (!b || !ms) { set_error("invalid argument"); return I2_ERR_INVALID; }
    if (!b->ran || !b->profile) { set_error("no profiled run"); return I2_ERR_STATE; }
    *ms = b->sweep_ms;
    return I2_OK;
}

int i2_batch_task_count(const i2_batch* b, int64_t* n) {
    if (!b || !n) { set_error("invalid argument"); return I2_ERR_INVALID; }
    int64_t s = 0;
    for (const i2_mesh* m : b->meshes) s += 2 * (m->pairs[0] + m->pairs[1] + m->pairs[2]);
    *n = s;
    return I2_OK;
}

}  // extern "C"
