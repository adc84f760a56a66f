// i2_evaluator.hip -- NumericalIntegrator3D + Evaluator3D/EvaluatorJ3DK behind
// the C ABI: the "plain" path with per-type, per-level launches.
//
// Control flow follows EvaluatorJ3DK::numericalIntegration
// (src/evaluators/evaluatorJ3DK.cu:895-1012): level 0 over all tasks, then
// refinement iterations 1..maxLevel, each integrating the 4^level sub-panels
// of the control panel of every task still unconverged and comparing with the
// previous level by the Runge rule.  Level k is written to buf[k % 2], which
// reproduces the reference's swapped result buffers exactly.  Unlike the
// reference, child tasks are never materialised: a task at level k is one
// group of lanes that walks its 4^k sub-panels by path digits and reduces in
// a fixed order, and nothing in a refined task depends on the order in which
// the lists of unconverged tasks were filled, so results are bitwise reproducible.
#include "i2_internal.hpp"
#include "i2_batch.hpp"
#include "i2_adjoint.hpp"

#include <algorithm>
#include <fstream>
#include <mutex>
#include <unordered_set>

namespace i2 {
using namespace i2d;

// ------------------------------------------------------------ per-pair integrand
template <int TYPE> struct PairCtx;
template <> struct PairCtx<I2_NOT_NEIGHBORS> {
    __device__ __forceinline__ void init(const Panel&, const Panel&) {}
    __device__ __forceinline__ q4 sing(d3, const i2m::MathTable*) const { return q4zero(); }
};
template <> struct PairCtx<I2_ATTACHED_NEIGHBORS> {
    EdgeCtx c;
    __device__ __forceinline__ void init(const Panel& I, const Panel& J) {
        int s1, s2;
        shifts_edge(I, J, &s1, &s2);
        c = edge_ctx(vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3));
    }
    __device__ __forceinline__ q4 sing(d3 p, const i2m::MathTable* lt) const { return sing_edge_fast(p, c, lt); }
};
template <> struct PairCtx<I2_SIMPLE_NEIGHBORS> {
    VertexCtx c;
    __device__ __forceinline__ void init(const Panel& I, const Panel& J) {
        int s1, s2;
        shifts_vertex(I, J, &s1, &s2);
        c = vertex_ctx(vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3), I.n, J.n, I.area);
    }
    __device__ __forceinline__ q4 sing(d3 p, const i2m::MathTable* lt) const { return sing_vertex_fast(p, c, lt); }
};

// Quadrature over one sub-panel: area * sum_k w_k (thetaPsi - singular part)(r_k)
// (NumericalIntegrator3d.cu:560-585, evaluatorJ3DK.cu:98-106).  thetaPsi is
// the cancellation-free form shared with the batched path: the reference's
// own FP64 form loses up to 1e-7 of a value to cancellation where a
// quadrature point lies near the extension of an edge line of K_j, which
// moves Runge decisions; both paths therefore take decisions on accurate values.
// Disjoint pairs sum the inner integral's terms, which the caller converts to
// (Psi, Theta) once per task.  Points k0, k0 + step, ...
template <int TYPE>
__device__ __forceinline__ q4 quad_sub(const Rule& R, const i2m::MathTable* lt, d3 a, d3 b, d3 c, double area,
                                       const JGeom& J, const PairCtx<TYPE>& ctx, int k0, int step) {
    q4 acc = q4zero();
    for (int k = k0; k < R.n; k += step) {
        d3 p = R.L1[k] * a;
        p = p + R.L2[k] * b;
        p = p + R.L3[k] * c;
        q4 f;
        if (TYPE == I2_NOT_NEIGHBORS) f = theta_terms(p, J, lt);
        else f = theta_psi_fast(p, J, lt) - ctx.sing(p, lt);
        acc = acc + R.w[k] * f;
    }
    return area * acc;
}

__device__ __forceinline__ q4 lanes_sum(q4 v, int lanes) {
    for (int m = 1; m < lanes; m <<= 1) {
        v.x += __shfl_xor(v.x, m);
        v.y += __shfl_xor(v.y, m);
        v.z += __shfl_xor(v.z, m);
        v.w += __shfl_xor(v.w, m);
    }
    return v;
}

// Level-`level` value of tasks: lanes per task = 1 << lanes_log2, of which
// 1 << per_log2 share a sub-panel's points; the groups walk the sub-panels
// < 4^level; butterfly reduction.
template <int TYPE, bool IMPLICIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(TYPE == I2_NOT_NEIGHBORS ? 3 : 2))) void k_level(int64_t nitems, const int32_t* __restrict__ list, TaskSource src,
                                               const Panel* __restrict__ panels, Rule R, int level, int lanes_log2, int per_log2,
                                               double4* __restrict__ out) {
    __shared__ i2m::MathTable lt;
    i2m::fill_mathtab(lt);
    __syncthreads();
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lanes = 1 << lanes_log2, step = 1 << per_log2, G = lanes >> per_log2;
    const int64_t slot = gid >> lanes_log2;
    const int sub = (int)(gid & (lanes - 1)) >> per_log2, k0 = (int)(gid & (step - 1));
    const bool active = slot < nitems;
    q4 acc = q4zero();
    int64_t z = 0;
    if (active) {
        z = list ? (int64_t)list[slot] : slot;
        int i, j;
        task_ij<IMPLICIT>(src, z, &i, &j);
        const Panel I = panels[i];
        const Panel J = panels[j];
        const JGeom JG = make_jgeom(J.a, J.b, J.c, J.ta, J.tb, J.tc);
        PairCtx<TYPE> ctx;
        ctx.init(I, J);
        double area = I.area;
        for (int l = 0; l < level; ++l) area *= 0.25;
        const uint32_t nsub = 1u << (2 * level);
        // Disjoint pairs: one loop per wavefront, in the form that holds for all its
        // pairs.  Those of a rest list each in its own form, because the list's
        // order changes from run to run (a wavefront holds four of them at level 2
        // above 8,192 tasks); a task list's pairs stand as the caller put them, and
        // four forms in turn cost 19 % there (1,280 panels at fixed level 2).
        int form = 0;
        if (TYPE == I2_NOT_NEIGHBORS) {
            const Ball ball = panel_ball(I.a, I.b, I.c, R.reach);
            form = list ? panel_far(ball, JG) : wave_form(true, ball, JG);
        }
        if (form != 0) {
            const FarFrame F = far_frame(I.a, I.b, I.c);
            const FarGeom FG = far_geom(F, JG);
            acc = area * far_scale(form == 1 ? quad_far<false>(R, R.n, level, sub, G, k0, step, F, FG)
                                               : quad_far<true>(R, R.n, level, sub, G, k0, step, F, FG), JG);
        } else {
            for (uint32_t c = sub; c < nsub; c += G) {
                d3 a = I.a, b = I.b, cc = I.c;
                sub_panel(a, b, cc, level, c);
                acc = acc + quad_sub<TYPE>(R, &lt, a, b, cc, area, JG, ctx, k0, step);
            }
        }
        if (TYPE == I2_NOT_NEIGHBORS) acc = psi_of_terms(acc, JG);
    }
    acc = lanes_sum(acc, lanes);
    if (active && sub == 0) out[z] = make_double4(acc.x, acc.y, acc.z, acc.w);
}

// Appends the wavefront's unconverged tasks to a rest list, one atomic per wavefront.
__device__ __forceinline__ void append_rest(bool unconv, int64_t z, int32_t* __restrict__ rest, unsigned long long* __restrict__ counter) {
    const unsigned long long mask = __ballot(unconv);
    const int lane = threadIdx.x & 63;
    const int before = __popcll(mask & ((1ull << lane) - 1ull));
    unsigned long long base = 0;
    if (lane == 0 && mask) base = atomicAdd(counter, (unsigned long long)__popcll(mask));
    base = __shfl(base, 0);
    if (unconv) rest[base + before] = (int32_t)z;
}

// Levels 0 and 1 of all tasks and their comparison (k_level for the two levels,
// then k_compare) in one launch: every task needs both, and the pair's
// geometry and the tasks' decoding serve both.  1 << lanes_log2 lanes per task
// share each level's points.  Plain run of 1,330 panels 1,250 -> 1,154 us, of 80
// panels 183 -> 134 (with one launch for the closed forms of all types).
template <int TYPE, bool IMPLICIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(TYPE == I2_NOT_NEIGHBORS ? 3 : 2))) void k_first_levels(
    int64_t nitems, TaskSource src, const Panel* __restrict__ panels, Rule R, int lanes_log2, double tol, int keep_converged,
    double4* __restrict__ out0, double4* __restrict__ out1, int8_t* __restrict__ conv, int32_t* __restrict__ rest_out,
    unsigned long long* __restrict__ counter) {
    __shared__ i2m::MathTable lt;
    i2m::fill_mathtab(lt);
    __syncthreads();
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lanes = 1 << lanes_log2, s = (int)(gid & (lanes - 1));
    const int per = max(1, lanes >> 2), subs = min(4, lanes), sub = s / per, k0 = s % per;   // level 1: per lanes a sub-panel
    const int64_t z = gid >> lanes_log2;
    const bool active = z < nitems;
    q4 v0 = q4zero(), v1 = q4zero();
    if (active) {
        int i, j;
        task_ij<IMPLICIT>(src, z, &i, &j);
        const Panel I = panels[i];
        const Panel J = panels[j];
        const JGeom JG = make_jgeom(J.a, J.b, J.c, J.ta, J.tb, J.tc);
        PairCtx<TYPE> ctx;
        ctx.init(I, J);
        const double area = I.area;
        const int form = TYPE == I2_NOT_NEIGHBORS ? wave_form(true, panel_ball(I.a, I.b, I.c, R.reach), JG) : 0;
        if (form != 0) {
            const FarFrame F = far_frame(I.a, I.b, I.c);
            const FarGeom FG = far_geom(F, JG);
            if (form == 1) {
                v0 = quad_far<false>(R, R.n, 0, 0, 1, s, lanes, F, FG);
                v1 = quad_far<false>(R, R.n, 1, sub, subs, k0, per, F, FG);
            } else {
                v0 = quad_far<true>(R, R.n, 0, 0, 1, s, lanes, F, FG);
                v1 = quad_far<true>(R, R.n, 1, sub, subs, k0, per, F, FG);
            }
            v0 = area * far_scale(v0, JG);
            v1 = (0.25 * area) * far_scale(v1, JG);
        } else {
            v0 = quad_sub<TYPE>(R, &lt, I.a, I.b, I.c, area, JG, ctx, s, lanes);
            for (uint32_t c = sub; c < 4; c += subs) {
                d3 a = I.a, b = I.b, cc = I.c;
                sub_panel(a, b, cc, 1, c);
                v1 = v1 + quad_sub<TYPE>(R, &lt, a, b, cc, 0.25 * area, JG, ctx, k0, per);
            }
        }
        if (TYPE == I2_NOT_NEIGHBORS) { v0 = psi_of_terms(v0, JG); v1 = psi_of_terms(v1, JG); }
    }
    v0 = lanes_sum(v0, lanes);
    v1 = lanes_sum(v1, lanes);
    bool unconv = false;
    if (active && s == 0) {
        unconv = runge_criterion(v1, v0, R.pow2p) > tol;
        conv[z] = 1;
        out1[z] = make_double4(v1.x, v1.y, v1.z, v1.w);
        const q4 p = !unconv && keep_converged ? v1 : v0;
        out0[z] = make_double4(p.x, p.y, p.z, p.w);
    }
    append_rest(unconv, z, rest_out, counter);
}

// Runge comparison of iteration `it` (evaluator3d.cu:76-99): items are all
// tasks (list == nullptr) or the previous rest list.  Unconverged tasks are
// appended to rest_out (one atomic per wave); with keep_converged the
// converged value is also written to the other buffer so that it survives
// later swaps (the reference's quirk disabled).
__global__ __launch_bounds__(256) void k_compare(int64_t nitems, const int32_t* __restrict__ list, double4* __restrict__ cur,
                                                 double4* __restrict__ prev, double pow2p, double tol, int keep_converged,
                                                 int it, int8_t* __restrict__ conv, int32_t* __restrict__ rest_out,
                                                 unsigned long long* __restrict__ counter) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = gid < nitems;
    bool unconv = false;
    int64_t z = 0;
    if (active) {
        z = list ? (int64_t)list[gid] : gid;
        const double4 c4 = cur[z], p4 = prev[z];
        const double crit = runge_criterion({c4.x, c4.y, c4.z, c4.w}, {p4.x, p4.y, p4.z, p4.w}, pow2p);
        unconv = crit > tol;
        conv[z] = (int8_t)it;
        if (!unconv && keep_converged) prev[z] = c4;
    }
    append_rest(unconv, z, rest_out, counter);
}

// Analytic singular part (vertex/edge-sharing) and conversion to J
// (evaluatorJ3DK.cu:22-56, 224-264).  The final integrals stay in `ints`.
template <int TYPE, bool IMPLICIT>
__device__ __forceinline__ void finalize_one(int64_t z, const TaskSource& src, const Panel* __restrict__ panels,
                                             double4* __restrict__ ints, double* __restrict__ results) {
    int i, j;
    task_ij<IMPLICIT>(src, z, &i, &j);
    const Panel I = panels[i];
    const Panel J = panels[j];
    const double4 v4 = ints[z];
    q4 v = {v4.x, v4.y, v4.z, v4.w};
    d3 res;
    if (TYPE == I2_ATTACHED_NEIGHBORS) {
        int s1, s2;
        shifts_edge(I, J, &s1, &s2);
        v = v + integrate_sing_edge(vtx(I, s1), vtx(I, (s1 + 1) % 3), vtx(I, (s1 + 2) % 3),
                                    vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3), I.n, J.n, I.area);
        res = finalize_plain(v, J.n);
    } else if (TYPE == I2_SIMPLE_NEIGHBORS) {
        int s1, s2;
        shifts_vertex(I, J, &s1, &s2);
        v = v + integrate_sing_vertex(vtx(I, s1), vtx(I, (s1 + 1) % 3), vtx(I, (s1 + 2) % 3),
                                      vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3), I.n, J.n, I.area);
        res = finalize_vertex(v, J.n, I.area);
    } else {
        res = finalize_plain(v, J.n);
    }
    ints[z] = make_double4(v.x, v.y, v.z, v.w);
    results[3 * z] = res.x; results[3 * z + 1] = res.y; results[3 * z + 2] = res.z;
}

// All types in one launch, a range of workgroups each, the closed forms first:
// one after another their 17 and 12 us on few tasks are latency.  `clock`, in the
// host's memory, receives when each type's first workgroup began and its last
// one ended, by which the launch's time is divided among the types.
struct FinalizeType { int64_t n; unsigned blocks; TaskSource src; double4* ints; double* results; };
struct FinalizeArgs { FinalizeType t[3]; bool implicit; long long* clock; };
__global__ __launch_bounds__(256) void k_finalize(FinalizeArgs A, const Panel* __restrict__ panels) {
    unsigned b = blockIdx.x;
    int t = 0;
    while (t < 2 && b >= A.t[t].blocks) b -= A.t[t++].blocks;
    const FinalizeType& T = A.t[t];
    const int64_t z = (int64_t)b * blockDim.x + threadIdx.x;
    if (z >= T.n) return;
    if (A.clock && b == 0 && threadIdx.x == 0) A.clock[2 * t] = wall_clock64();
    if (t == I2_SIMPLE_NEIGHBORS) finalize_one<I2_SIMPLE_NEIGHBORS, false>(z, T.src, panels, T.ints, T.results);
    else if (t == I2_ATTACHED_NEIGHBORS) finalize_one<I2_ATTACHED_NEIGHBORS, false>(z, T.src, panels, T.ints, T.results);
    else if (A.implicit) finalize_one<I2_NOT_NEIGHBORS, true>(z, T.src, panels, T.ints, T.results);
    else finalize_one<I2_NOT_NEIGHBORS, false>(z, T.src, panels, T.ints, T.results);
    if (A.clock && b + 1 == T.blocks && threadIdx.x == 0) {
        __threadfence();               // after the outputs
        A.clock[2 * t + 1] = wall_clock64();
    }
}

// (i,j)/(j,i) symmetry error (evaluator3d.cu:45-57)
__global__ void k_symmetry(int64_t n, const double* __restrict__ r, double* __restrict__ err) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const double ax = r[3 * q], ay = r[3 * q + 1], az = r[3 * q + 2];
    const double bx = r[3 * (n + q)], by = r[3 * (n + q) + 1], bz = r[3 * (n + q) + 2];
    const double num = fabs(ax + bx) + fabs(ay + by) + fabs(az + bz);
    const double den = fmax(fabs(ax) + fabs(ay) + fabs(az), fabs(bx) + fabs(by) + fabs(bz));
    const double d = num / den;
    err[q] = d;
    err[n + q] = d;
}

// ------------------------------------------------------------ host orchestration
constexpr int64_t LANES_FULL = 524288;   // eight wavefronts per SIMD
static unsigned blocks_for(int64_t threads, int bs) { return (unsigned)((threads + bs - 1) / bs); }

// Lanes per task of k_level: one for levels 0 and 1, 16 at level 2, a wavefront
// from level 3; more while the launch leaves most of the chip without work, down
// to one point per lane.  A lane repeats the pair's geometry, so few lanes are
// better once the chip is full.  Plain run of 80 panels 375 us with the fewest
// lanes, 249, 228 and 254 with the line at 2, 8 and 32 wavefronts per SIMD.
static int lanes_log2_for(int level, int64_t items) {
    int ll = level <= 1 ? 0 : std::min(2 * level, 6);
    const int most = std::min(2 * level + 4, 6);
    while (ll + 2 <= most && (items << (ll + 2)) <= LANES_FULL) ll += 2;
    return ll;
}
static int per_log2_for(int level, int lanes_log2) { return std::max(0, lanes_log2 - 2 * level); }

template <int TYPE, bool IMPLICIT>
static int launch_level(i2_evaluator* ev, int64_t nitems, const int32_t* list, const TaskSource& src, int level, double4* out) {
    if (nitems == 0) return I2_OK;
    const int ll = lanes_log2_for(level, nitems);
    const int64_t threads = nitems << ll;
    LaunchRecord rec{TYPE, level, nitems, nullptr, nullptr};
    if (ev->profile) {
        I2_HIP(hipEventCreate(&rec.e0));
        I2_HIP(hipEventCreate(&rec.e1));
        I2_HIP(hipEventRecord(rec.e0, ev->stream));
    }
    hipLaunchKernelGGL((k_level<TYPE, IMPLICIT>), dim3(blocks_for(threads, 256)), dim3(256), 0, ev->stream, nitems, list, src,
                       ev->mesh->d_panels.p, ev->integ->rule, level, ll, per_log2_for(level, ll), out);
    I2_TRY(check_launch("k_level"));
    if (ev->profile) {
        I2_HIP(hipEventRecord(rec.e1, ev->stream));
        ev->launches.push_back(rec);
    }
    return I2_OK;
}

// Lanes per task of k_first_levels, by the same rule: one to 64, disjoint pairs at
// most 16 (their points cost less than the geometry each lane repeats: 80 panels
// took 34 us with 64 lanes)
template <int TYPE, bool IMPLICIT>
static int launch_first_levels(hipStream_t st, const Panel* panels, const i2_integrator& it, int64_t n, const TaskSource& src,
                               double4* out0, double4* out1, int8_t* conv, int32_t* rest, unsigned long long* counter) {
    const int ll = std::min(lanes_log2_for(1, n), TYPE == I2_NOT_NEIGHBORS ? 4 : 6);
    hipLaunchKernelGGL((k_first_levels<TYPE, IMPLICIT>), dim3(blocks_for(n << ll, 256)), dim3(256), 0, st, n, src, panels, it.rule, ll,
                       it.tol, it.quirk ? 0 : 1, out0, out1, conv, rest, counter);
    return check_launch("k_first_levels");
}

static void clear_launches(i2_evaluator* ev) {
    for (auto& r : ev->launches) {
        if (r.e0) (void)hipEventDestroy(r.e0);
        if (r.e1) (void)hipEventDestroy(r.e1);
    }
    ev->launches.clear();
}

static int launch_level_of(i2_evaluator* ev, int type, bool implicit, int64_t nitems, const int32_t* list, const TaskSource& src,
                           int level, double4* out) {
    if (type == I2_SIMPLE_NEIGHBORS) return launch_level<I2_SIMPLE_NEIGHBORS, false>(ev, nitems, list, src, level, out);
    if (type == I2_ATTACHED_NEIGHBORS) return launch_level<I2_ATTACHED_NEIGHBORS, false>(ev, nitems, list, src, level, out);
    return implicit ? launch_level<I2_NOT_NEIGHBORS, true>(ev, nitems, list, src, level, out)
                    : launch_level<I2_NOT_NEIGHBORS, false>(ev, nitems, list, src, level, out);
}
static int launch_first_levels_of(i2_evaluator* ev, int type, TypeState& ts, const TaskSource& src, unsigned long long* counter) {
    const Panel* panels = ev->mesh->d_panels.p;
#define I2_FIRST(T, I) launch_first_levels<T, I>(ev->stream, panels, *ev->integ, ts.n, src, ts.buf[0].p, ts.buf[1].p, ts.conv.p, ts.rest[1].p, counter)
    if (type == I2_SIMPLE_NEIGHBORS) return I2_FIRST(I2_SIMPLE_NEIGHBORS, false);
    if (type == I2_ATTACHED_NEIGHBORS) return I2_FIRST(I2_ATTACHED_NEIGHBORS, false);
    return ts.implicit ? I2_FIRST(I2_NOT_NEIGHBORS, true) : I2_FIRST(I2_NOT_NEIGHBORS, false);
#undef I2_FIRST
}
static int launch_finalize(hipStream_t st, const Panel* panels, FinalizeArgs A) {
    unsigned blocks = 0;
    for (FinalizeType& T : A.t) { T.blocks = blocks_for(T.n, 256); blocks += T.blocks; }
    if (blocks == 0) return I2_OK;
    hipLaunchKernelGGL(k_finalize, dim3(blocks), dim3(256), 0, st, A, panels);
    return check_launch("k_finalize");
}

// The counters of all levels and the types' flags of unconverged control panels
__global__ void k_begin_run(unsigned long long* counters, int nc, uint8_t* f0, uint8_t* f1, uint8_t* f2, int nT) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < nc) counters[q] = 0ull;
    if (q < nT) {
        if (f0) f0[q] = 0;
        if (f1) f1[q] = 0;
        if (f2) f2[q] = 0;
    }
}

// Device time of the launches between marks on the evaluator's stream, by type
struct RunMarks {
    static constexpr int NONE = -1, ALL = 3;
    i2_evaluator* ev;
    size_t used = 0;
    std::vector<int> type;           // of the stretch that ends at the mark; ALL: k_finalize's, by its clock
    long long* clock() const { return reinterpret_cast<long long*>(ev->h_counter + 3); }
    int mark(int t) {
        if (used == ev->marks.size()) {
            hipEvent_t e;
            I2_HIP(hipEventCreate(&e));
            ev->marks.push_back(e);
        }
        I2_HIP(hipEventRecord(ev->marks[used++], ev->stream));
        type.push_back(t);
        return I2_OK;
    }
    int times() {
        double share[3], sum = 0.0;
        for (int t = 0; t < 3; ++t) {
            ev->type[t].ms = 0.0;
            share[t] = ev->type[t].n > 0 ? (double)std::max(clock()[2 * t + 1] - clock()[2 * t], 1ll) : 0.0;
            sum += share[t];
        }
        for (size_t q = 1; q < used; ++q) {
            if (type[q] == NONE) continue;
            float ms = 0.f;
            I2_HIP(hipEventElapsedTime(&ms, ev->marks[q - 1], ev->marks[q]));
            if (type[q] != ALL) ev->type[type[q]].ms += ms;
            else for (int t = 0; t < 3; ++t) if (share[t] > 0.0) ev->type[t].ms += ms * share[t] / sum;
        }
        return I2_OK;
    }
};

// The three types' levels in step: level 0 and 1 of each, then one level after
// the other for the types with tasks left, with one wait per level for the
// three counts.  A type at a time cost a wait per level and type and a clearing
// copy per level: a plain run of 80 panels 228 us against 186 in step, of 390
// 180 and 155.
static int run_types(i2_evaluator* ev, const TaskSource (&src)[3]) {
    const i2_integrator& it = *ev->integ;
    const int nT = (int)ev->mesh->nT;
    RunMarks marks{ev};
    for (int t = 0; t < 3; ++t) {
        TypeState& ts = ev->type[t];
        const int64_t n = ts.n;
        ts.K = 0; ts.final_buf = 0; ts.refined_tasks = 0; ts.ms = 0.0;
        if (n == 0) continue;
        if (n > (int64_t)INT32_MAX) { set_error("%lld tasks of one type exceed the plain path's 32-bit task lists", (long long)n); return I2_ERR_RANGE; }
        I2_TRY(ts.buf[0].ensure(n));
        I2_TRY(ts.buf[1].ensure(n));
        I2_TRY(ts.results.ensure(3 * n));
        I2_TRY(ts.conv.ensure(n));
        if (it.fixed) continue;
        I2_TRY(ts.rest[0].ensure(n));
        I2_TRY(ts.rest[1].ensure(n));
        I2_TRY(ts.unconv.ensure(nT));
    }
    I2_TRY(marks.mark(RunMarks::NONE));
    if (it.fixed) {
        for (int t = 0; t < 3; ++t) {
            TypeState& ts = ev->type[t];
            if (ts.n == 0) continue;
            I2_HIP(hipMemsetAsync(ts.conv.p, it.fixed_level, (size_t)ts.n, ev->stream));
            I2_TRY(launch_level_of(ev, t, ts.implicit, ts.n, nullptr, src[t], it.fixed_level, ts.buf[0].p));
            ts.refined_tasks = ts.n << (2 * it.fixed_level);
            ts.K = it.fixed_level;
            I2_TRY(marks.mark(t));
        }
    } else {
        const int nc = 3 * (it.max_level + 1);
        I2_TRY(ev->d_counter.ensure(nc));
        uint8_t* flags[3];
        for (int t = 0; t < 3; ++t) flags[t] = ev->type[t].n > 0 ? ev->type[t].unconv.p : nullptr;
        hipLaunchKernelGGL(k_begin_run, dim3(blocks_for(std::max(nc, nT), 256)), dim3(256), 0, ev->stream, ev->d_counter.p, nc,
                           flags[0], flags[1], flags[2], nT);
        I2_TRY(check_launch("k_begin_run"));
        int64_t remaining[3];
        int cur_rest[3] = {0, 0, 0};
        for (int t = 0; t < 3; ++t) remaining[t] = ev->type[t].n;
        // levels 0 and 1 in one launch per type, but for profiled runs, which list each level's
        const bool first = it.max_level > 0 && !ev->profile;
        for (int iter = first ? 1 : 0; iter <= it.max_level && (remaining[0] > 0 || remaining[1] > 0 || remaining[2] > 0); ++iter) {
            if (iter > 1) I2_TRY(marks.mark(RunMarks::NONE));
            for (int t = 0; t < 3; ++t) {
                TypeState& ts = ev->type[t];
                const int64_t n = remaining[t];
                if (n == 0) continue;
                const int32_t* list = iter <= 1 ? nullptr : ts.rest[cur_rest[t]].p;
                double4* cur = ts.buf[iter % 2].p;
                ts.K = iter;
                ts.final_buf = iter % 2;
                if (first && iter == 1) {
                    I2_TRY(launch_first_levels_of(ev, t, ts, src[t], ev->d_counter.p + 3 + t));
                    ts.refined_tasks = n + (n << 2);
                    I2_TRY(marks.mark(t));
                    continue;
                }
                I2_TRY(launch_level_of(ev, t, ts.implicit, n, list, src[t], iter, cur));
                ts.refined_tasks += n << (2 * iter);
                if (iter > 0) {
                    hipLaunchKernelGGL(k_compare, dim3(blocks_for(n, 256)), dim3(256), 0, ev->stream, n, list, cur, ts.buf[1 - iter % 2].p,
                                       it.rule.pow2p, it.tol, it.quirk ? 0 : 1, iter, ts.conv.p, ts.rest[1 - cur_rest[t]].p,
                                       ev->d_counter.p + 3 * iter + t);
                    I2_TRY(check_launch("k_compare"));
                } else if (it.max_level == 0) {
                    I2_HIP(hipMemsetAsync(ts.conv.p, 0, (size_t)n, ev->stream));
                }
                I2_TRY(marks.mark(t));
            }
            if (iter == 0) continue;
            I2_HIP(hipMemcpyAsync(ev->h_counter, ev->d_counter.p + 3 * iter, 3 * sizeof(unsigned long long), hipMemcpyDeviceToHost, ev->stream));
            I2_HIP(hipStreamSynchronize(ev->stream));
            for (int t = 0; t < 3; ++t) {
                if (remaining[t] > 0) cur_rest[t] = 1 - cur_rest[t];
                remaining[t] = (int64_t)ev->h_counter[t];
            }
        }
        for (int t = 0; t < 3; ++t) {
            TypeState& ts = ev->type[t];
            if (ts.n > 0 && remaining[t] > 0)   // still unconverged after the comparison at maxLevel (all tasks when maxLevel = 0)
                I2_TRY(mark_unconverged(ev, ts.implicit, src[t], remaining[t], it.max_level == 0 ? nullptr : ts.rest[cur_rest[t]].p, ts.unconv.p));
        }
    }
    I2_TRY(marks.mark(RunMarks::NONE));
    FinalizeArgs F{};
    F.implicit = ev->type[I2_NOT_NEIGHBORS].implicit;
    F.clock = marks.clock();
    for (int t = 0; t < 3; ++t) {
        TypeState& ts = ev->type[t];
        F.t[t] = {ts.n, 0, src[t], ts.buf[ts.final_buf].p, ts.results.p};
        F.clock[2 * t] = F.clock[2 * t + 1] = 0;
    }
    I2_TRY(launch_finalize(ev->stream, ev->mesh->d_panels.p, F));
    I2_TRY(marks.mark(RunMarks::ALL));
    I2_HIP(hipStreamSynchronize(ev->stream));
    return marks.times();
}

TaskSource task_source(const i2_evaluator* ev, int type) {
    const i2_mesh* m = ev->mesh;
    const TypeState& ts = ev->type[type];
    TaskSource src;
    src.nT = (int)m->nT;
    if (ts.implicit) {
        src.n_unordered = m->pairs[I2_NOT_NEIGHBORS];
        src.row_start = m->d_row_start.p;
        src.nbr_start = m->d_nbr_start.p;
        src.nbr = m->d_nbr.p;
    } else {
        src.ij3 = ts.tasks.p;
    }
    return src;
}

int results_current(const i2_evaluator* ev) {
    if (!ev->ran) { set_error("no results: run the evaluator first"); return I2_ERR_STATE; }
    if (!ev->mesh->prepared || ev->mesh->generation != ev->run_generation) {
        set_error("the mesh was changed or prepared again after the last run: run the evaluator again");
        return I2_ERR_STATE;
    }
    return I2_OK;
}

int evaluator_run(i2_evaluator* ev, bool all_pairs, bool check) {
    const i2_mesh* m = ev->mesh;
    DeviceGuard g(m->device);
    if (!g.ok) return I2_ERR_HIP;
    ev->ran = false;
    ev->all_pairs = all_pairs;
    clear_launches(ev);
    // the reference runs the types one after another (evaluator3d.cu:173-186)
    const TaskSource src[3] = {task_source(ev, 0), task_source(ev, 1), task_source(ev, 2)};
    for (int t = 0; t < 3; ++t) ev->type[t].has_errors = ev->type[t].refinements_ready = false;
    I2_TRY(run_types(ev, src));
    for (int t = 0; t < 3; ++t) {
        TypeState& ts = ev->type[t];
        if (check && all_pairs && ts.n > 0) {
            I2_TRY(ts.errors.ensure(ts.n));
            const int64_t half = ts.n / 2;
            hipLaunchKernelGGL(k_symmetry, dim3(blocks_for(half, 256)), dim3(256), 0, ev->stream, half, ts.results.p, ts.errors.p);
            I2_TRY(check_launch("k_symmetry"));
            ts.has_errors = true;
        }
    }
    if (check && all_pairs) I2_HIP(hipStreamSynchronize(ev->stream));
    ev->ran = true;
    ev->ran_path = 0;
    ev->run_generation = m->generation;
    ev->integ->last_ev = ev;
    return I2_OK;
}

// The ordered task list [(i,j,k)] ++ [(j,i,n+k)] of Evaluator3D::runAllPairs
// (evaluator3d.cu:22-31, 156-169) from the mesh's list.
__global__ void k_ordered_tasks(int64_t n, const int32_t* __restrict__ list, int32_t* __restrict__ tasks) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const int32_t i = list[3 * q], j = list[3 * q + 1];
    int32_t *a = tasks + 3 * q, *b = tasks + 3 * (n + q);
    a[0] = i; a[1] = j; a[2] = (int32_t)q;
    b[0] = j; b[1] = i; b[2] = (int32_t)(n + q);
}

static int set_ordered_tasks(i2_evaluator* ev, int t, const DBuf<int32_t>& list) {
    TypeState& ts = ev->type[t];
    const int64_t n = ev->mesh->pairs[t];
    ts.implicit = false;
    ts.task_list_ready = false;
    ts.n = 2 * n;
    I2_TRY(ts.tasks.ensure(3 * ts.n));
    if (n == 0) return I2_OK;
    hipLaunchKernelGGL(k_ordered_tasks, dim3(blocks_for(n, 256)), dim3(256), 0, ev->stream, n, list.p, ts.tasks.p);
    return check_launch("k_ordered_tasks");
}

// ------------------------------------------------------------ results to the host
// Pinned staging memory, two slots per buffer: up to STAGING_KEPT buffers stay
// allocated while any evaluator lives (a buffer's allocation costs 60-300 us);
// a call takes one for itself, so calls of several threads do not meet.
constexpr size_t STAGING_SLOT = (size_t)1 << 20;
constexpr int STAGING_KEPT = 4;
static std::mutex g_staging_mutex;
static unsigned char* g_staging[STAGING_KEPT];
static int g_staging_count = 0;
static int64_t g_evaluators = 0;

struct Staging {
    unsigned char* p = nullptr;
    int take() {
        {
            std::lock_guard<std::mutex> lock(g_staging_mutex);
            if (g_staging_count > 0) p = g_staging[--g_staging_count];
        }
        if (!p) I2_HIP(hipHostMalloc((void**)&p, 2 * STAGING_SLOT, hipHostMallocPortable));
        return I2_OK;
    }
    ~Staging() {
        if (!p) return;
        {
            std::lock_guard<std::mutex> lock(g_staging_mutex);
            if (g_evaluators > 0 && g_staging_count < STAGING_KEPT) { g_staging[g_staging_count++] = p; return; }
        }
        (void)hipHostFree(p);
    }
};
static void evaluator_count(int64_t d) {
    std::lock_guard<std::mutex> lock(g_staging_mutex);
    g_evaluators += d;
    if (g_evaluators == 0) while (g_staging_count > 0) (void)hipHostFree(g_staging[--g_staging_count]);
}

// A type's outputs of tasks z0 .. z0 + n - 1 into a staging slot, one array after
// the other: integrals, results, errors, tasks, convergence iterations (those
// asked for).  The device writes host memory, lines in order.  One launch instead
// of a copy per array (10-20 us each, whatever its size).
struct PackArgs {
    TaskSource src;
    bool implicit, tasks;
    const uint64_t *ints, *res, *err;
    const int8_t* conv;
};
__global__ __launch_bounds__(256) void k_pack(PackArgs P, int64_t z0, int64_t n, unsigned char* out) {
    __shared__ int32_t t3[3 * 256];
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
    uint64_t* o = reinterpret_cast<uint64_t*>(out);
    if (P.ints) { for (int64_t q = t; q < 4 * n; q += step) o[q] = P.ints[4 * z0 + q]; o += 4 * n; }
    if (P.res) { for (int64_t q = t; q < 3 * n; q += step) o[q] = P.res[3 * z0 + q]; o += 3 * n; }
    if (P.err) { for (int64_t q = t; q < n; q += step) o[q] = P.err[z0 + q]; o += n; }
    int32_t* o4 = reinterpret_cast<int32_t*>(o);
    if (P.tasks) {
        for (int64_t base = 256 * (int64_t)blockIdx.x; base < n; base += step) {
            const int64_t z = z0 + base + threadIdx.x;
            if (base + threadIdx.x < n) {
                int i, j;
                if (P.implicit) task_ij<true>(P.src, z, &i, &j);
                else task_ij<false>(P.src, z, &i, &j);
                t3[3 * threadIdx.x] = i; t3[3 * threadIdx.x + 1] = j;
                t3[3 * threadIdx.x + 2] = P.implicit ? (int32_t)z : P.src.ij3[3 * z + 2];
            }
            __syncthreads();
            const int64_t m = 3 * (n - base < 256 ? n - base : 256);
            for (int64_t q = threadIdx.x; q < m; q += 256) o4[3 * base + q] = t3[q];
            __syncthreads();
        }
        o4 += 3 * n;
    }
    if (P.conv) { int8_t* o1 = reinterpret_cast<int8_t*>(o4); for (int64_t q = t; q < n; q += step) o1[q] = P.conv[z0 + q]; }
}

static int read_back(hipStream_t st, const PackArgs& P, int64_t n, double* ints, double* res, double* err, int32_t* tasks, int8_t* conv) {
    const int64_t each = 32 * (ints != nullptr) + 24 * (res != nullptr) + 8 * (err != nullptr) + 12 * (tasks != nullptr) + (conv != nullptr);
    if (each == 0) return I2_OK;
    Staging S;
    I2_TRY(S.take());
    const int64_t most = (int64_t)STAGING_SLOT / each, chunks = (n + most - 1) / most;
    struct Events {
        hipEvent_t e[2] = {nullptr, nullptr};
        ~Events() { for (hipEvent_t x : e) if (x) (void)hipEventDestroy(x); }
    } E;
    // The slots are not coherent memory (Portable alone leaves that to
    // HIP_HOST_COHERENT): the host sees a chunk after a release to the system, which
    // a stream's synchronisation is and an event's record is only with the flag.
    if (chunks > 1) for (hipEvent_t& e : E.e) I2_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming | hipEventReleaseToSystem));
    auto launch = [&](int64_t c) -> int {
        const int64_t z0 = c * most, m = std::min(most, n - z0);
        hipLaunchKernelGGL(k_pack, dim3((unsigned)std::min<int64_t>((m + 255) / 256, 256)), dim3(256), 0, st, P, z0, m,
                           S.p + (c & 1) * STAGING_SLOT);
        I2_TRY(check_launch("k_pack"));
        if (chunks > 1) I2_HIP(hipEventRecord(E.e[c & 1], st));
        return I2_OK;
    };
    int status = launch(0);
    for (int64_t c = 0; c < chunks && status == I2_OK; ++c) {
        if (c + 1 < chunks) status = launch(c + 1);       // fills the other slot meanwhile
        if (status != I2_OK) break;
        I2_HIP(chunks > 1 ? hipEventSynchronize(E.e[c & 1]) : hipStreamSynchronize(st));
        const int64_t z0 = c * most, m = std::min(most, n - z0);
        const unsigned char* p = S.p + (c & 1) * STAGING_SLOT;
        auto take = [&](auto* dst, int64_t per) {
            if (!dst) return;
            memcpy(dst + per * z0, p, sizeof(*dst) * (size_t)(per * m));
            p += sizeof(*dst) * (size_t)(per * m);
        };
        take(ints, 4); take(res, 3); take(err, 1); take(tasks, 3); take(conv, 1);
    }
    if (status != I2_OK) (void)hipStreamSynchronize(st);  // before the slots are given back
    return status;
}

// ------------------------------------------------------------ allocation-free runPairs of one type
// Device scratch of i2_evaluator_run_tasks_noalloc: one level buffer (the
// caller's integrals are the other), the two lists of unconverged tasks, and
// counters.  Every GPU holds its own copy for the life of the process.  In
// host code the array's name is not a device address: the kernels get the
// address hipGetSymbolAddress returns for the current device.
constexpr size_t NOALLOC_REST0 = 32 * (size_t)I2_NOALLOC_MAX_TASKS;
constexpr size_t NOALLOC_REST1 = 36 * (size_t)I2_NOALLOC_MAX_TASKS;
constexpr size_t NOALLOC_COUNTERS = 40 * (size_t)I2_NOALLOC_MAX_TASKS;   // [0] unconverged tasks, [1] first bad task
constexpr size_t NOALLOC_BYTES = NOALLOC_COUNTERS + 256;
static_assert(sizeof(double4) == 32 && NOALLOC_COUNTERS % 256 == 0, "scratch layout");
static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

constexpr int NOALLOC_DEVICES = 64;
static std::mutex g_scratch_mutex;
static unsigned char* g_scratch[NOALLOC_DEVICES] = {};

// This device's scratch address, looked up on the first call with the device current.
static int scratch_address(int device, unsigned char** out) {
    if (device < 0 || device >= NOALLOC_DEVICES) {
        set_error("device %d is beyond the %d devices the scratch table holds", device, NOALLOC_DEVICES);
        return I2_ERR_RANGE;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            (void)hipGetLastError();
            set_error("hipGetSymbolAddress(scratch) failed on device %d: %s", device, hipGetErrorString(e));
            return I2_ERR_HIP;
        }
        g_scratch[device] = static_cast<unsigned char*>(p);
    }
    *out = g_scratch[device];
    return I2_OK;
}

// The task-list check of runPairs on the device: *bad receives the smallest
// 2 (q + 1) + kind over tasks q that fail, kind 0 for a cell outside [0, nT)
// and 1 for a pair that does not share `expect` vertices (all ones when none).
__global__ void k_check_tasks(int64_t n, const int32_t* __restrict__ tasks, int nT, const Panel* __restrict__ panels,
                              int expect, unsigned long long* bad) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const int i = tasks[3 * q], j = tasks[3 * q + 1];
    const unsigned long long key = 2ull * (unsigned long long)(q + 1);
    if (i < 0 || j < 0 || i >= nT || j >= nT) { atomicMin(bad, key); return; }
    if (shared_count(panels[i], panels[j]) != expect) atomicMin(bad, key + 1ull);
}

// The same for lists just uploaded, whose third entries are set as well.  The
// triangles' numbers are compared as the reference's lists define the types.
__global__ void k_take_tasks(int64_t n, int32_t* __restrict__ tasks, int64_t nT, const int32_t* __restrict__ tri, int expect,
                             unsigned long long* bad) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const int64_t i = tasks[3 * q], j = tasks[3 * q + 1];
    tasks[3 * q + 2] = (int32_t)q;
    const unsigned long long key = 2ull * (unsigned long long)(q + 1);
    if (i < 0 || j < 0 || i >= nT || j >= nT) { atomicMin(bad, key); return; }
    int cnt = 0;
    for (int x = 0; x < 3; ++x) {
        const int32_t a = tri[3 * i + x];
        cnt += a == tri[3 * j] || a == tri[3 * j + 1] || a == tri[3 * j + 2];
    }
    if (cnt != expect) atomicMin(bad, key + 1ull);
}

// run_types for one type's explicit device list, with the caller's integrals as level
// buffer 0 and the scratch as level buffer 1: the same launches in the same
// order, so the same values, levels and K.
template <int TYPE>
static int run_tasks_noalloc(i2_evaluator* ev, const int32_t* d_tasks3, int64_t n, unsigned char* S, double4* ints,
                             double* results, int8_t* conv, int* Kout) {
    const i2_integrator& it = *ev->integ;
    const Panel* panels = ev->mesh->d_panels.p;
    const hipStream_t st = ev->stream;
    TaskSource src;
    src.nT = (int)ev->mesh->nT;
    src.ij3 = d_tasks3;
    double4* buf[2] = {ints, reinterpret_cast<double4*>(S)};
    int32_t* rest[2] = {reinterpret_cast<int32_t*>(S + NOALLOC_REST0), reinterpret_cast<int32_t*>(S + NOALLOC_REST1)};
    unsigned long long* counter = reinterpret_cast<unsigned long long*>(S + NOALLOC_COUNTERS);
    auto level = [&](int64_t items, const int32_t* list, int L, double4* out) {
        const int ll = lanes_log2_for(L, items);
        hipLaunchKernelGGL((k_level<TYPE, false>), dim3(blocks_for(items << ll, 256)), dim3(256), 0, st, items, list, src,
                           panels, it.rule, L, ll, per_log2_for(L, ll), out);
        return check_launch("k_level");
    };
    int K = 0, final_buf = 0;
    if (it.fixed) {
        I2_HIP(hipMemsetAsync(conv, it.fixed_level, (size_t)n, st));
        I2_TRY(level(n, nullptr, it.fixed_level, buf[0]));
        K = it.fixed_level;
    } else {
        const bool first = it.max_level > 0 && !ev->profile;
        if (!first) {
            I2_HIP(hipMemsetAsync(conv, 0, (size_t)n, st));
            I2_TRY(level(n, nullptr, 0, buf[0]));
        }
        int64_t remaining = n;
        int iter = 0, cur_rest = 0;
        while (remaining > 0 && iter < it.max_level) {
            ++iter;
            const int32_t* list = (iter == 1) ? nullptr : rest[cur_rest];
            I2_HIP(hipMemsetAsync(counter, 0, sizeof(unsigned long long), st));
            if (first && iter == 1)
                I2_TRY((launch_first_levels<TYPE, false>(st, panels, it, n, src, buf[0], buf[1], conv, rest[1], counter)));
            else
                I2_TRY(level(remaining, list, iter, buf[iter % 2]));
            if (!(first && iter == 1)) hipLaunchKernelGGL(k_compare, dim3(blocks_for(remaining, 256)), dim3(256), 0, st, remaining, list, buf[iter % 2],
                               buf[(iter - 1) % 2], it.rule.pow2p, it.tol, it.quirk ? 0 : 1, iter, conv, rest[1 - cur_rest],
                               counter);
            I2_TRY(check_launch("k_compare"));
            I2_HIP(hipMemcpyAsync(ev->h_counter, counter, sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
            I2_HIP(hipStreamSynchronize(st));
            remaining = (int64_t)*ev->h_counter;
            cur_rest = 1 - cur_rest;
        }
        K = iter;
        final_buf = iter % 2;
    }
    if (final_buf == 1) I2_HIP(hipMemcpyAsync(buf[0], buf[1], sizeof(double4) * (size_t)n, hipMemcpyDeviceToDevice, st));
    FinalizeArgs F{};
    F.t[TYPE] = {n, 0, src, buf[0], results};
    I2_TRY(launch_finalize(st, panels, F));
    I2_HIP(hipStreamSynchronize(st));
    *Kout = K;
    return I2_OK;
}

}  // namespace i2

using namespace i2;

// Live integrators: an evaluator destroyed after its integrator must not touch it.
static std::mutex g_integrators_mutex;
static std::unordered_set<const i2_integrator*> g_integrators;

extern "C" {

int i2_integrator_create(i2_integrator** out, const i2_mesh* mesh, const double* L12, const double* w, int nPts, int order) {
    if (!out || !mesh || !L12 || !w) { set_error("null argument"); return I2_ERR_INVALID; }
    if (nPts < 1 || nPts > MAX_POINTS) { set_error("rule must have 1..%d points", MAX_POINTS); return I2_ERR_INVALID; }
    if (order < 0 || order > 30) { set_error("rule order out of range"); return I2_ERR_INVALID; }
    i2_integrator* it = new i2_integrator;
    it->mesh = mesh;
    it->rule.n = nPts;
    it->rule.order = order;
    it->rule.pow2p = (double)(1 << order);
    for (int k = 0; k < MAX_POINTS; ++k) {
        if (k < nPts) {
            it->rule.L1[k] = L12[2 * k];
            it->rule.L2[k] = L12[2 * k + 1];
            it->rule.L3[k] = 1.0 - L12[2 * k] - L12[2 * k + 1];
            it->rule.w[k] = w[k];
        } else {
            it->rule.L1[k] = it->rule.L2[k] = it->rule.L3[k] = it->rule.w[k] = 0.0;
        }
    }
    it->rule.centroid = i2d::rule_centroid(it->rule.L1, it->rule.L2, nPts);
    it->rule.reach = i2d::rule_reach(it->rule.L1, it->rule.L2, it->rule.L3, nPts);
    it->rule.pad = 0;
    {
        std::lock_guard<std::mutex> lock(g_integrators_mutex);
        g_integrators.insert(it);
    }
    *out = it;
    return I2_OK;
}
void i2_integrator_destroy(i2_integrator* it) {
    if (!it) return;
    {
        std::lock_guard<std::mutex> lock(g_integrators_mutex);
        g_integrators.erase(it);
    }
    release_refined_mesh(it);
    delete it;
}

int i2_integrator_set_fixed_refinement_level(i2_integrator* it, int level) {
    if (!it) { set_error("null integrator"); return I2_ERR_INVALID; }
    if (level < 0 || level > 12) { set_error("fixed refinement level %d out of range [0, 12]", level); return I2_ERR_RANGE; }
    it->fixed = 1;
    it->fixed_level = level;
    return I2_OK;
}
int i2_integrator_set_error_control(i2_integrator* it, int maxLevel, double tol, int refParityQuirk) {
    if (!it) { set_error("null integrator"); return I2_ERR_INVALID; }
    if (maxLevel < 0 || maxLevel > 12) { set_error("maxLevel %d out of range [0, 12]", maxLevel); return I2_ERR_RANGE; }
    if (!(tol > 0)) { set_error("tolerance must be positive"); return I2_ERR_INVALID; }
    it->fixed = 0;
    it->max_level = maxLevel;
    it->tol = tol;
    it->quirk = refParityQuirk ? 1 : 0;
    return I2_OK;
}

int i2_evaluator_create(i2_evaluator** out, const i2_mesh* m, i2_integrator* it) {
    if (!out || !m || !it) { set_error("null argument"); return I2_ERR_INVALID; }
    *out = nullptr;
    if (!m->prepared) { set_error("mesh not prepared (call i2_mesh_prepare)"); return I2_ERR_STATE; }
    DeviceGuard g(m->device);
    if (!g.ok) return I2_ERR_HIP;
    i2_evaluator* ev = new i2_evaluator;
    evaluator_count(1);
    ev->mesh = m;
    ev->integ = it;
    if (hipStreamCreateWithFlags(&ev->stream, hipStreamNonBlocking) != hipSuccess ||
        hipHostMalloc((void**)&ev->h_counter, 9 * sizeof(unsigned long long), hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        set_error("failed to create evaluator stream/events");
        i2_evaluator_destroy(ev);
        return I2_ERR_HIP;
    }
    if (ev->d_counter.ensure(1) != I2_OK) { i2_evaluator_destroy(ev); return I2_ERR_ALLOC; }
    *out = ev;
    return I2_OK;
}

void i2_evaluator_destroy(i2_evaluator* ev) {
    if (!ev) return;
    {
        DeviceGuard g(ev->mesh->device);
        if (ev->stream) (void)hipStreamSynchronize(ev->stream);
        for (auto& ts : ev->type) {
            ts.tasks.reset(); ts.new_tasks.reset(); ts.buf[0].reset(); ts.buf[1].reset(); ts.results.reset(); ts.errors.reset();
            ts.conv.reset(); ts.rest[0].reset(); ts.rest[1].reset();
            ts.unconv.reset(); ts.refinements.reset(); ts.task_list.reset();
        }
        {
            std::lock_guard<std::mutex> lock(g_integrators_mutex);
            if (g_integrators.count(ev->integ) && ev->integ->last_ev == ev) ev->integ->last_ev = nullptr;
        }
        clear_launches(ev);
        engine_release_evaluator(ev);
        adjoint_release(ev->adj);
        ev->d_counter.reset();
        if (ev->h_counter) (void)hipHostFree(ev->h_counter);
        for (hipEvent_t e : ev->marks) (void)hipEventDestroy(e);
        if (ev->stream) (void)hipStreamDestroy(ev->stream);
    }
    evaluator_count(-1);
    delete ev;
}

int i2_evaluator_run_all_pairs(i2_evaluator* ev, int checkCorrectness) {
    if (!ev) { set_error("null evaluator"); return I2_ERR_INVALID; }
    const i2_mesh* m = ev->mesh;
    if (!m->prepared) { set_error("mesh not prepared"); return I2_ERR_STATE; }
    DeviceGuard g(m->device);
    if (!g.ok) return I2_ERR_HIP;
    ev->ran = false;
    if (!ev->all_pairs_lists || ev->all_pairs_generation != m->generation) {
        // the ordered lists depend only on the mesh: written once per prepared mesh
        ev->all_pairs_lists = false;
        I2_TRY(set_ordered_tasks(ev, I2_SIMPLE_NEIGHBORS, m->d_simple));
        I2_TRY(set_ordered_tasks(ev, I2_ATTACHED_NEIGHBORS, m->d_attached));
        TypeState& d = ev->type[I2_NOT_NEIGHBORS];
        d.implicit = true;
        d.task_list_ready = false;
        d.n = 2 * m->pairs[I2_NOT_NEIGHBORS];
        d.tasks.reset();
        ev->all_pairs_lists = true;
        ev->all_pairs_generation = m->generation;
    }
    ev->tasks_generation = m->generation;
    if (ev->path == 0) return evaluator_run(ev, true, checkCorrectness != 0);
    // batched path: per-pair outputs in the same task order
    ev->ran = false;
    ev->all_pairs = true;
    clear_launches(ev);
    I2_TRY(engine_run_evaluator(ev));
    for (int t = 0; t < 3; ++t) {
        TypeState& ts = ev->type[t];
        ts.has_errors = false;
        ts.refinements_ready = false;
        if (checkCorrectness && ts.n > 0) {
            const double4* ints;
            const double* res;
            const int8_t* conv;
            engine_evaluator_outputs(ev, t, &ints, &res, &conv);
            I2_TRY(ts.errors.ensure(ts.n));
            const int64_t half = ts.n / 2;
            hipLaunchKernelGGL(k_symmetry, dim3(blocks_for(half, 256)), dim3(256), 0, ev->stream, half, res, ts.errors.p);
            I2_TRY(check_launch("k_symmetry"));
            ts.has_errors = true;
        }
    }
    I2_HIP(hipStreamSynchronize(ev->stream));
    ev->ran = true;
    ev->ran_path = 1;
    ev->run_generation = m->generation;
    ev->integ->last_ev = ev;
    return I2_OK;
}

int i2_evaluator_set_path(i2_evaluator* ev, int path) {
    if (!ev || (path != 0 && path != 1)) { set_error("invalid argument"); return I2_ERR_INVALID; }
    ev->path = path;
    return I2_OK;
}

int i2_evaluator_set_tuning(i2_evaluator* ev, int pairsPerWorkgroup, int pointsPerLane) {
    if (!ev) { set_error("null evaluator"); return I2_ERR_INVALID; }
    if (pairsPerWorkgroup < 1 || pairsPerWorkgroup > 4096 || (pairsPerWorkgroup & (pairsPerWorkgroup - 1)) != 0 ||
        (pointsPerLane != 1 && pointsPerLane != 2 && pointsPerLane != 4 && pointsPerLane != 13)) {
        set_error("invalid launch shape (%d pairs per workgroup, %d points per lane)", pairsPerWorkgroup, pointsPerLane);
        return I2_ERR_INVALID;
    }
    ev->fast_P = pairsPerWorkgroup;
    ev->fast_ppl = pointsPerLane;
    ev->fast_tuned = true;
    return I2_OK;
}

int i2_evaluator_run_pairs(i2_evaluator* ev, const int32_t* simple3, int64_t nSimple, const int32_t* attached3, int64_t nAttached,
                           const int32_t* not3, int64_t nNot) {
    if (!ev) { set_error("null evaluator"); return I2_ERR_INVALID; }
    if ((nSimple && !simple3) || (nAttached && !attached3) || (nNot && !not3) || nSimple < 0 || nAttached < 0 || nNot < 0) {
        set_error("invalid task lists");
        return I2_ERR_INVALID;
    }
    const i2_mesh* m = ev->mesh;
    if (!m->prepared) { set_error("mesh not prepared"); return I2_ERR_STATE; }
    const int32_t* lists[3] = {simple3, attached3, not3};
    const int64_t ns[3] = {nSimple, nAttached, nNot};
    DeviceGuard g(m->device);
    if (!g.ok) return I2_ERR_HIP;
    // Every list is checked before any is installed, so that a rejected call
    // leaves the previous run's tasks and outputs as they were.  The lists are
    // checked where they are used: host passes over 161,000 tasks and a copy of
    // them took 300 us.
    I2_TRY(ev->d_counter.ensure(3));
    I2_HIP(hipMemsetAsync(ev->d_counter.p, 0xff, 3 * sizeof(unsigned long long), ev->stream));
    for (int t = 0; t < 3; ++t) {
        if (ns[t] == 0) continue;
        I2_TRY(ev->type[t].new_tasks.ensure(3 * ns[t]));
        I2_HIP(hipMemcpyAsync(ev->type[t].new_tasks.p, lists[t], sizeof(int32_t) * 3 * (size_t)ns[t], hipMemcpyHostToDevice, ev->stream));
        // the integrand of each type is only valid for pairs of that type
        const int expect = (t == I2_SIMPLE_NEIGHBORS) ? 1 : (t == I2_ATTACHED_NEIGHBORS ? 2 : 0);
        hipLaunchKernelGGL(k_take_tasks, dim3(blocks_for(ns[t], 256)), dim3(256), 0, ev->stream, ns[t], ev->type[t].new_tasks.p,
                           m->nT, m->d_tri.p, expect, ev->d_counter.p + t);
        I2_TRY(check_launch("k_take_tasks"));
    }
    I2_HIP(hipMemcpyAsync(ev->h_counter, ev->d_counter.p, 3 * sizeof(unsigned long long), hipMemcpyDeviceToHost, ev->stream));
    I2_HIP(hipStreamSynchronize(ev->stream));
    for (int t = 0; t < 3; ++t) {
        const unsigned long long key = ev->h_counter[t];
        if (key == ~0ull) continue;
        const int64_t q = (int64_t)(key / 2) - 1;
        const int32_t i = lists[t][3 * q], j = lists[t][3 * q + 1];
        if (key % 2 == 0) { set_error("task %lld of type %d references a cell outside [0, %lld)", (long long)q, t, (long long)m->nT); return I2_ERR_INVALID; }
        const int32_t* a = &m->h_tri[3 * (int64_t)i];
        const int32_t* b = &m->h_tri[3 * (int64_t)j];
        int cnt = 0;
        for (int x = 0; x < 3; ++x) if (a[x] == b[0] || a[x] == b[1] || a[x] == b[2]) ++cnt;
        set_error("task %lld (%d, %d) shares %d vertices but was given as type %d", (long long)q, i, j, cnt, t);
        return I2_ERR_TOPOLOGY;
    }
    ev->ran = false;
    ev->all_pairs_lists = false;
    for (int t = 0; t < 3; ++t) {
        TypeState& ts = ev->type[t];
        ts.implicit = false;
        ts.task_list_ready = false;
        ts.n = ns[t];
        std::swap(ts.tasks, ts.new_tasks);
        I2_TRY(ts.tasks.ensure(3 * ns[t]));
    }
    ev->tasks_generation = m->generation;
    return evaluator_run(ev, false, false);
}

int i2_evaluator_run_tasks_noalloc(i2_evaluator* ev, int type, const int32_t* d_tasks3, int64_t n, double* d_integrals4,
                                   double* d_results3, int8_t* d_conv, int* K) {
    if (!ev || !K || type < 0 || type > 2 || n < 0) { set_error("invalid argument"); return I2_ERR_INVALID; }
    *K = 0;
    if (n > I2_NOALLOC_MAX_TASKS) {
        set_error("%lld tasks exceed the allocation-free limit of %d per call", (long long)n, I2_NOALLOC_MAX_TASKS);
        return I2_ERR_RANGE;
    }
    if (n > 0 && (!d_tasks3 || !d_integrals4 || !d_results3 || !d_conv)) { set_error("null device array"); return I2_ERR_INVALID; }
    if (reinterpret_cast<uintptr_t>(d_integrals4) % alignof(double4) || reinterpret_cast<uintptr_t>(d_results3) % alignof(double) ||
        reinterpret_cast<uintptr_t>(d_tasks3) % alignof(int32_t)) {
        set_error("misaligned device array (the integrals need %zu-byte alignment)", alignof(double4));
        return I2_ERR_INVALID;
    }
    const i2_mesh* m = ev->mesh;
    if (!m->prepared) { set_error("mesh not prepared"); return I2_ERR_STATE; }
    DeviceGuard g(m->device);
    if (!g.ok) return I2_ERR_HIP;
    unsigned char* S = nullptr;
    I2_TRY(scratch_address(m->device, &S));
    if (n == 0) return I2_OK;
    // the lists are checked where they are, on the device
    unsigned long long* bad = reinterpret_cast<unsigned long long*>(S + NOALLOC_COUNTERS) + 1;
    I2_HIP(hipMemsetAsync(bad, 0xff, sizeof(unsigned long long), ev->stream));
    const int expect = (type == I2_SIMPLE_NEIGHBORS) ? 1 : (type == I2_ATTACHED_NEIGHBORS ? 2 : 0);
    hipLaunchKernelGGL(k_check_tasks, dim3(blocks_for(n, 256)), dim3(256), 0, ev->stream, n, d_tasks3, (int)m->nT,
                       m->d_panels.p, expect, bad);
    I2_TRY(check_launch("k_check_tasks"));
    I2_HIP(hipMemcpyAsync(ev->h_counter, bad, sizeof(unsigned long long), hipMemcpyDeviceToHost, ev->stream));
    I2_HIP(hipStreamSynchronize(ev->stream));
    const unsigned long long key = *ev->h_counter;
    if (key != ~0ull) {
        const unsigned long long q = key / 2 - 1;
        if (key % 2 == 0) {
            set_error("task %llu of type %d references a cell outside [0, %lld)", q, type, (long long)m->nT);
            return I2_ERR_INVALID;
        }
        set_error("task %llu does not share %d vertices as pairs of type %d do", q, expect, type);
        return I2_ERR_TOPOLOGY;
    }
    double4* ints = reinterpret_cast<double4*>(d_integrals4);
    if (type == I2_SIMPLE_NEIGHBORS) return run_tasks_noalloc<I2_SIMPLE_NEIGHBORS>(ev, d_tasks3, n, S, ints, d_results3, d_conv, K);
    if (type == I2_ATTACHED_NEIGHBORS) return run_tasks_noalloc<I2_ATTACHED_NEIGHBORS>(ev, d_tasks3, n, S, ints, d_results3, d_conv, K);
    return run_tasks_noalloc<I2_NOT_NEIGHBORS>(ev, d_tasks3, n, S, ints, d_results3, d_conv, K);
}

int i2_evaluator_task_count(const i2_evaluator* ev, int type, int64_t* n) {
    if (!ev || !n || type < 0 || type > 2) { set_error("invalid argument"); return I2_ERR_INVALID; }
    *n = ev->type[type].n;
    return I2_OK;
}

int i2_evaluator_get_results(const i2_evaluator* ev, int type, int32_t* tasks3, double* integrals4, double* results3,
                             double* errors, int8_t* convLevel) {
    if (!ev || type < 0 || type > 2) { set_error("invalid argument"); return I2_ERR_INVALID; }
    I2_TRY(results_current(ev));
    const TypeState& ts = ev->type[type];
    const i2_mesh* m = ev->mesh;
    DeviceGuard g(m->device);
    if (!g.ok) return I2_ERR_HIP;
    if (ts.n == 0) return I2_OK;
    if (errors && !ts.has_errors) { set_error("symmetry errors were not computed (runAllPairs with checkCorrectness)"); return I2_ERR_STATE; }
    const double4* d_ints = ts.buf[ts.final_buf].p;
    const double* d_res = ts.results.p;
    const int8_t* d_conv = ts.conv.p;
    if (ev->ran_path == 1) engine_evaluator_outputs(ev, type, &d_ints, &d_res, &d_conv);
    PackArgs P{};
    P.src = task_source(ev, type);
    P.implicit = ts.implicit;
    if (integrals4) P.ints = reinterpret_cast<const uint64_t*>(d_ints);
    if (results3) P.res = reinterpret_cast<const uint64_t*>(d_res);
    if (errors) P.err = reinterpret_cast<const uint64_t*>(ts.errors.p);
    if (convLevel) P.conv = d_conv;
    P.tasks = tasks3 != nullptr;
    return read_back(ev->stream, P, ts.n, integrals4, results3, errors, tasks3, convLevel);
}

int i2_evaluator_refinement_iterations(const i2_evaluator* ev, int type, int* K) {
    if (!ev || !K || type < 0 || type > 2) { set_error("invalid argument"); return I2_ERR_INVALID; }
    I2_TRY(results_current(ev));
    *K = ev->type[type].K;
    return I2_OK;
}

int i2_evaluator_type_stats(const i2_evaluator* ev, int type, double* ms, int64_t* refinedTasks) {
    if (!ev || type < 0 || type > 2) { set_error("invalid argument"); return I2_ERR_INVALID; }
    I2_TRY(results_current(ev));
    if (ms) *ms = ev->type[type].ms;
    if (refinedTasks) *refinedTasks = ev->type[type].refined_tasks;
    return I2_OK;
}

int i2_evaluator_set_profiling(i2_evaluator* ev, int enable) {
    if (!ev) { set_error("null evaluator"); return I2_ERR_INVALID; }
    ev->profile = enable != 0;
    return I2_OK;
}

int i2_evaluator_sweep_ms(const i2_evaluator* ev, double* ms) {
    if (!ev || !ms) { set_error("null argument"); return I2_ERR_INVALID; }
    if (!ev->ran || ev->ran_path != 1 || !ev->profile) { set_error("no profiled batched run"); return I2_ERR_STATE; }
    *ms = ev->fast_sweep_ms;
    return I2_OK;
}

int i2_evaluator_launch_records(const i2_evaluator* ev, int64_t capacity, int32_t* type_level, int64_t* tasks, double* ms, int64_t* count) {
    if (!ev || !count) { set_error("null argument"); return I2_ERR_INVALID; }
    *count = (int64_t)ev->launches.size();
    const int64_t n = std::min<int64_t>(capacity, (int64_t)ev->launches.size());
    DeviceGuard g(ev->mesh->device);
    if (!g.ok) return I2_ERR_HIP;
    for (int64_t q = 0; q < n; ++q) {
        const LaunchRecord& r = ev->launches[q];
        if (type_level) { type_level[2 * q] = r.type; type_level[2 * q + 1] = r.level; }
        if (tasks) tasks[q] = r.tasks;
        if (ms) {
            float f = 0.f;
            I2_HIP(hipEventElapsedTime(&f, r.e0, r.e1));
            ms[q] = f;
        }
    }
    return I2_OK;
}

int i2_device_synchronize(int device) {
    DeviceGuard g(device);
    if (!g.ok) return I2_ERR_HIP;
    I2_HIP(hipDeviceSynchronize());
    return I2_OK;
}

int i2_evaluator_output_results_to_file(const i2_evaluator* ev, int type, int format, const char* dir) {
    if (!ev || type < 0 || type > 2 || (format != I2_OUTPUT_PLAIN_TEXT && format != I2_OUTPUT_CSV)) {
        set_error("invalid argument");
        return I2_ERR_INVALID;
    }
    I2_TRY(results_current(ev));
    const TypeState& ts = ev->type[type];
    if (ts.n == 0) { set_error("no tasks of type %d", type); return I2_ERR_STATE; }   // the reference returns false
    std::vector<int32_t> tasks(3 * ts.n);
    std::vector<double> res(3 * ts.n), err;
    I2_TRY(i2_evaluator_get_results(ev, type, tasks.data(), nullptr, res.data(), nullptr, nullptr));
    if (ts.has_errors) { err.resize(ts.n); I2_TRY(i2_evaluator_get_results(ev, type, nullptr, nullptr, nullptr, err.data(), nullptr)); }
    static const char* names[3] = {"SimpleNeighbors", "AttachedNeighbors", "NotNeighbors"};
    std::string path = dir ? std::string(dir) + "/" : std::string();
    path += names[type];
    path += (format == I2_OUTPUT_CSV) ? ".csv" : ".dat";
    std::ofstream f(path);
    if (!f.is_open()) { set_error("cannot open %s for writing", path.c_str()); return I2_ERR_IO; }
    // layout of evaluator3d.cu:418-441 (default stream precision)
    if (format == I2_OUTPUT_CSV) {
        f << "\"TaskI\";\"TaskJ\";\"IntegralX\";\"IntegralY\";\"IntegralZ\"";
        if (ts.has_errors) f << ";\"Error\"";
        f << "\n";
    }
    for (int64_t q = 0; q < ts.n; ++q) {
        if (format == I2_OUTPUT_PLAIN_TEXT) {
            f << "(" << tasks[3 * q] << ", " << tasks[3 * q + 1] << "): [" << res[3 * q] << ", " << res[3 * q + 1] << ", " << res[3 * q + 2] << "]";
            if (ts.has_errors) f << ", error = " << err[q];
        } else {
            f << tasks[3 * q] << ";" << tasks[3 * q + 1] << ";" << res[3 * q] << ";" << res[3 * q + 1] << ";" << res[3 * q + 2];
            if (ts.has_errors) f << ";" << err[q];
        }
        f << "\n";
    }
    if (!f.good()) { set_error("write to %s failed", path.c_str()); return I2_ERR_IO; }
    return I2_OK;
}

}  // extern "C"
