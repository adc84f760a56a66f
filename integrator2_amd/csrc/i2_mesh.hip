// i2_mesh.hip -- Mesh3D behind the C ABI: file loading, upload, the panel
// table kernel (normals, areas, edge tangents) and the neighbour lists.
#include "i2_internal.hpp"
#include "i2_math.hpp"

#include <algorithm>
#include <fstream>
#include <sstream>

namespace i2 {

static thread_local std::string g_last_error;

void set_error(const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
}
void clear_error() { g_last_error.clear(); }

// One thread per panel: vertices, tangents of the inner integral, unit
// normal n = (v2-v1)x(v3-v1)/|.| and area |.|/2 (src/Mesh3d.cu:23-32, 62-71).
__global__ void k_panel_table(int64_t nT, const double* __restrict__ xyz, const int32_t* __restrict__ tri,
                              i2d::Panel* __restrict__ panels, double* __restrict__ normals, double* __restrict__ measures) {
    using namespace i2d;
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nT) return;
    const int v0 = tri[3 * c], v1 = tri[3 * c + 1], v2 = tri[3 * c + 2];
    const d3 A = {xyz[3 * v0], xyz[3 * v0 + 1], xyz[3 * v0 + 2]};
    const d3 B = {xyz[3 * v1], xyz[3 * v1 + 1], xyz[3 * v1 + 2]};
    const d3 C = {xyz[3 * v2], xyz[3 * v2 + 1], xyz[3 * v2 + 2]};
    Panel P;
    P.a = A; P.b = B; P.c = C;
    P.ta = unit(C - B);
    P.tb = unit(A - C);
    P.tc = unit(B - A);
    const d3 cr = cross(B - A, C - A);
    P.n = unit(cr);
    P.area = vlen(cr) * 0.5;
    P.v0 = v0; P.v1 = v1; P.v2 = v2; P.pad = 0;
    panels[c] = P;
    normals[3 * c] = P.n.x; normals[3 * c + 1] = P.n.y; normals[3 * c + 2] = P.n.z;
    measures[c] = P.area;
}

// ------------------------------------------------------------ neighbour classification
// kDetermineNeighborType (src/Mesh3d.cu:93-142) counts, for every pair i < j,
// how many of cell i's three vertex slots occur in cell j: 1 -> vertex-sharing,
// 2 -> edge-sharing, 0 -> disjoint (3, a repeated cell, joins no list).  Here
// the count comes from vertex -> cell incidence in O(T * valence): the sorted
// cell lists of i's three slot vertices are merged, and a cell j > i occurring
// in m of them shares m slots.  Every merged j is a neighbour, so the disjoint
// pairs of row i are all j > i except those; they are never listed, only
// counted (row_start) and decoded on the fly from the sorted neighbour list.
// The vertex- and edge-sharing lists come out in lexicographic (i, j) order.

// Exclusive prefix sum of n counts into out[0..n] (out[n] = total), one
// workgroup: each thread scans a contiguous chunk.
template <class F>
__device__ __forceinline__ void scan_counts(int64_t n, F count, int64_t* __restrict__ out, int64_t* total) {
    __shared__ int64_t part[16];
    const int64_t chunk = (n + blockDim.x - 1) / blockDim.x;
    const int64_t b = threadIdx.x * chunk, e = b + chunk < n ? b + chunk : n;
    int64_t s = 0;
    for (int64_t q = b; q < e; ++q) s += count(q);
    const int lane = threadIdx.x & 63;
    int64_t run = s;                       // inclusive over the wavefront
    for (int d = 1; d < 64; d <<= 1) {
        const int64_t v = (int64_t)__shfl_up((long long)run, d);
        if (lane >= d) run += v;
    }
    if (lane == 63) part[threadIdx.x >> 6] = run;
    __syncthreads();
    int64_t before = 0;                    // the wavefronts before this one
    for (int w = 0; w < (int)(threadIdx.x >> 6); ++w) before += part[w];
    run += before;
    if (threadIdx.x == blockDim.x - 1) { out[n] = run; if (total) *total = run; }
    run -= s;
    for (int64_t q = b; q < e; ++q) { out[q] = run; run += count(q); }
}
__global__ __launch_bounds__(1024) void k_scan_degrees(int64_t n, const int32_t* __restrict__ cnt, int64_t* __restrict__ out) {
    scan_counts(n, [&](int64_t q) { return (int64_t)cnt[q]; }, out, nullptr);
}
// The offsets of the classification's lists, a workgroup each: vertex-sharing,
// edge-sharing and all sharing cells j > i and all sharing cells j < i from
// their counts (nT each), and the disjoint pairs of row i, the nT - 1 - i cells
// j > i less those sharing.
struct RowOffsets { int64_t* p[5]; };
__global__ __launch_bounds__(1024) void k_scan_rows(int64_t nT, const int32_t* __restrict__ counts, RowOffsets off, int64_t* totals) {
    const int w = blockIdx.x;
    if (w < 4) {
        const int32_t* c = counts + w * nT;
        scan_counts(nT, [&](int64_t q) { return (int64_t)c[q]; }, off.p[w], totals + w);
    } else {
        const int32_t* n = counts + 2 * nT;
        scan_counts(nT, [&](int64_t q) { return (nT - 1 - q) - (int64_t)n[q]; }, off.p[w], totals + w);
    }
}
__global__ void k_clear(int64_t n, int32_t* __restrict__ p) {
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) p[q] = 0;
}

__global__ void k_vertex_degree(int64_t nslots, const int32_t* __restrict__ tri, int32_t* __restrict__ deg) {
    for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < nslots; s += (int64_t)gridDim.x * blockDim.x)
        atomicAdd(&deg[tri[s]], 1);
}

__global__ void k_fill_incidence(int64_t nslots, const int32_t* __restrict__ tri, const int64_t* __restrict__ start,
                                 int32_t* __restrict__ cursor, int32_t* __restrict__ inc) {
    for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < nslots; s += (int64_t)gridDim.x * blockDim.x) {
        const int32_t v = tri[s];
        inc[start[v] + atomicAdd(&cursor[v], 1)] = (int32_t)(s / 3);
    }
}

// Per vertex: its cell list sorted ascending (insertion sort; lists are short).
__global__ void k_sort_incidence(int64_t nV, const int64_t* __restrict__ start, int32_t* __restrict__ inc) {
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nV; v += (int64_t)gridDim.x * blockDim.x) {
        const int64_t b = start[v], e = start[v + 1];
        for (int64_t q = b + 1; q < e; ++q) {
            const int32_t x = inc[q];
            int64_t r = q - 1;
            while (r >= b && inc[r] > x) { inc[r + 1] = inc[r]; --r; }
            inc[r + 1] = x;
        }
    }
}

// A vertex's cells from position q on, the next one held in a register
struct SlotList {
    const int32_t* p;
    int64_t q, e;
    int32_t head;
    __device__ void open(const int32_t* inc, int64_t b, int64_t end) { p = inc; q = b; e = end; read(); }
    __device__ void read() { head = q < e ? p[q] : INT32_MAX; }
    // to the first entry > i
    __device__ void seek(int32_t i) {
        int64_t lo = q, hi = e;
        while (lo < hi) { const int64_t mid = (lo + hi) >> 1; if (p[mid] <= i) lo = mid + 1; else hi = mid; }
        q = lo;
        read();
    }
    // advances past every copy of j (a cell with a repeated vertex is listed twice)
    __device__ int take(int32_t j) {
        if (head != j) return 0;
        do { ++q; read(); } while (head == j && q < e);
        return 1;
    }
};

// The three slots' cells of cell c, merged; each cell once.
struct SlotMerge {
    SlotList L[3];
    __device__ SlotMerge(int64_t c, const int32_t* tri, const int64_t* start, const int32_t* inc) {
        for (int k = 0; k < 3; ++k) {
            const int32_t v = tri[3 * c + k];
            L[k].open(inc, start[v], start[v + 1]);
        }
    }
    __device__ int32_t head() const { return min(L[0].head, min(L[1].head, L[2].head)); }
    __device__ int take(int32_t j) { return L[0].take(j) + L[1].take(j) + L[2].take(j); }
    // the number of cells before `end`, which are passed
    __device__ int32_t skip(int32_t end) {
        int32_t n = 0;
        for (int32_t j = head(); j < end; j = head()) { take(j); ++n; }
        return n;
    }
};

// WRITE = false: per cell i, the numbers of vertex-sharing, edge-sharing and
// all sharing cells j > i, and of all sharing cells j < i.  WRITE = true: the
// lists at the scanned offsets; the lists of earlier cells are cleared.
template <bool WRITE>
__global__ void k_classify(int64_t nT, const int32_t* __restrict__ tri, const int64_t* __restrict__ start,
                           const int32_t* __restrict__ inc, int32_t* __restrict__ counts, const int64_t* __restrict__ off_simple,
                           const int64_t* __restrict__ off_attached, const int64_t* __restrict__ off_shared,
                           const int64_t* __restrict__ off_back, int32_t* __restrict__ simple, int32_t* __restrict__ attached,
                           int32_t* __restrict__ nbr, int64_t* __restrict__ back) {
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < nT; c += (int64_t)gridDim.x * blockDim.x) {
        const int32_t i = (int32_t)c;
        SlotMerge S(c, tri, start, inc);
        int64_t ws = WRITE ? off_simple[c] : 0, wa = WRITE ? off_attached[c] : 0, wn = WRITE ? off_shared[c] : 0;
        int32_t cs = 0, ca = 0, cn = 0, cb = 0;
        if (WRITE) {
            for (auto& l : S.L) l.seek(i);
            for (int64_t q = off_back[c]; q < off_back[c + 1]; ++q) back[q] = -1;
        } else {
            cb = S.skip(i);
            S.take(i);
        }
        for (;;) {
            const int32_t j = S.head();
            if (j == INT32_MAX) break;
            const int m = S.take(j);
            ++cn;
            if (m == 1) ++cs;
            if (m == 2) ++ca;
            if (WRITE) {
                nbr[wn++] = j;
                if (m == 1) { simple[3 * ws] = i; simple[3 * ws + 1] = j; simple[3 * ws + 2] = (int32_t)ws; ++ws; }
                if (m == 2) { attached[3 * wa] = i; attached[3 * wa + 1] = j; attached[3 * wa + 2] = (int32_t)wa; ++wa; }
            }
        }
        if (!WRITE) { counts[c] = cs; counts[nT + c] = ca; counts[2 * nT + c] = cn; counts[3 * nT + c] = cb; }
    }
}

// The pairs of each cell with earlier cells, in the earlier cells' order: a pair
// (i, j), number k of its list, stands where i does among the cells before j
// that share a vertex with it, as 2 k (vertex-sharing) or 2 k + 1 (edge-sharing).
// Entries of cells that share all three stay -1.
__global__ void k_back_pairs(int64_t n0, int64_t n1, const int32_t* __restrict__ simple, const int32_t* __restrict__ attached,
                             const int32_t* __restrict__ tri, const int64_t* __restrict__ start, const int32_t* __restrict__ inc,
                             const int64_t* __restrict__ off_back, int64_t* __restrict__ back) {
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n0 + n1; q += (int64_t)gridDim.x * blockDim.x) {
        const int kind = q >= n0;
        const int64_t k = kind ? q - n0 : q;
        const int32_t* L = (kind ? attached : simple) + 3 * k;
        const int32_t i = L[0], j = L[1];
        SlotMerge S(j, tri, start, inc);
        back[off_back[j] + S.skip(i)] = 2 * k + kind;
    }
}

static unsigned grid_of(int64_t n) {
    const int64_t b = (n + 255) / 256;
    return (unsigned)(b < 1 ? 1 : (b > 65536 ? 65536 : b));
}

static int classify(i2_mesh* m) {
    const int64_t nT = m->nT, nV = m->nV, nslots = 3 * nT;
    hipStream_t st = m->stream;
    I2_TRY(m->d_degree.ensure(2 * nV)); I2_TRY(m->d_inc.ensure(nslots)); I2_TRY(m->d_inc_start.ensure(nV + 1));
    I2_TRY(m->d_counts.ensure(4 * nT)); I2_TRY(m->d_totals.ensure(5));
    for (DBuf<int64_t>* o : {&m->d_off[0], &m->d_off[1], &m->d_nbr_start, &m->d_back_start, &m->d_row_start}) I2_TRY(o->ensure(nT + 1));
    int32_t *deg = m->d_degree.p, *cursor = deg + nV;
    const int64_t* start = m->d_inc_start.p;
    hipLaunchKernelGGL(k_clear, dim3(grid_of(2 * nV)), dim3(256), 0, st, 2 * nV, deg);
    hipLaunchKernelGGL(k_vertex_degree, dim3(grid_of(nslots)), dim3(256), 0, st, nslots, m->d_tri.p, deg);
    I2_TRY(check_launch("k_vertex_degree"));
    hipLaunchKernelGGL(k_scan_degrees, dim3(1), dim3(1024), 0, st, nV, deg, m->d_inc_start.p);
    I2_TRY(check_launch("k_scan_degrees"));
    hipLaunchKernelGGL(k_fill_incidence, dim3(grid_of(nslots)), dim3(256), 0, st, nslots, m->d_tri.p, start, cursor, m->d_inc.p);
    I2_TRY(check_launch("k_fill_incidence"));
    hipLaunchKernelGGL(k_sort_incidence, dim3(grid_of(nV)), dim3(256), 0, st, nV, start, m->d_inc.p);
    I2_TRY(check_launch("k_sort_incidence"));
    hipLaunchKernelGGL(k_classify<false>, dim3(grid_of(nT)), dim3(256), 0, st, nT, m->d_tri.p, start, m->d_inc.p,
                       m->d_counts.p, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr);
    I2_TRY(check_launch("k_classify"));
    const RowOffsets off{{m->d_off[0].p, m->d_off[1].p, m->d_nbr_start.p, m->d_back_start.p, m->d_row_start.p}};
    hipLaunchKernelGGL(k_scan_rows, dim3(5), dim3(1024), 0, st, nT, m->d_counts.p, off, m->d_totals.p);
    I2_TRY(check_launch("k_scan_rows"));
    int64_t tot[5];
    I2_HIP(hipMemcpyAsync(tot, m->d_totals.p, sizeof tot, hipMemcpyDeviceToHost, st));
    I2_HIP(hipStreamSynchronize(st));
    if (tot[0] > (int64_t)INT32_MAX || tot[1] > (int64_t)INT32_MAX) {
        set_error("%lld vertex-sharing / %lld edge-sharing pairs exceed the 32-bit pair numbers", (long long)tot[0], (long long)tot[1]);
        return I2_ERR_RANGE;
    }
    I2_TRY(m->d_simple.ensure(3 * tot[0]));
    I2_TRY(m->d_attached.ensure(3 * tot[1]));
    I2_TRY(m->d_nbr.ensure(tot[2]));
    I2_TRY(m->d_back.ensure(tot[3]));
    hipLaunchKernelGGL(k_classify<true>, dim3(grid_of(nT)), dim3(256), 0, st, nT, m->d_tri.p, start, m->d_inc.p, nullptr,
                       off.p[0], off.p[1], off.p[2], off.p[3], m->d_simple.p, m->d_attached.p, m->d_nbr.p, m->d_back.p);
    I2_TRY(check_launch("k_classify"));
    if (tot[0] + tot[1] > 0) {
        hipLaunchKernelGGL(k_back_pairs, dim3(grid_of(tot[0] + tot[1])), dim3(256), 0, st, tot[0], tot[1], m->d_simple.p,
                           m->d_attached.p, m->d_tri.p, start, m->d_inc.p, off.p[3], m->d_back.p);
        I2_TRY(check_launch("k_back_pairs"));
    }
    m->pairs[I2_SIMPLE_NEIGHBORS] = tot[0];
    m->pairs[I2_ATTACHED_NEIGHBORS] = tot[1];
    m->pairs[I2_NOT_NEIGHBORS] = tot[4];
    return I2_OK;
}

template <class T>
static int upload(DBuf<T>& d, const std::vector<T>& h, hipStream_t s) {
    I2_TRY(d.ensure((int64_t)h.size()));
    if (!h.empty()) I2_HIP(hipMemcpyAsync(d.p, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice, s));
    return I2_OK;
}

int mesh_upload_and_prepare(i2_mesh* m) {
    DeviceGuard g(m->device);
    if (!g.ok) return I2_ERR_HIP;
    if (m->nT <= 0 || m->nV <= 0) { set_error("mesh is empty"); return I2_ERR_STATE; }
    if (m->nT > (int64_t)INT32_MAX) { set_error("more than 2^31-1 cells"); return I2_ERR_RANGE; }
    I2_TRY(upload(m->d_xyz, m->h_xyz, m->stream));
    I2_TRY(upload(m->d_tri, m->h_tri, m->stream));
    I2_TRY(classify(m));
    I2_TRY(m->d_normals.ensure(3 * m->nT));
    I2_TRY(m->d_measures.ensure(m->nT));
    I2_TRY(m->d_panels.ensure(m->nT));
    const int threads = 256;
    const int64_t blocks = (m->nT + threads - 1) / threads;
    hipLaunchKernelGGL(k_panel_table, dim3((unsigned)blocks), dim3(threads), 0, m->stream, m->nT, m->d_xyz.p, m->d_tri.p,
                       m->d_panels.p, m->d_normals.p, m->d_measures.p);
    I2_TRY(check_launch("k_panel_table"));
    I2_HIP(hipStreamSynchronize(m->stream));
    m->prepared = true;
    ++m->generation;
    return I2_OK;
}

}  // namespace i2

using namespace i2;

extern "C" {

const char* i2_last_error(void) { return g_last_error.c_str(); }

int i2_host_math(int fn, const double* x, const double* y, int64_t n, double* out) {
    if (!x || !out || n < 0 || ((fn == 1 || fn == 11) && !y)) { set_error("null argument"); return I2_ERR_INVALID; }
    for (int64_t q = 0; q < n; ++q) {
        if (fn == 0) out[q] = i2m::log_tab(x[q], &i2m::h_mathtab);
        else if (fn == 2) out[q] = i2m::sqrt_pos(x[q]);
        else if (fn == 1) out[q] = i2m::atan2_fast(y[q], x[q], &i2m::h_mathtab);
        else if (fn == 6) out[q] = i2m::rcp_pos(x[q]);
        else if (fn == 10) out[q] = i2m::log_tab_any(x[q], &i2m::h_mathtab);
        else if (fn == 11) out[q] = i2m::atan2_any(y[q], x[q], &i2m::h_mathtab);
        else { set_error("unknown function %d", fn); return I2_ERR_INVALID; }
    }
    return I2_OK;
}

int i2_host_theta_psi(int fast, const double* pts, int64_t n, const double* tri9, double* out4) {
    if (!pts || !tri9 || !out4 || n < 0) { set_error("null argument"); return I2_ERR_INVALID; }
    using namespace i2d;
    const d3 A = {tri9[0], tri9[1], tri9[2]}, B = {tri9[3], tri9[4], tri9[5]}, C = {tri9[6], tri9[7], tri9[8]};
    const JGeom J = make_jgeom(A, B, C, unit(C - B), unit(A - C), unit(B - A));
    for (int64_t q = 0; q < n; ++q) {
        const d3 p = {pts[3 * q], pts[3 * q + 1], pts[3 * q + 2]};
        q4 r;
        if (fast == 2 || fast == 3) {   // p as a point of a control panel of K_j's size and shape
            const double b0 = 0.3, b1 = -0.2;
            const d3 o = p - ((b0 + 1.0 / 3.0) * J.a + (b1 + 1.0 / 3.0) * J.b + (1.0 / 3.0 - b0 - b1) * J.c);
            const FarFrame F = far_frame(J.a + o, J.b + o, J.c + o);
            const FarGeom G = far_geom(F, J);
            const double pp = far_pp(F, far_point(b0, b1, 0.0));
            r = psi_of_terms(far_scale(fast == 3 ? theta_terms_far<true>(b0, b1, pp, G) : theta_terms_far<false>(b0, b1, pp, G), J), J);
        } else {
            r = fast ? theta_psi_fast(p, J, &i2m::h_mathtab) : theta_psi(p, J.a, J.b, J.c, J.ta, J.tb, J.tc);
        }
        out4[4 * q] = r.x; out4[4 * q + 1] = r.y; out4[4 * q + 2] = r.z; out4[4 * q + 3] = r.w;
    }
    return I2_OK;
}

// The kernels' math functions on the device, for checking (fn as in i2_host_math).
__global__ void k_math(int fn, int64_t n, const double* __restrict__ x, const double* __restrict__ y, double* __restrict__ out) {
    __shared__ i2m::MathTable lt;
    i2m::fill_mathtab(lt);
    __syncthreads();
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    if (fn == 0) out[q] = i2m::log_tab(x[q], &lt);
    else if (fn == 1) out[q] = i2m::atan2_fast(y[q], x[q], &lt);
    else if (fn == 2) out[q] = i2m::sqrt_pos(x[q]);
    else if (fn == 3) out[q] = log(x[q]);
    else if (fn == 4) out[q] = atan2(y[q], x[q]);
    else if (fn == 5) out[q] = sqrt(x[q]);
    else if (fn == 6) out[q] = i2m::rcp_pos(x[q]);
    else if (fn == 7) out[q] = 1.0 / x[q];
    else if (fn == 8) out[q] = i2m::rcp_estimate(x[q]);
    else if (fn == 9) out[q] = i2m::rsq_estimate(x[q]);
    else if (fn == 10) out[q] = i2m::log_tab_any(x[q], &lt);
    else out[q] = i2m::atan2_any(y[q], x[q], &lt);
}

int i2_device_math(int device, int fn, const double* x, const double* y, int64_t n, double* out) {
    if (!x || !out || n <= 0 || fn < 0 || fn > 11 || ((fn == 1 || fn == 4 || fn == 11) && !y)) { set_error("invalid argument"); return I2_ERR_INVALID; }
    DeviceGuard g(device);
    if (!g.ok) return I2_ERR_HIP;
    DBuf<double> dx, dy, dout;
    I2_TRY(dx.ensure(n)); I2_TRY(dy.ensure(n)); I2_TRY(dout.ensure(n));
    I2_HIP(hipMemcpy(dx.p, x, sizeof(double) * n, hipMemcpyHostToDevice));
    I2_HIP(hipMemcpy(dy.p, y ? y : x, sizeof(double) * n, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_math, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, nullptr, fn, n, dx.p, dy.p, dout.p);
    I2_TRY(check_launch("k_math"));
    I2_HIP(hipMemcpy(out, dout.p, sizeof(double) * n, hipMemcpyDeviceToHost));
    return I2_OK;
}

// Host evaluation of one ordered task's integrals with the kernels' device
// code compiled for the host: level-`level` quadrature of (thetaPsi -
// singular part) over K_i's sub-panels, points from the sub-panels' vertices
// and the inner integral's general form, plus the closed-form singular part.
// The kernels evaluate disjoint pairs by the terms and far ones by polynomials;
// this value agrees with theirs to rounding.  I9 and J9 are the two panels'
// vertices, vid6 their vertex ids (they decide the neighbour type and the
// rotations).  For checking.
int i2_host_task_value(const double* I9, const double* J9, const int32_t* vid6, int level, const double* L12,
                       const double* w, int nPts, double* out4) {
    if (!I9 || !J9 || !vid6 || !L12 || !w || !out4 || nPts < 1 || nPts > i2d::MAX_POINTS || level < 0 || level > 12) {
        set_error("invalid argument");
        return I2_ERR_INVALID;
    }
    using namespace i2d;
    auto panel = [](const double* X, const int32_t* v) {
        Panel P{};
        P.a = {X[0], X[1], X[2]}; P.b = {X[3], X[4], X[5]}; P.c = {X[6], X[7], X[8]};
        P.ta = unit(P.c - P.b); P.tb = unit(P.a - P.c); P.tc = unit(P.b - P.a);
        const d3 cr = cross(P.b - P.a, P.c - P.a);
        P.n = unit(cr);
        P.area = vlen(cr) * 0.5;
        P.v0 = v[0]; P.v1 = v[1]; P.v2 = v[2];
        return P;
    };
    const Panel I = panel(I9, vid6), J = panel(J9, vid6 + 3);
    const int shared = shared_count(I, J);
    const JGeom JG = make_jgeom(J.a, J.b, J.c, J.ta, J.tb, J.tc);
    int s1 = 0, s2 = 0;
    EdgeCtx ec{};
    VertexCtx vc{};
    if (shared == 2) { shifts_edge(I, J, &s1, &s2); ec = edge_ctx(vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3)); }
    if (shared == 1) {
        shifts_vertex(I, J, &s1, &s2);
        vc = vertex_ctx(vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3), I.n, J.n, I.area);
    }
    double area = I.area;
    for (int l = 0; l < level; ++l) area *= 0.25;
    q4 total = q4zero();
    const uint32_t nsub = 1u << (2 * level);
    for (uint32_t c = 0; c < nsub; ++c) {
        d3 a = I.a, b = I.b, cc = I.c;
        if (level == 1) {   // the sweep kernel's level-1 children
            const d3 mBC = 0.5 * (I.b + I.c), mCA = 0.5 * (I.c + I.a), mAB = 0.5 * (I.a + I.b);
            if (c == 0) { a = mAB; b = I.b; cc = mBC; }
            else if (c == 1) { a = mBC; b = I.c; cc = mCA; }
            else if (c == 2) { a = mCA; b = I.a; cc = mAB; }
            else { a = mBC; b = mCA; cc = mAB; }
        } else {
            sub_panel(a, b, cc, level, c);
        }
        q4 acc = q4zero();
        for (int k = 0; k < nPts; ++k) {
            const double l1 = L12[2 * k], l2 = L12[2 * k + 1], l3 = 1.0 - l1 - l2;
            d3 p = l1 * a;
            p = p + l2 * b;
            p = p + l3 * cc;
            q4 f = theta_psi_fast(p, JG, &i2m::h_mathtab);
            if (shared == 2) f = f - sing_edge_fast(p, ec, &i2m::h_mathtab);
            if (shared == 1) f = f - sing_vertex_fast(p, vc, &i2m::h_mathtab);
            acc = acc + w[k] * f;
        }
        total = total + area * acc;
    }
    if (shared == 2)
        total = total + integrate_sing_edge(vtx(I, s1), vtx(I, (s1 + 1) % 3), vtx(I, (s1 + 2) % 3),
                                           vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3), I.n, J.n, I.area);
    if (shared == 1)
        total = total + integrate_sing_vertex(vtx(I, s1), vtx(I, (s1 + 1) % 3), vtx(I, (s1 + 2) % 3),
                                             vtx(J, s2), vtx(J, (s2 + 1) % 3), vtx(J, (s2 + 2) % 3), I.n, J.n, I.area);
    out4[0] = total.x; out4[1] = total.y; out4[2] = total.z; out4[3] = total.w;
    return I2_OK;
}

int i2_host_point_split(int nPts, const int64_t* q, int64_t n, int64_t* sub, int64_t* point) {
    if (!q || !sub || !point || n < 0 || nPts < 1 || nPts > i2d::MAX_POINTS) { set_error("invalid argument"); return I2_ERR_INVALID; }
    const uint32_t factor = i2d::split_factor(nPts);
    for (int64_t k = 0; k < n; ++k) {
        if (q[k] < 0 || q[k] > (int64_t)1 << 28) { set_error("point number %lld out of range", (long long)q[k]); return I2_ERR_RANGE; }
        sub[k] = i2d::split_point((uint32_t)q[k], factor);
        point[k] = q[k] - sub[k] * nPts;
    }
    return I2_OK;
}

int i2_device_count(int* n) {
    if (!n) { set_error("null pointer"); return I2_ERR_INVALID; }
    int c = 0;
    if (hipGetDeviceCount(&c) != hipSuccess) { (void)hipGetLastError(); c = 0; }
    *n = c;
    return I2_OK;
}

int i2_mesh_create(i2_mesh** out, int device) {
    if (!out) { set_error("null pointer"); return I2_ERR_INVALID; }
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) {
        (void)hipGetLastError();
        set_error("no HIP device available");
        return I2_ERR_HIP;
    }
    if (device < 0 || device >= count) { set_error("device %d out of range (%d devices)", device, count); return I2_ERR_INVALID; }
    DeviceGuard g(device);
    if (!g.ok) return I2_ERR_HIP;
    i2_mesh* m = new i2_mesh;
    m->device = device;
    if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) {
        (void)hipGetLastError();
        delete m;
        set_error("hipStreamCreate failed");
        return I2_ERR_HIP;
    }
    *out = m;
    return I2_OK;
}

void i2_mesh_destroy(i2_mesh* m) {
    if (!m) return;
    {
        DeviceGuard g(m->device);
        (void)hipStreamSynchronize(m->stream);
        m->d_xyz.reset(); m->d_tri.reset(); m->d_normals.reset(); m->d_measures.reset(); m->d_panels.reset();
        m->d_simple.reset(); m->d_attached.reset(); m->d_nbr_start.reset(); m->d_row_start.reset(); m->d_nbr.reset(); m->d_not_list.reset();
        m->d_off[0].reset(); m->d_off[1].reset(); m->d_back_start.reset(); m->d_back.reset(); m->d_inc_start.reset(); m->d_inc.reset(); m->d_degree.reset(); m->d_counts.reset(); m->d_totals.reset();
        (void)hipStreamDestroy(m->stream);
    }
    delete m;
}

int i2_mesh_set_data(i2_mesh* m, const double* xyz, int64_t nV, const int32_t* tri, int64_t nT) {
    if (!m || !xyz || !tri || nV <= 0 || nT <= 0) { set_error("invalid mesh data"); return I2_ERR_INVALID; }
    if (nV > (int64_t)INT32_MAX || nT > (int64_t)INT32_MAX) { set_error("mesh too large for 32-bit indices"); return I2_ERR_RANGE; }
    for (int64_t q = 0; q < 3 * nT; ++q)
        if (tri[q] < 0 || tri[q] >= nV) { set_error("triangle %lld references vertex %d outside [0, %lld)", (long long)(q / 3), tri[q], (long long)nV); return I2_ERR_INVALID; }
    m->nV = nV; m->nT = nT;
    m->h_xyz.assign(xyz, xyz + 3 * nV);
    m->h_tri.assign(tri, tri + 3 * nT);
    m->prepared = false;
    return I2_OK;
}

int i2_mesh_load_file(i2_mesh* m, const char* path, double scale) {
    if (!m || !path) { set_error("null argument"); return I2_ERR_INVALID; }
    std::ifstream f(path);
    if (!f.is_open()) { set_error("cannot open mesh file %s", path); return I2_ERR_IO; }
    long long nv = 0, nc = 0;
    if (!(f >> nv >> nc) || nv <= 0 || nc < 0) { set_error("bad header in %s", path); return I2_ERR_IO; }
    std::vector<double> xyz(3 * nv);
    for (long long q = 0; q < nv; ++q) {
        long long idx;
        double x, y, z;
        if (!(f >> idx >> x >> y >> z)) { set_error("truncated vertex list in %s", path); return I2_ERR_IO; }
        xyz[3 * q] = scale * x; xyz[3 * q + 1] = scale * y; xyz[3 * q + 2] = scale * z;
    }
    // element records "idx type ..." (src/Mesh3d.cu:181-197): type 203 is a
    // triangle with three 1-based vertex indices; other entities carry two
    // more numbers and reduce the declared cell count.
    std::vector<int32_t> tri;
    long long declared = nc;
    long long idx, type;
    while (f >> idx >> type) {
        if (type == 203) {
            long long a, b, c;
            if (!(f >> a >> b >> c)) break;
            tri.push_back((int32_t)(a - 1)); tri.push_back((int32_t)(b - 1)); tri.push_back((int32_t)(c - 1));
        } else {
            --declared;
            long long s1, s2;
            if (!(f >> s1 >> s2)) break;
        }
    }
    const long long ncells = std::min<long long>(declared, (long long)tri.size() / 3);
    if (ncells <= 0) { set_error("no triangles in %s", path); return I2_ERR_IO; }
    tri.resize(3 * ncells);
    return i2_mesh_set_data(m, xyz.data(), nv, tri.data(), ncells);
}

int i2_mesh_prepare(i2_mesh* m) {
    if (!m) { set_error("null mesh"); return I2_ERR_INVALID; }
    return mesh_upload_and_prepare(m);
}

int i2_mesh_sizes(const i2_mesh* m, int64_t* nV, int64_t* nT, int64_t pairs[3]) {
    if (!m) { set_error("null mesh"); return I2_ERR_INVALID; }
    if (nV) *nV = m->nV;
    if (nT) *nT = m->nT;
    if (pairs) for (int t = 0; t < 3; ++t) pairs[t] = m->pairs[t];
    return I2_OK;
}

int i2_mesh_copy_vertices(const i2_mesh* m, double* xyz) {
    if (!m || !xyz) { set_error("null argument"); return I2_ERR_INVALID; }
    std::copy(m->h_xyz.begin(), m->h_xyz.end(), xyz);
    return I2_OK;
}
int i2_mesh_copy_cells(const i2_mesh* m, int32_t* tri) {
    if (!m || !tri) { set_error("null argument"); return I2_ERR_INVALID; }
    std::copy(m->h_tri.begin(), m->h_tri.end(), tri);
    return I2_OK;
}
static int copy_d2h(const void* d, void* h, size_t bytes, int device) {
    DeviceGuard g(device);
    if (!g.ok) return I2_ERR_HIP;
    I2_HIP(hipMemcpy(h, d, bytes, hipMemcpyDeviceToHost));
    return I2_OK;
}
int i2_mesh_copy_normals(const i2_mesh* m, double* n3) {
    if (!m || !n3) { set_error("null argument"); return I2_ERR_INVALID; }
    if (!m->prepared) { set_error("mesh not prepared"); return I2_ERR_STATE; }
    return copy_d2h(m->d_normals.p, n3, sizeof(double) * 3 * m->nT, m->device);
}
int i2_mesh_copy_measures(const i2_mesh* m, double* s) {
    if (!m || !s) { set_error("null argument"); return I2_ERR_INVALID; }
    if (!m->prepared) { set_error("mesh not prepared"); return I2_ERR_STATE; }
    return copy_d2h(m->d_measures.p, s, sizeof(double) * m->nT, m->device);
}
int i2_mesh_copy_neighbors(const i2_mesh* m, int type, int32_t* ijk) {
    if (!m || !ijk) { set_error("null argument"); return I2_ERR_INVALID; }
    if (!m->prepared) { set_error("mesh not prepared"); return I2_ERR_STATE; }
    if (type == I2_SIMPLE_NEIGHBORS || type == I2_ATTACHED_NEIGHBORS) {
        const DBuf<int32_t>& d = type == I2_SIMPLE_NEIGHBORS ? m->d_simple : m->d_attached;
        return m->pairs[type] ? copy_d2h(d.p, ijk, sizeof(int32_t) * 3 * m->pairs[type], m->device) : I2_OK;
    }
    if (type != I2_NOT_NEIGHBORS) { set_error("bad neighbour type %d", type); return I2_ERR_INVALID; }
    std::vector<int64_t> start((size_t)m->nT + 1);
    I2_TRY(copy_d2h(m->d_nbr_start.p, start.data(), sizeof(int64_t) * (m->nT + 1), m->device));
    std::vector<int32_t> nbr((size_t)start[m->nT]);
    if (!nbr.empty()) I2_TRY(copy_d2h(m->d_nbr.p, nbr.data(), sizeof(int32_t) * nbr.size(), m->device));
    int64_t k = 0;
    for (int64_t i = 0; i < m->nT; ++i) {
        int64_t q = start[i];
        const int64_t qe = start[i + 1];
        for (int64_t j = i + 1; j < m->nT; ++j) {
            if (q < qe && nbr[q] == j) { ++q; continue; }
            ijk[3 * k] = (int32_t)i; ijk[3 * k + 1] = (int32_t)j; ijk[3 * k + 2] = (int32_t)k;
            ++k;
        }
    }
    return I2_OK;
}
int i2_mesh_device_array(const i2_mesh* m, int what, const void** dptr, int64_t* n) {
    if (!m || !dptr || !n) { set_error("null argument"); return I2_ERR_INVALID; }
    if (!m->prepared) { set_error("mesh not prepared"); return I2_ERR_STATE; }
    switch (what) {
        case 0: *dptr = m->d_xyz.p; *n = m->nV; break;
        case 1: *dptr = m->d_tri.p; *n = m->nT; break;
        case 2: *dptr = m->d_normals.p; *n = m->nT; break;
        case 3: *dptr = m->d_measures.p; *n = m->nT; break;
        case 4: *dptr = m->d_simple.p; *n = m->pairs[I2_SIMPLE_NEIGHBORS]; break;
        case 5: *dptr = m->d_attached.p; *n = m->pairs[I2_ATTACHED_NEIGHBORS]; break;
        case 6: I2_TRY(materialize_disjoint_list(m)); *dptr = m->d_not_list.p; *n = m->pairs[I2_NOT_NEIGHBORS]; break;
        default: set_error("bad array id %d", what); return I2_ERR_INVALID;
    }
    return I2_OK;
}

}  // extern "C"
