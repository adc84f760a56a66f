// i2_internal.hpp -- host-side objects behind the C ABI.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <string>
#include <vector>

#include "../../include/integrator2_mi355x.h"
#include "i2_device.hpp"

namespace i2 {

// ------------------------------------------------------------ errors
void set_error(const char* fmt, ...);
void clear_error();

// Device buffer with RAII ownership; never copied (the reference's
// deviceVector is copyable and would double-free, src/common/device_vector.cuh:15-109).
template <class T> struct DBuf {
    T* p = nullptr;
    int64_t n = 0;
    DBuf() = default;
    DBuf(const DBuf&) = delete;
    DBuf& operator=(const DBuf&) = delete;
    DBuf(DBuf&& o) noexcept : p(o.p), n(o.n) { o.p = nullptr; o.n = 0; }
    DBuf& operator=(DBuf&& o) noexcept { if (this != &o) { reset(); p = o.p; n = o.n; o.p = nullptr; o.n = 0; } return *this; }
    ~DBuf() { reset(); }
    void reset() { if (p) (void)hipFree(p); p = nullptr; n = 0; }
    // (re)allocates when the capacity is too small; contents are not kept
    int ensure(int64_t count) {
        if (count <= n && p) return I2_OK;
        reset();
        if (count == 0) return I2_OK;
        if (hipMalloc((void**)&p, sizeof(T) * (size_t)count) != hipSuccess) {
            (void)hipGetLastError();
            p = nullptr;
            set_error("hipMalloc of %lld bytes failed", (long long)(sizeof(T) * (size_t)count));
            return I2_ERR_ALLOC;
        }
        n = count;
        return I2_OK;
    }
};

#define I2_HIP(call)                                                                           \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess) {                                                                \
            i2::set_error("%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, __LINE__); \
            return I2_ERR_HIP;                                                                 \
        }                                                                                      \
    } while (0)
#define I2_TRY(expr)            \
    do {                        \
        int s_ = (expr);        \
        if (s_ != I2_OK) return s_; \
    } while (0)

// Makes `device` current for the lifetime of the guard.
struct DeviceGuard {
    int prev = -1;
    bool ok = false;
    explicit DeviceGuard(int dev) {
        if (hipGetDevice(&prev) != hipSuccess) { (void)hipGetLastError(); prev = -1; }
        ok = hipSetDevice(dev) == hipSuccess;
        if (!ok) { (void)hipGetLastError(); set_error("hipSetDevice(%d) failed", dev); }
    }
    ~DeviceGuard() { if (prev >= 0) (void)hipSetDevice(prev); }
};

inline int check_launch(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { set_error("launch of %s failed: %s", what, hipGetErrorString(e)); return I2_ERR_HIP; }
    return I2_OK;
}

// A second stream beside a caller's, for kernels that do not depend on each
// other.  Forks and joins are events, so that a graph captured from the caller's
// stream gets two branches.
struct SideStream {
    hipStream_t stream = nullptr;
    hipEvent_t forked = nullptr, joined = nullptr;
    SideStream() = default;
    SideStream(const SideStream&) = delete;
    SideStream& operator=(const SideStream&) = delete;
    ~SideStream() { reset(); }
    int ensure() {
        if (!stream) I2_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
        if (!forked) I2_HIP(hipEventCreateWithFlags(&forked, hipEventDisableTiming));
        if (!joined) I2_HIP(hipEventCreateWithFlags(&joined, hipEventDisableTiming));
        return I2_OK;
    }
    int fork(hipStream_t from) {
        I2_HIP(hipEventRecord(forked, from));
        I2_HIP(hipStreamWaitEvent(stream, forked, 0));
        return I2_OK;
    }
    int join(hipStream_t to) {
        I2_HIP(hipEventRecord(joined, stream));
        I2_HIP(hipStreamWaitEvent(to, joined, 0));
        return I2_OK;
    }
    void reset() {
        if (stream) (void)hipStreamDestroy(stream);
        if (forked) (void)hipEventDestroy(forked);
        if (joined) (void)hipEventDestroy(joined);
        stream = nullptr;
        forked = joined = nullptr;
    }
};

// ------------------------------------------------------------ mesh
}  // namespace i2

struct i2_mesh {
    int device = 0;
    hipStream_t stream = nullptr;
    bool prepared = false;
    uint64_t generation = 0;            // incremented by every prepare (caches key on it)
    int64_t nV = 0, nT = 0;
    std::vector<double> h_xyz;          // host copy of vertices (AoS)
    std::vector<int32_t> h_tri;         // host copy of cells (AoS, 0-based)
    int64_t pairs[3] = {0, 0, 0};
    // device arrays
    i2::DBuf<double> d_xyz;             // vertices (double3 AoS)
    i2::DBuf<int32_t> d_tri;            // cells (int3 AoS)
    i2::DBuf<double> d_normals;         // double3 AoS
    i2::DBuf<double> d_measures;
    i2::DBuf<i2d::Panel> d_panels;      // kernel-side panel records
    // neighbour lists (i<j, k) for vertex- and edge-sharing pairs, lexicographic,
    // and where cell i's pairs start in them
    i2::DBuf<int32_t> d_simple, d_attached;
    i2::DBuf<int64_t> d_off[2];
    // per-cell sorted neighbour indices j > i (CSR) and disjoint-pair row offsets:
    // the k-th disjoint (i<j) pair in lexicographic order is found from these
    i2::DBuf<int64_t> d_nbr_start, d_row_start;
    i2::DBuf<int32_t> d_nbr;
    // cell j's vertex- and edge-sharing pairs (i, j) with earlier cells (CSR):
    // 2 k or 2 k + 1 for pair k of the one list or the other, or -1
    i2::DBuf<int64_t> d_back_start, d_back;
    // per-vertex cells, ascending (CSR; a cell is listed once per corner)
    i2::DBuf<int64_t> d_inc_start;
    i2::DBuf<int32_t> d_inc;
    // counts of the classification, kept for the next one
    i2::DBuf<int32_t> d_degree, d_counts;
    i2::DBuf<int64_t> d_totals;
    // disjoint (i < j, k) list, written out on request (the kernels decode it on the fly)
    mutable i2::DBuf<int32_t> d_not_list;
    mutable uint64_t not_list_generation = 0;
};

namespace i2 { struct RefinedMesh; }

// Plain settings struct (the batched engine keeps a copy of it as its
// configuration); the two pointers are owned by the i2_integrator_* calls only.
struct i2_integrator {
    const i2_mesh* mesh = nullptr;
    i2d::Rule rule{};
    int fixed = 0;          // 1: fixed refinement level
    int fixed_level = 0;
    int max_level = 5;      // MAX_REFINE_LEVEL (src/common/constants.h:56)
    double tol = 1e-5;      // EPS_INTEGRATION (src/common/constants.h:18)
    int quirk = 1;          // reproduce the result-buffer swap
    i2_evaluator* last_ev = nullptr;        // evaluator of the last run on this integrator (not owned)
    i2::RefinedMesh* refined = nullptr;     // fixed-level refined mesh, built on request (owned)
};

namespace i2 {

// Task source of one neighbour type: explicit ordered (i, j) list or, for
// all disjoint pairs, implicit decoding of task index t into (i, j).
struct TaskSource {
    const int32_t* ij3 = nullptr;     // explicit: (i, j, k) per task
    int64_t n_unordered = 0;          // implicit: number of i<j pairs; t >= n -> reversed
    const int64_t* row_start = nullptr;
    const int64_t* nbr_start = nullptr;
    const int32_t* nbr = nullptr;
    int nT = 0;
};

// ------------------------------------------------------------ task decoding
__device__ __forceinline__ int find_row(const int64_t* __restrict__ row_start, int nT, int64_t k) {
    int lo = 0, hi = nT - 1;   // largest i with row_start[i] <= k
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (row_start[mid] <= k) lo = mid; else hi = mid - 1;
    }
    return lo;
}
// k-th disjoint (i<j) pair in lexicographic order
__device__ __forceinline__ void decode_disjoint(const TaskSource& s, int64_t k, int* pi, int* pj) {
    const int i = find_row(s.row_start, s.nT, k);
    int64_t j = i + 1 + (k - s.row_start[i]);
    for (int64_t q = s.nbr_start[i]; q < s.nbr_start[i + 1]; ++q) {
        if (s.nbr[q] <= j) ++j; else break;
    }
    *pi = i; *pj = (int)j;
}
template <bool IMPLICIT>
__device__ __forceinline__ void task_ij(const TaskSource& s, int64_t t, int* i, int* j) {
    if (IMPLICIT) {
        if (t < s.n_unordered) decode_disjoint(s, t, i, j);
        else decode_disjoint(s, t - s.n_unordered, j, i);
    } else {
        *i = s.ij3[3 * t];
        *j = s.ij3[3 * t + 1];
    }
}

struct TypeState {
    int64_t n = 0;                 // ordered tasks
    bool implicit = false;         // disjoint all-pairs: tasks decoded on the fly
    DBuf<int32_t> tasks;           // explicit (i, j, k)
    DBuf<int32_t> new_tasks;       // runPairs: the next ones, until they are checked
    DBuf<double4> buf[2];          // level values, level k written to buf[k % 2]
    DBuf<double> results;          // J (double3 AoS)
    DBuf<double> errors;           // symmetry error
    DBuf<int8_t> conv;             // convergence iteration
    DBuf<int32_t> rest[2];         // rest lists
    DBuf<uint8_t> unconv;          // per control panel: a task still unconverged after the comparison at maxLevel
    DBuf<uint8_t> refinements;     // per control panel: refinement passes (computed on request)
    DBuf<int32_t> task_list;       // explicit (i, j, k) of an implicit type (materialised on request)
    int K = 0;                     // refinement iterations run
    int final_buf = 0;             // buffer holding the final integrals
    double ms = 0.0;
    int64_t refined_tasks = 0;
    bool has_errors = false;
    bool refinements_ready = false;
    bool task_list_ready = false;
};

}  // namespace i2

// One timed kernel launch of the plain path (profiling mode).
struct LaunchRecord {
    int type, level;
    int64_t tasks;
    hipEvent_t e0, e1;
};

namespace i2 { struct AdjState; }

struct i2_evaluator {
    const i2_mesh* mesh = nullptr;
    int path = 0;                  // 0: plain per-type launches, 1: batched persistent kernels
    i2_batch* fast = nullptr;      // engine of the batched path (one mesh)
    int fast_P = 64, fast_ppl = 13;
    bool fast_tuned = false;       // the caller set the launch shape
    double fast_sweep_ms = 0.0;    // disjoint sweep time of the last profiled batched run
    bool profile = false;
    std::vector<LaunchRecord> launches;
    i2_integrator* integ = nullptr;
    hipStream_t stream = nullptr;
    bool ran = false;
    bool all_pairs = false;
    int ran_path = 0;              // path of the last run (its outputs are the ones to read)
    uint64_t run_generation = 0;   // mesh generation the last run used
    uint64_t tasks_generation = 0; // mesh generation the installed task lists belong to
    // the runAllPairs task lists are on the device for this mesh generation
    bool all_pairs_lists = false;
    uint64_t all_pairs_generation = 0;
    i2::TypeState type[3];
    i2::DBuf<unsigned long long> d_counter;
    unsigned long long* h_counter = nullptr;   // pinned, one per type, then k_finalize's six clocks
    std::vector<hipEvent_t> marks;              // of the plain path's timing
    i2::SideStream side;           // of the batched path and the adjoint
    i2::AdjState* adj = nullptr;   // adjoint buffers (created by the first loss-and-gradient call)
};

namespace i2 {
// I2_OK if the evaluator's last run completed on the mesh as it is prepared
// now; a later i2_mesh_set_data or i2_mesh_prepare may have changed the pair
// counts and reallocated the arrays the outputs were sized for.
int results_current(const i2_evaluator* ev);
int evaluator_run(i2_evaluator* ev, bool all_pairs, bool check);
void release_refined_mesh(i2_integrator* it);
// Writes the mesh's disjoint (i < j, k) list to m->d_not_list (once per prepare).
int materialize_disjoint_list(const i2_mesh* m);
// Task source of one type of the evaluator's current task lists.
TaskSource task_source(const i2_evaluator* ev, int type);
// Sets flags[i] = 1 for the control panel i of each listed task (list == nullptr: tasks 0..n-1).
int mark_unconverged(i2_evaluator* ev, bool implicit, const TaskSource& src, int64_t n, const int32_t* list, uint8_t* flags);
int mesh_upload_and_prepare(i2_mesh* m);
}
