/*
 * integrator2_mi355x.h -- C ABI of the MI355X (gfx950) panel-pair integrator.
 *
 * Plain pointers and sizes only; host pointers are borrowed for the duration
 * of a call, device memory is owned by the objects.  Every function returns
 * I2_OK (0) or a negative status and never exits the process; the message of
 * the last failure on the calling thread is returned by i2_last_error().
 *
 * Each entry point names the reference interface it replaces
 * (andreyypopov/integrator2, paths relative to the repository root).
 */
#ifndef INTEGRATOR2_MI355X_H
#define INTEGRATOR2_MI355X_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* ---- status codes (the reference calls exit(EXIT_FAILURE) instead,
 *      src/common/cuda_helper.cuh:41-54) */
#define I2_OK 0
#define I2_ERR_INVALID (-1)  /* bad argument */
#define I2_ERR_HIP (-2)      /* HIP runtime error or no device */
#define I2_ERR_ALLOC (-3)    /* device or host allocation failed */
#define I2_ERR_STATE (-4)    /* call out of order (e.g. results before a run) */
#define I2_ERR_RANGE (-5)    /* size beyond a documented limit */
#define I2_ERR_IO (-6)       /* file could not be read or written */
#define I2_ERR_TOPOLOGY (-7) /* mesh topology the integrator cannot handle */

/* ---- neighbour types: the values of neighbour_type_enum (src/Mesh3d.cuh:18-23) */
#define I2_SIMPLE_NEIGHBORS 0   /* exactly one shared vertex ("vertex-sharing") */
#define I2_ATTACHED_NEIGHBORS 1 /* a shared edge ("edge-sharing") */
#define I2_NOT_NEIGHBORS 2      /* no shared vertex ("disjoint") */

/* ---- output formats: output_format_enum (src/evaluators/evaluator3d.cuh:19-22) */
#define I2_OUTPUT_PLAIN_TEXT 1
#define I2_OUTPUT_CSV 2

typedef struct i2_mesh i2_mesh;             /* Mesh3D */
typedef struct i2_integrator i2_integrator; /* NumericalIntegrator3D */
typedef struct i2_evaluator i2_evaluator;   /* Evaluator3D / EvaluatorJ3DK */
typedef struct i2_batch i2_batch;           /* batched path (no counterpart in the reference) */

/* Message of the last failed call on this thread ("" if none). */
const char* i2_last_error(void);
/* Number of visible HIP devices (0 without a GPU). */
int i2_device_count(int* n);
/* Host-side evaluation of the inner integral (Psi, Theta) of triangle tri9 at
 * n points, with the device formulas compiled for the CPU: fast = 0 is the
 * reference's expression (thetaPsi, src/evaluators/evaluatorJ3DK.cu:266-313),
 * fast = 1 the form the kernels use at any point, fast = 2 and 3 the forms they
 * use for points at least two and six of K_j's longest edges away from it.  For
 * checking. */
int i2_host_theta_psi(int fast, const double* pts, int64_t n, const double* tri9, double* out4);
/* Host-side evaluation of the kernels' FP64 logarithm (fn = 0, of x),
 * two-argument arctangent (fn = 1, atan2(y, x)), square root (fn = 2, of x;
 * the host uses the library's 1/sqrt as the estimate the device takes from
 * the hardware) and reciprocal (fn = 6, of x; the host starts from a
 * single-precision estimate); fn = 10 and 11: the table paths of the log and
 * atan2 without their range tests, which the inner integral runs on every
 * lane before it redoes the lanes outside the ranges.  For checking. */
int i2_host_math(int fn, const double* x, const double* y, int64_t n, double* out);
/* The same functions evaluated on the device (fn 0-2, 6, 10 and 11 as
 * above; 3, 4, 5, 7: the HIP library's log, atan2, sqrt and 1/x, for
 * comparison; 8, 9: the hardware estimates of 1/x and 1/sqrt(x) that
 * rcp_pos, div_pos and sqrt_pos refine).  For checking. */
int i2_device_math(int device, int fn, const double* x, const double* y, int64_t n, double* out);
/* Host-side evaluation of one ordered task's integrals (Psi, Theta) at
 * refinement level `level` with the kernels' device code compiled for the
 * host (the inner integral in its general form): I9, J9 the two panels' vertices, vid6 their vertex ids (which decide
 * the neighbour type).  For checking. */
int i2_host_task_value(const double* I9, const double* J9, const int32_t* vid6, int level, const double* L12,
                       const double* w, int nPts, double* out4);
/* Host-side evaluation of the adjoint kernels' numbering of a refined panel's
 * points: point q of a rule of nPts on the sub-panels, in order, is the rule's
 * point `point` on sub-panel `sub` (0 <= q <= 2^28).  For checking. */
int i2_host_point_split(int nPts, const int64_t* q, int64_t n, int64_t* sub, int64_t* point);

/* ======================================================================
 * Mesh3D (src/Mesh3d.cuh:55-126, src/Mesh3d.cu)
 * ==================================================================== */
int i2_mesh_create(i2_mesh** out, int device);
void i2_mesh_destroy(i2_mesh* m);
/* Mesh3D::loadMeshFromFile (src/Mesh3d.cu:159-217): "nV nC", then
 * "idx x y z" per vertex, then "idx 203 a b c" triangles (1-based indices);
 * entities of other types are skipped.  Coordinates are multiplied by scale. */
int i2_mesh_load_file(i2_mesh* m, const char* path, double scale);
/* Direct upload of vertices (xyz, nV*3 doubles) and 0-based triangles (nT*3). */
int i2_mesh_set_data(i2_mesh* m, const double* xyz, int64_t nV, const int32_t* tri, int64_t nT);
/* Mesh3D::prepareMesh (src/Mesh3d.cu:219-226): normals, areas and the three
 * neighbour lists (pairs i<j classified by the number of shared vertex indices). */
int i2_mesh_prepare(i2_mesh* m);
/* Sizes; pairs[t] = number of unordered (i<j) pairs of neighbour type t. */
int i2_mesh_sizes(const i2_mesh* m, int64_t* nV, int64_t* nT, int64_t pairs[3]);
/* Mesh3D getters (src/Mesh3d.cuh:70-126), copied to host buffers. */
int i2_mesh_copy_vertices(const i2_mesh* m, double* xyz);
int i2_mesh_copy_cells(const i2_mesh* m, int32_t* tri);
int i2_mesh_copy_normals(const i2_mesh* m, double* n3);
int i2_mesh_copy_measures(const i2_mesh* m, double* s);
/* getSimpleNeighbors / getAttachedNeighbors / getNotNeighbors: (i, j, k)
 * with i < j and k the position in the list, lexicographic order. */
int i2_mesh_copy_neighbors(const i2_mesh* m, int type, int32_t* ijk);
/* Device pointer and length of a mesh array for deviceVector-style getters:
 * what = 0 vertices (double3), 1 cells (int3), 2 normals (double3),
 * 3 measures (double), 4 simple, 5 attached, 6 disjoint neighbours (int3;
 * the disjoint list is written out on the first request, I2_ERR_RANGE beyond
 * 2^31 - 1 pairs). */
int i2_mesh_device_array(const i2_mesh* m, int what, const void** dptr, int64_t* n);
/* exportMeshToObj (src/Mesh3d.cu:264-276): OBJ text with 1-based faces. */
int i2_export_mesh_obj(const char* path, const double* xyz, int64_t nV, const int32_t* tri, int64_t nT);
/* exportMeshToVtk (src/Mesh3d.cu:278-343): VTK XML PolyData (ASCII) with one
 * Int32 cell array "<type>Refinements" per non-NULL count array (nT bytes). */
int i2_export_mesh_vtk(const char* path, const double* xyz, int64_t nV, const int32_t* tri, int64_t nT,
                       const uint8_t* simpleRefinements, const uint8_t* attachedRefinements, const uint8_t* notRefinements);

/* ======================================================================
 * NumericalIntegrator3D (src/NumericalIntegrator3d.cuh:89-327)
 * ==================================================================== */
/* The triangle rules qf3D1, qf3D3, qf3D4, qf3D6, qf3D7, qf3D9, qf3D12, qf3D13
 * (src/QuadratureFormula3d.cuh:34-213, same decimal literals): nPts (L1, L2)
 * pairs into L12, nPts weights into w, the order into *order (any may be NULL). */
int i2_quadrature_rule(int nPts, double* L12, double* w, int* order);
/* NumericalIntegrator3D(mesh, qf) (src/NumericalIntegrator3d.cu:197-216):
 * L12 = nPts (L1, L2) pairs, w = nPts weights, order = rule order (the Runge
 * factor is 2^order).  Default mode: automatic error control with the
 * reference's maxLevel 5 and tolerance 1e-5 (src/common/constants.h:18,56). */
int i2_integrator_create(i2_integrator** out, const i2_mesh* mesh, const double* L12, const double* w, int nPts, int order);
void i2_integrator_destroy(i2_integrator* it);
/* setFixedRefinementLevel (src/NumericalIntegrator3d.cu:225-229).  Level L
 * integrates over all 4^L sub-panels of each control panel. */
int i2_integrator_set_fixed_refinement_level(i2_integrator* it, int level);
/* Automatic error control with run-time maxLevel and Runge tolerance (compile-time
 * MAX_REFINE_LEVEL / EPS_INTEGRATION in the reference).  refParityQuirk != 0
 * reproduces the reference's result-buffer swap (src/evaluators/evaluatorJ3DK.cu:976-990). */
int i2_integrator_set_error_control(i2_integrator* it, int maxLevel, double tol, int refParityQuirk);
/* NumericalIntegrator3D::getRefinementsRequired (src/NumericalIntegrator3d.cuh:316-324):
 * per original cell, how many refinement passes of the last automatic run
 * on this integrator refined it for `type` (the counts of
 * determineCellsToBeRefined, src/NumericalIntegrator3d.cu:461-499: a task
 * converged at iteration c counts c, one unconverged after the comparison at
 * maxLevel counts maxLevel + 1; a cell takes the largest over its tasks).
 * *n = nT, or 0 in fixed-level mode or before a run (the reference allocates
 * the counts for automatic error control only).  d_counts receives a device
 * pointer valid until the next run; h_counts (nT bytes) a host copy; either
 * may be NULL.  The evaluator of that run must still exist. */
int i2_integrator_refinements_required(i2_integrator* it, int type, const void** d_counts, uint8_t* h_counts, int64_t* n);
/* getRefinedVertices / getRefinedCells / getRefinedCellMeasures
 * (src/NumericalIntegrator3d.cuh:243-274) in fixed-level mode: the mesh split
 * L times by kSplitCell (src/NumericalIntegrator3d.cu:37-87): nV + nT (4^L - 1)
 * vertices (double3) and nT 4^L cells (int3) with measures (double).  The
 * slots of the new vertices and cells of cell idx are fixed at 3 idx and 4 idx
 * of each pass (the reference takes them from atomic counters).  Device
 * pointers owned by the integrator; built on the first call per (mesh, level).
 * I2_ERR_STATE in automatic mode (the reference's arrays then hold the
 * working state of the last refined type). */
int i2_integrator_refined_mesh(i2_integrator* it, const void** d_vertices, const void** d_cells, const void** d_measures,
                               int64_t* nV, int64_t* nT);

/* ======================================================================
 * Evaluator3D / EvaluatorJ3DK (src/evaluators/evaluator3d.cuh:42-100,
 * src/evaluators/evaluatorJ3DK.cuh:151-185)
 * ==================================================================== */
int i2_evaluator_create(i2_evaluator** out, const i2_mesh* m, i2_integrator* it);
void i2_evaluator_destroy(i2_evaluator* ev);
/* Evaluator3D::runAllPairs (src/evaluators/evaluator3d.cu:120-204): ordered
 * task list per type = [(i,j,k) for the i<j list] ++ [(j,i,n+k)], integrated
 * per type (vertex-sharing, edge-sharing, disjoint) with per-level launches;
 * checkCorrectness computes the (i,j)/(j,i) symmetry error. */
int i2_evaluator_run_all_pairs(i2_evaluator* ev, int checkCorrectness);
/* Evaluator3D::runPairs (src/evaluators/evaluator3d.cu:213-288): user task
 * lists (i, j, k) per type; k is ignored (tasks are numbered by position). */
int i2_evaluator_run_pairs(i2_evaluator* ev, const int32_t* simple3, int64_t nSimple,
                           const int32_t* attached3, int64_t nAttached, const int32_t* not3, int64_t nNot);
/* No counterpart in the reference.  For callers that cannot allocate device
 * memory (code under HIP graph capture, tight serving loops, harnesses that
 * forbid hipMalloc): runPairs for one type with everything on the device.
 * d_tasks3 holds n device (i, j, k) triples (k is ignored); the outputs are
 * the caller's device arrays d_integrals4 (n x (Psi, Theta), 32-byte
 * aligned), d_results3 (n x J) and d_conv (n convergence iterations); *K
 * receives the refinement iterations run.  Values, levels and K equal those
 * of i2_evaluator_run_pairs on the same list, computed by the same kernels.
 * The refinement state (a level buffer, the lists of unconverged tasks, the
 * counters) lives in a static device array of the library, one per GPU,
 * which bounds n to I2_NOALLOC_MAX_TASKS (I2_ERR_RANGE above it).  The call
 * allocates nothing, returns when the outputs are complete, and leaves the
 * evaluator's own results alone.  Calls that overlap on one GPU share that
 * array and race.  Errors as runPairs: I2_ERR_INVALID for a cell outside
 * the mesh, I2_ERR_TOPOLOGY for a pair of another neighbour type. */
#define I2_NOALLOC_MAX_TASKS 262144
int i2_evaluator_run_tasks_noalloc(i2_evaluator* ev, int type, const int32_t* d_tasks3, int64_t n,
                                   double* d_integrals4, double* d_results3, int8_t* d_conv, int* K);
int i2_evaluator_task_count(const i2_evaluator* ev, int type, int64_t* n);
/* Evaluator3D::getTasks (src/evaluators/evaluator3d.cuh:89-101): device
 * pointer to the (i, j, k) list of a type (int3, *n entries).  The disjoint
 * list of runAllPairs is decoded on the fly by the kernels; this call writes
 * it out once per run (I2_ERR_RANGE beyond 2^31 - 1 tasks). */
int i2_evaluator_device_tasks(i2_evaluator* ev, int type, const void** d_tasks, int64_t* n);
/* Results of the last run for one type, in task order; any output may be NULL.
 * tasks3: (i, j, k); integrals4: (Psi_x, Psi_y, Psi_z, Theta); results3: J;
 * errors: symmetry error (only after runAllPairs with checkCorrectness);
 * convLevel: refinement iteration at which the task converged (or the last). */
int i2_evaluator_get_results(const i2_evaluator* ev, int type, int32_t* tasks3, double* integrals4,
                             double* results3, double* errors, int8_t* convLevel);
/* Number of refinement iterations K run for a type in the last run. */
int i2_evaluator_refinement_iterations(const i2_evaluator* ev, int type, int* K);
/* Device time (ms) of the last run for a type and the number of refined
 * (sub-panel, panel) tasks integrated. */
int i2_evaluator_type_stats(const i2_evaluator* ev, int type, double* ms, int64_t* refinedTasks);
/* Profiling mode: record HIP events around every integration launch
 * (GpuTimer of src/common/gpu_timer.cuh:14-77 times whole types only). */
int i2_evaluator_set_profiling(i2_evaluator* ev, int enable);
/* Launch records of the last run: (type, level) pairs, task counts and device
 * milliseconds; *count receives the number of records (capacity may be 0). */
int i2_evaluator_launch_records(const i2_evaluator* ev, int64_t capacity, int32_t* type_level, int64_t* tasks,
                                double* ms, int64_t* count);
/* Batched path in profiling mode: device milliseconds of the disjoint-pair
 * sweep kernel (levels 0 and 1) of the last run. */
int i2_evaluator_sweep_ms(const i2_evaluator* ev, double* ms);
/* hipDeviceSynchronize on `device`. */
int i2_device_synchronize(int device);
/* copy_d2h (src/common/cuda_memory.cuh:104-109) for the device pointers the
 * getters return: `bytes` from device memory `src` to host memory `dst`. */
int i2_copy_to_host(void* dst, const void* src, int64_t bytes);
/* Evaluator3D::outputResultsToFile (src/evaluators/evaluator3d.cu:354-457):
 * writes SimpleNeighbors/AttachedNeighbors/NotNeighbors .dat or .csv into dir
 * (NULL = current directory). */
int i2_evaluator_output_results_to_file(const i2_evaluator* ev, int type, int format, const char* dir);

/* Integration path of runAllPairs / runPairs: 0 = plain per-type, per-level
 * launches (the reference's structure, src/evaluators/evaluatorJ3DK.cu:895-1012);
 * 1 = the batched persistent kernels (runAllPairs only).  Both produce the same
 * outputs in the same task order. */
int i2_evaluator_set_path(i2_evaluator* ev, int path);
/* Launch shape of the batched path: pairs per workgroup and quadrature points
 * per lane (1, 2, 4 or 13 = the whole 13-point rule in one lane).  Until
 * the first call the shape follows the mesh's size: 64 pairs of one lane each,
 * fewer pairs and more lanes per pair on small meshes. */
int i2_evaluator_set_tuning(i2_evaluator* ev, int pairsPerWorkgroup, int pointsPerLane);

/* ---- shape sensitivity (no counterpart in the reference) --------------
 * Scalar loss over every ordered pair of the last runAllPairs,
 *   L = sum_ij w_ij Theta_ij + v_ij . J_ij,
 * Theta_ij the Theta channel of the pair's integrals, J_ij its result,
 * w_ij ~ N(0,1), v_ij ~ N(0,1)^3 drawn from (seed, pair id i*nT + j), and
 * dL/dX (3*nV doubles, vertex-major) by the hand-written adjoint kernels.
 * Refinement levels, the vertex-sharing 2*pi*p wrap and all branches are
 * frozen at the forward pass's choices.  Both integration paths.  The sums
 * have a fixed order: two calls on the same mesh give the same bits.  Device
 * memory: about nT*(nT/jt + nT/64)*72 bytes of partial-cotangent slots, with
 * jt = 32 above 16,384 panels, 16 above some 2,900 and less below. */
int i2_evaluator_loss_and_grad(i2_evaluator* ev, uint64_t seed, double* loss, double* dLdX);
/* Device milliseconds of the last adjoint run. */
int i2_evaluator_adjoint_ms(const i2_evaluator* ev, double* ms);
/* The loss weights (w, v) of n ordered pairs ij (2 ints each) of a mesh with nT cells. */
int i2_host_loss_weights(uint64_t seed, const int32_t* ij, int64_t n, int nT, double* out4);
/* Host-side reverse mode of one per-point function, for checking: kind 0
 * thetaPsi (params: A, B, C, tau_a, tau_b, tau_c; 18), 1 edge-sharing singular
 * part (JB, JC, tau_a, tau_b, tau_c, 1/|JC-JB|; 16), 2 vertex-sharing singular
 * part (JA, tau_a, tau_b, e, 1/sqrt(S_i); 13), 3, 4 and 5 the terms of thetaPsi
 * (line integrals of 1/r along AB, BC, CA and Theta/2) in the general form and
 * in the far ones from two and six longest edges (A, B, C; 9).  The kernels run
 * kinds 1 to 5; kind 0 is the formula with free tangents.  Returns f(p) and gbar4 . df
 * with respect to p (pbar3) and to every parameter (parbar). */
int i2_host_point_adjoint(int kind, const double* p3, const double* params, const double* gbar4, double* f4,
                          double* pbar3, double* parbar);

/* ======================================================================
 * Batched path: many meshes, all neighbour types and refinement levels in one
 * captured HIP graph of persistent kernels fed by device work queues (no
 * counterpart in the reference, which runs one mesh type by type).
 * ==================================================================== */
#define I2_BATCH_PER_PAIR 0  /* per-pair integrals and J, reference task order */
#define I2_BATCH_ROW_SUMS 1  /* per control panel i: sum over j of (J, Theta) */
int i2_batch_create(i2_batch** out, int device);
void i2_batch_destroy(i2_batch* b);
/* Adds a prepared mesh (same device); meshes are borrowed and must outlive the batch. */
int i2_batch_add_mesh(i2_batch* b, const i2_mesh* m, int* index);
int i2_batch_clear(i2_batch* b);
/* Rule and error control are taken from an integrator object. */
int i2_batch_configure(i2_batch* b, const i2_integrator* it, int outputMode);
/* Launch shape (see i2_evaluator_set_tuning). */
int i2_batch_set_tuning(i2_batch* b, int pairsPerWorkgroup, int pointsPerLane);
/* Runs every task of every mesh; the first run after a change captures the
 * graph, later runs replay it.  ms receives the device time of the run. */
int i2_batch_run(i2_batch* b, double* ms);
/* Appends the adjoint of the loss of i2_evaluator_loss_and_grad (weights from
 * `seed`) to the batch's graph: one replay runs the forward pass and dL/dX
 * of every mesh, with per-pair terms recomputed, not stored (row-sum mode
 * keeps one convergence byte per pair).  No counterpart in the reference. */
int i2_batch_enable_adjoint(i2_batch* b, int enable, uint64_t seed);
/* Loss and dL/dX (3*nV doubles) of one mesh of the last run. */
int i2_batch_get_loss_and_grad(const i2_batch* b, int mesh, double* loss, double* dLdX);
/* Autotuner (no counterpart in the reference): times the batch's graph for
 * pairs per workgroup {16, 32, 64, 128} x points per lane {1, 2, 4} (and 13,
 * the whole rule per lane, when includeWholeRule), the median of `reps`
 * replays each, and leaves the batch on the fastest.  table_ms receives the
 * medians, row-major over (pairs per workgroup, points per lane). */
int i2_batch_autotune(i2_batch* b, int reps, int includeWholeRule, int* bestP, int* bestPPL, double* table_ms);
int i2_batch_get_pair_results(const i2_batch* b, int mesh, int type, double* integrals4, double* results3, int8_t* conv);
/* rows4[i] = (sum_j J_ij, sum_j Theta_ij) over all three types. */
int i2_batch_get_row_sums(const i2_batch* b, int mesh, double* rows4);
int i2_batch_refinement_iterations(const i2_batch* b, int mesh, int type, int* K);
/* counts[3*L + t]: tasks of type t integrated at level L in the last run. */
int i2_batch_level_counts(const i2_batch* b, int64_t* counts);
/* Total ordered tasks of the batch. */
int i2_batch_task_count(const i2_batch* b, int64_t* n);
/* Profiling mode: runs the kernels without the graph, with events around the
 * disjoint sweep; i2_batch_sweep_ms returns its device time. */
int i2_batch_set_profiling(i2_batch* b, int enable);
int i2_batch_sweep_ms(const i2_batch* b, double* ms);

/* ======================================================================
 * Synthetic meshes (no counterpart in the reference, which loads files)
 * Call once with NULL buffers to get nV and nT.
 * ==================================================================== */
/* Geodesic icosphere subdivided `level` times, scaled to semi-axes
 * (ax, ay, az), each vertex moved along the ellipsoid normal by
 * N(0, (jitter_rel * mean edge length)^2) from mt19937_64(seed). */
int i2_meshgen_icosphere(int level, double ax, double ay, double az, double jitter_rel, uint64_t seed,
                         double* xyz, int32_t* tri, int64_t* nV, int64_t* nT);
/* Torus with major radius R, minor radius r on an nmajor x nminor grid, each
 * quad split along a fixed diagonal, jittered along the surface normal. */
int i2_meshgen_torus(int nmajor, int nminor, double R, double r, double jitter_rel, uint64_t seed,
                     double* xyz, int32_t* tri, int64_t* nV, int64_t* nT);
/* Subdivision levels (uniform on {2,3,4,5}) and semi-axes (uniform on
 * (0.5, 3.0)) of a batch of nmeshes icospheres, drawn from mt19937_64(seed). */
int i2_meshgen_batch_spec(int nmeshes, uint64_t seed, int32_t* levels, double* axes3);

#ifdef __cplusplus
}
#endif

#endif /* INTEGRATOR2_MI355X_H */
