"""Python binding of the MI355X panel-pair integrator (ctypes over the C ABI).

This is plumbing for tests and benchmarks: every computation runs in the HIP
library ``libintegrator2_mi355x.so`` built by ``integrator2_amd.build``.  The
classes mirror the reference's C++ API (Mesh3D, NumericalIntegrator3D,
EvaluatorJ3DK in andreyypopov/integrator2 src/) with the same names and
argument meaning.  There is no fallback: if the library is missing or no GPU
is present, the calls raise.
"""
import ctypes
import os

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libintegrator2_mi355x.so")

SIMPLE_NEIGHBORS = 0     # one shared vertex (vertex-sharing)
ATTACHED_NEIGHBORS = 1   # shared edge (edge-sharing)
NOT_NEIGHBORS = 2        # disjoint
TYPE_NAMES = {0: "vertex-sharing", 1: "edge-sharing", 2: "disjoint"}

# tasks per call of the allocation-free runPairs (I2_NOALLOC_MAX_TASKS)
NOALLOC_MAX_TASKS = 262144

PLAIN_TEXT = 1
CSV = 2

# Cowper's 13-point rule (7th order) with the reference's 15-digit literals,
# src/QuadratureFormula3d.cuh:181-213 (qf3D13).
QF3D13_L12 = np.array([
    [0.333333333333333, 0.333333333333333],
    [0.479308067841923, 0.260345966079038],
    [0.260345966079038, 0.479308067841923],
    [0.260345966079038, 0.260345966079038],
    [0.869739794195598, 0.065130102902216],
    [0.065130102902216, 0.869739794195598],
    [0.065130102902216, 0.065130102902216],
    [0.638444188569809, 0.312865496004875],
    [0.312865496004875, 0.638444188569809],
    [0.638444188569809, 0.048690315425316],
    [0.048690315425316, 0.638444188569809],
    [0.312865496004875, 0.048690315425316],
    [0.048690315425316, 0.312865496004875],
])
QF3D13_W = np.array([-0.149570044467670] + [0.175615257433204] * 3 + [0.053347235608839] * 3 + [0.077113760890257] * 6)
QF3D13_ORDER = 7

_P = ctypes.c_void_p
_I64 = ctypes.c_int64
_D = ctypes.c_double
_lib = None


class I2Error(RuntimeError):
    pass


def _ptr(a):
    return None if a is None else a.ctypes.data_as(_P)


def lib():
    """Loads the HIP library (raises if it has not been built)."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise I2Error(f"{LIB_PATH} is missing: run integrator2_amd.build.build() first")
    L = ctypes.CDLL(LIB_PATH)
    L.i2_last_error.restype = ctypes.c_char_p
    _lib = L
    return L


def _check(status):
    if status != 0:
        msg = lib().i2_last_error().decode(errors="replace")
        raise I2Error(f"status {status}: {msg}")


def synchronize(device=0):
    _check(lib().i2_device_synchronize(ctypes.c_int(device)))


def device_count():
    n = ctypes.c_int(0)
    _check(lib().i2_device_count(ctypes.byref(n)))
    return n.value


# ---------------------------------------------------------------- meshes
def icosphere(level, axes=(1.0, 1.0, 1.0), jitter=0.0, seed=0):
    """Icosphere subdivided `level` times mapped to an ellipsoid, jittered along its normal."""
    L = lib()
    nV, nT = _I64(), _I64()
    args = [ctypes.c_int(level), _D(axes[0]), _D(axes[1]), _D(axes[2]), _D(jitter), ctypes.c_uint64(seed)]
    _check(L.i2_meshgen_icosphere(*args, None, None, ctypes.byref(nV), ctypes.byref(nT)))
    xyz = np.zeros((nV.value, 3))
    tri = np.zeros((nT.value, 3), np.int32)
    _check(L.i2_meshgen_icosphere(*args, _ptr(xyz), _ptr(tri), ctypes.byref(nV), ctypes.byref(nT)))
    return xyz, tri


def torus(nmajor=256, nminor=128, R=1.0, r=0.25, jitter=0.0, seed=0):
    L = lib()
    nV, nT = _I64(), _I64()
    args = [ctypes.c_int(nmajor), ctypes.c_int(nminor), _D(R), _D(r), _D(jitter), ctypes.c_uint64(seed)]
    _check(L.i2_meshgen_torus(*args, None, None, ctypes.byref(nV), ctypes.byref(nT)))
    xyz = np.zeros((nV.value, 3))
    tri = np.zeros((nT.value, 3), np.int32)
    _check(L.i2_meshgen_torus(*args, _ptr(xyz), _ptr(tri), ctypes.byref(nV), ctypes.byref(nT)))
    return xyz, tri


def quadrature_rule(nPts):
    """The reference's triangle rule with nPts points (qf3D1 ... qf3D13,
    src/QuadratureFormula3d.cuh): (L12 of shape (nPts, 2), weights, order)."""
    L12 = np.zeros((nPts, 2)) if nPts > 0 else np.zeros((0, 2))
    w = np.zeros(max(nPts, 0))
    order = ctypes.c_int()
    _check(lib().i2_quadrature_rule(ctypes.c_int(nPts), _ptr(L12), _ptr(w), ctypes.byref(order)))
    return L12, w, order.value


def export_mesh_obj(filename, xyz, tri):
    """exportMeshToObj (src/Mesh3d.cu:264-276)."""
    xyz = np.ascontiguousarray(xyz, np.float64)
    tri = np.ascontiguousarray(tri, np.int32)
    _check(lib().i2_export_mesh_obj(filename.encode(), _ptr(xyz), _I64(len(xyz)), _ptr(tri), _I64(len(tri))))


def export_mesh_vtk(filename, xyz, tri, refinements=(None, None, None)):
    """exportMeshToVtk (src/Mesh3d.cu:278-343); refinements: three per-cell count arrays or None."""
    xyz = np.ascontiguousarray(xyz, np.float64)
    tri = np.ascontiguousarray(tri, np.int32)
    refs = [None if r is None or len(r) == 0 else np.ascontiguousarray(r, np.uint8) for r in refinements]
    for r in refs:
        if r is not None and len(r) != len(tri):
            raise I2Error("a refinement-count array needs one entry per cell")
    _check(lib().i2_export_mesh_vtk(filename.encode(), _ptr(xyz), _I64(len(xyz)), _ptr(tri), _I64(len(tri)),
                                    _ptr(refs[0]), _ptr(refs[1]), _ptr(refs[2])))


def _device_to_host(dptr, shape, dtype):
    out = np.zeros(shape, dtype)
    if out.size:
        _check(lib().i2_copy_to_host(_ptr(out), dptr, _I64(out.nbytes)))
    return out


def batch_spec(nmeshes=64, seed=0):
    levels = np.zeros(nmeshes, np.int32)
    axes = np.zeros((nmeshes, 3))
    _check(lib().i2_meshgen_batch_spec(ctypes.c_int(nmeshes), ctypes.c_uint64(seed), _ptr(levels), _ptr(axes)))
    return levels, axes


# ---------------------------------------------------------------- Mesh3D
class Mesh3D:
    """Mesh3D (src/Mesh3d.cuh:55-126): vertices, cells, normals, areas, neighbour lists."""

    def __init__(self, device=0):
        self._h = _P()
        _check(lib().i2_mesh_create(ctypes.byref(self._h), ctypes.c_int(device)))

    def __del__(self):
        if getattr(self, "_h", None) and _lib is not None:
            _lib.i2_mesh_destroy(self._h)
            self._h = None

    def loadMeshFromFile(self, filename, scale=1.0):
        st = lib().i2_mesh_load_file(self._h, filename.encode(), _D(scale))
        if st != 0:
            return False
        return True

    def setData(self, xyz, tri):
        xyz = np.ascontiguousarray(xyz, np.float64)
        tri = np.ascontiguousarray(tri, np.int32)
        _check(lib().i2_mesh_set_data(self._h, _ptr(xyz), _I64(len(xyz)), _ptr(tri), _I64(len(tri))))

    def prepareMesh(self):
        _check(lib().i2_mesh_prepare(self._h))

    def sizes(self):
        nV, nT = _I64(), _I64()
        pairs = (ctypes.c_int64 * 3)()
        _check(lib().i2_mesh_sizes(self._h, ctypes.byref(nV), ctypes.byref(nT), pairs))
        return nV.value, nT.value, [pairs[0], pairs[1], pairs[2]]

    def getVertices(self):
        out = np.zeros((self.sizes()[0], 3))
        _check(lib().i2_mesh_copy_vertices(self._h, _ptr(out)))
        return out

    def getCells(self):
        out = np.zeros((self.sizes()[1], 3), np.int32)
        _check(lib().i2_mesh_copy_cells(self._h, _ptr(out)))
        return out

    def getCellNormals(self):
        out = np.zeros((self.sizes()[1], 3))
        _check(lib().i2_mesh_copy_normals(self._h, _ptr(out)))
        return out

    def getCellMeasures(self):
        out = np.zeros(self.sizes()[1])
        _check(lib().i2_mesh_copy_measures(self._h, _ptr(out)))
        return out

    def _neighbors(self, t):
        n = self.sizes()[2][t]
        out = np.zeros((n, 3), np.int32)
        _check(lib().i2_mesh_copy_neighbors(self._h, ctypes.c_int(t), _ptr(out)))
        return out

    def getSimpleNeighbors(self):
        return self._neighbors(SIMPLE_NEIGHBORS)

    def getAttachedNeighbors(self):
        return self._neighbors(ATTACHED_NEIGHBORS)

    def getNotNeighbors(self):
        return self._neighbors(NOT_NEIGHBORS)


# ---------------------------------------------------------------- NumericalIntegrator3D
class NumericalIntegrator3D:
    """NumericalIntegrator3D(mesh, qf) (src/NumericalIntegrator3d.cuh:89-327)."""

    def __init__(self, mesh, L12=QF3D13_L12, weights=QF3D13_W, order=QF3D13_ORDER):
        self.mesh = mesh
        self._L12 = np.ascontiguousarray(L12, np.float64)
        self._w = np.ascontiguousarray(weights, np.float64)
        self._h = _P()
        _check(lib().i2_integrator_create(ctypes.byref(self._h), mesh._h, _ptr(self._L12), _ptr(self._w),
                                          ctypes.c_int(len(self._w)), ctypes.c_int(order)))

    def __del__(self):
        if getattr(self, "_h", None) and _lib is not None:
            _lib.i2_integrator_destroy(self._h)
            self._h = None

    def setFixedRefinementLevel(self, refinementLevel=0):
        _check(lib().i2_integrator_set_fixed_refinement_level(self._h, ctypes.c_int(refinementLevel)))

    def setErrorControl(self, maxLevel=5, tol=1e-5, refParityQuirk=True):
        _check(lib().i2_integrator_set_error_control(self._h, ctypes.c_int(maxLevel), _D(tol), ctypes.c_int(int(refParityQuirk))))

    def getRefinementsRequired(self, t):
        """Per original cell, the refinement passes of the last automatic run for type t
        (empty in fixed-level mode), as uint8."""
        n = _I64()
        _check(lib().i2_integrator_refinements_required(self._h, ctypes.c_int(t), None, None, ctypes.byref(n)))
        out = np.zeros(n.value, np.uint8)
        if n.value:
            _check(lib().i2_integrator_refinements_required(self._h, ctypes.c_int(t), None, _ptr(out), ctypes.byref(n)))
        return out

    def refinedMesh(self):
        """(vertices (nV, 3), cells (nT, 3), measures (nT,)) of the mesh split to the fixed level."""
        dv, dc, dm = _P(), _P(), _P()
        nV, nT = _I64(), _I64()
        _check(lib().i2_integrator_refined_mesh(self._h, ctypes.byref(dv), ctypes.byref(dc), ctypes.byref(dm),
                                                ctypes.byref(nV), ctypes.byref(nT)))
        return (_device_to_host(dv, (nV.value, 3), np.float64), _device_to_host(dc, (nT.value, 3), np.int32),
                _device_to_host(dm, (nT.value,), np.float64))


# ---------------------------------------------------------------- EvaluatorJ3DK
class EvaluatorJ3DK:
    """EvaluatorJ3DK(mesh, integrator) (src/evaluators/evaluatorJ3DK.cuh:151-185)."""

    def __init__(self, mesh, integrator):
        self.mesh, self.integrator = mesh, integrator
        self._h = _P()
        _check(lib().i2_evaluator_create(ctypes.byref(self._h), mesh._h, integrator._h))

    def __del__(self):
        if getattr(self, "_h", None) and _lib is not None:
            _lib.i2_evaluator_destroy(self._h)
            self._h = None

    def runAllPairs(self, checkCorrectness=False):
        _check(lib().i2_evaluator_run_all_pairs(self._h, ctypes.c_int(int(checkCorrectness))))

    def runPairs(self, simple, attached, notn):
        arrs = [np.ascontiguousarray(np.asarray(a, np.int32).reshape(-1, 3)) for a in (simple, attached, notn)]
        _check(lib().i2_evaluator_run_pairs(self._h, _ptr(arrs[0]), _I64(len(arrs[0])), _ptr(arrs[1]), _I64(len(arrs[1])),
                                            _ptr(arrs[2]), _I64(len(arrs[2]))))

    def runTasksNoAlloc(self, t, d_tasks, n, d_integrals, d_results, d_conv):
        """runPairs for one type on device arrays, with no device allocation
        (i2_evaluator_run_tasks_noalloc): d_* are device addresses (integers)
        of n (i, j, k) int32 triples and of the outputs (n x 4 doubles, n x 3
        doubles, n int8).  Returns the refinement iterations K."""
        K = ctypes.c_int()
        _check(lib().i2_evaluator_run_tasks_noalloc(self._h, ctypes.c_int(t), _P(d_tasks), _I64(n), _P(d_integrals),
                                                    _P(d_results), _P(d_conv), ctypes.byref(K)))
        return K.value

    def taskCount(self, t):
        n = _I64()
        _check(lib().i2_evaluator_task_count(self._h, ctypes.c_int(t), ctypes.byref(n)))
        return n.value

    def getTasks(self, t):
        """Host copy of the device (i, j, k) task list of type t (Evaluator3D::getTasks)."""
        d = _P()
        n = _I64()
        _check(lib().i2_evaluator_device_tasks(self._h, ctypes.c_int(t), ctypes.byref(d), ctypes.byref(n)))
        return _device_to_host(d, (n.value, 3), np.int32)

    def results(self, t, errors=False):
        """Dict with tasks (n,3), integrals (n,4), results (n,3), conv (n,), errors (n,) if requested."""
        n = self.taskCount(t)
        # not zeroed: the call writes every element
        out = dict(tasks=np.empty((n, 3), np.int32), integrals=np.empty((n, 4)), results=np.empty((n, 3)),
                   conv=np.empty(n, np.int8))
        err = np.empty(n) if errors else None
        _check(lib().i2_evaluator_get_results(self._h, ctypes.c_int(t), _ptr(out["tasks"]), _ptr(out["integrals"]),
                                              _ptr(out["results"]), _ptr(err), _ptr(out["conv"])))
        if errors:
            out["errors"] = err
        return out

    def refinementIterations(self, t):
        K = ctypes.c_int()
        _check(lib().i2_evaluator_refinement_iterations(self._h, ctypes.c_int(t), ctypes.byref(K)))
        return K.value

    def typeStats(self, t):
        ms = _D()
        n = _I64()
        _check(lib().i2_evaluator_type_stats(self._h, ctypes.c_int(t), ctypes.byref(ms), ctypes.byref(n)))
        return ms.value, n.value

    def setPath(self, path):
        """0: plain per-type, per-level launches; 1: batched persistent kernels."""
        _check(lib().i2_evaluator_set_path(self._h, ctypes.c_int(path)))

    def setTuning(self, pairsPerWorkgroup=64, pointsPerLane=13):
        _check(lib().i2_evaluator_set_tuning(self._h, ctypes.c_int(pairsPerWorkgroup), ctypes.c_int(pointsPerLane)))

    def setProfiling(self, enable=True):
        _check(lib().i2_evaluator_set_profiling(self._h, ctypes.c_int(int(enable))))

    def sweepMs(self):
        ms = _D()
        _check(lib().i2_evaluator_sweep_ms(self._h, ctypes.byref(ms)))
        return ms.value

    def launchRecords(self):
        """List of (type, level, tasks, ms) of the last run's integration launches (profiling mode)."""
        cnt = _I64()
        _check(lib().i2_evaluator_launch_records(self._h, _I64(0), None, None, None, ctypes.byref(cnt)))
        n = cnt.value
        tl = np.zeros((n, 2), np.int32)
        tasks = np.zeros(n, np.int64)
        ms = np.zeros(n)
        _check(lib().i2_evaluator_launch_records(self._h, _I64(n), _ptr(tl), _ptr(tasks), _ptr(ms), ctypes.byref(cnt)))
        return [(int(tl[q, 0]), int(tl[q, 1]), int(tasks[q]), float(ms[q])) for q in range(n)]

    def outputResultsToFile(self, t, fmt, directory=None):
        st = lib().i2_evaluator_output_results_to_file(self._h, ctypes.c_int(t), ctypes.c_int(fmt),
                                                       None if directory is None else directory.encode())
        return st == 0

    def lossAndGrad(self, seed=1):
        """Loss L = sum_ij w_ij Theta_ij + v_ij . J_ij over all ordered pairs of the last
        runAllPairs (weights drawn from seed) and dL/dX, shape (nV, 3), from the adjoint kernels."""
        nV = self.mesh.sizes()[0]
        grad = np.zeros((nV, 3))
        loss = ctypes.c_double()
        _check(lib().i2_evaluator_loss_and_grad(self._h, ctypes.c_uint64(seed), ctypes.byref(loss), _ptr(grad)))
        return loss.value, grad

    def adjointMs(self):
        ms = ctypes.c_double()
        _check(lib().i2_evaluator_adjoint_ms(self._h, ctypes.byref(ms)))
        return ms.value


# ---------------------------------------------------------------- batched path
BATCH_PER_PAIR = 0
BATCH_ROW_SUMS = 1


class Batch:
    """Many meshes in one captured graph of persistent kernels (i2_batch_*)."""

    def __init__(self, device=0):
        self._h = _P()
        _check(lib().i2_batch_create(ctypes.byref(self._h), ctypes.c_int(device)))
        self.meshes = []

    def __del__(self):
        if getattr(self, "_h", None) and _lib is not None:
            _lib.i2_batch_destroy(self._h)
            self._h = None

    def addMesh(self, mesh):
        idx = ctypes.c_int()
        _check(lib().i2_batch_add_mesh(self._h, mesh._h, ctypes.byref(idx)))
        self.meshes.append(mesh)
        return idx.value

    def configure(self, integrator, outputMode=BATCH_PER_PAIR):
        self._integrator = integrator
        _check(lib().i2_batch_configure(self._h, integrator._h, ctypes.c_int(outputMode)))

    def setTuning(self, pairsPerWorkgroup=64, pointsPerLane=13):
        _check(lib().i2_batch_set_tuning(self._h, ctypes.c_int(pairsPerWorkgroup), ctypes.c_int(pointsPerLane)))

    def run(self):
        ms = _D()
        _check(lib().i2_batch_run(self._h, ctypes.byref(ms)))
        return ms.value

    def enableAdjoint(self, enable=True, seed=1):
        """Append the adjoint of L = sum w Theta + v . J (weights from seed) to the batch graph."""
        _check(lib().i2_batch_enable_adjoint(self._h, ctypes.c_int(int(enable)), ctypes.c_uint64(seed)))

    def lossAndGrad(self, mesh):
        nV = self.meshes[mesh].sizes()[0]
        grad = np.zeros((nV, 3))
        loss = ctypes.c_double()
        _check(lib().i2_batch_get_loss_and_grad(self._h, ctypes.c_int(mesh), ctypes.byref(loss), _ptr(grad)))
        return loss.value, grad

    def autotune(self, reps=2, includeWholeRule=True):
        """Times pairs-per-workgroup {16, 32, 64, 128} x points-per-lane {1, 2, 4} (+ 13) and keeps
        the fastest; returns (pairsPerWorkgroup, pointsPerLane, {(P, ppl): median ms})."""
        ppls = [1, 2, 4, 13] if includeWholeRule else [1, 2, 4]
        table = np.zeros(4 * len(ppls))
        bp, bl = ctypes.c_int(), ctypes.c_int()
        _check(lib().i2_batch_autotune(self._h, ctypes.c_int(reps), ctypes.c_int(int(includeWholeRule)),
                                       ctypes.byref(bp), ctypes.byref(bl), _ptr(table)))
        grid = {(P, l): float(table[a * len(ppls) + k]) for a, P in enumerate([16, 32, 64, 128]) for k, l in enumerate(ppls)}
        return bp.value, bl.value, grid

    def setProfiling(self, enable=True):
        _check(lib().i2_batch_set_profiling(self._h, ctypes.c_int(int(enable))))

    def sweepMs(self):
        ms = _D()
        _check(lib().i2_batch_sweep_ms(self._h, ctypes.byref(ms)))
        return ms.value

    def pairResults(self, mesh, t):
        n = 2 * self.meshes[mesh].sizes()[2][t]
        ints = np.zeros((n, 4))
        res = np.zeros((n, 3))
        conv = np.zeros(n, np.int8)
        _check(lib().i2_batch_get_pair_results(self._h, ctypes.c_int(mesh), ctypes.c_int(t), _ptr(ints), _ptr(res), _ptr(conv)))
        return dict(integrals=ints, results=res, conv=conv)

    def rowSums(self, mesh):
        out = np.zeros((self.meshes[mesh].sizes()[1], 4))
        _check(lib().i2_batch_get_row_sums(self._h, ctypes.c_int(mesh), _ptr(out)))
        return out

    def refinementIterations(self, mesh, t):
        K = ctypes.c_int()
        _check(lib().i2_batch_refinement_iterations(self._h, ctypes.c_int(mesh), ctypes.c_int(t), ctypes.byref(K)))
        return K.value

    def levelCounts(self):
        c = np.zeros((13, 3), np.int64)
        _check(lib().i2_batch_level_counts(self._h, _ptr(c)))
        return c

    def taskCount(self):
        n = _I64()
        _check(lib().i2_batch_task_count(self._h, ctypes.byref(n)))
        return n.value
