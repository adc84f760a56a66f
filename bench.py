"""Benchmark of the panel-pair integrator on one MI355X.

Workload (one "step"): all 26,209,280 ordered panel pairs of the jittered
ellipsoid -- icosphere subdivided 4x (2,562 vertices, 5,120 triangles), semi-axes
(3, 1, 0.5), vertices moved along the normal by N(0, (0.05 * mean edge)^2) from
seed 0 -- integrated in FP64 with the 13-point rule and automatic Runge error
control (up to 3 refinement levels, tolerance 1e-8): all three neighbour types,
analytic singular parts and the final J, per-pair outputs in the reference's
task order, inputs resident in HBM.

Prints one JSON line.  value = ordered pair-integrals per second of the batched
persistent path; plain_value is the same step through the plain per-type,
per-level launches.  `roofline` is for the dominant kernel (the disjoint-pair
sweep, refinement levels 0 and 1), timed with HIP events on the library's
stream.  `cpu_baseline` times the CPU oracle (FP64 OpenMP restatement of the
reference, all host threads) on the whole step, median of 3 runs.

`autotune` is the batch autotuner's table for this workload (pairs per
workgroup x points per lane, median ms of graph replays); the timed steps use
its choice.  `batch64` is 64 ragged meshes (icosphere levels U{2,3,4,5},
semi-axes U(0.5, 3.0), about 7e9 ordered pairs) in one captured graph with
row-sum outputs, tuned by the autotuner on its first 4 meshes.

`adjoint` is the shape-sensitivity step on the jittered unit sphere of the
same size (icosphere-4, axes (1, 1, 1), same jitter and refinement): the
forward pass, then the loss L = sum w Theta + v . J over all ordered pairs
and dL/dX by the adjoint kernels; `ratio` = adjoint time / forward time.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

import integrator2_amd as i2  # noqa: E402

N_PAIRS = 26_209_280
N_DISJOINT = 26_147_900
FP64_PEAK_TFLOPS = 78.6

# The reference formula's FP64 work per quadrature point of the inner integral
# as written (thetaPsi, evaluatorJ3DK.cu:266-313, edge tangents recomputed per
# point, plus the Gauss point and the weighted sum): 188 basic operations, 6
# square roots, 3 logarithms and 1 atan2, the transcendentals weighted by the
# FP64 VALU instructions the HIP math library spends on them on gfx950 (sqrt
# 16, log 92, atan2 99).  Reported as `reference_equivalent_tflops` only: this
# build executes far less than that work, so its rate is not a fraction of the
# peak.
BASIC_OPS_PER_POINT = 188
TRANS_PER_POINT = {"sqrt": 6, "log": 3, "atan2": 1}
TRANS_WEIGHTS = {"sqrt": 16, "log": 92, "atan2": 99}
POINTS = 13
# Integrand evaluations of the sweep per disjoint pair: 13 points at level 0
# and 4 x 13 at level 1, less one, since the rule's centroid is also the
# centroid of the central level-1 child and is evaluated once for both.
EVALS_PER_PAIR = 5 * POINTS - 1
# FP64 operations the sweep executes per evaluation, from rocprofv3 counters of
# one dispatch on this workload (profiles/valu_counters_sweep_icosphere4.md):
# (2 SQ_INSTS_VALU_FMA_F64 + SQ_INSTS_VALU_MUL_F64 + SQ_INSTS_VALU_ADD_F64) x 64
# lanes / evaluations.  roofline.achieved = this x evaluations / the kernel's
# live HIP-event time.  VALU_ISSUE is the share of the VALU issue capacity the
# same dispatch used (SQ_INSTS_VALU x 4 cycles / (SIMDs x busy cycles)).
COUNTER_FLOPS_PER_EVAL = 126.2
COUNTER_VALU_PER_EVAL = 97.2
VALU_ISSUE = 0.82
# HBM bytes per sweep dispatch on this workload, measured with rocprofv3
# FETCH_SIZE and WRITE_SIZE and scaled by a 1 GiB copy's readings
# (0.61 GB read + 3.09 GB written; the algorithmic figure is 2.33 GB)
SWEEP_HBM_BYTES = 3.70e9


def flops_per_point():
    return BASIC_OPS_PER_POINT + sum(TRANS_PER_POINT[k] * TRANS_WEIGHTS[k] for k in TRANS_PER_POINT)


def make_mesh():
    xyz, tri = i2.icosphere(4, (3.0, 1.0, 0.5), 0.05, 0)
    mesh = i2.Mesh3D(0)
    mesh.setData(xyz, tri)
    mesh.prepareMesh()
    return xyz, tri, mesh


def time_steps(ev, steps, warmup):
    for _ in range(warmup):
        ev.runAllPairs(False)
    i2.synchronize(0)
    t0 = time.perf_counter()
    for _ in range(steps):
        ev.runAllPairs(False)
    i2.synchronize(0)
    return (time.perf_counter() - t0) / steps


def progress(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def batch64_step():
    """64 ragged meshes in one graph (row sums), autotuned on the first 4."""
    levels, axes = i2.batch_spec(64, 0)
    meshes = []
    for m in range(64):
        x, t = i2.icosphere(int(levels[m]), tuple(axes[m]), 0.05, 1000 + m)
        mesh = i2.Mesh3D(0)
        mesh.setData(x, t)
        mesh.prepareMesh()
        meshes.append(mesh)
    integ = i2.NumericalIntegrator3D(meshes[0])
    integ.setErrorControl(3, 1e-8, True)
    sub = i2.Batch(0)
    for mesh in meshes[:4]:
        sub.addMesh(mesh)
    sub.configure(integ, i2.BATCH_ROW_SUMS)
    progress("batch64: autotuning on 4 meshes")
    P, ppl, grid = sub.autotune(reps=1)
    del sub
    progress(f"batch64: tuned {P}x{ppl}; running 64 meshes")
    b = i2.Batch(0)
    for mesh in meshes:
        b.addMesh(mesh)
    b.configure(integ, i2.BATCH_ROW_SUMS)
    b.setTuning(P, ppl)
    b.run()
    t0 = time.perf_counter()
    ms = b.run()
    wall = time.perf_counter() - t0
    n = b.taskCount()
    del b
    # the same 64 meshes one after another through the plain per-type, per-level
    # path (per-pair outputs), device time of each type summed
    progress("batch64: plain path, mesh by mesh")
    plain_ms = 0.0
    for mesh in meshes:
        it = i2.NumericalIntegrator3D(mesh)
        it.setErrorControl(3, 1e-8, True)
        ev = i2.EvaluatorJ3DK(mesh, it)
        ev.setPath(0)
        ev.runAllPairs(False)
        plain_ms += sum(ev.typeStats(t)[0] for t in range(3))
        del ev, it
    return {"workload": "64 icospheres, levels U{2,3,4,5} (seed 0): " + ",".join(str(int(x)) for x in levels) +
                        "; semi-axes U(0.5, 3.0); jitter 0.05 mean edge (seed 1000 + mesh); refinement up to 3 "
                        "levels at tol 1e-8; row-sum outputs",
            "ordered_pairs": int(n), "ms": ms, "wall_ms": 1e3 * wall, "value": n / wall, "unit": "pair-integrals/s",
            "plain_ms": plain_ms, "plain_value": n / (plain_ms * 1e-3), "batched_over_plain": plain_ms / ms,
            "tuning": [P, ppl], "autotune_table_ms": {f"{k[0]}x{k[1]}": round(v, 2) for k, v in grid.items()}}


def adjoint_step(args):
    """Forward (batched path) and adjoint on the 5,120-triangle jittered sphere."""
    xyz, tri = i2.icosphere(4, (1.0, 1.0, 1.0), 0.05, 0)
    mesh = i2.Mesh3D(0)
    mesh.setData(xyz, tri)
    mesh.prepareMesh()
    integ = i2.NumericalIntegrator3D(mesh)
    integ.setErrorControl(3, 1e-8, True)
    ev = i2.EvaluatorJ3DK(mesh, integ)
    ev.setPath(1)
    ev.setTuning(args.pairs_per_workgroup, args.points_per_lane)
    t_fwd = time_steps(ev, args.steps, args.warmup)
    for _ in range(args.warmup):
        ev.lossAndGrad(1)
    reps = max(1, args.steps)
    t0 = time.perf_counter()
    adj_ms = []
    results = []
    for _ in range(reps):
        L, G = ev.lossAndGrad(1)
        adj_ms.append(ev.adjointMs())
        results.append((L, G))
    t_adj = (time.perf_counter() - t0) / reps
    # the adjoint's sums have a fixed order: every run gives the same bits
    same_bits = all(Lr == results[0][0] and np.array_equal(Gr, results[0][1]) for Lr, Gr in results)
    return {"workload": "jittered unit sphere, icosphere-4 (5,120 triangles), refinement up to 3 levels at tol 1e-8; "
                        "loss sum w Theta + v . J over 26,209,280 ordered pairs, weights N(0,1) from seed 1",
            "forward_ms": 1e3 * t_fwd, "adjoint_ms": 1e3 * t_adj, "adjoint_device_ms": float(np.median(adj_ms)),
            "ratio": t_adj / t_fwd, "loss": L, "grad_norm": float(np.linalg.norm(G)),
            "runs_bitwise_equal": bool(same_bits), "runs": reps}


def cpu_baseline(xyz, tri, reps=3):
    """CPU oracle (FP64 OpenMP restatement of the reference, all host threads)
    on the whole step: every ordered pair of all three types with automatic
    refinement; the median of `reps` runs."""
    import oracle
    orc = oracle.Oracle(xyz, tri)
    threads = oracle.lib().o_max_threads()
    tasks = [orc.ordered_tasks(t) for t in range(3)]
    times = []
    for _ in range(reps):
        t0 = time.perf_counter()
        for t in range(3):
            orc.run_tasks(t, tasks[t], i2.QF3D13_L12, i2.QF3D13_W, 7, mode=1, level=3, tol=1e-8, nthreads=threads)
        times.append(time.perf_counter() - t0)
    med = float(np.median(times))
    cpu = ""
    try:
        with open("/proc/cpuinfo") as fh:
            cpu = next((l.split(":", 1)[1].strip() for l in fh if l.startswith("model name")), "")
    except OSError:
        pass
    return {"value": N_PAIRS / med, "unit": "pair-integrals/s", "cores": threads, "kind": "port",
            "sample": f"the whole step: all {N_PAIRS:,} ordered pairs with automatic refinement (maxLevel 3, "
                      f"tol 1e-8), median of {reps} runs ({', '.join(f'{x:.2f}' for x in times)} s)",
            "cpu": cpu}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--pairs-per-workgroup", type=int, default=64)
    ap.add_argument("--points-per-lane", type=int, default=13)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-autotune", action="store_true")
    ap.add_argument("--no-batch64", action="store_true")
    args = ap.parse_args()
    if args.gpus != 1:
        print(json.dumps({"error": "the path runs on one GPU; run with --gpus 1"}))
        sys.exit(2)
    if i2.device_count() < 1:
        raise SystemExit("no HIP device")

    xyz, tri, mesh = make_mesh()
    integ = i2.NumericalIntegrator3D(mesh)
    integ.setErrorControl(3, 1e-8, True)

    tune = None
    progress("ellipsoid: autotuning")
    if not args.no_autotune:
        tb = i2.Batch(0)
        tb.addMesh(mesh)
        tb.configure(integ, i2.BATCH_PER_PAIR)
        P, ppl, grid = tb.autotune(reps=3)
        args.pairs_per_workgroup, args.points_per_lane = P, ppl
        tune = {"choice": [P, ppl], "table_ms": {f"{k[0]}x{k[1]}": round(v, 3) for k, v in grid.items()}}
        del tb

    fast = i2.EvaluatorJ3DK(mesh, integ)
    fast.setPath(1)
    fast.setTuning(args.pairs_per_workgroup, args.points_per_lane)
    progress("ellipsoid: batched path")
    t_fast = time_steps(fast, args.steps, args.warmup)
    progress("ellipsoid: plain path")

    plain = i2.EvaluatorJ3DK(mesh, integ)
    plain.setPath(0)
    t_plain = time_steps(plain, max(1, args.steps // 2), 1)

    # dominant kernel: the disjoint sweep (levels 0 and 1), HIP events on the library stream
    fast.setProfiling(True)
    sweep_ms = []
    for _ in range(3):
        fast.runAllPairs(False)
        sweep_ms.append(fast.sweepMs())
    fast.setProfiling(False)
    sweep_ms = float(np.median(sweep_ms))
    points = N_DISJOINT * POINTS * 5      # quadrature points: level 0 (13) and level 1 (4 x 13)
    evals = N_DISJOINT * EVALS_PER_PAIR   # integrand evaluations the kernel executes
    achieved = evals * COUNTER_FLOPS_PER_EVAL / (sweep_ms * 1e-3) / 1e12
    # algorithmic HBM bytes of the sweep: 192-byte panel records of both panels and
    # the per-pair outputs (two double4, J and the convergence level)
    traffic_bytes = N_DISJOINT * (2 * 32 + 24 + 1) + 2 * tri.shape[0] * 192
    Ks = {i2.TYPE_NAMES[t]: fast.refinementIterations(t) for t in range(3)}

    out = {
        "metric": "FP64 pair-integrals/s (<=1e-11 rel err) batched vs plain; adjoint/forward ratio",
        "value": N_PAIRS / t_fast,
        "unit": "pair-integrals/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": 1e3 * t_fast,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": "jittered ellipsoid (3, 1, 0.5), icosphere-4: 5,120 triangles, 26,209,280 ordered pairs, "
                               "13-point rule, automatic refinement up to 3 levels at tol 1e-8",
                   "path": "batched persistent kernels in one HIP graph",
                   "pairs_per_workgroup": args.pairs_per_workgroup, "points_per_lane": args.points_per_lane,
                   "refinement_iterations": Ks},
        "plain_value": N_PAIRS / t_plain,
        "plain_ms_per_step": 1e3 * t_plain,
        "batched_over_plain": t_plain / t_fast,
        "roofline": {"bound": "valu", "achieved": achieved, "peak": FP64_PEAK_TFLOPS,
                     "unit": "TFLOP/s", "frac": achieved / FP64_PEAK_TFLOPS, "traffic": SWEEP_HBM_BYTES,
                     "kernel": "k_sweep_disjoint (levels 0 and 1 of all disjoint pairs)", "kernel_ms": sweep_ms,
                     "points": points, "evaluations": evals, "flops_per_evaluation": COUNTER_FLOPS_PER_EVAL,
                     "flops_source": "rocprofv3 SQ_INSTS_VALU_{FMA,MUL,ADD}_F64 (FMA = 2) x 64 lanes per "
                                     "evaluation; profiles/valu_counters_sweep_icosphere4.md",
                     "valu_instructions_per_evaluation": COUNTER_VALU_PER_EVAL,
                     "valu_issue_frac": VALU_ISSUE,
                     "traffic_source": "rocprofv3 --pmc FETCH_SIZE (x2.0) + WRITE_SIZE (x1.0), copy-calibrated; "
                                       "profiles/valu_counters_sweep_icosphere4.md",
                     "algorithmic_bytes": traffic_bytes,
                     # the reference formula's work (library transcendentals weighted by their
                     # instruction counts) over this kernel's time: not a fraction of the peak
                     "reference_equivalent_flops_per_point": flops_per_point(),
                     "reference_equivalent_tflops": points * flops_per_point() / (sweep_ms * 1e-3) / 1e12},
    }
    out["autotune"] = tune
    # the reference's (i, j)/(j, i) symmetry check (runAllPairs(true)), outside the
    # timed steps: largest delta per type and reported level of the batched run
    fast.runAllPairs(True)
    delta = {}
    for t in range(3):
        r = fast.results(t, errors=True)
        K = fast.refinementIterations(t)
        c = r["conv"].astype(np.int64)
        rl = np.where((c >= 1) & (((K - c) & 1) == 1), c - 1, c)
        delta[i2.TYPE_NAMES[t]] = {f"level {int(L)}": float(r["errors"][rl == L].max()) for L in np.unique(rl)}
    out["symmetry_delta_max"] = delta
    progress("adjoint")
    out["adjoint"] = adjoint_step(args)
    if not args.no_batch64:
        out["batch64"] = batch64_step()
    if not args.no_cpu_baseline:
        progress("CPU baseline")
        out["cpu_baseline"] = cpu_baseline(xyz, tri)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
