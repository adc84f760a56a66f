"""Refined values with a rule that refines pairs at all distances: a task's
value is its own, whichever tasks share its wavefront."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", [0, 1])
def test_weak_rule_bitwise_reproducible(gpu, path):
    """3-point rule at a tight tolerance on 1,280 panels, with K = 2, so that tasks
    report their level-2 value: many times the 8,192 disjoint tasks from which
    four share a wavefront at level 2, near and far ones in the order in which
    they were found, which changes from run to run."""
    xyz, tri = gpu.icosphere(3, (1.4, 1.0, 0.8), 0.05, 7)
    L12, W, order = gpu.quadrature_rule(3)
    m = gpu.Mesh3D()
    m.setData(xyz, tri)
    m.prepareMesh()
    it = gpu.NumericalIntegrator3D(m, L12.ravel(), W, order)
    it.setErrorControl(2, 1e-6, True)
    ev = gpu.EvaluatorJ3DK(m, it)
    ev.setPath(path)
    first = None
    for rep in range(4):
        print(f"path {path}, run {rep}", flush=True)
        ev.runAllPairs(False)
        r = ev.results(gpu.NOT_NEIGHBORS)
        if first is None:
            first = r
            deep = np.nonzero(r["conv"] >= 2)[0]
            i, j = r["tasks"][deep, 0], r["tasks"][deep, 1]
            c = xyz[tri].mean(axis=1)
            edge = np.linalg.norm(xyz[tri] - xyz[np.roll(tri, 1, axis=1)], axis=2).max(axis=1)
            d = np.linalg.norm(c[i] - c[j], axis=1) / edge[j]
            print(f"{len(deep)} tasks at level 2, {(d < 2).sum()} near, {(d > 10).sum()} distant", flush=True)
            assert len(deep) > 8192 and (d < 2).sum() > 1000 and (d > 10).sum() > 1000
        for k in first:
            assert np.array_equal(first[k], r[k]), (rep, k, int((first[k] != r[k]).sum()))
