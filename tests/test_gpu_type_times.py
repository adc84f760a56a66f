"""The plain path's times by type: closed forms count with their own type."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_closed_forms_count_with_their_type(gpu):
    """Half a million vertex-sharing tasks at one point each, whose closed forms
    are most of the run, and one disjoint task, which has none: its time is that
    of two launches of one workgroup, well under half of the others'."""
    xyz, tri = gpu.icosphere(1, (1.3, 1.0, 0.8), 0.04, 3)
    m = gpu.Mesh3D()
    m.setData(xyz, tri)
    m.prepareMesh()
    L12, W, order = gpu.quadrature_rule(1)
    it = gpu.NumericalIntegrator3D(m, L12.ravel(), W, order)
    it.setFixedRefinementLevel(0)
    ev = gpu.EvaluatorJ3DK(m, it)
    simple = np.tile(m.getSimpleNeighbors(), (2000, 1))
    for rep in range(2):
        ev.runPairs(simple, np.zeros((0, 3), np.int32), m.getNotNeighbors()[:1])
        ms = [ev.typeStats(t)[0] for t in range(3)]
        print(len(simple), ms, flush=True)
    assert ms[1] == 0.0 and 0.0 < ms[2] < 0.5 * ms[0]
