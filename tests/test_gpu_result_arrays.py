"""The arrays that results() returns stand by themselves."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_each_array_owns_its_memory(gpu):
    """Keeping one output keeps no other, an array can be resized in place, and
    any true value asks for the errors."""
    xyz, tri = gpu.icosphere(1, (1.3, 1.0, 0.8), 0.04, 3)
    m = gpu.Mesh3D()
    m.setData(xyz, tri)
    m.prepareMesh()
    ev = gpu.EvaluatorJ3DK(m, gpu.NumericalIntegrator3D(m))
    ev.runAllPairs(True)
    for t in range(3):
        n = ev.taskCount(t)
        want = ev.results(t, errors=True)
        assert set(ev.results(t)) == {"tasks", "integrals", "results", "conv"}
        for errors in (1, 2, np.int64(3), "yes"):
            r = ev.results(t, errors=errors)
            assert {k: (a.shape, a.dtype) for k, a in r.items()} == {
                "tasks": ((n, 3), np.int32), "integrals": ((n, 4), np.float64), "results": ((n, 3), np.float64),
                "conv": ((n,), np.int8), "errors": ((n,), np.float64)}
            for k, a in r.items():
                assert np.array_equal(a, want[k]) and a.flags.owndata
                a.resize((1,) + a.shape[1:], refcheck=False)
