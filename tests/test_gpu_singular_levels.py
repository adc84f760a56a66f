"""A singular pair's levels on the batched path stand apart."""
import numpy as np
import pytest

from tests.helpers import rel_err_rows

pytestmark = pytest.mark.gpu


def test_not_finite_at_level_0_only(gpu):
    """A rule with a point at the first vertex: where that is the shared one, the
    integrand is not finite there, but level 1, whose sub-panels begin at edge
    midpoints, is.  Level 1 is reported (a NaN quotient is not above the
    tolerance), by both paths where the plain path has it, within the 1e-11 of
    the parity checks."""
    xyz, tri = gpu.icosphere(1, (1.3, 1.0, 0.8), 0.04, 3)
    m = gpu.Mesh3D()
    m.setData(xyz, tri)
    m.prepareMesh()
    it = gpu.NumericalIntegrator3D(m, np.array([1.0, 0.0, 1 / 3, 1 / 3]), np.array([0.25, 0.75]), 1)
    it.setErrorControl(1, 1e-6, False)
    out = []
    for path in (0, 1):
        ev = gpu.EvaluatorJ3DK(m, it)
        ev.setPath(path)
        print(f"path {path}", flush=True)
        ev.runAllPairs(False)
        out.append(ev.results(gpu.SIMPLE_NEIGHBORS))
    plain, batched = out
    i, j = plain["tasks"][:, 0], plain["tasks"][:, 1]
    at_vertex = (tri[j] == tri[i][:, :1]).any(axis=1)
    assert 0 < at_vertex.sum() < len(i) and np.isfinite(plain["integrals"]).all()
    assert np.isfinite(batched["integrals"]).all()
    assert rel_err_rows(batched["integrals"], plain["integrals"]).max() <= 1e-11
