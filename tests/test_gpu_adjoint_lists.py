"""The adjoint's list of refined disjoint pairs: pairs within it, pairs beyond
its end (more than 65,536 refined pairs), two refinement depths, against central
differences of the loss, and the same bits whatever order the list has."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level", [2, 3])
@pytest.mark.parametrize("subdivisions", [1, 2])
def test_refined_pairs_listed_and_beyond_the_list(gpu, level, subdivisions):
    xyz, tri = gpu.icosphere(subdivisions, (1.3, 1.0, 0.8), 0.04, 3)
    rng = np.random.default_rng(4)
    step = rng.normal(size=xyz.shape)

    def run(x, grad):
        m = gpu.Mesh3D()
        m.setData(x, tri)
        m.prepareMesh()
        it = gpu.NumericalIntegrator3D(m)
        it.setFixedRefinementLevel(level)
        ev = gpu.EvaluatorJ3DK(m, it)
        ev.setPath(1)
        print(f"level {level}, {len(tri)} panels", flush=True)
        ev.runAllPairs(False)
        L, g = ev.lossAndGrad(7)
        return (L, g, ev.lossAndGrad(7)) if grad else L

    L, g, (L2, g2) = run(xyz, True)
    assert L == L2 and np.array_equal(g, g2)
    # central differences with h = 2^-12 of the edge scale 0.1..0.5: the quotient's
    # truncation is h^2 f'''/6, about (h/edge)^2 = 1e-5 of the derivative at most
    # for the random direction's terms, and its rounding eps |L|/h below that
    h = 2.0 ** -12 * 0.1
    fd = (run(xyz + h * step, False) - run(xyz - h * step, False)) / (2 * h)
    scale = np.linalg.norm(g) * np.linalg.norm(step) / np.sqrt(g.size)
    assert abs(fd - (g * step).sum()) <= 1e-5 * scale
