"""The vertex gather of the adjoint on lists of unusual shape: a vertex of
sixteen panels (more than the gather's eight lanes), a panel listed twice (a
pair that shares all three vertices is no task), a vertex without panels; the
gradient against central differences of the loss, and the mesh's own lists."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _fan(twice):
    """A cone of 16 panels around its apex over a ring, with a second ring below it."""
    n = 16
    a = 2 * np.pi * np.arange(n) / n
    ring = lambda r, z: np.stack([r * np.cos(a), r * np.sin(a) * 0.8, np.full(n, z)], axis=1)
    xyz = np.concatenate([[[0.1, 0.05, 1.0]], ring(1.0, 0.3), ring(1.2, -0.6), [[5.0, 5.0, 5.0]]])
    xyz += np.random.default_rng(1).normal(scale=0.01, size=xyz.shape)
    tri = []
    for k in range(n):
        b, c = 1 + k, 1 + (k + 1) % n
        tri += [[0, b, c], [b, b + n, c], [c, b + n, c + n]]
    if twice:
        tri.append(tri[5])
    return xyz, np.array(tri, np.int32)


@pytest.mark.parametrize("path", [0, 1])
@pytest.mark.parametrize("twice", [False, True])
def test_gather(gpu, path, twice):
    xyz, tri = _fan(twice)
    step = np.random.default_rng(2).normal(size=xyz.shape)

    def run(x, grad=False):
        m = gpu.Mesh3D()
        m.setData(x, tri)
        m.prepareMesh()
        it = gpu.NumericalIntegrator3D(m)
        it.setFixedRefinementLevel(2)
        ev = gpu.EvaluatorJ3DK(m, it)
        ev.setPath(path)
        print(f"path {path}, {len(tri)} panels", flush=True)
        ev.runAllPairs(False)
        if grad:
            share = (tri[:, None, :, None] == tri[None, :, None, :]).any(axis=3).sum(axis=2)
            upper = np.triu(np.ones((len(tri), len(tri)), bool), 1)
            for t, count in ((gpu.SIMPLE_NEIGHBORS, 1), (gpu.ATTACHED_NEIGHBORS, 2), (gpu.NOT_NEIGHBORS, 0)):
                ij = np.argwhere((share == count) & upper)
                tasks = ev.results(t)["tasks"]
                assert np.array_equal(tasks[: len(ij), :2], ij) and np.array_equal(tasks[len(ij):, :2], ij[:, ::-1])
        return ev.lossAndGrad(3)

    L, g = run(xyz, True)
    assert np.isfinite(g).all() and (g[-1] == 0).all()
    # step 2^-12 * 0.1 of the edge scale 0.4: truncation (h/edge)^2, 1e-5 allowed (as for closed meshes)
    h = 2.0 ** -12 * 0.1
    fd = (run(xyz + h * step)[0] - run(xyz - h * step)[0]) / (2 * h)
    assert abs(fd - (g * step).sum()) <= 1e-5 * np.linalg.norm(g) * np.linalg.norm(step) / np.sqrt(g.size)
