"""Far pairs depend on differences of coordinates only."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", [0, 1])
@pytest.mark.parametrize("level", [0, 1, 2, None])
def test_translated_mesh_same_bits(gpu, path, level):
    """Two spheres of 320 panels ten radii apart, as they are and 2,400 radii off.
    The coordinates are multiples of 2^-20, so that the translation is exact and
    every difference of coordinates the same number: the pairs of the one sphere
    with the other, all in the far forms (tiles of 64 panels lie in one
    sphere), give the same bits.  A panel's centroid rounded at the distance of the
    origin would shift its points by some 1e-13."""
    x, t = gpu.icosphere(2, (1.0, 1.0, 1.0), 0.05, 1)
    x = np.round(np.concatenate([x, x + [10.0, 0.0, 0.0]]) * 2 ** 20) / 2 ** 20
    tri = np.concatenate([t, t + len(x) // 2]).astype(np.int32)
    n = len(t)
    out = []
    for shift in ([0.0, 0.0, 0.0], [1024.0, -2048.0, 512.0]):
        m = gpu.Mesh3D()
        m.setData(x + np.array(shift), tri)
        m.prepareMesh()
        it = gpu.NumericalIntegrator3D(m)
        if level is None:
            it.setErrorControl(2, 1e-9, False)
        else:
            it.setFixedRefinementLevel(level)
        ev = gpu.EvaluatorJ3DK(m, it)
        ev.setPath(path)
        print(f"path {path}, level {level}, shift {shift}", flush=True)
        if path == 0:
            pairs = m.getNotNeighbors()
            pairs = pairs[(pairs[:, 0] < n) & (pairs[:, 1] >= n)]
            ev.runPairs(pairs[:0], pairs[:0], np.concatenate([pairs, pairs[:, [1, 0, 2]]]))
        else:
            ev.runAllPairs(False)
        r = ev.results(gpu.NOT_NEIGHBORS)
        cross = (r["tasks"][:, 0] < n) != (r["tasks"][:, 1] < n)
        assert cross.sum() == 2 * n * n
        out.append({k: r[k][cross] for k in ("tasks", "integrals", "results", "conv")})
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), (k, np.abs(out[0][k] - out[1][k]).max())
