"""Disjoint pairs by a tile's shared distances against the panels' own: tiles
of up to 64 vertices, of up to 96 and of more (panels in random order), ragged
last tiles, one or several wavefronts per workgroup."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(gpu, shape):
    if shape == "ico":
        return gpu.icosphere(2, (1.3, 1.0, 0.8), 0.05, 1)
    xyz, tri = gpu.torus(13, 15 if shape != "wide" else 33, 1.0, 0.3, 0.01, 1)
    if shape == "random":
        tri = tri[np.random.default_rng(3).permutation(len(tri))]
    return xyz, tri[:-7] if shape == "open" else tri


@pytest.mark.parametrize("shape", ["ico", "torus", "wide", "random", "open"])
@pytest.mark.parametrize("rule", [13, 3])
def test_shared_and_own_distances(gpu, shape, rule):
    xyz, tri = _mesh(gpu, shape)
    m = gpu.Mesh3D()
    m.setData(xyz, tri)
    m.prepareMesh()
    # with and without the centroid among its points
    three = (np.array([1 / 6, 1 / 6, 2 / 3, 1 / 6, 1 / 6, 2 / 3]), np.full(3, 1 / 3), 2)
    it = gpu.NumericalIntegrator3D(m) if rule == 13 else gpu.NumericalIntegrator3D(m, *three)
    it.setFixedRefinementLevel(1)
    out = []
    for P in (32, 64, 128, 256):     # 32: less than a wavefront, the panels' own distances
        ev = gpu.EvaluatorJ3DK(m, it)
        ev.setPath(1)
        ev.setTuning(P, 13)
        print(f"{shape}, {len(tri)} panels, rule {rule}, {P} pairs per workgroup", flush=True)
        ev.runAllPairs(False)
        out.append(ev.results(2)["integrals"])
    # a term t = 2 atanh(L/S) is below 8 on these meshes and carries some 8
    # roundings; the sums' weights add to K_i's area
    scale = 8 * m.getCellMeasures().max()
    assert np.isfinite(out[0]).all()
    for o in out[1:]:
        assert np.abs(o - out[0]).max() <= 16 * 2.0 ** -52 * scale
