"""Refinement of disjoint pairs with two and with three wavefronts per SIMD: a
small mesh alone, and in a batch whose pairs are many enough for the other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level", [2, 3])
@pytest.mark.parametrize("rule", [13, 3])
def test_row_sums_alone_and_beside_a_large_mesh(gpu, level, rule):
    meshes = []
    for shape in (gpu.torus(6, 5, 1.0, 0.3, 0.01, 1), gpu.icosphere(2, (1.3, 1.0, 0.8), 0.05, 1), gpu.icosphere(3, (1.0, 1.0, 1.0), 0.05, 2)):
        m = gpu.Mesh3D()
        m.setData(*shape)
        m.prepareMesh()
        meshes.append(m)
    three = (np.array([1 / 6, 1 / 6, 2 / 3, 1 / 6, 1 / 6, 2 / 3]), np.full(3, 1 / 3), 2)
    it = gpu.NumericalIntegrator3D(meshes[0]) if rule == 13 else gpu.NumericalIntegrator3D(meshes[0], *three)
    it.setFixedRefinementLevel(level)
    sums = []
    for group in (meshes[:2], meshes):
        b = gpu.Batch()
        for m in group:
            b.addMesh(m)
        b.configure(it, gpu.BATCH_ROW_SUMS)
        print(f"{len(group)} meshes, level {level}, rule {rule}", flush=True)
        b.run()
        sums.append([b.rowSums(k) for k in range(2)])
    for k in range(2):
        # a pair's terms are below 8 with weights that add to K_i's area; a lane's
        # sum, the butterfly and the row's additions are some 64 roundings
        bound = 64 * 2.0 ** -52 * 8 * len(sums[0][k]) * meshes[k].getCellMeasures().max()
        assert np.isfinite(sums[0][k]).all()
        assert np.abs(sums[1][k] - sums[0][k]).max() <= bound
