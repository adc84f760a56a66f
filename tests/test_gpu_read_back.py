"""Results read through the staging slots: all arrays of a type together, each
alone (other chunk lengths), and the device's own lists, around a slot's size."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SLOT = (1 << 20) // 57      # tasks per slot when all arrays but the errors are read


@pytest.mark.parametrize("n", [1, 255, SLOT, SLOT + 1, 2 * SLOT + 7])
def test_arrays_together_and_alone(gpu, n):
    xyz, tri = gpu.icosphere(2, (1.3, 1.0, 0.8), 0.05, 1)
    m = gpu.Mesh3D()
    m.setData(xyz, tri)
    m.prepareMesh()
    it = gpu.NumericalIntegrator3D(m)
    it.setErrorControl(2, 1e-6, True)
    ev = gpu.EvaluatorJ3DK(m, it)
    pairs = m.getNotNeighbors()
    lists = [np.zeros((0, 3), np.int32)] * 2 + [np.concatenate([pairs, pairs[:, [1, 0, 2]]])[:n]]
    print(f"{n} tasks", flush=True)
    ev.runPairs(*lists)
    r = ev.results(2)
    assert np.array_equal(r["tasks"][:, :2], lists[2][:, :2]) and np.array_equal(r["tasks"][:, 2], np.arange(n))
    keys = ["tasks", "integrals", "results", None, "conv"]
    for k, name in enumerate(keys):
        if name is None:
            continue
        a = np.full_like(r[name], 77)
        args = [ctypes.c_void_p(a.ctypes.data) if q == k else None for q in range(5)]
        assert gpu.lib().i2_evaluator_get_results(ev._h, ctypes.c_int(2), *args) == 0
        assert np.array_equal(a, r[name]), name
    # the same pairs by the general path: the lists decoded on the device
    ev.runAllPairs(True)
    full = ev.results(2, errors=True)
    assert len(full["tasks"]) == 2 * len(pairs) and np.array_equal(full["tasks"][:, 2], np.arange(2 * len(pairs)))
    assert np.array_equal(full["tasks"][: len(pairs), :2], pairs[:, :2])
    assert np.array_equal(full["tasks"][len(pairs):, :2], pairs[:, 1::-1])
    assert np.array_equal(full["conv"][:n], r["conv"])
    assert np.isfinite(full["errors"]).all() and full["errors"].shape == (2 * len(pairs),)
