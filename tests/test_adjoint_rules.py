"""The adjoint with each of the rules: the numbering of a refined panel's
points on the host, and loss and gradient on the device against the oracle at
fixed levels, where every pair's points are spread over sub-panels."""
import ctypes

import numpy as np
import pytest


@pytest.mark.parametrize("npts", range(1, 17))
def test_points_of_a_refined_panel(i2, npts):
    """q = npts sub + point, around every sub-panel's first and last point where
    there are few and around random ones up to level 12, exactly."""
    rng = np.random.default_rng(npts)
    last = (npts << 24) - 1
    q = np.concatenate([np.arange(min(last + 1, 1 << 16)), last - np.arange(64), rng.integers(0, last + 1, 20000),
                        npts * rng.integers(0, 1 << 24, 20000) + npts - 1, npts * rng.integers(0, 1 << 24, 20000)]).astype(np.int64)
    sub, point = np.empty_like(q), np.empty_like(q)
    P = ctypes.c_void_p
    assert i2.lib().i2_host_point_split(ctypes.c_int(npts), q.ctypes.data_as(P), ctypes.c_int64(len(q)),
                                        sub.ctypes.data_as(P), point.ctypes.data_as(P)) == 0
    assert np.array_equal(sub, q // npts) and np.array_equal(point, q % npts)


@pytest.mark.gpu
@pytest.mark.parametrize("level", [1, 2, 3])
@pytest.mark.parametrize("npts", [1, 3, 4, 6, 7, 9, 12, 13])
def test_loss_and_gradient(gpu, oracle_mod, npts, level):
    """Eighty panels, all pairs, both paths.  The loss is a sum of some 25,000
    terms of order |L|/100 at most, each within 1e-11 of the oracle's value
    (the forward pass's gate): 1e-10 of max(|L|, 1).  The derivatives within 1e-8
    and eight times the FP64 noise of the oracle's own, the adjoint's gate with
    the 13-point rule."""
    L12, W, order = gpu.quadrature_rule(npts)
    xyz, tri = gpu.icosphere(1, (1.3, 1.0, 0.8), 0.04, 3)
    orc = oracle_mod.Oracle(xyz, tri)
    rng = np.random.default_rng(npts)
    coords = [(int(rng.integers(len(xyz))), int(rng.integers(3))) for _ in range(6)]
    want = None
    for path in (0, 1):
        m = gpu.Mesh3D()
        m.setData(xyz, tri)
        m.prepareMesh()
        it = gpu.NumericalIntegrator3D(m, L12.ravel(), W, order)
        it.setFixedRefinementLevel(level)
        ev = gpu.EvaluatorJ3DK(m, it)
        ev.setPath(path)
        print(f"{npts} points, level {level}, path {path}", flush=True)
        ev.runAllPairs(False)
        tasks = [ev.results(t)["tasks"] for t in range(3)]
        L, G = ev.lossAndGrad(5)
        if want is None:
            args = [(t, tasks[t], np.full(len(tasks[t]), level, np.int8), L12.ravel(), W, order, 5) for t in range(3)]
            L_orc, ld, dual = sum(orc.loss_tasks(*a) for a in args), [], []
            for v, axis in coords:
                near = []
                for t, tk, rl, *rest in args:
                    k = (tri[tk[:, 0]] == v).any(axis=1) | (tri[tk[:, 1]] == v).any(axis=1)
                    near.append((t, tk[k], rl[k], *rest))
                ld.append(sum(orc.loss_tasks(*a, vtx=v, axis=axis, dual=True, long_double=True) for a in near))
                dual.append(sum(orc.loss_tasks(*a, vtx=v, axis=axis, dual=True) for a in near))
            want = L_orc, np.array(ld), np.array(dual)
        L_orc, ld, dual = want
        assert abs(L - L_orc) <= 1e-10 * max(abs(L_orc), 1.0), (path, L, L_orc)
        scale = np.maximum(np.abs(ld), 1e-2 * np.abs(ld).max())
        g = np.array([G[v, a] for v, a in coords])
        assert (np.abs(g - ld) / scale <= 1e-8 + 8 * np.abs(dual - ld) / scale).all(), (path, g, ld)
