"""The kernels' two forms of the inner integral: the far one (points at least
twice the panel's longest edge away) and the general one next to an edge, on
the host against 40-digit arithmetic; and a rule with points outside the
triangle, whose reach decides between them on the device."""
import ctypes

import numpy as np
import pytest

from tests.helpers import parity_gate

EPS = 2.0 ** -53
SHAPES = {"equilateral": [(0, 0), (1, 0), (0.5, 0.75 ** 0.5)], "right": [(0, 0), (1, 0), (0, 0.3)],
          "sliver": [(0, 0), (1, 0), (0.4, 1e-4)]}


def _form(i2, fast, pts, T):
    pts, T = np.ascontiguousarray(pts), np.ascontiguousarray(T)
    out = np.zeros((len(pts), 4))
    P = ctypes.c_void_p
    assert i2.lib().i2_host_theta_psi(ctypes.c_int(fast), pts.ctypes.data_as(P), ctypes.c_int64(len(pts)),
                                      T.ctypes.data_as(P), out.ctypes.data_as(P)) == 0
    return out


def _exact(p, T):
    """Line integrals t of the three edges, Psi, Theta and the scales of their
    rounding errors, in 40 digits."""
    import mpmath as mp
    mp.mp.dps = 40
    v = [mp.matrix([mp.mpf(float(c)) for c in x]) for x in T]
    q = mp.matrix([mp.mpf(float(c)) for c in p])
    dot = lambda a, b: sum(a[k] * b[k] for k in range(3))
    cross = lambda a, b: mp.matrix([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])
    d = [q - x for x in v]
    l = [mp.sqrt(dot(x, x)) for x in d]
    t, psi = [], mp.matrix([0, 0, 0])
    for k in range(3):
        m = (k + 1) % 3
        e = v[m] - v[k]
        L, S = mp.sqrt(dot(e, e)), l[k] + l[m]
        t.append(mp.log((S + L) / (S - L)))
        psi += t[-1] / L * e
    n2 = cross(v[1] - v[0], v[2] - v[0])
    x = l[0] * l[1] * l[2] + dot(d[0], d[1]) * l[2] + dot(d[1], d[2]) * l[0] + dot(d[2], d[0]) * l[1]
    y = dot(d[0], n2)
    dx = 16 * EPS * l[0] * l[1] * l[2]
    dy = 8 * EPS * l[0] * mp.sqrt(dot(n2, n2))
    return ([float(c) for c in psi], float(2 * mp.atan2(y, x)), float(sum(abs(c) for c in t)),
            float(2 * (dx + dy) / mp.sqrt(x * x + y * y)))


def _panel(shape, rng, scale=1.0):
    Q = np.linalg.qr(rng.normal(size=(3, 3)))[0]
    T = np.array(SHAPES[shape])
    return scale * (np.concatenate([T, np.zeros((3, 1))], axis=1) @ Q.T + rng.normal(size=3))


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("scale", [1e-20, 1.0, 1e20])
def test_far_form(i2, shape, scale):
    """At the limit distance and far beyond.  Per edge the form keeps t to a
    few rounding errors (8 ulp allowed), so Psi to those of sum |t|; Theta to the
    rounding of its two arguments and 8 ulp of its own."""
    rng = np.random.default_rng(5)
    T = _panel(shape, rng, scale)
    M = max(np.linalg.norm(T[k] - T[k - 1]) for k in range(3))
    u = rng.normal(size=(40, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    r = M * np.repeat([8 / 3 * (1 + 1e-6), 3.0, 30.0, 1e4], 10)
    pts = T.mean(axis=0) + r[:, None] * u
    got = _form(i2, 2, pts, T)
    for p, g in zip(pts, got):
        psi, theta, t, dth = _exact(p, T)
        assert np.abs(g[:3] - psi).max() <= 8 * 2 * EPS * t
        assert abs(g[3] - theta) <= dth + 8 * 2 * EPS * abs(theta)


@pytest.mark.parametrize("shape", ["equilateral", "right"])
@pytest.mark.parametrize("delta", [0.3, 0.05, 0.03, 1e-3, 1e-5])
def test_general_form_beside_an_edge(i2, shape, delta):
    """Points at a distance delta (in edge lengths) from each edge's interior
    and around the switch of S - L to the cross product at S/1024: t loses at
    most 2^10 ulps of S - L above the switch, and the relative rounding
    |u||v|/(delta L^2) of the cross product below it."""
    rng = np.random.default_rng(6)
    T = _panel(shape, rng)
    n = np.cross(T[1] - T[0], T[2] - T[0])
    n /= np.linalg.norm(n)
    for k in range(3):
        e = T[(k + 1) % 3] - T[k]
        L = np.linalg.norm(e)
        side = np.cross(n, e / L)
        s, a = rng.uniform(0.2, 0.8, 12), rng.uniform(0, 2 * np.pi, 12)
        pts = T[k] + s[:, None] * e + delta * L * (np.cos(a)[:, None] * side + np.sin(a)[:, None] * n)
        got = _form(i2, 1, pts, T)
        for p, g in zip(pts, got):
            psi, theta, t, dth = _exact(p, T)
            assert np.abs(g[:3] - psi).max() <= 4 * EPS * (2 ** 10 + 2 / delta + t)
            assert abs(g[3] - theta) <= dth + 8 * 2 * EPS * abs(theta)


@pytest.mark.parametrize("far", [False, True])
@pytest.mark.parametrize("shape", ["equilateral", "right"])
def test_reverse_mode_of_the_terms(i2, shape, far):
    """The gradient of a random combination of the terms in the point and the
    vertices against central differences in 40 digits (step 1e-12: exact to
    1e-24).  Every derivative is a sum of terms of at most 8 |g|/d each, d the
    distance to the panel, and loses some ten roundings (2^-44 allowed)."""
    import mpmath as mp
    mp.mp.dps = 40
    rng = np.random.default_rng(8)
    T = _panel(shape, rng)
    P = ctypes.c_void_p

    def value(x, g):
        p, v = x[:3], [x[3:6], x[6:9], x[9:12]]
        sub = lambda a, b: [a[k] - b[k] for k in range(3)]
        dot = lambda a, b: sum(a[k] * b[k] for k in range(3))
        cross = lambda a, b: [a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]]
        d = [sub(p, w) for w in v]
        l = [mp.sqrt(dot(w, w)) for w in d]
        out = 0
        for k in range(3):
            e = sub(v[(k + 1) % 3], v[k])
            L, S = mp.sqrt(dot(e, e)), l[k] + l[(k + 1) % 3]
            out += g[k] * mp.log((S + L) / (S - L))
        y = dot(d[0], cross(sub(v[1], v[0]), sub(v[2], v[0])))
        z = l[0] * l[1] * l[2] + dot(d[0], d[1]) * l[2] + dot(d[1], d[2]) * l[0] + dot(d[2], d[0]) * l[1]
        return out + g[3] * mp.atan2(y, z)

    for r in ((2.7, 8.0, 100.0) if far else (0.4, 1.0, 3.0)):
        u = rng.normal(size=3)
        p, g = T.mean(axis=0) + r * u / np.linalg.norm(u), rng.normal(size=4)
        f, pb, par, tri = np.zeros(4), np.zeros(3), np.zeros(9), np.ascontiguousarray(T)
        assert i2.lib().i2_host_point_adjoint(ctypes.c_int(4 if far else 3), *(a.ctypes.data_as(P) for a in (p, tri, g, f, pb, par))) == 0
        x = [mp.mpf(float(c)) for c in np.concatenate([p, T.ravel()])]
        h, ref = mp.mpf(10) ** -12, []
        for k in range(12):
            up, dn = list(x), list(x)
            up[k] += h
            dn[k] -= h
            ref.append(float((value(up, g) - value(dn, g)) / (2 * h)))
        d = min(np.linalg.norm(p - w) for w in T) if not far else r / 2
        d = min(d, min(np.linalg.norm(np.cross(p - T[k], T[k] - T[k - 1])) / np.linalg.norm(T[k] - T[k - 1]) for k in range(3))) if not far else d
        assert np.abs(np.concatenate([pb, par]) - ref).max() <= 2.0 ** -44 * 8 * np.abs(g).sum() / d


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("scale", [1e-20, 1.0, 1e20])
def test_distant_form(i2, shape, scale):
    """From six longest edges on, with the bounds of test_far_form."""
    rng = np.random.default_rng(11)
    T = _panel(shape, rng, scale)
    M = max(np.linalg.norm(T[k] - T[k - 1]) for k in range(3))
    u = rng.normal(size=(30, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    pts = T.mean(axis=0) + (M * np.repeat([20 / 3 * (1 + 1e-6), 30.0, 1e4], 10))[:, None] * u
    for p, g in zip(pts, _form(i2, 3, pts, T)):
        psi, theta, t, dth = _exact(p, T)
        assert np.abs(g[:3] - psi).max() <= 8 * 2 * EPS * t
        assert abs(g[3] - theta) <= dth + 8 * 2 * EPS * abs(theta)


@pytest.mark.parametrize("shape", ["equilateral", "right"])
def test_reverse_mode_distant_against_far(i2, shape):
    """The two polynomial forms' gradients, each within the far form's bound of
    the exact ones (test_reverse_mode_of_the_terms), from six longest edges on."""
    rng = np.random.default_rng(12)
    T = np.ascontiguousarray(_panel(shape, rng))
    P = ctypes.c_void_p
    for r in (6.7 * 1.05, 12.0, 300.0):
        u = rng.normal(size=3)
        p, g = np.ascontiguousarray(T.mean(axis=0) + r * u / np.linalg.norm(u)), rng.normal(size=4)
        out = []
        for kind in (4, 5):
            f, pb, par = np.zeros(4), np.zeros(3), np.zeros(9)
            assert i2.lib().i2_host_point_adjoint(ctypes.c_int(kind), *(a.ctypes.data_as(P) for a in (p, T, g, f, pb, par))) == 0
            out.append(np.concatenate([f, pb, par]))
        assert np.abs(out[0] - out[1]).max() <= 2 * 2.0 ** -44 * 8 * np.abs(g).sum() / (r / 2)


@pytest.mark.gpu
@pytest.mark.parametrize("path", [0, 1])
def test_rule_with_points_outside_the_triangle(gpu, oracle_mod, path):
    """The far form is only for points within its distance: a rule that reaches
    3 circumradii out of the control panel, against the oracle."""
    rule = (np.array([[2.0, -0.5], [-0.5, 2.0], [-0.5, -0.5], [1 / 3, 1 / 3]]), np.array([0.1, 0.2, 0.15, 0.55]), 3)
    xyz, tri = gpu.icosphere(2, (2.0, 1.0, 0.7), 0.05, 0)
    orc = oracle_mod.Oracle(xyz, tri)
    m = gpu.Mesh3D()
    m.setData(xyz, tri)
    m.prepareMesh()
    it = gpu.NumericalIntegrator3D(m, rule[0].ravel(), rule[1], rule[2])
    it.setFixedRefinementLevel(1)
    ev = gpu.EvaluatorJ3DK(m, it)
    ev.setPath(path)
    ev.runAllPairs(False)
    r = ev.results(gpu.NOT_NEIGHBORS)
    I4, J3, conv, K = orc.run_tasks(2, r["tasks"], rule[0].ravel(), rule[1], rule[2], mode=0, level=1)
    parity_gate(orc, gpu, 2, r["tasks"], r["integrals"], I4, np.ones(len(conv), np.int8), f"outside points path {path}",
                rule=(rule[0].ravel(), rule[1], rule[2]))
