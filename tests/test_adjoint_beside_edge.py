"""Reverse mode of the inner integral's terms, the form the adjoint kernels run,
beside an edge of the panel, where S - L comes from the cross product."""
import ctypes

import numpy as np
import pytest

EPS = 2.0 ** -53


def _value(mp, x, g):
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


@pytest.mark.parametrize("delta", [0.1, 0.05, 0.03, 1e-2, 1e-3, 1e-5])
def test_reverse_mode_beside_an_edge(i2, delta):
    """Against central differences in 40 digits (step 1e-14: exact to 1e-18 of
    a derivative's scale).  A derivative is a sum of terms of at most 8 |g|/d, d =
    delta L the distance to the edge, each with the relative rounding of S - L: at
    most 2^10 ulps where it is a difference, |u||v|/(delta L^2) <= 2/delta of them
    where it is the cross product, and the adjoint's few others."""
    import mpmath as mp
    mp.mp.dps = 40
    rng = np.random.default_rng(13)
    P = ctypes.c_void_p
    T = np.ascontiguousarray(rng.normal(size=3) + np.array([[0.0, 0, 0], [1, 0, 0], [0.4, 0.8, 0]]) @ np.linalg.qr(rng.normal(size=(3, 3)))[0])
    n = np.cross(T[1] - T[0], T[2] - T[0])
    n /= np.linalg.norm(n)
    for k in range(3):
        e = T[(k + 1) % 3] - T[k]
        L = np.linalg.norm(e)
        a = rng.uniform(0, 2 * np.pi)
        p = np.ascontiguousarray(T[k] + rng.uniform(0.2, 0.8) * e + delta * L * (np.cos(a) * np.cross(n, e / L) + np.sin(a) * n))
        g = rng.normal(size=4)
        f, pb, par = np.zeros(4), np.zeros(3), np.zeros(9)
        assert i2.lib().i2_host_point_adjoint(ctypes.c_int(3), *(q.ctypes.data_as(P) for q in (p, T, g, f, pb, par))) == 0
        x = [mp.mpf(float(c)) for c in np.concatenate([p, T.ravel()])]
        h, ref = mp.mpf(10) ** -14, []
        for q in range(12):
            up, dn = list(x), list(x)
            up[q] += h
            dn[q] -= h
            ref.append(float((_value(mp, up, g) - _value(mp, dn, g)) / (2 * h)))
        bound = 8 * np.abs(g).sum() / (delta * L) * 4 * EPS * (2 ** 10 + 2 / delta)
        assert np.abs(np.concatenate([pb, par]) - ref).max() <= bound
