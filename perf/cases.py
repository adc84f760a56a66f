"""The work this library is measured on: what a program that integrates over
the panel pairs of a surface mesh has it do, through the public classes.

Kinds of work (`case["kind"]`):

  pairs   a prepared mesh, `runAllPairs`, and the per-pair integrals, J and
          convergence iterations of all three neighbour types read back
  list    the same for lists of pairs that the caller chooses (`runPairs`)
  rows    a batch of meshes in one graph, one (sum J, sum Theta) per panel
  step    `runAllPairs` and then the loss and its gradient (`lossAndGrad`)
  graph   a batch of meshes, forward pass, loss and gradient in one graph
  shape   one iteration of a shape optimisation: new vertex coordinates into a
          mesh (`setData`, `prepareMesh`), then as `step`

Meshes are icospheres mapped to ellipsoids ("ico", `size` = subdivisions) and
tori ("torus", `size` x `size2` quads), every vertex moved along the radius by
a random part of the mean edge: closed surfaces like those of this
repository's tests and benchmark.  Several meshes of a batch take sizes from
`size` down.  Rules are the reference's triangle rules by their number of
points; `level` >= 0 fixes the refinement level, otherwise the Runge rule with
`max_level` and `tol` controls it.

`exact` computes the same integrals with torch in 64 bits from the published
formulas: the potential of an edge as log1p(2 L / (la + lb - L)) and the solid
angle from its tangent formula, quadrature of the difference to the singular
part where panels touch, the closed form of the latter, and autograd.
"""
import math

import numpy as np
import torch

import integrator2_amd as i2

SIMPLE, ATTACHED, DISJOINT = i2.SIMPLE_NEIGHBORS, i2.ATTACHED_NEIGHBORS, i2.NOT_NEIGHBORS
# the reference's defaults (largest level, Runge tolerance) and the tighter
# control of this repository's workloads
COARSE = {"max_level": 5, "tol": 1e-5, "level": -1}
FINE = {"max_level": 3, "tol": 1e-8, "level": -1}
LEVEL2 = {"max_level": 2, "tol": 1e-8, "level": -1}


def _fixed(level):
    return {"max_level": 0, "tol": 1e-8, "level": level}


def _case(name, kind, shape, size, size2=0, *, meshes=1, path=1, rule=13, control=FINE, share=1.0):
    return {"name": name, "kind": kind, "shape": shape, "size": size, "size2": size2, "meshes": meshes, "path": path,
            "rule": rule, "share": share, **control}


def listed():
    return [
        # the smallest call: an 80-triangle body with the reference's default
        # error control on the default (plain) path, everything read back
        _case("pairs_80_plain", "pairs", "ico", 1, path=0, control=COARSE),
        # the reference's driver on a mesh of a few hundred panels
        _case("pairs_320_batched", "pairs", "ico", 2),
        # a ragged mesh (390 panels, no multiple of a wavefront) with a cheaper
        # rule and a fixed level, the plain path
        _case("pairs_390_rule7_fixed", "pairs", "torus", 15, 13, path=0, rule=7, control=_fixed(1)),
        # a caller's own lists: half of all pairs of a 574-panel torus
        _case("list_574", "list", "torus", 41, 7, path=0, share=0.5),
        # the headline forward pass: 26.2 million ordered pairs of an ellipsoid
        _case("rows_5120", "rows", "ico", 4),
        # many bodies of uneven size in one launch
        _case("rows_ragged_8", "rows", "ico", 4, meshes=8),
        # a large surface, coarser control: 6.0e8 ordered pairs
        _case("rows_24576", "rows", "torus", 128, 96, control=LEVEL2),
        # sensitivities after a forward pass on either path: the size of the
        # repository's differentiation workload, and an ordinary ragged one
        _case("step_5120", "step", "ico", 4),
        _case("step_1330_plain", "step", "torus", 35, 19, path=0),
        # forward and adjoint of two bodies in one graph
        _case("graph_torus_2", "graph", "torus", 48, 32, meshes=2, control=LEVEL2),
        # a shape-optimisation iteration on a small and on an ordinary body
        _case("shape_320", "shape", "ico", 2),
        _case("shape_1280", "shape", "ico", 3),
    ]


def draw(rng):
    def between(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["pairs", "list", "rows", "rows", "step", "graph", "shape"])
    most = {"pairs": 800, "list": 800, "rows": 16000, "step": 5000, "graph": 3000, "shape": 2500}[kind]
    panels = between(72, most)
    if rng.random() < 0.25:
        shape, size, size2 = "ico", max(1, min(4, int(math.log(panels / 20.0, 4) + 0.5))), 0
        if 20 * 4 ** size > most:
            size -= 1
    else:
        shape = "torus"
        size2 = max(5, min(96, between(0.4 * math.sqrt(panels / 2), 1.1 * math.sqrt(panels / 2))))
        size = max(6, panels // (2 * size2))
    control = rng.choice([FINE, FINE, LEVEL2, COARSE, _fixed(rng.choice([0, 1, 2]))])
    return {"kind": kind, "shape": shape, "size": size, "size2": size2,
            "meshes": rng.choice([1, 2, 3, 5]) if kind in ("rows", "graph") and panels < 2000 else 1,
            "path": rng.choice([0, 1]), "rule": rng.choice([13, 13, 13, 7, 12]), "share": round(rng.uniform(0.05, 1.0), 3),
            **control}


# ---------------------------------------------------------------- meshes
def _icosphere(level):
    phi = (1.0 + math.sqrt(5.0)) / 2.0
    v = np.array([p for a in (-1.0, 1.0) for b in (-phi, phi) for p in ((0.0, a, b), (a, b, 0.0), (b, 0.0, a))])
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    d = ((v[:, None] - v[None]) ** 2).sum(2)
    near = (d < 1.001 * d[d > 1e-9].min()) & (d > 1e-9)
    tri = []
    for a in range(12):
        for b in range(a + 1, 12):
            for c in range(b + 1, 12):
                if near[a, b] and near[b, c] and near[a, c]:
                    out = np.dot(np.cross(v[b] - v[a], v[c] - v[a]), v[a] + v[b] + v[c]) > 0
                    tri.append((a, b, c) if out else (a, c, b))
    tri = np.array(tri)
    for _ in range(level):
        e = np.sort(np.stack([tri, np.roll(tri, -1, axis=1)], axis=2).reshape(-1, 2), axis=1)
        edge, at = np.unique(e, axis=0, return_inverse=True)
        mid = v[edge].sum(1)
        m = at.reshape(-1, 3) + len(v)
        v = np.concatenate([v, mid / np.linalg.norm(mid, axis=1, keepdims=True)])
        a, b, c = tri.T
        ab, bc, ca = m.T
        tri = np.stack([a, ab, ca, ab, b, bc, ca, bc, c, ab, bc, ca], axis=1).reshape(-1, 3)
    return v, tri


def _torus(n, m, minor=0.3):
    th, ph = np.meshgrid(2 * np.pi * np.arange(n) / n, 2 * np.pi * np.arange(m) / m, indexing="ij")
    r = 1.0 + minor * np.cos(ph)
    v = np.stack([r * np.cos(th), r * np.sin(th), minor * np.sin(ph)], axis=-1).reshape(-1, 3)
    a, b = np.meshgrid(np.arange(n), np.arange(m), indexing="ij")
    p00, p10 = a * m + b, (a + 1) % n * m + b
    p11, p01 = (a + 1) % n * m + (b + 1) % m, a * m + (b + 1) % m
    tri = np.stack([p00, p10, p11, p00, p11, p01], axis=-1).reshape(-1, 3)
    return v, tri


def _panels(case):
    """The number of panels of each mesh of the case."""
    if case["shape"] == "ico":
        return [20 * 4 ** max(1, case["size"] - k % 3) for k in range(case["meshes"])]
    return [2 * max(6, case["size"] - 3 * k) * max(5, case["size2"] - 2 * k) for k in range(case["meshes"])]


def _meshes(case, seed):
    """[(vertices, triangles)] of the case, made from the seed alone."""
    rng = np.random.default_rng([seed, case["size"], case["size2"]])
    found = []
    for k in range(case["meshes"]):
        if case["shape"] == "ico":
            v, tri = _icosphere(max(1, case["size"] - k % 3))
            v = v * rng.uniform(0.5, 3.0, 3)
        else:
            v, tri = _torus(max(6, case["size"] - 3 * k), max(5, case["size2"] - 2 * k))
        edge = np.linalg.norm(v[tri] - v[np.roll(tri, -1, axis=1)], axis=2).mean()
        centre = np.zeros_like(v) if case["shape"] == "ico" else _ring(v)
        out = v - centre
        out /= np.linalg.norm(out, axis=1, keepdims=True)
        v = v + 0.03 * edge * np.clip(rng.standard_normal((len(v), 1)), -3, 3) * out
        found.append((np.ascontiguousarray(v), np.ascontiguousarray(tri, np.int32)))
    return found


def _ring(v):
    """The nearest point of the unit circle in the plane z = 0."""
    r = v.copy()
    r[:, 2] = 0.0
    return r / np.linalg.norm(r, axis=1, keepdims=True)


# ---------------------------------------------------------------- the measured calls
def _mesh(v, tri):
    mesh = i2.Mesh3D(0)
    mesh.setData(v, tri)
    mesh.prepareMesh()
    return mesh


def _integrator(case, mesh):
    integ = i2.NumericalIntegrator3D(mesh, *i2.quadrature_rule(case["rule"]))
    if case["level"] >= 0:
        integ.setFixedRefinementLevel(case["level"])
    else:
        integ.setErrorControl(case["max_level"], case["tol"], True)
    return integ


def _chosen(case, seed, mesh):
    """The ordered pairs of a `list` case, by neighbour type."""
    rng = np.random.default_rng([seed, 77])
    lists = []
    for half in (mesh.getSimpleNeighbors(), mesh.getAttachedNeighbors(), mesh.getNotNeighbors()):
        both = np.concatenate([half[:, :2], half[:, 1::-1]])
        pick = np.sort(rng.choice(len(both), max(1, int(case["share"] * len(both))), replace=False))
        lists.append(np.concatenate([both[pick], np.zeros((len(pick), 1), both.dtype)], axis=1).astype(np.int32))
    return lists


def prepare(case, seed):
    kind = case["kind"]
    data = _meshes(case, seed)
    state = {"kind": kind, "weights": seed % 1000 + 1}
    meshes = [_mesh(v, t) for v, t in data]
    integ = _integrator(case, meshes[0])
    if kind in ("rows", "graph"):
        batch = i2.Batch(0)
        for mesh in meshes:
            batch.addMesh(mesh)
        batch.configure(integ, i2.BATCH_ROW_SUMS)
        if kind == "graph":
            batch.enableAdjoint(True, state["weights"])
        state.update(batch=batch, count=len(meshes))
        return state
    ev = i2.EvaluatorJ3DK(meshes[0], integ)
    ev.setPath(case["path"])
    state.update(ev=ev, mesh=meshes[0], data=data[0])
    if kind == "list":
        state["lists"] = _chosen(case, seed, meshes[0])
    return state


def _read(ev):
    """Integrals, J and convergence iterations per type, and the iterations K."""
    out = []
    for t in (SIMPLE, ATTACHED, DISJOINT):
        r = ev.results(t)
        out.append({"integrals": r["integrals"], "J": r["results"], "conv": r["conv"], "K": ev.refinementIterations(t)})
    return out


def run(state):
    kind = state["kind"]
    if kind == "pairs":
        state["ev"].runAllPairs()
        return _read(state["ev"])
    if kind == "list":
        state["ev"].runPairs(*state["lists"])
        return _read(state["ev"])
    if kind in ("rows", "graph"):
        batch = state["batch"]
        batch.run()
        out = [{"rows": batch.rowSums(m)} for m in range(state["count"])]
        if kind == "graph":
            for m, o in enumerate(out):
                o["loss"], o["grad"] = batch.lossAndGrad(m)
        return out
    if kind == "shape":
        state["mesh"].setData(*state["data"])
        state["mesh"].prepareMesh()
    state["ev"].runAllPairs()
    loss, grad = state["ev"].lossAndGrad(state["weights"])
    return {"loss": loss, "grad": grad}


# One evaluation of the integrand: three differences, squared lengths and
# distances, three edge terms, one solid angle and the weighted sums, with
# square root, logarithm, arctangent and division counted as ten operations.
FLOPS_PER_POINT = 9 + 15 + 30 + 3 * 24 + 35 + 8


def work(case):
    pairs = [n * (n - 1) for n in _panels(case)]
    if case["kind"] == "list":
        pairs = [int(case["share"] * n) for n in pairs]
    points = case["rule"] * (4 ** case["level"] if case["level"] >= 0 else 5 if case["max_level"] else 1)
    grad = case["kind"] in ("step", "graph", "shape")
    flops = sum(pairs) * points * FLOPS_PER_POINT * (2 if grad else 1)
    mesh = sum(12 * n + 12 * n for n in _panels(case))       # about half as many vertices as panels
    if case["kind"] in ("pairs", "list"):
        out = 57 * sum(pairs) + (12 * sum(pairs) if case["kind"] == "list" else 0)
    else:
        out = sum((32 * n if case["kind"] in ("rows", "graph") else 0) + (12 * n if grad else 0) for n in _panels(case))
    return {"bytes": mesh + out, "flops": flops}


# ---------------------------------------------------------------- the same in 64 bits, by torch alone
DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
CHUNK = 1 << 20


def _dot(a, b):
    return (a * b).sum(-1)


def _cross(a, b):
    return torch.linalg.cross(a, b)


def _len(a):
    return torch.sqrt(_dot(a, a))


def _unit(a):
    return a / _len(a)[..., None]


class _Geometry:
    def __init__(self, xyz, tri):
        self.v = xyz[tri]                                   # (T, 3, 3): corner, axis
        n2 = _cross(self.v[:, 1] - self.v[:, 0], self.v[:, 2] - self.v[:, 0])
        self.n2, self.n, self.area = n2, _unit(n2), 0.5 * _len(n2)
        self.tri = tri


def _theta_psi(p, A, B, C, n2):
    """(Psi, Theta) of the panels (A, B, C) at the points p."""
    a, b, c = p - A, p - B, p - C
    la, lb, lc = _len(a), _len(b), _len(c)
    psi = 0.0
    for u, v, lu, lv in ((A, B, la, lb), (B, C, lb, lc), (C, A, lc, la)):
        e = v - u
        L = _len(e)
        psi = psi + (torch.log1p(2 * L / (lu + lv - L)) / L)[..., None] * e
    theta = 2 * torch.atan2(_dot(a, n2), la * lb * lc + _dot(a, b) * lc + _dot(b, c) * la + _dot(c, a) * lb)
    return torch.cat([psi, theta[..., None]], -1)


def _sub_panels(V, level):
    """The 4^level sub-panels of the panels V (n, 3, 3), one after another."""
    if level == 0:
        yield V
        return
    a, b, c = V[:, 0], V[:, 1], V[:, 2]
    ab, bc, ca = 0.5 * (a + b), 0.5 * (b + c), 0.5 * (c + a)
    for corners in ((ab, b, bc), (bc, c, ca), (ca, a, ab), (bc, ca, ab)):
        yield from _sub_panels(torch.stack(corners, 1), level - 1)


def _corner_of(G, I, J, kind):
    """The corners of the panels I and J rotated so that the first is the
    shared vertex (vertex-sharing) or the one off the shared edge."""
    same = G.tri[I][:, :, None] == G.tri[J][:, None, :]
    si, sj = same.any(2), same.any(1)
    if kind == ATTACHED:
        si, sj = ~si, ~sj
    turn = torch.arange(3, device=I.device)
    out = []
    for P, s in ((I, si), (J, sj)):
        k = (s.to(torch.int64).argmax(1)[:, None] + turn) % 3
        out.append(torch.gather(G.v[P], 1, k[:, :, None].expand(-1, -1, 3)))
    return out


def _edge_direction(nI, nJ, ta, tb):
    """The direction e of a vertex-sharing pair and its two angles."""
    with torch.no_grad():
        flat = (_cross(nI, nJ) ** 2).sum(-1) < 1e-10
    e = torch.where(flat[:, None], tb, _unit(torch.where(flat[:, None], tb, _cross(nI, nJ))))

    def angles(e):
        return (torch.atan2(_dot(_cross(ta, e), nJ), -_dot(e, ta)), torch.atan2(_dot(_cross(e, tb), nJ), _dot(e, tb)))

    for turned in (lambda x, y: (math.pi - x.abs() < 1e-6) | (math.pi - y.abs() < 1e-6),
                   lambda x, y: (x * y < 0) & ((x - y).abs() > math.pi)):
        x, y = angles(e)
        e = torch.where(turned(x, y)[:, None], -e, e)
    return (e, *angles(e))


def _singular(G, I, J, kind):
    """The singular part as a function of the point, and its closed-form
    integral over the panels I."""
    VI, VJ = _corner_of(G, I, J, kind)
    nI, nJ, S = G.n[I], G.n[J], G.area[I]
    A, B, C = VJ[:, 0], VJ[:, 1], VJ[:, 2]
    ta, tb = _unit(A - C), _unit(B - A)
    if kind == ATTACHED:
        tc, il = _unit(C - B), 1 / _len(C - B)

        def part(p):
            va, vb = p - B, p - C
            la, lb = _len(va), _len(vb)
            l1 = torch.log((lb - _dot(tc, vb)) / (la - _dot(tc, va)))
            l2, l3 = torch.log((la + _dot(tb, va)) * il), torch.log((lb - _dot(ta, vb)) * il)
            va, vb = va / la[:, None], vb / lb[:, None]
            th = torch.atan2(_dot(_cross(va, tb), tc), _dot(tb - tc, tb + va)) - torch.atan2(
                _dot(_cross(vb, ta), tc), _dot(ta - tc, ta - vb))
            return torch.cat([l1[:, None] * tc - l2[:, None] * tb - l3[:, None] * ta, 2 * th[:, None]], -1)

        return part, _closed_edge(VI, VJ, nI, nJ, S, ta, tb, tc)
    e, dA, dB = _edge_direction(nI, nJ, ta, tb)
    inv = 1 / torch.sqrt(S)

    def part(p):
        d = p - A
        l = _len(d)
        la, lb = torch.log((l + _dot(ta, d)) * inv), torch.log((l - _dot(tb, d)) * inv)
        o = d / l[:, None]
        th = torch.atan2(_dot(_cross(o, ta), e), _dot(e - o, e - ta)) + torch.atan2(_dot(_cross(o, tb), e), _dot(e - o, e + tb))
        return torch.cat([-(la[:, None] * ta + lb[:, None] * tb), 2 * th[:, None]], -1)

    return part, _closed_vertex(VI, nI, nJ, S, ta, tb, e, dA, dB)


def _angle(a, b):
    return torch.acos((_dot(a, b) / torch.sqrt(_dot(a, a) * _dot(b, b))).clamp(-1, 1))


def _closed_edge(VI, VJ, nI, nJ, S, ta, tb, tc):
    IA, IB, IC = VI[:, 0], VI[:, 1], VI[:, 2]
    JA, JB, JC = VJ[:, 0], VJ[:, 1], VJ[:, 2]
    alpha, beta = _angle(IA - IC, IB - IC), _angle(IC - IB, IA - IB)
    gamma, delta = _angle(JC - JB, JA - JB), _angle(JB - JC, JA - JC)
    nu = math.pi - alpha - beta
    xi = torch.atan2(_dot(_cross(nI, nJ), tc), _dot(nI, nJ))
    sX, cX = torch.sin(xi), torch.cos(xi)
    sA, cA, sB, cB = torch.sin(alpha), torch.cos(alpha), torch.sin(beta), torch.cos(beta)
    sN, cN = torch.sin(alpha + beta), -torch.cos(alpha + beta)

    def q(sA, cA, sB, cB, g):
        sG, cG = torch.sin(g), torch.cos(g)
        mu, lam = -(cB * cG + cX * sB * sG), -(cA * cG - cX * sA * sG)

        def phi(cA, cG):
            return 2 * torch.atan2(sX * sA * sG, 1 - cA + cG + lam)

        phi1, phi2, iS = phi(cA, cG), phi(-cA, -cG), 1 / (sA * (1 - mu * mu))
        qT = phi1 + sG * sN * iS * ((cB * sG - cX * sB * cG) * phi2 + sX * sB * (
            0.5 * (1 + mu) * torch.log((1 + cB) / (1 - cN)) + 0.5 * (1 - mu) * torch.log((1 - cB) / (1 + cN)) +
            torch.log((1 + lam) / (1 - cG))))
        qP = 1.5 - iS * (sB * (cN + mu * lam) * torch.log(1 + lam) + sN * (cB + mu * cG) * torch.log(1 - cG) +
                         sB * (1 - mu) * (cN - lam) * torch.log(sB / sN) +
                         sN * sB * (sB * cG - cX * sG * cB) * torch.log((1 - cN) / (1 + cB)) + phi2 * sX * sG * sN * sB)
        return qT, qP

    qAT, qAP = q(sA, cA, sB, cB, gamma)
    qBT, qBP = q(sB, cB, sA, cA, delta)
    ha, hb, hn = torch.tan(0.5 * alpha), torch.tan(0.5 * beta), torch.tan(0.5 * nu)
    qab = sN * torch.log(ha * hn) / sB + sN * torch.log(hb * hn) / sA + torch.log(ha * hb)
    psi = qAP[:, None] * tb + qBP[:, None] * ta - qab[:, None] * tc
    return S[:, None] * torch.cat([psi, (qAT + qBT)[:, None]], -1)


def _closed_vertex(VI, nI, nJ, S, ta, tb, e, dA, dB):
    IA, IB, IC = VI[:, 0], VI[:, 1], VI[:, 2]
    xi = torch.atan2(_dot(_cross(nI, nJ), e), _dot(nI, nJ))
    sX, cX = torch.sin(xi), torch.cos(xi)
    s = IC - IB
    nu, mu, kappa = _angle(IA - IB, IC - IB), _angle(IB - IC, IA - IC), _angle(IB - IA, IC - IA)
    psi = torch.atan2(_dot(_cross(e, s), nI), _dot(e, s))
    sM, cM, sN, cN, sK = torch.sin(mu), torch.cos(mu), torch.sin(nu), torch.cos(nu), torch.sin(kappa)
    sP, cP = torch.sin(psi), torch.cos(psi)

    def q(d):
        sD, cD, snp, cnp, smp, cmp_ = (torch.sin(d), torch.cos(d), torch.sin(nu + psi), torch.cos(nu + psi),
                                       torch.sin(mu - psi), torch.cos(mu - psi))
        sigma, chi, eta = sD * sP * cX + cD * cP, sD * cP * cX - cD * sP, cD * sP * cX - sD * cP
        lo_t, lo_l = torch.log(1 + sD * snp * cX + cD * cnp), torch.log(1 + sD * smp * cX - cD * cmp_)
        lsn, lsm = torch.log(sN), torch.log(sM)
        L1 = lo_l - lo_t + lsn - lsm
        L2 = torch.log(torch.tan(0.5 * nu) * torch.tan(0.5 * mu))
        td = torch.tan(0.5 * d)
        hm, hn = 0.5 * (mu - psi), 0.5 * (nu + psi)
        Am = torch.atan2(td * torch.cos(hm) * sX, td * torch.cos(hm) * cX + torch.sin(hm))
        An = torch.atan2(td * torch.sin(hn) * sX, td * torch.sin(hn) * cX + torch.cos(hn))
        W = torch.atan2(sD * torch.sin(0.5 * kappa) * sX,
                        torch.cos(0.5 * kappa) + sD * torch.cos(hm - hn) * cX + cD * torch.sin(hm - hn))
        sdp, cdp = torch.sin(d - psi), torch.cos(d - psi)
        D = 1 / (sdp * sdp + sD * sP * (1 - cX) * (cdp + sigma))
        Gc = cP * (sD * sigma * cX + cD * chi - sD * sD / sP)
        qT = 2 * (An * sM * snp - Am * sN * smp - D * sM * sN * sD * (W * eta + 0.5 * sP * sX * (L1 - L2 * sigma))) / (sP * sK)
        qP = 0.5 * (3 - math.log(2.0)) + (sM * sN / sK) * ((lo_l - lo_t) * cP / sP + D * (
            L1 * sD * eta / sP + L2 * chi - 2 * W * sD * sX - Gc * (lsn - lsm))) - (
            cM * sN * (lo_l - lsm) + sM * cN * (lo_t - lsn)) / sK - 0.5 * (lsm + lsn - torch.log(sK))
        return qT, qP

    qAT, qAP = q(dA)
    qBT, qBP = q(dB)
    v = qAP[:, None] * ta + qBP[:, None] * tb
    return S[:, None] * torch.cat([v, (qAT - qBT)[:, None]], -1)


def _quadrature(G, I, J, level, L, w, part=None):
    """The quadrature at one refinement level, without the closed form."""
    VJ, n2 = G.v[J], G.n2[J]
    total = 0.0
    for sub in _sub_panels(G.v[I], level):
        for l, wk in zip(L, w):
            p = l[0] * sub[:, 0] + l[1] * sub[:, 1] + l[2] * sub[:, 2]
            f = _theta_psi(p, VJ[:, 0], VJ[:, 1], VJ[:, 2], n2)
            if part is not None:
                f = f - part(p)
            total = total + wk * f
    return (G.area[I] / 4.0 ** level)[:, None] * total


def _criterion(cur, prev, power):
    num, den = cur - prev, power * prev - cur
    eps = torch.tensor([2e-6, 2e-6, 2e-6, 1e-10], dtype=cur.dtype, device=cur.device)
    return torch.where((num.abs() < eps) & (den.abs() < eps), torch.zeros_like(num), num / den).abs().sum(-1)


def _tasks(tri):
    """Ordered (I, J) of each neighbour type, in the order of the library."""
    T = len(tri)
    shared = np.zeros((T, T), np.int8)
    for k in range(3):
        for l in range(3):
            shared += tri[:, k][:, None] == tri[:, l][None]
    upper = np.triu(np.ones((T, T), bool), 1)
    out = []
    for count in (1, 2, 0):
        a, b = np.nonzero(upper & (shared == count))
        out.append((np.concatenate([a, b]), np.concatenate([b, a])))
    return out


def _levels(G, I, J, kind, case, L, w, order):
    """Values, convergence iterations and K of the tasks of one type."""
    n = len(I)
    value = torch.zeros(n, 4, dtype=torch.float64, device=DEVICE)
    other = value.clone()
    conv = torch.zeros(n, dtype=torch.int64, device=DEVICE)
    closed = torch.zeros_like(value)
    for at in range(0, n, CHUNK):
        s = slice(at, min(n, at + CHUNK))
        i, j = I[s], J[s]
        part = None
        if kind != DISJOINT:
            part, closed[s] = _singular(G, i, j, kind)
        if case["level"] >= 0:
            value[s] = _quadrature(G, i, j, case["level"], L, w, part)
            conv[s] = case["level"]
            continue
        value[s] = _quadrature(G, i, j, 0, L, w, part)
        rest = torch.arange(s.start, s.stop, device=DEVICE)
        for level in range(1, case["max_level"] + 1):
            if not len(rest):
                break
            part = _singular(G, I[rest], J[rest], kind)[0] if kind != DISJOINT else None
            new = _quadrature(G, I[rest], J[rest], level, L, w, part)
            other[rest], value[rest] = value[rest], new
            conv[rest] = level
            rest = rest[_criterion(new, other[rest], 2.0 ** order) > case["tol"]]
    K = case["level"] if case["level"] >= 0 else int(conv.max()) if n else 0
    swap = (conv >= 1) & ((K - conv) % 2 == 1)
    if case["level"] >= 0:
        swap[:] = False
    return torch.where(swap[:, None], other, value) + closed, conv, K, torch.where(swap, conv - 1, conv)


def _result(G, I, J, kind, v):
    theta = v[:, 3]
    if kind == SIMPLE:
        ref = 2 * math.pi * G.area[I]
        with torch.no_grad():
            turns = torch.where(theta > ref, -(torch.trunc((theta - ref) / (2 * ref)) + 1), torch.where(
                theta < -ref, torch.trunc((-ref - theta) / (2 * ref)) + 1, torch.zeros_like(theta)))
        theta = theta + 2 * turns * ref
    return (theta[:, None] * G.n[J] + _cross(v[:, :3], G.n[J])) / (4 * math.pi)


def _mix(z):
    z = z + np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _weights(seed, I, J, T):
    """The normal weights (w, v) of the loss: splitmix64 of (seed, pair, stream) and Box-Muller."""
    pid = I.astype(np.uint64) * np.uint64(T) + J.astype(np.uint64)
    out = []
    with np.errstate(over="ignore"):
        for stream in range(4):
            base = _mix(np.uint64(seed) ^ _mix(pid * np.uint64(4) + np.uint64(stream)))
            u, v = (((_mix(base ^ np.uint64(k)) >> np.uint64(11)).astype(np.float64) + 0.5) * 2.0 ** -53 for k in (1, 2))
            out.append(np.sqrt(-2 * np.log(u)) * np.cos(2 * np.pi * v))
    return torch.from_numpy(np.stack(out, 1)).to(DEVICE)


def _loss_and_grad(xyz, tri, tasks, reported, seed, L, w):
    x = xyz.clone().requires_grad_(True)
    total = 0.0
    for kind, ((i, j), levels) in enumerate(zip(tasks, reported)):
        for level in torch.unique(levels).tolist():
            which = torch.nonzero(levels == level)[:, 0]
            step = max(512, int(3e6) // (len(w) * 4 ** level))
            for at in range(0, len(which), step):
                pick = which[at:at + step].cpu().numpy()
                G = _Geometry(x, tri)
                I, J = (torch.from_numpy(t[pick]).to(DEVICE) for t in (i, j))
                part, v = _singular(G, I, J, kind) if kind != DISJOINT else (None, 0.0)
                v = v + _quadrature(G, I, J, level, L, w, part)
                W = _weights(seed, i[pick], j[pick], len(tri))
                loss = (W[:, 0] * v[:, 3]).sum() + (W[:, 1:] * _result(G, I, J, kind, v)).sum()
                loss.backward()
                total += float(loss.detach())
    return total, x.grad.cpu().numpy()


def exact(case, seed):
    kind, grad = case["kind"], case["kind"] in ("step", "graph", "shape")
    panels = _panels(case)
    points = case["rule"] * (4 ** case["level"] if case["level"] >= 0 else 5)
    # what stays under about 20 seconds on the GPU, forward and with autograd
    if sum(n * n for n in panels) * points > (1.3e8 if grad else 1.8e9) or max(panels) > 6000:
        return None
    bary, weight, order = i2.quadrature_rule(case["rule"])
    L = [(float(a), float(b), 1.0 - float(a) - float(b)) for a, b in bary]
    w = [float(x) for x in weight]
    seeds, out = seed % 1000 + 1, []
    for v, t in _meshes(case, seed):
        xyz, tri = torch.from_numpy(v).to(DEVICE), torch.from_numpy(t.astype(np.int64)).to(DEVICE)
        G = _Geometry(xyz, tri)
        tasks = _tasks(t)
        if kind == "list":
            tasks = _subset(case, seed, tasks)
        rows = torch.zeros(len(t), 4, dtype=torch.float64, device=DEVICE)
        types, reported = [], []
        for q, (i, j) in enumerate(tasks):
            I, J = torch.from_numpy(i).to(DEVICE), torch.from_numpy(j).to(DEVICE)
            val, conv, K, rep = _levels(G, I, J, q, case, L, w, order)
            res = _result(G, I, J, q, val)
            reported.append(rep)
            types.append({"integrals": val, "J": res, "conv": conv.to(torch.int8), "K": K})
            rows.index_add_(0, I, torch.cat([res, val[:, 3:]], -1))
        if kind in ("pairs", "list"):
            return types
        one = {"rows": rows}
        if grad:
            one["loss"], one["grad"] = _loss_and_grad(xyz, tri, tasks, reported, seeds, L, w)
        out.append(one)
    return out if kind in ("rows", "graph") else {"loss": out[0]["loss"], "grad": out[0]["grad"]}


def _subset(case, seed, tasks):
    """The pairs _chosen takes, from the same draws."""
    rng = np.random.default_rng([seed, 77])
    out = []
    for i, j in tasks:
        pick = np.sort(rng.choice(len(i), max(1, int(case["share"] * len(i))), replace=False))
        out.append((i[pick], j[pick]))
    return out
