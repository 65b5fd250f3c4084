"""The framework's work as its users have it done, in sizes from the smallest to the largest.

A case is one call, or the short sequence of calls that a program makes as one step:

``rhs``       the plane-wave right-hand side of one excitation
``matrix``    a dense matrix on the host, ``assemble(op, X, Y)``
``solve``     right-hand sides, resident matrix, factorisation and solve of one problem
``batch``     the same for several problems in shared launches, as the solve service runs them
``resident``  further right-hand sides on factors that stay on the GPU
``farfield``  ``potential`` of a current for a set of directions

Shapes, sizes, wavenumbers and tolerances are those of the benchmark, the serving workloads and
the tests: spheres, 2 x 1 x 1 ellipsoids and cubes, wavenumbers from 0.5 to 8.
"""
import math

import numpy as np
import torch

import __graft_entry__

bj = __graft_entry__.load_package()


def listed():
    return [
        # the excitation of a small sphere: the smallest call there is
        dict(name="rhs 702", kind="rhs", op="efie", shape="sphere", dofs=702, k=2.0),
        # a first look at a coarse mesh: the whole matrix to the host
        dict(name="matrix efie 318", kind="matrix", op="efie", shape="sphere", dofs=318, k=2.0, loss=0.0, other="",
             other_dofs=0, precision="fp64"),
        # coupling of two bodies in a lossy medium, single precision, uneven sizes
        dict(name="matrix mfie 1515x2400", kind="matrix", op="mfie_k", shape="ellipsoid", dofs=1515, k=3.0, loss=0.3,
             other="sphere", other_dofs=2400, precision="fp32"),
        # a small problem in plain double precision
        dict(name="solve fp64 702", kind="solve", op="efie", shape="sphere", dofs=702, k=2.0, precision="fp64", nrhs=1),
        # a jittered sphere at k = 2 pi in plain double precision
        dict(name="solve fp64 17406", kind="solve", op="efie", shape="sphere", dofs=17406, k=2 * math.pi,
             precision="fp64", nrhs=1),
        # a cube with single-precision products and two excitations
        dict(name="solve fp32 4050", kind="solve", op="efie", shape="cube", dofs=4050, k=4.0, precision="fp32", nrhs=2),
        # the RT-tested MFIE, mixed precision, four excitations
        dict(name="solve mfie 9003", kind="solve", op="mfie", shape="ellipsoid", dofs=9003, k=3.0,
             precision="fp32split", nrhs=4),
        # the benchmark's problem: 26,664 triangles, mixed precision
        dict(name="solve efie 39996", kind="solve", op="efie", shape="sphere", dofs=39996, k=4.0,
             precision="fp32split", nrhs=1),
        # one batch of the solve service: 16 problems of 500 to 8000 unknowns
        dict(name="batch 16", kind="batch", count=16, mix=4),
        # the service's repeat customers: new excitations on factors that are there
        dict(name="resident 12000", kind="resident", op="efie", shape="sphere", dofs=12000, k=4.0,
             precision="fp32split", nrhs=4),
        # the full pattern of the benchmark's current, every degree
        dict(name="farfield 181x361", kind="farfield", op="single", shape="sphere", dofs=39996, k=4.0, loss=0.0,
             theta=181, phi=361),
        # a coarse pattern of magnetic currents in a lossy medium
        dict(name="farfield lossy 37x73", kind="farfield", op="double", shape="ellipsoid", dofs=3003, k=5.0, loss=0.2,
             theta=37, phi=73),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["rhs", "matrix", "matrix", "solve", "solve", "solve", "batch", "resident", "farfield", "farfield"])
    c = dict(kind=kind, shape=rng.choice(["sphere", "ellipsoid", "cube"]), k=round(rng.uniform(0.5, 8.0), 3))
    if kind == "rhs":
        return dict(c, op=rng.choice(["efie", "mfie"]), dofs=size(300, 40000))
    if kind == "matrix":
        other = rng.choice(["", "", "sphere", "ellipsoid", "cube"])
        return dict(c, op=rng.choice(["efie", "efie", "mfie_k", "nxk"]), dofs=size(300, 4000), loss=rng.choice([0.0, 0.0, 0.25]),
                    other=other, other_dofs=size(300, 4000) if other else 0, precision=rng.choice(["fp64", "fp64", "fp32"]))
    if kind == "solve":
        p = rng.choice(["fp64", "fp32", "fp32split", "fp32split"])
        return dict(c, op=rng.choice(["efie", "mfie"]), dofs=size(500, 12000 if p == "fp64" else 24000), precision=p,
                    nrhs=rng.randint(1, 4))
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(3, 16), mix=rng.randint(10, 9999))
    if kind == "resident":
        return dict(c, op=rng.choice(["efie", "mfie"]), dofs=size(500, 20000), precision=rng.choice(["fp64", "fp32", "fp32split"]),
                    nrhs=rng.randint(1, 4))
    return dict(c, op=rng.choice(["single", "double", "rotated"]), dofs=size(500, 24000), loss=rng.choice([0.0, 0.0, 0.25]),
                theta=size(5, 91), phi=size(9, 181))


# ------------------------------------------------------------------ what a program has in hand

TOL = 1e-12   # relative residual of the mixed-precision solves


def _mesh(shape, dofs, seed):
    """About ``dofs`` edges: spheres and ellipsoids have 3 (nv - 2) of them, cubes 18 n^2."""
    if shape == "cube":
        return bj.meshcube(max(1, int(round(math.sqrt(dofs / 18.0)))))
    nv = max(8, int(round(dofs / 3.0 + 2)))
    if shape == "ellipsoid":
        return bj.meshellipsoid(2.0, 1.0, 1.0, nv=nv, jitter=0.02, seed=seed)
    return bj.meshsphere(1.0, nv=nv, jitter=0.02, seed=seed)


def _dofs(shape, dofs):
    return 18 * max(1, int(round(math.sqrt(dofs / 18.0)))) ** 2 if shape == "cube" else 3 * (max(8, int(round(dofs / 3.0 + 2))) - 2)


def _waves(rng, count):
    """Directions and polarisations of ``count`` plane waves."""
    d = rng.normal(size=(count, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    p = np.cross(d, rng.normal(size=(count, 3)))
    return d, p / np.linalg.norm(p, axis=1, keepdims=True)


def _operator(op, gamma):
    if op == "efie":
        return bj.Maxwell3D.singlelayer(gamma=gamma)
    if op == "mfie_k":
        return bj.Maxwell3D.doublelayer(gamma=gamma)
    if op == "nxk":
        return bj.cross(bj.n, bj.Maxwell3D.doublelayer(gamma=gamma))
    return bj.cross(bj.n, bj.Maxwell3D.doublelayer(gamma=gamma)) - 0.5 * bj.Identity()


def _excitation(op, k, d, p):
    """(n x E) x n for the EFIE, n x H with H = -1/(i k) curl E for the MFIE."""
    E = bj.Maxwell3D.planewave(direction=d, polarization=p, wavenumber=k)
    if op == "efie":
        return bj.cross(bj.cross(bj.n, E), bj.n)
    return bj.cross(bj.n, (-1.0 / (1j * k)) * bj.curl(E))


def _problem(op, shape, dofs, k, nrhs, rng):
    k *= 1.0 + 0.02 * rng.uniform(-1, 1)
    mesh = _mesh(shape, dofs, int(rng.integers(1 << 30)))
    d, p = _waves(rng, nrhs)
    return dict(op=op, k=k, mesh=mesh, X=bj.raviartthomas(mesh), d=d, p=p, operator=_operator(op, 1j * k),
                excitations=[_excitation(op, k, *w) for w in zip(d, p)])


def _batch(case, rng):
    """Problems as the batched service gets them: up to 16, at most 6.4e8 summed unknowns squared."""
    mix, out, work = np.random.default_rng(case["mix"]), [], 0.0
    for _ in range(case["count"]):
        shape = ["sphere", "ellipsoid", "cube"][mix.integers(3)]
        dofs = int(round(math.exp(mix.uniform(math.log(500), math.log(8000)))))
        k, nrhs = float(mix.uniform(0.5, 8.0)), int(mix.integers(1, 5))
        work += float(_dofs(shape, dofs)) ** 2
        if out and work > 6.4e8:
            break
        out.append(("efie", shape, dofs, k, nrhs) if rng is None else _problem("efie", shape, dofs, k, nrhs, rng))
    return out


def _directions(nth, nph):
    th, ph = np.meshgrid(np.linspace(0, np.pi, nth), np.linspace(0, 2 * np.pi, nph), indexing="ij")
    return np.stack([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th)], -1)


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "batch":
        return dict(kind=kind, problems=_batch(case, rng))
    if kind in ("rhs", "solve", "resident"):
        s = _problem(case["op"], case["shape"], case["dofs"], case["k"], case.get("nrhs", 1), rng)
        return dict(s, kind=kind, precision=case.get("precision"))
    k = case["k"] * (1.0 + 0.02 * rng.uniform(-1, 1))
    gamma = 1j * k + case["loss"]
    X = bj.raviartthomas(_mesh(case["shape"], case["dofs"], int(rng.integers(1 << 30))))
    if kind == "matrix":
        Y = X
        if case["other"]:   # a second body beside the first
            m = _mesh(case["other"], case["other_dofs"], int(rng.integers(1 << 30)))
            Y = bj.raviartthomas(bj.Mesh(m.vertices + np.array([0.4, 3.0, -0.3]), m.cells))
        return dict(kind=kind, op=case["op"], gamma=gamma, operator=_operator(case["op"], gamma), X=X, Y=Y,
                    precision=case["precision"])
    N = X.numfunctions()
    op = {"single": bj.MWFarField3D, "double": bj.MWDoubleLayerFarField3D, "rotated": bj.MWDoubleLayerRotatedFarField3D}
    return dict(kind=kind, op=case["op"], gamma=gamma, operator=op[case["op"]](gamma=gamma), X=X,
                points=_directions(case["theta"], case["phi"]), coeffs=rng.normal(size=N) + 1j * rng.normal(size=N))


def _rhs(s):
    return np.stack([bj.assemble(e, s["X"]) for e in s["excitations"]], axis=1)


def prepare(case, seed):
    s = _inputs(case, seed)
    if s["kind"] == "resident":
        s["M"] = bj.DeviceMatrix.assemble(s["operator"], s["X"]).factor(s["precision"])
        s["B"] = _rhs(s)
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    kind = s["kind"]
    if kind == "rhs":
        return bj.assemble(s["excitations"][0], s["X"])
    if kind == "matrix":
        return bj.assemble(s["operator"], s["X"], s["Y"], precision=s["precision"])
    if kind == "farfield":
        return bj.potential(s["operator"], s["points"], s["coeffs"], s["X"])
    if kind == "resident":
        return s["M"].solve(s["B"], tol=TOL, maxit=10)
    if kind == "solve":
        B = _rhs(s)
        M = bj.DeviceMatrix.assemble(s["operator"], s["X"]).factor(s["precision"])
        return {"b": B, "x": M.solve(B, tol=TOL, maxit=10)}
    mats = bj.DeviceMatrix.assemble_batch([(p["operator"], p["X"]) for p in s["problems"]])
    bj.DeviceMatrix.factor_batch(mats)
    return [M.solve(_rhs(p), tol=TOL, maxit=10) for M, p in zip(mats, s["problems"])]


# ------------------------------------------------------------------ work

def _solve_work(op, n, nrhs, precision):
    """Kernel evaluations of the far rule (170 operations each for the single layer, 210 for the double
    layer), the factorisation, and two passes over the factors; the matrix is written once and read once."""
    pairs = (2.0 * n / 3.0) ** 2
    flops = pairs * (12 * 170 if op == "efie" else 156 * 210) + 8.0 * n ** 3 / 3 + nrhs * 16.0 * n * n
    return {"bytes": 2 * (16.0 if precision == "fp64" else 8.0) * n * n + 32.0 * n * nrhs, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind == "batch":
        w = [_solve_work(op, _dofs(shape, dofs), nrhs, "fp32split") for op, shape, dofs, k, nrhs in _batch(case, None)]
        return {q: sum(x[q] for x in w) for q in ("bytes", "flops")}
    n = _dofs(case["shape"], case["dofs"])
    cells = 2 * n // 3
    if kind == "rhs":
        return {"bytes": 16.0 * n + 120.0 * cells, "flops": 2.0 * n * 16 * 40}
    if kind == "matrix":
        m = _dofs(case["other"], case["other_dofs"]) if case["other"] else n
        per = {"efie": 12 * 170, "mfie_k": 12 * 210, "nxk": 156 * 210}[case["op"]]
        return {"bytes": (16.0 if case["precision"] == "fp64" else 8.0) * n * m, "flops": float(cells) * (2 * m // 3) * per}
    if kind == "solve":
        return _solve_work(case["op"], n, case["nrhs"], case["precision"])
    if kind == "resident":   # the factors once and, to refine, the matrix once
        size = 16.0 if case["precision"] == "fp64" else 24.0
        return {"bytes": size * n * n + 32.0 * n * case["nrhs"], "flops": case["nrhs"] * 8.0 * n * n * (1 if size == 16.0 else 2)}
    dirs = float(case["theta"] * case["phi"])   # per direction and cell: a phase, and the cell's three moments in it
    return {"bytes": 48.0 * dirs + 24.0 * dirs + 16.0 * n + 96.0 * cells, "flops": dirs * cells * 120.0}


# ------------------------------------------------------------------ the same in 64 bits, in plain torch

# Dunavant's rules of degree 2, 3, 6, 7, 8, 10: weight and barycentric coordinates of each orbit
_ORBITS = {
    2: [(0.333333333333333, (0.666666666666667, 0.166666666666667))],
    3: [(-0.5625, ()), (0.520833333333333, (0.6, 0.2))],
    6: [(0.116786275726379, (0.501426509658179, 0.249286745170910)), (0.050844906370207, (0.873821971016996, 0.063089014491502)),
        (0.082851075618374, (0.053145049844817, 0.310352451033784, 0.636502499121399))],
    7: [(-0.149570044467682, ()), (0.175615257433208, (0.479308067841920, 0.260345966079040)),
        (0.053347235608838, (0.869739794195568, 0.065130102902216)),
        (0.077113760890257, (0.048690315425316, 0.312865496004874, 0.638444188569810))],
    8: [(0.144315607677787, ()), (0.095091634267285, (0.081414823414554, 0.459292588292723)),
        (0.103217370534718, (0.658861384496480, 0.170569307751760)), (0.032458497623198, (0.898905543365938, 0.050547228317031)),
        (0.027230314174435, (0.008394777409958, 0.263112829634638, 0.728492392955404))],
    10: [(0.090817990382754, ()), (0.036725957756467, (0.028844733232685, 0.485577633383657)),
         (0.045321059435528, (0.781036849029926, 0.109481575485037)),
         (0.072757916845420, (0.141707219414880, 0.307939838764121, 0.550352941820999)),
         (0.028327242531057, (0.025003534762686, 0.246672560639903, 0.728323904597411)),
         (0.009421666963733, (0.009540815400299, 0.066803251012200, 0.923655933587500))],
}
_CELLS = 12000   # cells of the largest matrix that is formed and solved here
_PERM = ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0))


def _rule(degree):
    """Barycentric points [Q, 3] and weights [Q] that sum to one."""
    pts, wts = [], []
    for w, c in _ORBITS[degree]:
        if not c:
            orbit = [(1 / 3, 1 / 3, 1 / 3)]
        elif len(c) == 2:
            orbit = [tuple(c[0] if i == j else c[1] for i in range(3)) for j in range(3)]
        else:
            orbit = [tuple(c[i] for i in p) for p in _PERM]
        pts += [(a, b, 1.0 - a - b) for a, b, _ in orbit]
        wts += [w] * len(orbit)
    return torch.tensor(pts, dtype=torch.float64), torch.tensor(wts, dtype=torch.float64)


class _Cells:
    """Vertices [F, 3, 3], areas, normals and centroids of a mesh's triangles, and a space's shapes."""

    def __init__(self, X, dev):
        self.dev, self.n = dev, X.numfunctions()
        self.v = torch.as_tensor(X.geo.vertices[X.geo.cells], device=dev)
        nrm = torch.linalg.cross(self.v[:, 0] - self.v[:, 2], self.v[:, 1] - self.v[:, 2])
        self.area = 0.5 * nrm.norm(dim=1)
        self.normal = nrm / nrm.norm(dim=1, keepdim=True)
        self.slot = torch.as_tensor(3 * X.shape_cell.astype(np.int64) + X.shape_ref, device=dev)
        self.coef = torch.as_tensor(X.shape_coeff, device=dev)
        self.dof = torch.as_tensor(np.repeat(np.arange(self.n), np.diff(X.shape_ptr)), device=dev)

    def points(self, degree, cells=slice(None)):
        """Points [F, Q, 3] and weights [F, Q] of a rule."""
        b, w = (t.to(self.dev) for t in _rule(degree))
        return torch.einsum("qa,fak->fqk", b, self.v[cells]), self.area[cells, None] * w

    def gather(self, local):
        """sum over a function's shapes of coefficient times local[..., 3 cell + shape], for each function."""
        out = torch.zeros(*local.shape[:-1], self.n, dtype=local.dtype, device=self.dev)
        return out.index_add_(out.dim() - 1, self.dof, local[..., self.slot] * self.coef)


def _blocks(op, gamma, tv, sv, ta, sa, tn, x, y, w, regular=False):
    """sum over points of w K(x, y) for the 3 x 3 local shapes (x - v_i)/(2A), (y - u_j)/(2A).

    tv, sv [P, 3, 3]: vertices; x, y [P, S, 3], w [P, S]: points in pairs and their weights."""
    r = x - y
    R = r.norm(dim=-1)
    gR = gamma * R
    f = (x[:, :, None, :] - tv[:, None]) / (2 * ta)[:, None, None, None]
    g = (y[:, :, None, :] - sv[:, None]) / (2 * sa)[:, None, None, None]
    if op == "efie":
        green = torch.exp(-gR) / R if not regular else -gamma ** 3 * R ** 2 * _tail(gR, 3)
        green = green * w / (4 * math.pi)
        z = -gamma * torch.einsum("ps,psic,psjc->pij", green, f.to(green), g.to(green))
        return z - (green.sum(1) / (gamma * ta * sa))[:, None, None]
    if not regular:
        h = -(gamma + 1 / R) * torch.exp(-gR) / R ** 2
    else:   # -(gR + 1) e^-gR + 1 - (gR)^2 / 2, over R^3
        h = gamma ** 3 * (_tail(gR, 2) + gR * _tail(gR, 3))
    h = h * w / (4 * math.pi)
    c = torch.linalg.cross(r[:, :, None, :].expand_as(g), g)
    if op == "nxk":
        c = torch.linalg.cross(tn[:, None, None, :].expand_as(c), c)
    return torch.einsum("ps,psic,psjc->pij", h, f.to(h), c.to(h))


def _tail(z, n):
    """sum over m >= n of (-z)^(m - n) / m!, negated for n = 2: what is left of e^-z without its first terms."""
    out = torch.zeros_like(z)
    for m in range(n + 24, n - 1, -1):
        out = out * -z + 1.0 / math.factorial(m)
    return out if n == 3 else -out


def _far(op, gamma, T, S, cells, degrees):
    """Blocks [P, F, 3, 3] of some test cells with all trial cells, by two rules, expanded in moments about the vertices."""
    x, wx = T.points(degrees[0], cells)
    y, wy = S.points(degrees[1])
    tv, ta, tn = T.v[cells], T.area[cells], T.normal[cells]
    P, F = len(tv), len(S.v)
    z = torch.zeros(P, F, 3, 3, dtype=torch.complex128, device=T.dev)
    for q in range(x.shape[1]):
        f = (x[:, q, None, :] - tv) / (2 * ta)[:, None, None]                     # [P, 3, 3]
        s0 = torch.zeros(P, F, dtype=torch.complex128, device=T.dev)
        s1 = torch.zeros(P, F, 3, dtype=torch.complex128, device=T.dev)
        for m in range(y.shape[1]):
            r = x[:, q, None, :] - y[None, :, m, :]
            R = r.norm(dim=-1).clamp_min(1e-300)
            h = torch.exp(-gamma * R) / R * (wx[:, q, None] * wy[None, :, m] / (4 * math.pi))
            if op == "efie":
                s0 += h
                s1 += h[..., None] * y[None, :, m, :]
            else:
                h = h * -(gamma + 1 / R) / R
                s1 += h[..., None] * r
        if op == "efie":
            g = (s1[:, :, None, :] - s0[:, :, None, None] * S.v[None]) / (2 * S.area)[None, :, None, None]
            z += -gamma * torch.einsum("pic,pfjc->pfij", f.to(g), g)
            z += (-1 / gamma) * (s0 / (ta[:, None] * S.area))[:, :, None, None]
        else:   # r x (y - u) = r x (x - u), as r = x - y
            g = ((x[:, q, None, None, :] - S.v[None]) / (2 * S.area)[None, :, None, None]).to(s1)
            c = torch.linalg.cross(s1[:, :, None, :].expand_as(g), g)
            if op == "nxk":
                c = torch.linalg.cross(tn[:, None, None, :].to(c).expand_as(c), c)
            z += torch.einsum("pic,pfjc->pfij", f.to(c), c)
    return z


def _classes(T, S, cells, gamma):
    """Shared vertices of each pair, and whether it is near: closer than 0.2 wavelengths/2 pi and 0.8 root areas."""
    d = (T.v[cells][:, None, :, None, :] - S.v[None, :, None, :, :]).norm(dim=-1)   # [P, F, 3, 3]
    hits = (d < 1e3 * 2.220446049250313e-16).sum((2, 3))
    d2 = d.amin((2, 3)) ** 2
    near = torch.maximum(d2 * abs(gamma) ** 2, d2 / (16 * S.area)) < 0.2 * 0.2
    return hits, near & (hits == 0)


def _singular(op, gamma, tv, sv, hits):
    """Pairs with ``hits`` common vertices in Sauter and Schwab's coordinates (Boundary Element Methods, 5.2)."""
    n = {3: 5, 2: 4, 1: 3}[hits]
    gx, gw = np.polynomial.legendre.leggauss(n)
    grid = torch.as_tensor(np.stack(np.meshgrid(*[0.5 * (gx + 1)] * 4, indexing="ij")).reshape(4, -1), device=tv.device)
    w4 = torch.as_tensor(np.einsum("a,b,c,d->abcd", *[0.5 * gw] * 4).reshape(-1), device=tv.device)
    t, a, b, c = grid
    if hits == 3:
        j = t ** 3 * a ** 2 * b
        r = [((t, t * (1 - a + a * b)), (t * (1 - a * b * c), t * (1 - a))),
             ((t, t * a * (1 - b + b * c)), (t * (1 - a * b), t * a * (1 - b))),
             ((t * (1 - a * b * c), t * a * (1 - b * c)), (t, t * a * (1 - b)))]
        r = [(p, q, j) for p, q in r] + [(q, p, j) for p, q in r]
    elif hits == 2:
        j = t ** 3 * a ** 2
        r = [((t, t * a * c), (t * (1 - a * b), t * a * (1 - b)), j),
             ((t, t * a), (t * (1 - a * b * c), t * a * b * (1 - c)), j * b),
             ((t * (1 - a * b), t * a * (1 - b)), (t, t * a * b * c), j * b),
             ((t * (1 - a * b * c), t * a * b * (1 - c)), (t, t * a), j * b),
             ((t * (1 - a * b * c), t * a * (1 - b * c)), (t, t * a * b), j * b)]
    else:
        j = t ** 3 * b
        r = [((t, t * a), (t * b, t * b * c), j), ((t * b, t * b * c), (t, t * a), j)]
    # vertices in common first, in the test cell's order; then the others as they come
    same = (tv[:, :, None, :] - sv[:, None, :, :]).norm(dim=-1) < 1e3 * 2.220446049250313e-16
    ti = torch.argsort((~same.any(2)).to(torch.int8), dim=1, stable=True)
    rank = torch.where(same.any(1), torch.gather(torch.argsort(ti, 1), 1, same.to(torch.int8).argmax(1)), 3)
    si = torch.argsort(rank, dim=1, stable=True)
    pt, ps = (torch.gather(v, 1, i[:, :, None].expand_as(v)) for v, i in ((tv, ti), (sv, si)))

    def at(p, u):
        return p[:, None, 0] + u[0][None, :, None] * (p[:, 1] - p[:, 0])[:, None] + u[1][None, :, None] * (p[:, 2] - p[:, 1])[:, None]

    ta, sa = (0.5 * torch.linalg.cross(v[:, 0] - v[:, 2], v[:, 1] - v[:, 2]).norm(dim=1) for v in (tv, sv))
    z = 0
    for p, q, jac in r:   # each cell's map has the Jacobian 2 A
        z = z + _blocks(op, gamma, tv, sv, ta, sa, None, at(pt, p), at(ps, q), (w4 * jac)[None] * (4 * ta * sa)[:, None])
    return z


def _near(op, gamma, tv, sv):
    """Pairs that nearly touch: what is left of the kernel without its first terms by two rules, the first
    terms' integrals over the trial triangle in closed form (Wilton et al., IEEE Trans. AP 32, 1984; Graglia, 41, 1993)."""
    area = lambda v: 0.5 * torch.linalg.cross(v[:, 0] - v[:, 2], v[:, 1] - v[:, 2]).norm(dim=1)  # noqa: E731
    ta, sa = area(tv), area(sv)
    (bx, ux), (by, uy) = ((t.to(tv.device) for t in _rule(d)) for d in (6, 7))
    x = torch.einsum("qa,fak->fqk", bx, tv)
    y = torch.einsum("qa,fak->fqk", by, sv)
    X, W = len(ux), len(uy)
    P = len(tv)
    w = (ux[:, None] * uy[None, :]).reshape(-1)[None] * (ta * sa)[:, None]
    z = _blocks(op, gamma, tv, sv, ta, sa, None, x.repeat_interleave(W, 1), y.repeat(1, X, 1), w, regular=True)
    n = torch.linalg.cross(sv[:, 1] - sv[:, 0], sv[:, 2] - sv[:, 0])
    n = (n / n.norm(dim=1, keepdim=True))[:, None, :].expand(P, X, 3)
    d = ((x - sv[:, None, 0]) * n).sum(-1)
    rho = x - d[..., None] * n
    D = d.abs()
    zero = torch.zeros_like(d)
    s3, s1, s0, sp = zero.clone(), zero.clone(), zero.clone(), zero.clone()      # d/R^3, 1/R, 1, R
    v3, v1, v0, vp = (torch.zeros_like(x) for _ in range(4))                     # (y - rho) times R^-3, R^-1, 1, R
    for e in range(3):
        p, q = sv[:, e], sv[:, (e + 1) % 3]
        t = ((q - p) / (q - p).norm(dim=1, keepdim=True))[:, None, :].expand(P, X, 3)
        m = torch.linalg.cross(t, n)
        xa, xb = (((c[:, None] - rho) * t).sum(-1) for c in (p, q))
        h = ((p[:, None] - rho) * m).sum(-1)
        w2 = h * h + d * d
        ra, rb = (xa * xa + w2).sqrt(), (xb * xb + w2).sqrt()
        lg = torch.where(xa + xb > 0, torch.log((xb + rb) / (xa + ra)), torch.log((ra - xa) / (rb - xb)))
        flat = D < 1e3 * 2.220446049250313e-16
        # the angle's part, with the solid angle in it: |d| (atan(...) at b less at a)
        ang = torch.atan(h * xb / (w2 + D * rb)) - torch.atan(h * xa / (w2 + D * ra))
        s3 += torch.where(flat, zero, torch.sign(d) * ang)
        s1 += h * lg - D * ang
        s0 += 0.5 * h * (xb - xa)
        sp += h * (xb * rb - xa * ra) / 6 + (0.5 * d * d + h * h / 6) * h * lg - D ** 3 * ang / 3
        v3 -= lg[..., None] * m
        v1 += 0.5 * (xb * rb - xa * ra + w2 * lg)[..., None] * m
        v0 += (0.5 * xb * (xb * xb / 3 + h * h) - 0.5 * xa * (xa * xa / 3 + h * h))[..., None] * m
        vp += ((xb * rb ** 3 - xa * ra ** 3) / 12 + 0.125 * w2 * (xb * rb - xa * ra) + 0.125 * w2 * w2 * lg)[..., None] * m
    f = (x[:, :, None, :] - tv[:, None]) / (2 * ta)[:, None, None, None] * (ux[None, :] * ta[:, None])[..., None, None]
    if op == "efie":
        i0 = (s1 - gamma * s0 + 0.5 * gamma ** 2 * sp) / (4 * math.pi)
        i1 = (v1 - gamma * v0 + 0.5 * gamma ** 2 * vp) / (4 * math.pi) + i0[..., None] * rho
        g = (i1[:, :, None, :] - i0[:, :, None, None] * sv[:, None]) / (2 * sa)[:, None, None, None]
        z = z - gamma * torch.einsum("pqic,pqjc->pij", f.to(g), g)
        return z - ((i0 * ux).sum(1) / (gamma * sa))[:, None, None]
    # integrals of the gradients, in x, of 1/R and of R
    gm = v3 - s3[..., None] * n
    gp = -(v1 - d[..., None] * s1[..., None] * n)
    dg = (gm + 0.5 * gamma ** 2 * gp) / (4 * math.pi)
    g = ((x[:, :, None, :] - sv[:, None]) / (2 * sa)[:, None, None, None]).to(dg)
    return z + torch.einsum("pqic,pqjc->pij", f.to(dg), torch.linalg.cross(dg[:, :, None, :].expand_as(g), g))


def _matrix(op, gamma, X, Y, dev):
    T, S = _Cells(X, dev), _Cells(Y, dev)
    kernel = "nxk" if op == "mfie" else op
    Z = torch.zeros(T.n, S.n, dtype=torch.complex128, device=dev)
    step = max(1, int(4e6 if dev != "cpu" else 4e5) // len(S.v))
    for p0 in range(0, len(T.v), step):
        cells = torch.arange(p0, min(p0 + step, len(T.v)), device=dev)
        z = _far(kernel, gamma, T, S, cells, (6, 7) if kernel == "nxk" else (2, 3))
        if kernel != "nxk":
            hits, near = _classes(T, S, cells, gamma)
            for h in (0, 1, 2, 3):
                p, q = torch.nonzero(near if h == 0 else hits == h, as_tuple=True)
                for k in range(0, len(p), 4000):
                    i, j = p[k:k + 4000], q[k:k + 4000]
                    tv, sv = T.v[cells[i]], S.v[j]
                    z[i, j] = _near(kernel, gamma, tv, sv) if h == 0 else _singular(kernel, gamma, tv, sv, h)
        rows = S.gather(z.permute(0, 2, 1, 3).reshape(3 * len(cells), -1))        # [3 cells, N]
        for k in range(3):
            mine = (T.slot % 3 == k) & (T.slot // 3 >= p0) & (T.slot // 3 < p0 + len(cells))
            at = T.slot[mine]
            Z.index_add_(0, T.dof[mine], rows[3 * (at // 3 - p0) + k] * T.coef[mine, None])
    if op == "mfie":   # less half of the Gram matrix
        x, w = T.points(6)
        f = (x[:, :, None, :] - T.v[:, None]) / (2 * T.area)[:, None, None, None]
        gram = torch.einsum("fq,fqic,fqjc->fij", w, f, f)
        for i in range(3):
            for j in range(3):
                m = torch.full((3 * len(T.v),), -1, dtype=torch.int64, device=dev)
                c = torch.zeros(3 * len(T.v), dtype=torch.float64, device=dev)
                m[T.slot], c[T.slot] = T.dof, T.coef
                a, b = m[i::3], m[j::3]
                ok = (a >= 0) & (b >= 0)
                Z.index_put_((a[ok], b[ok]), (-0.5 * gram[:, i, j] * c[i::3] * c[j::3])[ok].to(Z.dtype), accumulate=True)
    return Z


def _right_hand_sides(s, dev):
    """(n x E) x n, or n x H, of plane waves, tested: H = (d x p) exp(-i k d.x)."""
    T = _Cells(s["X"], dev)
    x, w = T.points(8)
    f = (x[:, :, None, :] - T.v[:, None]) / (2 * T.area)[:, None, None, None]
    out = []
    for d, p in zip(s["d"], s["p"]):
        d, p = torch.as_tensor(d, device=dev), torch.as_tensor(p, device=dev)
        ph = torch.exp(-1j * s["k"] * (x * d).sum(-1)) * w
        if s["op"] == "efie":
            e = p.expand(len(T.v), 3)
        else:
            e = torch.linalg.cross(T.normal, torch.linalg.cross(d, p).expand(len(T.v), 3))
        out.append(T.gather(((f * e[:, None, None, :]).sum(-1) * ph[..., None]).sum(1).reshape(-1)))
    return torch.stack(out, 1)


def _far_field(s, dev):
    T = _Cells(s["X"], dev)
    x, w = T.points(10)
    f = (x[:, :, None, :] - T.v[:, None]) / (2 * T.area)[:, None, None, None]
    a = torch.zeros(3 * len(T.v), dtype=torch.complex128, device=dev)
    a.index_add_(0, T.slot, T.coef * torch.as_tensor(s["coeffs"], device=dev)[T.dof])
    J = torch.einsum("fi,fqic->fqc", a.reshape(-1, 3), f.to(a)) * w[..., None]
    if s["op"] == "rotated":
        J = torch.linalg.cross(J, T.normal[:, None, :].to(J).expand_as(J))
    J, x = J.reshape(-1, 3), x.reshape(-1, 3)
    Y = torch.as_tensor(s["points"], device=dev).reshape(-1, 3)
    out = torch.zeros(len(Y), 3, dtype=torch.complex128, device=dev)
    for y, o in zip(Y.split(max(1, 100_000_000 // len(x))), out.split(max(1, 100_000_000 // len(x)))):
        k = torch.exp(s["gamma"] * (y @ x.T))
        v = torch.stack([(k * J[:, c]).sum(1) for c in range(3)], 1)
        c = torch.linalg.cross(y.to(v), v)
        o.copy_(torch.linalg.cross(c, y.to(v)) if s["op"] == "single" else c)
    return out.reshape(s["points"].shape)


def _solution(s, dev):
    if s["X"].geo.numcells > (_CELLS if dev != "cpu" else 700):
        return None
    Z = _matrix(s["op"], 1j * s["k"], s["X"], s["X"], dev)
    return torch.linalg.solve(Z, _right_hand_sides(s, dev)).cpu().numpy()


def exact(case, seed):
    dev = "cuda:0" if torch.cuda.is_available() else "cpu"
    s = _inputs(case, seed)
    kind = s["kind"]
    if kind == "rhs":
        return _right_hand_sides(s, dev)[:, 0].cpu().numpy()
    if kind == "matrix":
        return _matrix(s["op"], s["gamma"], s["X"], s["Y"], dev).cpu().numpy()
    if kind == "farfield":
        return _far_field(s, dev).cpu().numpy()
    if kind == "solve":
        return {"b": _right_hand_sides(s, dev).cpu().numpy(), "x": _solution(s, dev)}
    if kind == "resident":
        return _solution(s, dev)
    return [_solution(p, dev) for p in s["problems"]]
