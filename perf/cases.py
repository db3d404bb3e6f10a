"""The framework's main path as measurable cases: the dense collocation assembly of F, G and
C (one wavenumber, sweeps, k-derivatives, uneven batches, field points), its derivatives
(vector-Jacobian product, batched dF/dk), the sparse near field and the dense apply, each
through the entry points of bie_amd on device buffers that the caller owns.

Bodies are geodesic meshes deformed smoothly by the seed, so that another seed is another
shape and another wavenumber.  exact() restates each result in plain torch in 64 bits.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "boundaryintegralequations.jl_amd"))
import bie_amd  # noqa: E402
from bie_amd import adjoint, operators, taylor  # noqa: E402
from bie_amd.mesh import Mesh3d, fibonacci_sphere, with_discontinuous_physics  # noqa: E402

DEVICE = "cuda"
# values of one complex work array of exact() at a time
CHUNK = 12_000_000


def listed():
    return [
        # the smallest call: pulsating sphere of 642 nodes, four-point rule, launches count
        dict(name="assemble_linear_642", kind="dense", f=8, order="linear", n=2, m=2,
             k=1.0, ki=0.0, g=True),
        # field operator of a scattering objective: few rows, explicit targets, F only
        dict(name="field_linear_100x2562", kind="field", f=16, order="linear", n=4, m=4,
             k=5.0, ki=0.0, points=100),
        # an ordinary call: linear sphere at the reference's default orders
        dict(name="assemble_linear_4002", kind="dense", f=20, order="linear", n=4, m=4,
             k=10.0, ki=0.0, g=True),
        # the full-size quadratic sphere with the 6-point rule
        dict(name="assemble_quadratic_10242", kind="dense", f=16, order="quadratic", n=3, m=2,
             k=10.0, ki=0.0, g=True),
        # a lossy mode: complex wavenumber, quadratic elements, default orders, odd size
        dict(name="assemble_lossy_3242", kind="dense", f=9, order="quadratic", n=4, m=4,
             k=4.0, ki=0.3, g=True),
        # frequency sweep on one mesh, F and G of every wavenumber
        dict(name="sweep_linear_4002x16", kind="sweep", f=20, order="linear", n=4, m=4, nk=16,
             k=0.5, k1=30.0, g=True),
        # k-derivatives of F as a reduced-order model needs them
        dict(name="taylor_linear_4002x26", kind="taylor", f=20, order="linear", n=2, m=2,
             orders=26, k=4.12, ki=0.0, g=False),
        # an uneven batch of ellipsoids in one launch
        dict(name="batch_linear_24", kind="batch", count=24, n_min=500, n_max=6000, n=4, m=4),
        # its k-derivatives, contracted with each instance's adjoint
        dict(name="batch_dfdk_24", kind="dfdk", count=24, n_min=500, n_max=6000, n=4, m=4),
        # shape gradient of the assembled operator (the adjoint direction)
        dict(name="vjp_linear_2562", kind="vjp", f=16, order="linear", n=4, m=4, k=5.0),
        # sparse near field of a fast operator on the quadratic sphere
        dict(name="near_quadratic_10242", kind="near", f=16, order="quadratic",
             physics="geometry", depth=1, k=10.0, ki=0.0, gauss=40),
        # the assembled operator applied to 32 right-hand sides
        dict(name="apply_10242x32", kind="apply", rows=10242, cols=10242, rhs=32),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dense", "dense", "dense", "field", "sweep", "taylor", "batch", "dfdk",
                       "vjp", "near", "near", "apply"])
    k = round(rng.uniform(0.5, 20.0), 4)
    if kind == "dense":
        order = rng.choice(["linear", "quadratic"])
        n, m = rng.choice([(2, 2), (3, 3), (4, 4)] if order == "linear" else [(3, 2), (4, 4)])
        f = _log_int(rng, 8, 30) if order == "linear" else _log_int(rng, 4, 16)
        return dict(kind=kind, f=f, order=order, n=n, m=m, k=k,
                    ki=rng.choice([0.0, 0.0, round(rng.uniform(0.05, 1.0), 4)]),
                    g=rng.random() < 0.75)
    if kind == "field":
        return dict(kind=kind, f=_log_int(rng, 8, 16), order=rng.choice(["linear", "quadratic"]),
                    n=4, m=4, k=k, ki=0.0, points=_log_int(rng, 20, 2000))
    if kind == "sweep":
        return dict(kind=kind, f=_log_int(rng, 6, 20), order="linear", n=4, m=4,
                    nk=rng.randint(3, 16), k=0.5, k1=round(rng.uniform(5.0, 30.0), 4),
                    g=rng.random() < 0.5)
    if kind == "taylor":
        return dict(kind=kind, f=_log_int(rng, 6, 20), order="linear",
                    n=2, m=2, orders=rng.randint(3, 26), k=round(rng.uniform(0.5, 6.0), 4),
                    ki=0.0, g=rng.random() < 0.25)
    if kind in ("batch", "dfdk"):
        return dict(kind=kind, count=rng.randint(4, 24), n_min=rng.randint(162, 500),
                    n_max=_log_int(rng, 1500, 6000), n=4, m=4)
    if kind == "vjp":
        order = rng.choice(["linear", "quadratic"])
        f = _log_int(rng, 6, 18) if order == "linear" else _log_int(rng, 4, 9)
        return dict(kind=kind, f=f, order=order, n=4, m=4, k=k)
    if kind == "near":
        physics = rng.choice(["geometry", "disctrilinear", "disctriconstant"])
        order = rng.choice(["linear", "quadratic"])
        # (on flat elements the double layer of depth 1 is zero but for rounding)
        return dict(kind=kind, f=_log_int(rng, 4, 14), order=order, physics=physics,
                    depth=2 if order == "linear" else rng.choice([1, 2]), k=k, ki=0.0, gauss=40)
    return dict(kind=kind, rows=_log_int(rng, 400, 10242), cols=_log_int(rng, 400, 10242),
                rhs=rng.choice([1, 8, 17, 32, 40, 64]))


# ---- bodies --------------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _sphere(f, order):
    return bie_amd.icosphere(f, order)


def _body(f, order, rng, physics="geometry", axes=(1.0, 1.0, 1.0)):
    """A geodesic mesh with its radius modulated by three smooth waves."""
    base = _sphere(f, order)
    x = base.coordinates
    s = np.ones(x.shape[1])
    for _ in range(3):
        d = rng.standard_normal(3)
        s = s + 0.03 * np.sin(2.0 * (d / np.linalg.norm(d)) @ x + rng.uniform(0.0, 6.28))
    x = x * s * np.asarray(axes)[:, None]
    mesh = Mesh3d(x, base.topology, x.copy(), base.topology.copy(), base.geometry_kind,
                  base.geometry_kind)
    return mesh if physics == "geometry" else with_discontinuous_physics(mesh, physics)


def _nodes(f, order):
    return 10 * f * f + 2 if order == "linear" else 40 * f * f + 2


def _batch_sizes(case):
    """Subdivisions whose node counts run log-uniformly from n_min to n_max, interleaved."""
    c = case["count"]
    ns = [case["n_min"] * (case["n_max"] / case["n_min"]) ** (i / max(1, c - 1))
          for i in range(c)]
    fs = [max(2, round(math.sqrt((x - 2) / 10))) for x in ns]
    return fs[::2] + fs[1::2][::-1]


def _batch_bodies(case, rng):
    return [(_body(f, "linear", rng, axes=rng.uniform(0.5, 2.0, 3)), float(rng.uniform(1, 20)))
            for f in _batch_sizes(case)]


def _empty(*shape):
    return torch.empty(shape, dtype=torch.complex128, device=DEVICE)


def _normal(seed, *shape):
    g = torch.Generator(device=DEVICE).manual_seed(int(seed) % (1 << 62))
    return torch.randn(*shape, dtype=torch.complex128, device=DEVICE, generator=g)


def _inputs(case, seed):
    """The mesh and numbers that a case's seed stands for (host side)."""
    rng = np.random.default_rng(int(seed))
    kind = case["kind"]
    if kind in ("batch", "dfdk"):
        return dict(bodies=_batch_bodies(case, rng))
    if kind == "apply":
        return {}
    mesh = _body(case["f"], case["order"], rng, case.get("physics", "geometry"))
    got = dict(mesh=mesh, k=case["k"] * (1.0 + 0.02 * rng.uniform()))
    if kind == "field":
        got["points"] = np.asfortranarray(
            fibonacci_sphere(case["points"], 3.0 + 0.1 * rng.uniform()))
    if kind == "sweep":
        got["ks"] = np.linspace(got["k"], case["k1"], case["nk"])
    if kind == "vjp":
        N = mesh.n_sources
        got.update({x: rng.standard_normal(N) + 1j * rng.standard_normal(N)
                    for x in ("alpha", "beta", "p")})
    return got


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, **_inputs(case, seed))
    if kind == "apply":
        M, K, R = case["rows"], case["cols"], case["rhs"]
        # column-major matrices: a row of the tensor is a column of the matrix
        s.update(A=_normal(seed, K, M), X=_normal(seed + 7919, R, K), Y=_empty(R, M))
        return s
    if kind in ("batch", "dfdk"):
        meshes = [b[0] for b in s["bodies"]]
        s["ks"] = [b[1] for b in s["bodies"]]
        s["dms"] = [bie_amd.DeviceMesh(x) for x in meshes]
        s["batch"] = bie_amd.Batch(s["dms"], n=case["n"], m=case["m"])
        Ns = [x.n_sources for x in meshes]
        at = np.concatenate([[0], np.cumsum(Ns)])
        if kind == "dfdk":
            s["alpha"], s["p"] = _normal(seed, at[-1]), _normal(seed + 7919, at[-1])
            s["w"] = _empty(len(Ns))
            for v in ("alpha", "p"):
                s[v + "_ptrs"] = [s[v].data_ptr() + 16 * int(o) for o in at[:-1]]
            return s
        sq = np.concatenate([[0], np.cumsum([N * N for N in Ns])])
        s.update(F=_empty(int(sq[-1])), G=_empty(int(sq[-1])), C=_empty(int(at[-1])))
        for v, off in (("F", sq), ("G", sq), ("C", at)):
            s[v + "_ptrs"] = [s[v].data_ptr() + 16 * int(o) for o in off[:-1]]
        return s
    mesh = s["mesh"]
    N = mesh.n_sources
    s["dm"] = bie_amd.DeviceMesh(mesh)
    if kind == "vjp":
        s["nodes"] = np.arange(N, dtype=np.int32)
    elif kind == "near":
        s["near"] = bie_amd.SparsePattern(s["dm"], depth=case["depth"], Ngauss=case["gauss"])
        s.update(F=_empty(s["near"].nnz), G=_empty(s["near"].nnz))
    elif kind == "taylor":
        s.update(F=_empty(case["orders"], N, N), C=_empty(N),
                 G=_empty(case["orders"], N, N) if case["g"] else None)
    elif kind == "sweep":
        s["k_dev"] = torch.from_numpy(s["ks"]).to(DEVICE)
        s.update(F=_empty(case["nk"], N, N), C=_empty(N),
                 G=_empty(case["nk"], N, N) if case["g"] else None)
    else:
        M = N
        if kind == "field":
            M = s["points"].shape[1]
            s["targets"] = torch.from_numpy(s["points"].T.copy()).to(DEVICE)
        s.update(F=_empty(N, M), G=_empty(N, M), C=_empty(M))
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "apply":
        M, K, R = case["rows"], case["cols"], case["rhs"]
        operators.zgemm_device(M, R, K, s["A"].data_ptr(), M, s["X"].data_ptr(), K,
                               s["Y"].data_ptr(), M, stream)
        return s["Y"]
    if kind == "batch":
        s["batch"].assemble(s["ks"], s["F_ptrs"], s["G_ptrs"], s["C_ptrs"], stream=stream)
        return s["F"], s["G"], s["C"]
    if kind == "dfdk":
        s["batch"].dfdk(s["ks"], s["alpha_ptrs"], s["p_ptrs"], s["w"].data_ptr(), stream=stream)
        return s["w"]
    dm = s["dm"]
    if kind == "vjp":
        return adjoint.assembly_vjp(dm, s["k"], s["alpha"], s["p"], beta=s["beta"],
                                    target_node=s["nodes"], n=case["n"], m=case["m"])
    if kind == "near":
        s["near"].assemble_device(complex(s["k"], case["ki"]), s["F"].data_ptr(),
                                  s["G"].data_ptr(), stream=stream)
        return s["F"], s["G"]
    orders = dict(n=case["n"], m=case["m"])
    if kind in ("sweep", "taylor"):
        N = dm.n_sources
        G = s["G"].data_ptr() if case["g"] else 0
        if kind == "sweep":
            dm.assemble_sweep(s["k_dev"].data_ptr(), case["nk"], s["F"].data_ptr(), G, N * N,
                              s["C"].data_ptr(), gOn=case["g"], stream=stream, **orders)
        else:
            taylor.assemble_taylor_device(dm, complex(s["k"], case["ki"]), case["orders"],
                                          s["F"].data_ptr(), G, N * N, s["C"].data_ptr(),
                                          gOn=case["g"], stream=stream, **orders)
        return (s["F"], s["G"], s["C"]) if case["g"] else (s["F"], s["C"])
    k = complex(s["k"], case["ki"])
    if kind == "field":
        dm.assemble(k, s["F"].data_ptr(), s["G"].data_ptr(), s["C"].data_ptr(),
                    targets_ptr=s["targets"].data_ptr(), n_targets=case["points"], gOn=False,
                    cOn=False, stream=stream, **orders)
        return s["F"]
    dm.assemble(k, s["F"].data_ptr(), s["G"].data_ptr(), s["C"].data_ptr(), gOn=case["g"],
                stream=stream, **orders)
    return (s["F"], s["G"], s["C"]) if case["g"] else (s["F"], s["C"])


# ---- the work that cannot be left out ------------------------------------------------------

def _mesh_bytes(E, N, nodes):
    return 24.0 * N + 16.0 * E * nodes


def work(case):
    """Outputs written once and inputs read once; per quadrature point 35 operations (sqrt,
    reciprocal, sin and cos one each) and 4 per accumulated real value and node, per pair
    10 per node for the choice of its rule."""
    kind = case["kind"]
    if kind == "apply":
        M, K, R = case["rows"], case["cols"], case["rhs"]
        return {"bytes": 16.0 * (M * K + K * R + M * R), "flops": 8.0 * M * K * R}
    if kind in ("batch", "dfdk"):
        b = f = 0.0
        for x in _batch_sizes(case):
            N, E, Q = 10 * x * x + 2, 20 * x * x, case["n"] * case["m"]
            out = 32.0 * N * N + 16 * N if kind == "batch" else 32.0 * N
            b += _mesh_bytes(E, N, 3) + out
            f += N * E * (Q * (35 + (24 if kind == "batch" else 20)) + 30.0)
        return {"bytes": b, "flops": f}
    f, order = case["f"], case["order"]
    E, N, nd = 20.0 * f * f, float(_nodes(f, order)), 3 if order == "linear" else 6
    mesh = _mesh_bytes(E, N, nd)
    if kind == "near":
        npk = {"geometry": nd, "disctrilinear": 3, "disctriconstant": 1}[case["physics"]]
        rules = _near_rules(case["physics"], nd, case["gauss"])
        points = sum(len(r[0]) for r in rules[:npk]) / npk
        if case["physics"] == "geometry":
            pairs = E * nd * (1 if case["depth"] == 1 else 13 / 3 if nd == 3 else 17 / 3)
            nnz = N * (7 if nd == 3 else 11.5) * (1 if case["depth"] == 1 else 2.7)
        else:
            pairs = E * npk * (1 if case["depth"] == 1 else 13)
            nnz = pairs * npk
        return {"bytes": mesh + 32.0 * nnz,
                "flops": pairs * points * (18.0 * nd + 60 + 8 * npk)}
    Q = float(case["n"] * case["m"])
    if kind == "vjp":
        return {"bytes": 2 * mesh + 48.0 * N,
                "flops": N * E * (Q * (36.0 * nd + 4 * nd + 110) + 10 * nd)}
    M = float(case["points"]) if kind == "field" else N
    outs = 2 if case.get("g", False) else 1
    many = case["nk"] if kind == "sweep" else case["orders"] if kind == "taylor" else 1
    return {"bytes": mesh + 16.0 * outs * M * N * many + 16 * M,
            "flops": M * E * (Q * (35 + many * (8.0 + 4 * nd * outs)) + 10 * nd)}


# ---- the same results in plain torch -------------------------------------------------------

def _gauss01(n):
    x, w = np.polynomial.legendre.leggauss(n)
    return 0.5 * (x + 1.0), 0.5 * w


def _tensor(n, m):
    (x, wx), (y, wy) = _gauss01(n), _gauss01(m)
    return np.tile(x, m), np.repeat(y, n), np.outer(wy, wx).ravel()


def _vertex_rules(n, m, nodes):
    """Duffy rules clustered at the corners (n x m points) and, on six-node elements, the
    two-triangle rules clustered at the edge midpoints."""
    u, v, w = _tensor(n, m)
    rules = [(u * v, (1 - u) * v, w * v), (u, v * (1 - u), w * (1 - u)),
             (v * (1 - u), u, w * (1 - u))]
    if nodes == 6:
        u, v, w = _tensor(n, 2 * ((m + 1) // 2))
        x = np.concatenate([0.5 * u, (u - 0.5) * v + 0.5])
        y = np.concatenate([v * (1 - u), v * (1 - u)])
        w = np.concatenate([w * 0.5 * (1 - u), w * 0.5 * v])
        rules += [(x, y, w), (1 - x - y, x, w), (y, 1 - x - y, w)]
    return rules


def _subdivision_rule(src):
    """The reference triangle split in four while a part's longest side exceeds a quarter of
    its distance from src, three points around each part's centre."""
    def lift(p):
        return np.stack([1 - p[..., 0] - p[..., 1], p[..., 0], p[..., 1]], -1)

    def side(a, b):
        return np.linalg.norm(a - b, axis=-1)

    todo = np.array([[[0.0, 0.0], [1.0, 0.0], [0.0, 1.0]]])
    done = []
    while len(todo):
        t3 = lift(todo)
        cen = todo.sum(1) / 3.0
        dist = np.minimum(side(lift(cen), src), side(t3, src).min(1))
        size = np.stack([side(t3[:, a], t3[:, b]) for a, b in ((1, 0), (2, 1), (0, 2))]).max(0)
        size = np.where(size < math.sqrt(2.0) * 1e-6, 0.0, size)
        more = size > dist / 4
        done.append(todo[~more])
        t = todo[more]
        ab, bc, ca = (0.5 * (t[:, i] + t[:, j]) for i, j in ((0, 1), (1, 2), (2, 0)))
        todo = np.concatenate([np.stack(x, 1) for x in (
            (t[:, 0], ab, ca), (ab, t[:, 1], bc), (ca, bc, t[:, 2]), (ab, bc, ca))])
    t = np.concatenate(done)
    dim = np.stack([side(t[:, a], t[:, b]) for a, b in ((1, 0), (2, 1), (0, 2))]).min(0)
    cen = t.sum(1) / 3.0
    g = np.array([[1, 1], [4, 1], [1, 4]]) / 6.0 - 1 / 3
    p = cen[:, None, :] + g[None] * dim[:, None, None]
    return p[..., 0].ravel(), p[..., 1].ravel(), np.repeat(dim * dim / 6.0, 3)


def _polar_rule(P, n):
    """Polar rules on the three triangles between the node P and the sides."""
    n = 2 * ((n + 1) // 2)
    g, w = np.polynomial.legendre.leggauss(n)
    th, tw = np.pi / 4 * (1 + g), np.pi / 4 * w
    rm = 1 / (np.cos(th) + np.sin(th))
    r = 0.5 * rm[:, None] * (1 + g)[None, :]
    W = (tw[:, None] * 0.5 * rm[:, None] * w[None, :] * r).ravel()
    X, Y = (r * np.cos(th)[:, None]).ravel(), (r * np.sin(th)[:, None]).ravel()
    out = []
    c = np.array([[0.0, 0.0], [1.0, 0.0], [0.0, 1.0]])
    for a, b in ((2, 0), (1, 2), (0, 1)):
        A, B = c[a] - P, c[b] - P
        out.append((P[0] + A[0] * X + B[0] * Y, P[1] + A[1] * X + B[1] * Y,
                    W * abs(A[0] * B[1] - A[1] * B[0])))
    return tuple(np.concatenate(x) for x in zip(*out))


@functools.lru_cache(maxsize=None)
def _near_rules(physics, nodes, gauss):
    """The rule of each geometry node that may be the nearest one to the source."""
    if physics == "geometry":
        mid = [[0.5, 0.5, 0.0], [0.0, 0.5, 0.5], [0.5, 0.0, 0.5]]
        return [_subdivision_rule(np.array(s)) for s in np.eye(3).tolist() + mid][:nodes]
    b = 0.5 * (1.0 - 1.0 / math.sqrt(3.0))
    at = [[1 / 3, 1 / 3]] if physics == "disctriconstant" else [[b, b], [1 - 2 * b, b],
                                                                 [b, 1 - 2 * b]]
    rules = [_polar_rule(np.array(p), gauss) for p in at]
    return [rules[c % len(rules)] for c in range(nodes)]


def _basis(nodes, u, v):
    """Lagrange bases on three or six nodes and their derivatives, each (points, nodes)."""
    o, z, l = np.ones_like(u), np.zeros_like(u), 1 - u - v
    if nodes == 3:
        return [np.stack(x, 1) for x in ((l, u, v), (-o, o, z), (-o, z, o))]
    return [np.stack(x, 1) for x in (
        (l * (2 * l - 1), u * (2 * u - 1), v * (2 * v - 1), 4 * u * l, 4 * u * v, 4 * v * l),
        (1 - 4 * l, 4 * u - 1, z, 4 * (l - u), 4 * v, -4 * v),
        (1 - 4 * l, z, 4 * v - 1, -4 * u, 4 * u, 4 * (l - v)))]


def _physics_basis(mesh, u, v):
    if mesh.physics_kind == 0x101:
        return np.ones((u.size, 1))
    if mesh.physics_kind == 0x103:
        b = mesh.physics_beta
        return (np.stack([1 - u - v, u, v], 1) - b) / (1 - 3 * b)
    return _basis(mesh.physics_kind & 0xFF, u, v)[0]


def _dev(x):
    return torch.as_tensor(np.ascontiguousarray(x), device=DEVICE)


def _nearest(P, x):
    """Index of the node nearest to each x: (pairs..., nodes) distances as
    max * sqrt(sum (x / max)^2), the first of equal ones."""
    best, at = None, None
    for s in range(P.shape[-2]):
        a, b, c = (P[..., s, :] - x).abs().unbind(-1)
        m = torch.maximum(torch.maximum(a, b), c)
        d = m.clamp_min(1e-300)
        t = (a / d) * (a / d)
        t = t + (b / d) * (b / d)
        t = t + (c / d) * (c / d)
        d = m * t.sqrt()
        if best is None:
            best, at = d, torch.zeros_like(d, dtype=torch.int64)
        else:
            at = torch.where(d < best, s, at)
            best = torch.minimum(best, d)
    return at


class _Surface:
    """Points, normals and weights of every rule on every element of a mesh."""

    def __init__(self, mesh, rules):
        X = _dev(mesh.coordinates[:, mesh.topology].transpose(2, 1, 0))   # E, nodes, 3
        self.rules = []
        for u, v, w in rules:
            N, du, dv = (_dev(b) for b in _basis(mesh.topology.shape[0], u, v))
            y, tu, tv = (torch.matmul(b, X) for b in (N, du, dv))
            c = torch.linalg.cross(tu, tv)
            J = c.norm(dim=-1)
            self.rules.append((y, -c / J[..., None], J * _dev(w) / (4 * math.pi),
                               _dev(_physics_basis(mesh, u, v))))

    def pairs(self, c, e, x):
        """r, n.d / r^2, J w / (4 pi r) and the basis for elements e and targets x, rule c."""
        y, n, jw, phi = self.rules[c]
        d = y[e] - x[:, None, :]
        r2 = (d * d).sum(-1)
        r = r2.sqrt()
        return r, (n[e] * d).sum(-1) / r2, jw[e] / r, phi


def _dense_pairs(mesh, targets, n, m):
    """Yields (rows, elements, r, n.d / r^2, J w / (4 pi r), basis) over all pairs."""
    sel = _dev(mesh.sources[:, mesh.physics_topology].transpose(2, 1, 0))
    surf = _Surface(mesh, _vertex_rules(n, m, mesh.topology.shape[0]))
    x = _dev(targets.T)
    step = max(1, CHUNK // (mesh.n_elements * n * m))
    for i0 in range(0, x.shape[0], step):
        xs = x[i0:i0 + step]
        c = _nearest(sel[None], xs[:, None, :])
        for q in range(len(surf.rules)):
            i, e = torch.nonzero(c == q, as_tuple=True)
            if i.numel():
                yield (i + i0, e) + surf.pairs(q, e, xs[i])


def _dense(mesh, targets, n, m, values, many, g=True):
    """F and G (many x N x M, column-major), C: values(r, t, a, b) are f and g of matrix b."""
    N, M = mesh.n_sources, targets.shape[1]
    cols = _dev(mesh.physics_topology.T)
    F = torch.zeros(many, N * M, dtype=torch.complex128, device=DEVICE)
    G = torch.zeros_like(F) if g else None
    C = torch.zeros(M, dtype=torch.complex128, device=DEVICE)
    for i, e, r, t, a, phi in _dense_pairs(mesh, targets, n, m):
        C.index_add_(0, i, -(t * a).sum(1).to(torch.complex128))
        at = (cols[e] * M + i[:, None]).reshape(-1)
        phi = phi.to(torch.complex128)
        for b in range(many):
            fv, gv = values(r, t, a, b)
            F[b].index_add_(0, at, (fv @ phi).reshape(-1))
            if g:
                G[b].index_add_(0, at, (gv @ phi).reshape(-1))
    return F.view(many, N, M), G.view(many, N, M) if g else None, C


def _helmholtz(ks):
    def values(r, t, a, b):
        k = complex(ks[b])
        gv = torch.polar(a * torch.exp(-k.imag * r), k.real * r)
        return gv * torch.complex(-k.imag * r - 1.0, k.real * r) * t, gv
    return values


def _derivatives(k):
    """Orders of the k-derivative: (i r)^b e^{ikr} and (i k r - 1 + b) times it."""
    k = complex(k)

    def values(r, t, a, b):
        gv = torch.polar(a * torch.exp(-k.imag * r) * r ** b, k.real * r) * (1j ** b)
        return gv * torch.complex(b - 1.0 - k.imag * r, k.real * r) * t, gv
    return values


def _near_pairs(mesh, depth):
    """(row, element) pairs of the near field."""
    E = mesh.n_elements
    P = mesh.physics_topology
    touch = {}
    key = P if mesh.physics_kind < 0x100 else mesh.topology[:3]
    for e in range(E):
        for j in key[:, e]:
            touch.setdefault(int(j), []).append(e)
    around = [np.unique(np.concatenate([touch[int(j)] for j in key[:, e]])) for e in range(E)]
    rows, els = [], []
    if mesh.physics_kind < 0x100:
        for i in range(mesh.n_sources):
            el = np.array(touch[i])
            if depth == 2:
                el = np.unique(np.concatenate([around[e] for e in el]))
            rows.append(np.full(len(el), i))
            els.append(el)
    else:
        for e in range(E):
            el = np.array([e]) if depth == 1 else around[e]
            for i in P[:, e]:
                rows.append(np.full(len(el), i))
                els.append(el)
    return np.concatenate(rows), np.concatenate(els)


def _near(mesh, k, case):
    rows, els = (_dev(x) for x in _near_pairs(mesh, case["depth"]))
    N = mesh.n_sources
    cols = _dev(mesh.physics_topology.T)
    keys, at = torch.unique((rows[:, None] * N + cols[els]).reshape(-1), return_inverse=True)
    at = at.view(cols[els].shape)
    F = torch.zeros(keys.numel(), dtype=torch.complex128, device=DEVICE)
    G = torch.zeros_like(F)
    X = _dev(mesh.coordinates[:, mesh.topology].transpose(2, 1, 0))
    x = _dev(mesh.sources.T)
    c = _nearest(X[els], x[rows])
    values = _helmholtz([k])
    nodes = X.shape[1]
    for q, rule in enumerate(_near_rules(case["physics"], nodes, case["gauss"])):
        mine = torch.nonzero(c == q).view(-1)
        u, v, w = rule
        phi = _dev(_physics_basis(mesh, u, v)).to(torch.complex128)
        B = [_dev(b) for b in _basis(nodes, u, v)]
        w = _dev(w) / (4 * math.pi)
        step = max(1, CHUNK // (4 * len(u)))
        for p in mine.split(step):
            y, tu, tv = (torch.matmul(b, X[els[p]]) for b in B)
            cr = torch.linalg.cross(tu, tv)
            J = cr.norm(dim=-1)
            d = y - x[rows[p]][:, None, :]
            r2 = (d * d).sum(-1)
            r = r2.sqrt()
            fv, gv = values(r, -(cr * d).sum(-1) / (J * r2), J * w / r, 0)
            F.index_add_(0, at[p].reshape(-1), (fv @ phi).reshape(-1))
            G.index_add_(0, at[p].reshape(-1), (gv @ phi).reshape(-1))
    return F, G


def _vjp(mesh, k, s, n, m):
    """Gradient of Re[alpha^T F p + beta^T C] by torch's reverse mode, rules held fixed."""
    nodes = mesh.topology.shape[0]
    Xc = _dev(mesh.coordinates.T).requires_grad_(True)
    topo = _dev(mesh.topology.T)
    kk = torch.tensor(float(k), dtype=torch.float64, device=DEVICE, requires_grad=True)
    alpha, beta, p = (_dev(s[x]) for x in ("alpha", "beta", "p"))
    with torch.no_grad():
        sel = Xc[topo]
    rules = _vertex_rules(n, m, nodes)
    step = max(1, CHUNK // (6 * mesh.n_elements * n * m))
    for i0 in range(0, mesh.n_sources, step):
        c = _nearest(sel[None], Xc.detach()[i0:i0 + step, None, :])
        for q, (u, v, w) in enumerate(rules):
            i, e = torch.nonzero(c == q, as_tuple=True)
            if not i.numel():
                continue
            N, du, dv = (_dev(b) for b in _basis(nodes, u, v))
            X = Xc[topo]
            y, tu, tv = (torch.matmul(b, X) for b in (N, du, dv))
            cr = torch.linalg.cross(tu, tv)
            d = y[e] - Xc[i + i0][:, None, :]
            r2 = (d * d).sum(-1)
            r = r2.sqrt()
            cd = (cr[e] * d).sum(-1) * (_dev(w) / (4 * math.pi)) / (r2 * r)
            ph = torch.matmul(p[topo[e]], N.T.to(torch.complex128)) * alpha[i + i0][:, None]
            # f = -(c.d) e^{ikr} (ikr - 1) / (4 pi r^3), C's integrand (c.d) / (4 pi r^3)
            kr = kk * r
            re = -(kr * torch.sin(kr) + torch.cos(kr))
            im = kr * torch.cos(kr) - torch.sin(kr)
            val = -cd * (ph.real * re - ph.imag * im) + cd * beta.real[i + i0][:, None]
            val.sum().backward()
    return Xc.grad.T.contiguous(), kk.grad


def exact(case, seed):
    kind = case["kind"]
    if kind == "apply":
        A = _normal(seed, case["cols"], case["rows"])
        return _normal(seed + 7919, case["rhs"], case["cols"]) @ A
    s = _inputs(case, seed)
    if kind == "batch":
        out = [_dense(x, x.sources, case["n"], case["m"], _helmholtz([k]), 1)
               for x, k in s["bodies"]]
        return tuple(torch.cat([o[j].reshape(-1) for o in out]) for j in range(3))
    if kind == "dfdk":
        Ns = [x.n_sources for x, _ in s["bodies"]]
        alpha, p = (_normal(t, sum(Ns)).split(Ns) for t in (seed, seed + 7919))
        w = torch.zeros(len(Ns), dtype=torch.complex128, device=DEVICE)
        for b, (mesh, k) in enumerate(s["bodies"]):
            cols = _dev(mesh.physics_topology.T)
            for i, e, r, t, a, phi in _dense_pairs(mesh, mesh.sources, case["n"], case["m"]):
                v = torch.polar(-k * t * a * r * r, k * r)
                w[b] += (((v @ phi.to(torch.complex128)) * p[b][cols[e]]).sum(1) *
                         alpha[b][i]).sum()
        return w
    mesh, k = s["mesh"], s["k"]
    if kind == "vjp":
        return _vjp(mesh, k, s, case["n"], case["m"])
    if kind == "near":
        return _near(mesh, complex(k, case["ki"]), case)
    n, m = case["n"], case["m"]
    if kind == "field":
        return _dense(mesh, s["points"], n, m, _helmholtz([complex(k, case["ki"])]), 1,
                      False)[0][0]
    if kind == "sweep":
        F, G, C = _dense(mesh, mesh.sources, n, m, _helmholtz(s["ks"]), case["nk"], case["g"])
    elif kind == "taylor":
        F, G, C = _dense(mesh, mesh.sources, n, m, _derivatives(complex(k, case["ki"])),
                         case["orders"], case["g"])
    else:
        F, G, C = _dense(mesh, mesh.sources, n, m, _helmholtz([complex(k, case["ki"])]), 1,
                         case["g"])
        F, G = F[0], G[0] if case["g"] else None
    return (F, G, C) if case["g"] else (F, C)
