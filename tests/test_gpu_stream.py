"""The dense, sweep and derivative kernels where their work splits: rule lengths around the
points taken at a time and the rows staged, odd lengths, partial blocks of wavenumbers and
orders, spaced and scattered wavenumbers, tiles left to the launch for large arguments, and
tiles with more mid-edge pairs than they queue."""
import numpy as np
import pytest

import oracle
from bie_amd import mesh as M
from bie_amd.assembly import DeviceMesh, assemble_parallel
from bie_amd.taylor import taylor_assemble
from gpu_helpers import TOL, DevBuf, rel, sync

pytestmark = pytest.mark.gpu


def sweep(mesh, ks, targets, n, m, gOn=True):
    dm = DeviceMesh(mesh)
    N, Mt, nk = mesh.n_sources, targets.shape[1], len(ks)
    kb, tb = DevBuf(8 * nk), DevBuf(24 * Mt)
    kb.upload(np.asarray(ks, dtype=np.float64))
    tb.upload(np.ascontiguousarray(targets.T))
    F, G, C = DevBuf(16 * Mt * N * nk), DevBuf(16 * Mt * N * nk), DevBuf(16 * Mt)
    dm.assemble_sweep(kb.ptr, nk, F.ptr, G.ptr, Mt * N, C.ptr, targets_ptr=tb.ptr, n_targets=Mt,
                      n=n, m=m, gOn=gOn)
    sync()
    out = [b.download(np.empty(s, dtype=np.complex128)) for b, s in
           ((F, (nk, N, Mt)), (G, (nk, N, Mt)), (C, (Mt,)))]
    return out[0].transpose(0, 2, 1), out[1].transpose(0, 2, 1), out[2]


def some_targets(mesh, count, seed=3):
    """Mesh nodes and field points, not a multiple of a tile's rows."""
    rng = np.random.default_rng(seed)
    x = 1.5 * rng.standard_normal((3, count))
    x[:, ::2] = mesh.sources[:, rng.integers(0, mesh.n_sources, x[:, ::2].shape[1])]
    return np.asfortranarray(x)


@pytest.mark.parametrize("kind", ["linear", "quadratic"])
@pytest.mark.parametrize("nm", [(1, 1), (2, 1), (3, 1), (3, 3), (4, 4), (5, 5)])
def test_rule_lengths(kind, nm):
    mesh = M.perturb_radial(M.icosphere(3 if kind == "linear" else 2, kind), 0.02, 4)
    n, m = nm
    t = some_targets(mesh, 75)
    for k in (3.0, 2.0 + 0.4j):
        Fo, Go, Co = oracle.assemble(mesh, k, targets=t, n=n, m=m)
        F, G, C = assemble_parallel(mesh, k, t, n=n, m=m)
        assert rel(F, Fo) <= TOL and rel(G, Go) <= TOL and rel(C, Co) <= TOL, k


@pytest.mark.parametrize("kind", ["linear", "quadratic"])
@pytest.mark.parametrize("nk,spaced", [(1, True), (5, True), (7, False), (9, True), (12, False)])
def test_sweep_blocks(kind, nk, spaced):
    """Partial last blocks, with and without G."""
    mesh = M.icosphere(3 if kind == "linear" else 2, kind)
    t = some_targets(mesh, 67)
    ks = np.linspace(0.5, 7.0, nk) if spaced else np.sort(
        np.random.default_rng(nk).uniform(0.5, 7.0, nk))
    F, G, C = sweep(mesh, ks, t, 3, 3)
    Fx, _, Cx = sweep(mesh, ks, t, 3, 3, gOn=False)
    for q, k in enumerate(ks):
        Fo, Go, Co = oracle.assemble(mesh, k, targets=t, n=3, m=3)
        assert rel(F[q], Fo) <= TOL and rel(G[q], Go) <= TOL and rel(Fx[q], Fo) <= TOL, q
    assert rel(C, Co) <= TOL and rel(Cx, Co) <= TOL


@pytest.mark.parametrize("kind", ["linear", "quadratic"])
@pytest.mark.parametrize("orders", [1, 4, 6, 12, 13])
def test_derivative_blocks(kind, orders):
    """Orders in full, half and partial blocks, with and without G, real and complex k."""
    mesh = M.icosphere(2 if kind == "linear" else 1, kind)
    t = some_targets(mesh, 67)
    for k in (2.5, 2.0 + 0.3j):
        F, G, _ = taylor_assemble(mesh, k, t, M=orders - 1, n=3, m=3)
        Fx = taylor_assemble(mesh, k, t, M=orders - 1, n=3, m=3, gOn=False)[0]
        for q in range(orders):
            Fo, Go = oracle.assemble_taylor(mesh, k, q, targets=t, n=3, m=3)
            assert rel(F[:, :, q], Fo) <= TOL and rel(G[:, :, q], Go) <= TOL, q
            assert rel(Fx[:, :, q], Fo) <= TOL, q


@pytest.mark.parametrize("kind", ["linear", "quadratic"])
def test_tiles_with_a_far_target(kind):
    """One target so far off that its |k| r leaves the range of the branch-free sincos: its
    tile's other rows come from the launch for large arguments."""
    mesh = M.icosphere(3 if kind == "linear" else 2, kind)
    t = some_targets(mesh, 150)
    t[:, 70] = (0.0, 3e14, 0.0)
    near = np.arange(150) != 70
    Fo, Go, Co = oracle.assemble(mesh, 3.0, targets=t, n=3, m=3)
    F, G, C = assemble_parallel(mesh, 3.0, t, n=3, m=3)
    Fs, Gs, Cs = sweep(mesh, [3.0, 3.5], t, 3, 3)
    for X, Xo in ((F, Fo), (Fs[0], Fo), (G, Go), (Gs[0], Go)):
        assert rel(X[near], Xo[near]) <= TOL
        assert np.max(np.abs(X[70])) <= np.max(np.abs(Xo[70])) * (1 + 1e-9)
    assert rel(C[near], Co[near]) <= TOL and rel(Cs[near], Co[near]) <= TOL


def test_more_mid_edge_pairs_than_a_tile_queues():
    """Targets about the centre: every node is about as far, so a good part of all pairs has a
    mid-edge rule."""
    mesh = M.icosphere(4, "quadratic")
    t = np.asfortranarray(1e-2 * np.random.default_rng(8).standard_normal((3, 130)))
    for k in (2.0, 2.0 + 0.3j):
        Fo, Go, Co = oracle.assemble(mesh, k, targets=t, n=3, m=2)
        F, G, C = assemble_parallel(mesh, k, t, n=3, m=2)
        assert rel(F, Fo) <= TOL and rel(G, Go) <= TOL and rel(C, Co) <= TOL
    Fo, Go, Co = oracle.assemble(mesh, 2.0, targets=t, n=3, m=2)
    F, G, C = sweep(mesh, [2.0, 3.0], t, 3, 2)
    assert rel(F[0], Fo) <= TOL and rel(G[0], Go) <= TOL and rel(C, Co) <= TOL
    F, G, C = taylor_assemble(mesh, 2.0, t, M=1, n=3, m=2)
    assert rel(F[:, :, 0], Fo) <= TOL and rel(G[:, :, 0], Go) <= TOL


@pytest.mark.parametrize("f,nm,k", [(2, (1, 1), 3.0), (4, (3, 1), 2.0 + 0.3j), (5, (2, 2), 4.0),
                                    (5, (3, 3), 3.0 + 0.2j)])
def test_flat_adjoint_sizes(f, nm, k):
    """Elements short of a workgroup's 256 and past it, one point and odd lengths; targets
    given as points attached to nodes, one more so far off that its row is the other
    launch's (weight 0: finite there, nothing added)."""
    from bie_amd.adjoint import assembly_vjp, source_nodes
    from dual_oracle import assemble_F_C
    mesh = M.perturb_radial(M.icosphere(f, "linear"), 0.01, 4)
    n, m = nm
    rng = np.random.default_rng(f)
    N = mesh.n_sources
    alpha, beta, p = (rng.standard_normal(N) + 1j * rng.standard_normal(N) for _ in range(3))
    t = np.asfortranarray(np.concatenate([mesh.sources, [[0.0], [3e14], [0.0]]], axis=1))
    node = np.append(source_nodes(mesh), -1).astype(np.int32)
    dm = DeviceMesh(mesh)
    g, gk = assembly_vjp(dm, k, alpha, p, beta=beta, target_node=source_nodes(mesh), n=n, m=m)
    g2, gk2 = assembly_vjp(dm, k, np.append(alpha, 0.0), p, beta=np.append(beta, 0.0), targets=t,
                           target_node=node, n=n, m=m)
    assert rel(g2, g) <= 1e-12 and rel(np.atleast_1d(gk2), np.atleast_1d(gk)) <= 1e-12
    V = rng.standard_normal(mesh.coordinates.shape)
    rules = oracle.select(mesh, None)
    F, C = assemble_F_C(mesh, mesh.coordinates, V, k, 0.0, rules, targets=None, n=n, m=m)
    dd = np.real(alpha @ (F.d @ p) + beta @ C.d)
    assert abs(float(np.sum(g * V)) - dd) <= 1e-10 * abs(dd)


@pytest.mark.parametrize("kind", ["linear", "quadratic"])
@pytest.mark.parametrize("nm", [(1, 1), (3, 1), (3, 3), (5, 5)])
def test_batched_k_derivative(kind, nm):
    """Real and complex wavenumbers side by side, and one instance whose |k| r leaves the range
    of the branch-free sincos."""
    from bie_amd.assembly import Batch
    meshes = [M.icosphere(f, kind) for f in ((1, 2, 4) if kind == "linear" else (1, 2, 2))]
    ks = [3.0, 2.0 + 0.4j, 1e14]
    n, m = nm
    rng = np.random.default_rng(6)
    al, ps, w = [], [], DevBuf(16 * 3)
    for x in meshes:
        for out in (al, ps):
            v = rng.standard_normal(x.n_sources) + 1j * rng.standard_normal(x.n_sources)
            buf = DevBuf(16 * x.n_sources)
            buf.upload(v)
            out.append((v, buf))
    dms = [DeviceMesh(x) for x in meshes]
    b = Batch(dms, n=n, m=m)
    b.dfdk(ks, [x[1].ptr for x in al], [x[1].ptr for x in ps], w.ptr)
    got = w.download(np.empty(3, dtype=np.complex128))
    assert np.isfinite(got).all()
    for i in range(2):
        D = oracle.assemble_taylor(meshes[i], ks[i], 1, n=n, m=m)[0]
        ref = al[i][0] @ (D @ ps[i][0])
        scale = np.abs(al[i][0]) @ (np.abs(D) @ np.abs(ps[i][0]))
        assert abs(got[i] - ref) <= 1e-12 * scale, i


@pytest.mark.parametrize("kind,physics", [("linear", "geometry"), ("quadratic", "geometry"),
                                          ("quadratic", "linear")])
@pytest.mark.parametrize("depth", [1, 2])
def test_near_field_out_of_the_middle_of_the_range(kind, physics, depth):
    """The near field of a mesh 2^200 times as large, at k / 2^200: a power of two commutes with
    every rounding, so the normals formed by division (the Jacobian is beyond the range of the
    reciprocal form) give the same F, and G 2^200 times as large, but for the order of the
    additions to an entry."""
    from bie_amd.assembly import sparse_assemble_parallel
    kw = {} if physics == "geometry" else dict(physics=physics)
    mesh = M.ellipsoid(2, axes=(1.2, 1.0, 0.7), order=kind, **kw)
    s = 2.0 ** 200
    big = M.Mesh3d(mesh.coordinates * s, mesh.topology, mesh.sources * s, mesh.physics_topology,
                   mesh.geometry_kind, mesh.physics_kind)
    F, G = sparse_assemble_parallel(mesh, 3.0, mesh.sources, depth=depth)
    Fb, Gb = sparse_assemble_parallel(big, 3.0 / s, big.sources, depth=depth)
    fs = max(np.max(np.abs(F.data)), np.max(np.abs(G.data)))
    assert np.max(np.abs(F.data - Fb.data)) <= 1e-14 * fs
    assert np.max(np.abs(G.data - Gb.data / s)) <= 1e-14 * fs


def test_near_field_of_a_far_source():
    """An explicit source whose |k| r leaves the range of the branch-free sincos, among others
    (its wave takes the other one)."""
    from bie_amd.assembly import sparse_assemble_parallel
    mesh = M.icosphere(2, "quadratic")
    pts = np.array(mesh.sources, order="F")
    F, G = sparse_assemble_parallel(mesh, 3.0, pts, depth=1)
    pts[:, 7] = (0.0, 0.0, 5e14)
    F2, G2 = sparse_assemble_parallel(mesh, 3.0, pts, depth=1)
    rows = np.repeat(np.arange(F.shape[0]), np.diff(F.indptr))
    near = rows != 7
    assert np.max(np.abs(G.data - G2.data)[near]) <= 1e-14 * np.max(np.abs(G.data))
    assert np.max(np.abs(F.data - F2.data)[near]) <= 1e-14 * np.max(np.abs(G.data))
    assert np.isfinite(F2.data).all() and 0 < np.max(np.abs(G2.data[~near])) < 1e-12


@pytest.mark.parametrize("kind", ["linear", "quadratic"])
def test_a_source_that_is_not_a_number(kind):
    """Its row is NaN, its elements take the rules the reference's comparisons leave them; the
    other rows are the oracle's.  (No bound on |k| r holds for its tile, and no second launch
    exists to leave it to.)"""
    mesh = M.icosphere(3 if kind == "linear" else 2, kind)
    src = mesh.sources.copy()
    src[:, 5] = np.nan
    mesh = M.Mesh3d(mesh.coordinates, mesh.topology, src, mesh.physics_topology,
                    mesh.geometry_kind, mesh.physics_kind)
    rows = np.arange(mesh.n_sources) != 5
    Fo, Go, Co = oracle.assemble(mesh, 3.0, n=3, m=3)
    F, G, C = assemble_parallel(mesh, 3.0, n=3, m=3)
    T = taylor_assemble(mesh, 3.0, M=0, n=3, m=3)
    for X, Xo in ((F, Fo), (G, Go), (C, Co), (T[0][:, :, 0], Fo), (T[1][:, :, 0], Go)):
        assert rel(X[rows], Xo[rows]) <= TOL
        assert np.isnan(X[5]).any()


@pytest.mark.parametrize("nm", [(22, 23), (16, 32), (40, 41), (64, 64)])
@pytest.mark.parametrize("k", [3.0, 2.0 + 0.3j])
def test_flat_adjoint_of_long_rules(nm, k):
    """Rules on both sides of what the kernel takes into LDS, and up to the longest there are.
    (The oracle's n.d of a node's own elements is rounding noise, 1e-17, which its derivative
    takes times 3 w / r^4: with Gauss points 3.5e-4 from the corner about 1e-11 of the
    functional's terms; held to 1e-9 of their sum.)"""
    from bie_amd.adjoint import assembly_vjp, source_nodes
    from dual_oracle import assemble_F_C
    mesh = M.perturb_radial(M.icosphere(1, "linear"), 0.01, 4)
    n, m = nm
    rng = np.random.default_rng(n)
    N = mesh.n_sources
    alpha, beta, p = (rng.standard_normal(N) + 1j * rng.standard_normal(N) for _ in range(3))
    g, gk = assembly_vjp(DeviceMesh(mesh), k, alpha, p, beta=beta,
                         target_node=source_nodes(mesh), n=n, m=m)
    rules = oracle.select(mesh, None)
    V = rng.standard_normal(mesh.coordinates.shape)
    for dX, dk, got in ((V, 0.0, float(np.sum(g * V))),
                        (np.zeros_like(V), 1.0, float(np.atleast_1d(gk)[0]))):
        F, C = assemble_F_C(mesh, mesh.coordinates, dX, k, dk, rules, targets=None, n=n, m=m)
        dd = np.real(alpha @ (F.d @ p) + beta @ C.d)
        scale = np.abs(alpha) @ (np.abs(F.d) @ np.abs(p)) + np.abs(beta) @ np.abs(C.d)
        assert abs(got - dd) <= 1e-9 * scale


@pytest.mark.parametrize("f,rows", [(1, None), (3, 3), (3, 5), (6, None), (10, 37), (11, 33)])
def test_flat_adjoint_of_few_elements(f, rows):
    """Waves that share their elements and divide the rows: elements short of a wave, rows short
    of a workgroup's, both sides of the sizes (2048 elements, 4 rows) where it begins."""
    from bie_amd.adjoint import assembly_vjp, source_nodes
    from dual_oracle import assemble_F_C
    mesh = M.perturb_radial(M.icosphere(f, "linear"), 0.01, 4)
    rng = np.random.default_rng(f)
    t = None if rows is None else np.asfortranarray(M.fibonacci_sphere(rows, 1.7))
    N, Mt = mesh.n_sources, rows or mesh.n_sources
    alpha, beta = (rng.standard_normal(Mt) + 1j * rng.standard_normal(Mt) for _ in range(2))
    p = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    rules = oracle.select(mesh, t)
    V = rng.standard_normal(mesh.coordinates.shape)
    dm = DeviceMesh(mesh)
    for k in (3.0, 2.0 + 0.3j):
        g, _ = assembly_vjp(dm, k, alpha, p, beta=beta, targets=t, n=3, m=3,
                            target_node=source_nodes(mesh) if t is None else None)
        F, C = assemble_F_C(mesh, mesh.coordinates, V, k, 0.0, rules, targets=t, n=3, m=3)
        dd = np.real(alpha @ (F.d @ p) + beta @ C.d)
        scale = np.abs(alpha) @ (np.abs(F.d) @ np.abs(p)) + np.abs(beta) @ np.abs(C.d)
        assert abs(float(np.sum(g * V)) - dd) <= 1e-10 * scale


@pytest.mark.parametrize("kind,physics", [("linear", "geometry"), ("quadratic", "geometry"),
                                          ("quadratic", "disctrilinear"),
                                          ("linear", "disctriconstant")])
@pytest.mark.parametrize("k", [3.0, 2.0 + 0.3j])
def test_near_field_batches_with_far_sources(kind, physics, k):
    """Explicit sources of batches of pairs: those with a source beyond the range of the
    branch-free sincos, or one that is not a number, are the other launch's; each pair is some
    launch's, once."""
    from bie_amd.assembly import sparse_assemble_parallel
    mesh = M.ellipsoid(3 if kind == "linear" else 2, axes=(1.2, 1.0, 0.7), order=kind)
    if physics != "geometry":
        mesh = M.with_discontinuous_physics(mesh, physics)
    pts = np.array(mesh.sources, order="F")
    F0, G0 = sparse_assemble_parallel(mesh, k, depth=2)
    F, G = sparse_assemble_parallel(mesh, k, pts, depth=2)
    scale = max(np.max(np.abs(F0.data)), np.max(np.abs(G0.data)))
    assert np.max(np.abs(F.data - F0.data)) <= 1e-14 * scale
    assert np.max(np.abs(G.data - G0.data)) <= 1e-14 * scale
    pts[:, 7] = (0.0, 0.0, 5e14)
    pts[:, 20] = np.nan
    F2, G2 = sparse_assemble_parallel(mesh, k, pts, depth=2)
    rows = np.repeat(np.arange(F.shape[0]), np.diff(F.indptr))
    others = (rows != 7) & (rows != 20)
    assert np.max(np.abs(F2.data - F0.data)[others]) <= 1e-14 * scale
    assert np.max(np.abs(G2.data - G0.data)[others]) <= 1e-14 * scale
    assert np.isfinite(G2.data[rows == 7]).all() and np.max(np.abs(G2.data[rows == 7])) < 1e-12
    assert np.isnan(G2.data[rows == 20]).all() and np.isnan(F2.data[rows == 20]).all()


def with_collapsed_element(kind):
    """A sphere and one more element, of no area: its first two vertices are the origin.  (The
    third is at powers of two: the tangent's terms then cancel whether they are rounded or
    fused.)"""
    mesh = M.icosphere(3 if kind == "linear" else 2, kind)
    B = np.array([0.25, 0.5, -0.125])
    extra = [0 * B, 0 * B, B] + ([0 * B, B / 2, B / 2] if kind == "quadratic" else [])
    X = np.concatenate([mesh.coordinates, np.array(extra).T], axis=1)
    T = np.concatenate([mesh.topology, mesh.n_coordinates + np.arange(len(extra))[:, None]], axis=1)
    return M.Mesh3d(X, T, X.copy(), T.copy(), mesh.geometry_kind, mesh.physics_kind)


@pytest.mark.parametrize("kind", ["linear", "quadratic"])
def test_an_element_of_no_area(kind, monkeypatch):
    """The reference divides by the Jacobian: F in its columns and C are not numbers, G is what
    the other elements leave, on every path and for every rule (mid-edge ones among them).  (But
    for the rows of its own mid-edge nodes, which lie on points of its rules: 0 / 0.)"""
    from bie_amd.assembly import Batch
    mesh = with_collapsed_element(kind)
    N, k = mesh.n_sources, 3.0
    Fo, Go, Co = oracle.assemble(mesh, k, n=3, m=2)
    hole, some = np.isnan(Fo), np.isfinite(Go)
    assert np.isnan(Co).all() and hole.any() and some[:-2].all()
    rules = oracle.select(mesh, None)[:, -1]
    assert kind == "linear" or (rules > 3).any()

    def check(F, G, C):
        assert (np.isnan(F) == hole).all() and np.isnan(C).all()
        assert rel(F[~hole], Fo[~hole]) <= TOL
        assert G is None or rel(G[some], Go[some]) <= TOL

    check(*assemble_parallel(mesh, k, n=3, m=2))
    F, _, C = assemble_parallel(mesh, k, n=3, m=2, gOn=False)
    check(F, None, C)
    F, G, C = sweep(mesh, [k, 4.0], mesh.sources, 3, 2)
    check(F[0], G[0], C)
    F, G, C = taylor_assemble(mesh, k, M=1, n=3, m=2)
    check(F[:, :, 0], G[:, :, 0], C)
    F, _, C = taylor_assemble(mesh, k, M=1, n=3, m=2, gOn=False)
    check(F[:, :, 0], None, C)
    monkeypatch.setenv("BIE_AMD_KERNEL", "atomic")
    check(*assemble_parallel(mesh, k, n=3, m=2))
    monkeypatch.delenv("BIE_AMD_KERNEL")
    b = Batch([DeviceMesh(mesh)], n=3, m=2)
    F, G, C, w = DevBuf(16 * N * N), DevBuf(16 * N * N), DevBuf(16 * N), DevBuf(16)
    b.assemble([k], [F.ptr], [G.ptr], [C.ptr])
    sync()
    check(*[x.download(np.empty(s, dtype=np.complex128, order="F"))
            for x, s in ((F, (N, N)), (G, (N, N)), (C, (N,)))])
    one = DevBuf(16 * N)
    one.upload(np.ones(N, dtype=np.complex128))
    b.dfdk([k], [one.ptr], [one.ptr], w.ptr)
    assert np.isnan(w.download(np.empty(1, dtype=np.complex128))).all()


@pytest.mark.parametrize("kind", ["linear", "quadratic"])
@pytest.mark.parametrize("far,down", [(210, 110), (365, 220)])
def test_targets_far_beyond_the_range_of_one_over_r_cubed(kind, far, down):
    """Targets at 2^far times the body's size, others near: F and C are the same, G is 2^down
    times as large, an order's derivative and the shape gradient in their units, as for the
    body and targets 2^down times smaller (every rounding is the same there, so they agree but
    for the order of operations: 1e-12.  C of a target outside a closed body is 0: it is held
    to its terms, which are F's.  (The gradient forms 1 / r^4 by itself: up to 2^250.)"""
    from bie_amd.adjoint import assembly_vjp
    body = M.perturb_radial(M.icosphere(3 if kind == "linear" else 2, kind), 0.02, 4)
    rng = np.random.default_rng(far)
    t = 1.5 * rng.standard_normal((3, 70))
    t[:, 3::5] *= 2.0 ** far
    s = 2.0 ** -down
    small = M.Mesh3d(body.coordinates * s, body.topology, body.sources * s, body.physics_topology,
                     body.geometry_kind, body.physics_kind)
    k = 2.0 ** (1 - far)
    ks = [k, 1.5 * k, 1.75 * k, 3.0 * k, 4.0 * k]
    alpha = rng.standard_normal(70) + 1j * rng.standard_normal(70)
    p = rng.standard_normal(body.n_sources) + 1j * rng.standard_normal(body.n_sources)
    far_rows = np.arange(70) % 5 == 3

    def everything(mesh, u):
        x = np.asfortranarray(t * u)
        out = {}
        for c, kk in (("", k / u), ("c", (k + 0.5j * k) / u)):
            F, G, C = assemble_parallel(mesh, kk, x, n=3, m=2)
            out.update({"F" + c: F, "G" + c: G / u, "C" + c: C})
            F, G, _ = taylor_assemble(mesh, kk, x, M=2, n=3, m=2)
            Fx = taylor_assemble(mesh, kk, x, M=2, n=3, m=2, gOn=False)[0]
            for q in range(3):
                v = u ** -q * (k if q else 1.0) ** q
                out.update({f"TF{q}" + c: F[:, :, q] * v, f"TG{q}" + c: G[:, :, q] / u * v,
                            f"TX{q}" + c: Fx[:, :, q] * v})
            for rows, name in ((far_rows, "far"), (~far_rows, "near")) if far < 250 else ():
                g, _ = assembly_vjp(DeviceMesh(mesh), kk, alpha[rows], p, targets=x[:, rows], n=3,
                                    m=2)
                out[f"V{name}{c}"] = g * u
        F, G, C = sweep(mesh, np.array(ks) / u, x, 3, 2)
        Fx = sweep(mesh, np.array(ks) / u, x, 3, 2, gOn=False)[0]
        for q in range(len(ks)):
            out.update({f"SF{q}": F[q], f"SG{q}": G[q] / u, f"SX{q}": Fx[q]})
        out["SC"] = C
        return out

    big, ref = everything(body, 1.0), everything(small, s)
    for name, x in big.items():
        y = ref[name]
        for rows in ([slice(None)] if name[0] == "V" else [far_rows, ~far_rows]):
            a, b = x[rows], y[rows]
            if name in ("C", "Cc", "SC"):
                b = np.abs(ref["F"][rows]).sum(axis=1)
                a = x[rows] - y[rows] + b
            m = np.max(np.abs(b))
            assert 0 < m < np.inf, name
            assert np.linalg.norm(a / m - b / m) <= 1e-12 * np.linalg.norm(b / m), name


@pytest.mark.parametrize("kind", ["linear", "quadratic"])
@pytest.mark.parametrize("polls", [0, 1, 2])
def test_waits_that_give_up(kind, polls, monkeypatch):
    """With so few polls that waves give up waiting for each other, an entry is not a number or
    it is right (C, which no wave waits for, is right).  Sixteen waves at once always meet: with
    no poll after the first look some entries are not numbers."""
    from bie_amd.assembly import Batch
    mesh = M.perturb_radial(M.icosphere(12 if kind == "linear" else 5, kind), 0.01, 2)
    N, k, n, m = mesh.n_sources, 3.0, 2, 2
    dms = [DeviceMesh(mesh), DeviceMesh(M.icosphere(3, kind))]
    bufs = [[DevBuf(16 * s) for s in (d.n_sources**2, d.n_sources**2, d.n_sources)] for d in dms]

    def batch():
        b = Batch(dms, n=n, m=m)
        b.assemble([k, k], *[[x[q].ptr for x in bufs] for q in range(3)])
        sync()
        return [x.download(np.empty(s, dtype=np.complex128, order="F"))
                for x, s in zip(bufs[0], ((N, N), (N, N), (N,)))]

    def sweeps(gOn):
        F, G, C = sweep(mesh, [k, 4.0, 5.0], mesh.sources, n, m, gOn=gOn)
        return F[2], (G[2] if gOn else None), C

    def orders(gOn):
        F, G, C = taylor_assemble(mesh, k, M=2, n=n, m=m, gOn=gOn)
        return F[:, :, 2], (G[:, :, 2] if gOn else None), C

    calls = [lambda: assemble_parallel(mesh, k, n=n, m=m),
             lambda: assemble_parallel(mesh, k + 0.2j, n=n, m=m), batch,
             lambda: sweeps(True), lambda: sweeps(False), lambda: orders(True),
             lambda: orders(False)]
    given_up = 0
    for number, call in enumerate(calls):
        monkeypatch.delenv("BIE_AMD_POLLS", raising=False)
        ref = call()
        monkeypatch.setenv("BIE_AMD_POLLS", str(polls))
        for x, y in zip(call(), ref):
            if y is None:
                continue
            bad = np.isnan(x)
            assert np.max(np.abs(x - y)[~bad], initial=0.0) <= 1e-12 * np.max(np.abs(y)), number
            assert y.ndim == 2 or not bad.any(), number
            given_up += int(bad.sum())
    print(f"  {given_up} entries given up", flush=True)
    assert polls > 0 or given_up > 0


@pytest.mark.parametrize("physics", ["linear", "disctriconstant", "disctrilinear"])
@pytest.mark.parametrize("nm", [(3, 2), (5, 5)])
def test_targets_that_are_not_numbers_on_quadratic_geometry(physics, nm):
    """Such a row falls to the last of six rules, of which fewer than six nodes have three: it is
    NaN, and the other rows are those of a call without it (rules staged, and read from
    memory).  C, 0 outside a closed body, is held to the solid angles it cancels from."""
    n, m = nm
    mesh = (M.icosphere(3, "quadratic", physics="linear") if physics == "linear"
            else M.with_discontinuous_physics(M.icosphere(3, "quadratic"), physics))
    t = np.asfortranarray(M.fibonacci_sphere(130, 1.6))
    t[:, 70], t[1, 5] = np.nan, np.inf
    rows = np.isfinite(t).all(axis=0)
    Fo, Go, Co = assemble_parallel(mesh, 3.0, t[:, rows], n=n, m=m)
    F, G, C = assemble_parallel(mesh, 3.0, t, n=n, m=m)
    Fs, Gs, Cs = sweep(mesh, [3.0, 4.0], t, n, m)
    for X, Xo in ((F, Fo), (G, Go), (C, Co), (Fs[0], Fo), (Gs[0], Go), (Cs, Co)):
        assert (np.max(np.abs(X[rows] - Xo)) if X.ndim == 1 else rel(X[rows], Xo)) <= TOL
        assert np.isnan(X[~rows]).all()


@pytest.mark.parametrize("kind", ["linear", "quadratic"])
@pytest.mark.parametrize("im", [0.0, 0.3])
def test_batches_beyond_the_branch_free_sincos(kind, im):
    """One instance's |k| r is beyond it: its tiles are the launch for large arguments', which
    has its own number of waves; the other's are not."""
    from bie_amd.assembly import Batch
    meshes = [M.icosphere(4, kind), M.perturb_radial(M.icosphere(3, kind), 0.02, 1)]
    ks, n, m = [1e14, 3.0 + 1j * im], 3, 2
    bufs = [[DevBuf(16 * s) for s in (x.n_sources**2, x.n_sources**2, x.n_sources)]
            for x in meshes]
    b = Batch([DeviceMesh(x) for x in meshes], n=n, m=m)
    b.assemble(ks, *[[x[q].ptr for x in bufs] for q in range(3)])
    sync()
    out = [[x.download(np.empty(x.nbytes // 16, dtype=np.complex128)) for x in y] for y in bufs]
    for x, y in zip(out[1], oracle.assemble(meshes[1], ks[1], n=n, m=m)):
        assert rel(x.reshape(y.shape, order="F"), y) <= TOL
    # (phases of 1e14 keep few digits: the single-mesh call takes the same steps)
    for x, y in zip(out[0], assemble_parallel(meshes[0], ks[0], n=n, m=m)):
        assert np.isfinite(x).all() and rel(x.reshape(y.shape, order="F"), y) <= TOL
    assert rel(out[0][2], oracle.assemble(meshes[0], 1.0, n=n, m=m)[2]) <= TOL
