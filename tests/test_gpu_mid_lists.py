"""Mid-edge pairs (split rules 4-6) beyond what a tile queues in LDS (2048) and beyond what a
call's list holds (a sixteenth of all pairs and 2^18): those tiles' pairs are selected again.
Bodies with dimpled edges, seen from about their centre, have them in any number."""
import numpy as np
import pytest

import oracle
from bie_amd import mesh as M
from bie_amd.assembly import Batch, DeviceMesh, assemble_parallel
from bie_amd.taylor import taylor_assemble
from gpu_helpers import TOL, DevBuf, rel, sync
from test_gpu_stream import sweep

pytestmark = pytest.mark.gpu

QUEUE, LIST = 2048, 1 << 18


def dimpled(f, share, seed=1):
    """A quadratic sphere with the given share of its edge nodes a little further in."""
    mesh = M.icosphere(f, "quadratic")
    edge = np.unique(mesh.topology[3:])
    edge = edge[np.random.default_rng(seed).random(edge.size) < share]
    X = mesh.coordinates.copy()
    X[:, edge] *= 0.97
    return M.Mesh3d(X, mesh.topology, X.copy(), mesh.topology.copy(), 6, 6)


def about_the_centre(n):
    return np.asfortranarray(1e-3 * np.random.default_rng(n).standard_normal((3, n)))


def check(got, ref):
    for x, y in zip(got, ref):
        assert rel(x, y) <= TOL


@pytest.mark.parametrize("share", [0.26, 1.0])
def test_more_pairs_than_the_list_holds(share):
    """Two blocks of rows, so that tiles have few elements: at the smaller share most queue their
    pairs (some 1500 each) until the list is full.  The sweep's and the derivatives' tiles have
    many elements and queue too much at either share."""
    mesh, t = dimpled(16, share), about_the_centre(128)
    mids = int((oracle.select(mesh, t) > 3).sum())
    pairs = 128 * mesh.n_elements
    assert mids > pairs // 16 + LIST
    for k in (2.0, 2.0 + 0.3j):
        check(assemble_parallel(mesh, k, t, n=3, m=2), oracle.assemble(mesh, k, targets=t, n=3, m=2))
    ref = oracle.assemble(mesh, 2.0, targets=t, n=3, m=2)
    F, G, C = sweep(mesh, [2.0, 3.0], t, 3, 2)
    check((F[0], G[0], C), ref)
    F, G, C = taylor_assemble(mesh, 2.0, t, M=1, n=3, m=2)
    check((F[:, :, 0], G[:, :, 0], C), ref)
    F1, G1 = oracle.assemble_taylor(mesh, 2.0, 1, targets=t, n=3, m=2)
    check((F[:, :, 1], G[:, :, 1]), (F1, G1))


@pytest.mark.parametrize("graph", [False, True])
def test_more_pairs_than_a_batch_tile_queues(graph):
    """A body within another one, in one mesh and one segment (or so): the inner one's rows see
    the outer one's dimples."""
    outer, inner = dimpled(4, 1.0), M.icosphere(4, "quadratic", radius=1e-2)
    X = np.concatenate([outer.coordinates, inner.coordinates], axis=1)
    T = np.concatenate([outer.topology, inner.topology + outer.n_coordinates], axis=1)
    mesh = M.Mesh3d(X, T, X.copy(), T.copy(), 6, 6)
    N, k = mesh.n_sources, 2.0
    other = M.icosphere(2, "quadratic")
    dms = [DeviceMesh(mesh), DeviceMesh(other)]
    b = Batch(dms, n=3, m=2)
    b.configure(1 << 20, 0, 0)
    bufs = [[DevBuf(16 * s) for s in (d.n_sources**2, d.n_sources**2, d.n_sources)] for d in dms]
    args = ([k, 3.0], *[[x[q].ptr for x in bufs] for q in range(3)])
    b.assemble(*args)
    blocks = -(-N // 64)
    segments = (b.info()["n_tiles"] - -(-other.n_sources // 64)) / blocks
    rules = oracle.select(mesh, None)[64 * (blocks - 2):64 * (blocks - 1)]
    assert (rules > 3).sum() > QUEUE * segments
    g = b.graph(*args) if graph else None
    for _ in range(3 if graph else 1):
        if graph:
            for x in bufs[0]:
                x.upload(np.full(x.nbytes // 8, np.nan))
            g.launch()
        sync()
        F, G, C = [x.download(np.empty(s, dtype=np.complex128, order="F"))
                   for x, s in zip(bufs[0], ((N, N), (N, N), (N,)))]
        check((F, G, C), oracle.assemble(mesh, k, n=3, m=2))
