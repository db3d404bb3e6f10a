"""Schedules and lists that several users of one mesh hold side by side: what one of them asks
for leaves the others' alone."""
import numpy as np
import pytest

from bie_amd import mesh as M
from bie_amd.assembly import Batch, DeviceMesh
from gpu_helpers import DevBuf, rel, sync

pytestmark = pytest.mark.gpu


def outputs(meshes):
    return [(DevBuf(16 * x.n_sources**2), DevBuf(16 * x.n_sources**2), DevBuf(16 * x.n_sources))
            for x in meshes]


def pointers(bufs):
    return [[b[i].ptr for b in bufs] for i in range(3)]


def values(bufs):
    sync()
    return [[x.download(np.empty(x.nbytes // 16, dtype=np.complex128)) for x in b] for b in bufs]


def spoil(bufs):
    for b in bufs:
        for x in b:
            x.upload(np.full(x.nbytes // 8, np.nan))


@pytest.mark.parametrize("kind", ["linear", "quadratic"])
def test_a_batch_graph_and_another_batch_on_its_mesh(kind):
    """Unconfigured batches that share a mesh fit different segments to it.  A graph of one is
    replayed between eager calls of the others, and every result stays the first one's."""
    small, large = (8, 16) if kind == "linear" else (4, 8)
    meshes = [M.icosphere(small, kind), M.ellipsoid(large, (1.0, 0.7, 1.3), kind)]
    dms = [DeviceMesh(x) for x in meshes]
    a, b, c = Batch(dms[:1], n=3, m=2), Batch(dms, n=3, m=2), Batch(dms[1:], n=3, m=2)
    ka, kb = [2.0], [3.0, 1.5]
    ba, bb, bc = outputs(meshes[:1]), outputs(meshes), outputs(meshes[1:])
    a.assemble(ka, *pointers(ba))
    ref_a = values(ba)
    g = a.graph(ka, *pointers(ba))
    b.assemble(kb, *pointers(bb))
    ref_b = values(bb)
    c.assemble(kb[1:], *pointers(bc))
    # the case that is meant: the batches cut the shared meshes into different segments
    assert a.info()["n_tiles"] + c.info()["n_tiles"] != b.info()["n_tiles"]
    gb = b.graph(kb, *pointers(bb))
    for _ in range(3):
        spoil(ba), spoil(bb), spoil(bc)
        sync()
        g.launch()
        gb.launch()
        c.assemble(kb[1:], *pointers(bc))
        for got, ref in zip(values(ba) + values(bb) + values(bc), ref_a + ref_b + ref_b[1:]):
            for x, y in zip(got, ref):
                assert rel(x, y) < 1e-14
        b.assemble(kb, *pointers(bb))
        a.assemble([4.0], *pointers(ba))
    # schedules are let go of with the last that holds them
    b.configure(32, 0, 0)
    b.assemble(kb, *pointers(bb))
    b.close()
    spoil(ba), spoil(bb)
    sync()
    g.launch()
    gb.launch()
    for got, ref in zip(values(ba) + values(bb), ref_a + ref_b):
        for x, y in zip(got, ref):
            assert rel(x, y) < 1e-14
    g.close()
    gb.close()
    a.close()
    c.close()


def test_a_captured_assembly_and_calls_of_other_rows():
    """A caller's own capture of the collocation assembly, replayed between calls with other
    rows (some of them more than the mesh's) and without G, whose pair lists are larger: they
    are not the captured call's."""
    import torch
    mesh = M.icosphere(4, "quadratic")
    N, n, m, k = mesh.n_sources, 3, 2, 3.0
    dm = DeviceMesh(mesh)
    F, G, C = outputs([mesh])[0]
    more = 6 * N
    t = DevBuf(24 * more)
    t.upload(1.5 * np.random.default_rng(1).standard_normal((more, 3)))
    Ff, Gf, Cf = DevBuf(16 * more * N), DevBuf(16 * more * N), DevBuf(16 * more)
    dm.assemble(k, F.ptr, G.ptr, C.ptr, n=n, m=m)
    ref = values([(F, G, C)])[0]
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        dm.assemble(k, F.ptr, G.ptr, C.ptr, n=n, m=m, stream=stream.cuda_stream)
    for rows in (more, 70, N + 1):
        dm.assemble(k, Ff.ptr, Gf.ptr, Cf.ptr, n=n, m=m, targets_ptr=t.ptr, n_targets=rows)
        dm.assemble(k, Ff.ptr, Gf.ptr, Cf.ptr, n=n, m=m, gOn=False)
        spoil([(F, G, C)])
        sync()
        graph.replay()
        torch.cuda.synchronize()
        for x, y in zip(values([(F, G, C)])[0], ref):
            assert rel(x, y) < 1e-14


@pytest.mark.parametrize("kind", ["linear", "quadratic"])
def test_a_sweep_graph_and_sweeps_of_other_lengths(kind):
    """Sweeps of few and of many wavenumbers cut a small mesh into different segments, more kinds
    of them than a mesh keeps: a graph's replays stay right beside them, and so do they."""
    import oracle
    mesh = M.icosphere(4 if kind == "linear" else 2, kind)
    N, n, m, most = mesh.n_sources, 3, 2, 44
    dm = DeviceMesh(mesh)
    ks = np.linspace(0.5, 6.0, most)
    kb = DevBuf(8 * most)
    kb.upload(ks)
    F, G, C = DevBuf(16 * N * N * most), DevBuf(16 * N * N * most), DevBuf(16 * N)
    Fg, Gg, Cg = DevBuf(16 * N * N * 40), DevBuf(16 * N * N * 40), DevBuf(16 * N)
    g = dm.sweep_graph(kb.ptr, 40, Fg.ptr, Gg.ptr, N * N, Cg.ptr, n=n, m=m)
    ref = {q: oracle.assemble(mesh, ks[q], n=n, m=m) for q in (0, 2, 33, 39)}

    def check(bufs, nk):
        for q, (Fo, Go, Co) in ref.items():
            if q < nk:
                for x, y in zip(bufs[:2], (Fo, Go)):
                    v = x.download(np.empty(nk * N * N, dtype=np.complex128)).reshape(nk, N, N)
                    assert rel(v[q].T, y) < 1e-12
        assert rel(bufs[2].download(np.empty(N, dtype=np.complex128)), ref[0][2]) < 1e-12

    for nk in (1, 3, 34, 35, 36, 37, 38, 39, 41, 42, 43, 44):
        for gOn in (False, True):
            dm.assemble_sweep(kb.ptr, nk, F.ptr, G.ptr, N * N, C.ptr, n=n, m=m, gOn=gOn)
        sync()
        check((F, G, C), nk)
        if nk in (3, 38, 44):
            spoil([(Fg, Gg, Cg)])
            sync()
            g.launch()
            sync()
            check((Fg, Gg, Cg), 40)
    g.close()
