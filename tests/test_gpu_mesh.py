"""Device mesh generation equals the host generator and table builders bit
for bit (util.py:17-50 stand-in, build_adjacency util.py:590-613,
sort_adjacency util.py:638-662), including the reference's append order
for a triangle list in an arbitrary order."""
import ctypes

import numpy as np
import pytest
import torch

from nixis_amd import _lib, erosion, util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [1, 2, 3, 8, 57, 400])
def test_device_icosphere_equals_host(d):
    pts, cells = util.create_mesh(d)
    dp, dc = util.create_mesh_device(d)
    assert (dp.cpu().numpy() == pts).all()
    assert (dc.cpu().numpy() == cells).all()


@pytest.mark.parametrize("d", [1, 5, 64])
def test_device_adjacency_equals_host(d):
    pts, cells = util.create_mesh(d)
    adj = util.build_adjacency(cells)
    dadj = util.build_adjacency_device(torch.from_numpy(cells).cuda(), pts.shape[0])
    assert (dadj.cpu().numpy() == adj).all()
    util.sort_adjacency(adj)
    sadj = util.sort_adjacency_device(dadj)
    assert (sadj.cpu().numpy() == adj).all()


def test_device_adjacency_keeps_triangle_order(oracle):
    """Rows follow the triangle order of the input, whatever it is."""
    pts, cells = util.create_mesh(9)
    perm = np.random.default_rng(3).permutation(cells.shape[0])
    shuffled = np.ascontiguousarray(cells[perm])
    ref = oracle.build_adjacency(shuffled, pts.shape[0])
    dadj = util.build_adjacency_device(torch.from_numpy(shuffled).cuda(), pts.shape[0])
    assert (dadj.cpu().numpy() == ref).all()
    oracle.sort_adjacency(ref)
    assert (util.sort_adjacency_device(dadj).cpu().numpy() == ref).all()


def test_device_adjacency_rejects_degree_over_six():
    cells = np.array([[0, k, k + 1] for k in range(1, 9)], dtype=np.int32)   # fan of 8
    with pytest.raises(_lib.NixisArgError):
        util.build_adjacency_device(torch.from_numpy(cells).cuda(), 12)


def test_device_mesh_at_scale():
    """d=2000 (40,000,002 vertices): points, triangles and sorted table."""
    d = 2000
    pts, nb = util.icosphere_with_neighbors(d)
    dp, dn = util.icosphere_with_neighbors_device(d)
    assert (dp.cpu().numpy() == pts).all()
    assert (dn.cpu().numpy() == nb).all()


@pytest.mark.parametrize("d", [3, 40, 300])
def test_device_sfc_order_and_layout_equal_host(d):
    from nixis_amd import erosion
    pts, nb = util.icosphere_with_neighbors(d)
    dp, dn = util.icosphere_with_neighbors_device(d)
    order = util.sfc_order(pts)
    dorder = util.sfc_order_device(dp)
    assert (dorder.cpu().numpy() == order).all()
    g_host = erosion.ErosionGraph(pts, nb)
    g_dev = erosion.ErosionGraph.from_device(dp, dn)
    assert (g_dev.order == g_host.order).all()
    assert (g_dev.col.cpu().numpy() == g_host.col.cpu().numpy()).all()
    assert (g_dev.elen.cpu().numpy() == g_host.elen.cpu().numpy()).all()
    assert (g_dev.plan is None) == (g_host.plan is None)
    if g_host.plan is not None:
        assert (g_dev._plan_blob.cpu().numpy() == g_host._plan_blob.cpu().numpy()).all()


def test_mesh_cache_device_equals_host_path():
    from nixis_amd import batch
    job = batch.Job(d=48, seed=5, n_octaves=6, erosion_iters=17, rain=1.0)
    outs = []
    for on_device in (True, False):
        meshes = batch.MeshCache(on_device=on_device)
        run = batch.PlanetRun(job, meshes)
        batch.BatchRunner().run([run])
        outs.append(run.heights())
        assert (meshes.verts(48).cpu().numpy() ==
                util.create_points(48)[meshes.order(48)]).all()
    assert (outs[0] == outs[1]).all()


@pytest.mark.parametrize("d,chunk", [(1, 0), (2, 0), (11, 0), (17, 300), (64, 0), (64, 97), (90, 1400),
                                     (120, 2048), (200, 700)])
def test_device_tile_plan_equals_host(d, chunk):
    """The four-step plan made on the device against the host planner's, byte
    for byte: one tile and many, chunks that are halved and a short last one."""
    dp, dn = util.icosphere_with_neighbors_device(d)
    print("d", d, "chunk", chunk, flush=True)
    g = erosion.ErosionGraph.from_device(dp, dn, chunk=chunk)
    col, elen, L = g.col.cpu().numpy(), g.elen.cpu().numpy(), _lib.lib()
    q = _lib.NxTilePlan()
    rc = L.nx_tile_plan_build_chunk(_lib.ptr(col), _lib.ptr(elen), g.V, 4, chunk, None, 0,
                                    ctypes.byref(q))
    if rc == _lib.NX_ERANGE:
        assert g.plan is None or g.steps == 2
        return
    assert rc == _lib.NX_OK and g.steps == 4
    img = np.zeros(q.bytes, np.uint8)
    _lib.check(L.nx_tile_plan_build_chunk(_lib.ptr(col), _lib.ptr(elen), g.V, 4, chunk,
                                          _lib.ptr(img), q.bytes, ctypes.byref(q)))
    for name, _ in _lib.NxTilePlan._fields_:
        assert name == "blob" or getattr(g.plan, name) == getattr(q, name), name
    assert np.array_equal(g._plan_blob.cpu().numpy(), img)
    assert g.stream_bytes_per_launch == erosion._plan_stream_bytes(q, img, g.V)


def test_device_tile_plan_refusals():
    """Tables the device planner leaves to the host: without locality, not
    symmetric, an index out of range."""
    _, nb = util.icosphere_with_neighbors(60)
    V = nb.shape[0]
    base = np.where(nb >= 0, nb, np.arange(V)[:, None]).T.astype(np.int32)
    rng = np.random.default_rng(3)
    p = rng.permutation(V).astype(np.int32)
    inv = np.argsort(p)
    one_way = base.copy()
    one_way[2, 5] = (base[2, 5] + V // 2) % V
    outside = base.copy()
    outside[1, V - 1] = V
    for name, col in (("shuffled", inv[base[:, p]].astype(np.int32)), ("one way", one_way),
                      ("outside", outside)):
        print(name, flush=True)
        c = torch.from_numpy(np.ascontiguousarray(col)).cuda()
        e = torch.zeros((6, V), dtype=torch.float64, device="cuda")
        L = _lib.lib()
        ws = torch.empty(L.nx_tile_plan_device_workspace_bytes(V, 0), dtype=torch.uint8, device="cuda")
        q = _lib.NxTilePlan()
        rc = L.nx_tile_plan_build_device(_lib.Context.get(c.device).handle, _lib.ptr(c), _lib.ptr(e),
                                         V, 0, _lib.ptr(ws), None, 0, ctypes.byref(q),
                                         _lib.stream_ptr())
        assert rc == _lib.NX_ERANGE
