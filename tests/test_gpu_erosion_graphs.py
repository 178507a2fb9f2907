"""Captured hipGraphs of erosion steps, which runs without a tile plan replay
(runs over a plan launch eagerly): replays equal eager launches and the oracle
bit for bit, with other work in between, over runs that continue one another,
and where another mesh's tables lie at a freed mesh's addresses."""
import numpy as np
import pytest
import torch

from nixis_amd import _lib, erosion, util

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _graph_chunk():
    yield
    _lib.Context.get().set_graph_chunk(32)


def _mesh(d, seed=3):
    pts, nb = util.icosphere_with_neighbors(d)
    return pts, nb, np.random.default_rng(seed).uniform(-9000, 9000, pts.shape[0])


def _fields(g, st):
    out = [torch.empty(g.V, dtype=torch.float64, device="cuda") for _ in range(3)]
    st.store(*out)
    st.ctx.sync_check()
    return [g.unpermute(t.cpu().numpy()) for t in out]


@pytest.mark.parametrize("rule", [3, 4])
@pytest.mark.parametrize("chunk,iters", [(16, 100), (7, 29), (2, 5), (32, 33)])
def test_replays_match_eager(chunk, iters, rule):
    """Full chunks and remainders of 0, 1 and more steps, replayed from the same
    workspace three times with eager work and synchronisations in between."""
    pts, nb, h = _mesh(20)
    g = erosion.ErosionGraph(pts, nb, tiled=False)
    assert g.plan is None
    ctx = _lib.Context.get(g.device)
    dh = torch.from_numpy(g.permute(h)).cuda()
    st = erosion.ErosionState(g.V)
    ctx.set_graph_chunk(0)
    st.load(dh)
    st.run(g, iters, 1.0, rule=rule)
    eager = _fields(g, st)
    ctx.set_graph_chunk(chunk)
    for rep in range(3):
        st.load(dh)
        st.run(g, iters, 1.0, rule=rule)
        util.rescale_device(dh, -1, 1)
        torch.cuda.synchronize()
        assert all((a == b).all() for a, b in zip(_fields(g, st), eager)), f"replay {rep} differs"


def test_runs_continue_one_another(oracle):
    """Runs of odd and even lengths, captured and eager, over a plan and without
    one, each from where the last one left the workspace."""
    pts, nb, h = _mesh(24)
    graphs = [erosion.ErosionGraph(pts, nb, tiled=False), erosion.ErosionGraph(pts, nb)]
    ctx = _lib.Context.get(graphs[0].device)
    st = erosion.ErosionState(graphs[0].V)
    st.load(torch.from_numpy(graphs[0].permute(h)).cuda())
    steps = 0
    for chunk, tiled, iters in ((8, 0, 17), (0, 1, 5), (8, 0, 8), (8, 1, 4), (0, 0, 3), (8, 0, 1),
                                (3, 0, 10), (8, 1, 2), (8, 0, 17)):
        ctx.set_graph_chunk(chunk)
        st.run(graphs[tiled], iters, 1.0)
        steps += iters
    href = h.copy()
    oracle.erode_terrain3(pts, nb, href, steps, 1.0)
    assert (_fields(graphs[0], st)[0] == href).all()


def test_meshes_of_one_size_back_to_back(oracle):
    """Two meshes with the same vertex count and other edge lengths and order,
    eroded in turn with captured graphs, tables and state freed before the next
    are made: a graph captured for one reads the tables that now lie at its
    addresses, or is not used."""
    pts, nb, h = _mesh(24)
    jit = pts + np.random.default_rng(5).normal(scale=0.02, size=pts.shape)
    jit /= np.linalg.norm(jit, axis=1, keepdims=True)
    at = []
    for k, p in enumerate((pts, jit, pts, jit)):
        g = erosion.ErosionGraph(p, nb, tiled=False)
        assert g.plan is None
        st = erosion.ErosionState(g.V)
        st.load(torch.from_numpy(g.permute(h)).cuda())
        st.run(g, 70, 1.0)                 # 32 + 32 + 6 steps, each a cached graph
        got = _fields(g, st)[0]
        at.append((st.buf.data_ptr(), g.col.data_ptr(), g.elen.data_ptr()))
        del g, st
        torch.cuda.synchronize()
        href = h.copy()
        oracle.erode_terrain3(p, nb, href, 70, 1.0)
        assert (got == href).all(), f"run {k} differs from the oracle"
    assert len(set(at)) < len(at)          # addresses, and with them graphs, were reused
