"""A graph's tile plan is complete when ErosionGraph.from_device returns, so a
run on any stream may read it.

On the CPU the library is replaced by one that records its calls: the planner's
stream is waited for after the last call that writes the image, with a stream
of the caller's and without one.  On the GPU a graph made on the current stream
runs on another one at once and gives the oracle's fields.
"""
import contextlib
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from nixis_amd import _lib, erosion, util


@pytest.mark.parametrize("given", [False, True])
def test_planner_waits_for_the_image(monkeypatch, given):
    calls = []
    stream = object() if given else None

    class Library:
        @staticmethod
        def nx_tile_plan_device_workspace_bytes(V, chunk):
            return 256

        @staticmethod
        def nx_tile_plan_build_device(ctx, col, elen, V, chunk, ws, out, cap, plan, s):
            plan._obj.bytes = 512
            calls.append(("write" if out is not None else "size", s))
            return _lib.NX_OK

    monkeypatch.setattr(_lib, "lib", lambda: Library)
    monkeypatch.setattr(_lib, "stream_ptr", lambda s=None: s)
    monkeypatch.setattr(_lib.Context, "get", lambda device=None: SimpleNamespace(
        handle=None, sync_check=lambda s=None: calls.append(("wait", s))))
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    g = erosion.ErosionGraph.__new__(erosion.ErosionGraph)
    g.V, g.chunk, g.device = 12, 0, torch.device("cpu")
    g.col = torch.zeros((6, 12), dtype=torch.int32)
    g.elen = torch.zeros((6, 12), dtype=torch.float64)
    g._set_plan = lambda plan, blob: calls.append(("use", None))
    assert g._build_plan_device(stream)
    assert calls == [("size", stream), ("write", stream), ("wait", stream), ("use", None)]


def test_no_memory_for_the_planner(monkeypatch):
    """Without device memory for the planner's workspace the plan is left to the
    host planner, which needs none."""
    def empty(*args, **kw):
        raise torch.OutOfMemoryError("full")

    monkeypatch.setattr(_lib, "lib", lambda: SimpleNamespace(
        nx_tile_plan_device_workspace_bytes=lambda V, chunk: 256))
    monkeypatch.setattr(_lib.Context, "get", lambda device=None: SimpleNamespace(handle=None))
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    monkeypatch.setattr(torch, "empty", empty)
    g = erosion.ErosionGraph.__new__(erosion.ErosionGraph)
    g.V, g.chunk, g.device = 12, 0, torch.device("cpu")
    assert g._build_plan_device(None) is False


@pytest.mark.gpu
def test_run_on_another_stream_after_the_build(oracle):
    """The state is loaded and run on a second stream, which waits for nothing
    of the first, as soon as the graph is built there."""
    pts, nb = util.icosphere_with_neighbors_device(64)
    V = pts.shape[0]
    h = np.random.default_rng(5).uniform(-9000, 9000, V)
    href = h.copy()
    oracle.erode_terrain3(pts.cpu().numpy(), nb.cpu().numpy(), href, 9, 1.0)
    side = _lib.side_stream()
    st = erosion.ErosionState(V)
    dh = torch.from_numpy(h[util.sfc_order(pts.cpu().numpy())]).cuda()
    out = torch.empty_like(dh)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g = erosion.ErosionGraph.from_device(pts, nb)
        st.load(dh, stream=side)
        st.run(g, 9, 1.0, stream=side)
        st.store(out, stream=side)
        st.ctx.sync_check(side)
        assert g.steps == 4 and g.plan is not None
        assert (g.unpermute(out.cpu().numpy()) == href).all()
