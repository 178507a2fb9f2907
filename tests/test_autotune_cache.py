"""The erosion autotuner's cache entries (CPU only): lookups by step count,
entries written before plans had a step count, and the merge that keeps a
faster tuning of step counts a later search did not cover."""
import json

from nixis_amd import autotune


def _write(tmp_path, entries):
    path = str(tmp_path / "tune.json")
    with open(path, "w") as f:
        json.dump(entries, f)
    return path


def test_lookup_by_step_count(tmp_path):
    V = 10_000_002
    key = autotune.erosion_key(V)
    path = _write(tmp_path, {key: {"chunk": 896, "variant": 0, "graph_chunk": 32, "steps": 4,
                                   "us_per_step": 92.0,
                                   "steps2": {"chunk": 768, "variant": 5, "graph_chunk": 32,
                                              "steps": 2, "us_per_step": 117.0}}})
    assert autotune.lookup_erosion(V, path=path) == autotune.ErosionTuning(896, 0, 32, 4)
    assert autotune.lookup_erosion(V, path=path, steps=4) == autotune.ErosionTuning(896, 0, 32, 4)
    assert autotune.lookup_erosion(V, path=path, steps=2) == autotune.ErosionTuning(768, 5, 32, 2)
    assert autotune.lookup_erosion(V // 4, path=path) is None
    kw = autotune.lookup_erosion(V, path=path).graph_kwargs()
    assert kw == {"chunk": 896, "variant": 0, "graph_chunk": 32, "steps": 4}


def test_entry_without_step_count_is_two_step(tmp_path):
    V = 2_560_002
    path = _write(tmp_path, {autotune.erosion_key(V): {"chunk": 768, "variant": 0,
                                                       "graph_chunk": 64, "us_per_step": 30.0}})
    assert autotune.lookup_erosion(V, path=path) == autotune.ErosionTuning(768, 0, 64, 2)
    assert autotune.lookup_erosion(V, path=path, steps=2).steps == 2
    assert autotune.lookup_erosion(V, path=path, steps=4) is None


def test_merge_keeps_faster_unsearched_step_count():
    four = {"chunk": 896, "variant": 0, "graph_chunk": 32, "steps": 4, "us_per_step": 92.0}
    two = {"chunk": 768, "variant": 5, "graph_chunk": 32, "steps": 2, "us_per_step": 117.0}
    # a two-step-only search (the multi-planet form) keeps the faster four-step entry first
    m = autotune.merge_erosion_entry(four, two, {2: None})
    assert m["steps"] == 4 and m["chunk"] == 896 and m["steps2"] == two
    # a search that covered four-step plans replaces the entry
    assert autotune.merge_erosion_entry(four, two, {4: None, 2: None}) == two
    # a slower cached entry of another step count is replaced
    slow = dict(four, us_per_step=130.0)
    assert autotune.merge_erosion_entry(slow, two, {2: None}) == two
    assert autotune.merge_erosion_entry(None, two, {2: None}) == two


def test_mesh_cache_cuts_plans_as_tuned(monkeypatch):
    """MeshCache.graph takes a tuning's chunk as it was timed, 0 (the library's
    default) too, as MeshCache.tune_erosion does; without a tuning plans start
    from full tiles."""
    from nixis_amd import batch
    made = []
    meshes = batch.MeshCache(device="cpu")
    monkeypatch.setattr(meshes, "_build_graph", lambda d, **kw: made.append((d, kw.get("chunk"))))
    monkeypatch.setattr(autotune, "tune_erosion", lambda make, **kw: (autotune.ErosionTuning(0, 0, 32, 4), []))
    monkeypatch.setattr(autotune, "lookup_erosion", lambda V: None)
    meshes.graph(32)
    meshes.graph(64, tuning=autotune.ErosionTuning(0, 0, 32, 4))
    meshes.graph(66, tuning=autotune.ErosionTuning(640, 0, 32, 2))
    meshes.tune_erosion(68)
    monkeypatch.setattr(autotune, "lookup_erosion", lambda V: autotune.ErosionTuning(0, 0, 32, 4))
    meshes.graph(70)
    assert made == [(32, batch.BATCH_CHUNK), (64, 0), (66, 640), (68, 0), (70, 0)]


def test_tuner_times_graph_chunks_without_a_plan_only(monkeypatch, tmp_path):
    """Runs over a plan replay no graphs: the tuner runs nothing for the graph
    chunks and keeps the default, where every one would have measured noise.
    Without a plan it times each."""
    from types import SimpleNamespace

    import torch
    from nixis_amd import erosion
    runs = []

    class State:
        def __init__(self, V, device=None):
            pass

        def load(self, heights):
            pass

        def run(self, graph, iters, rain):
            runs.append(graph.graph_chunk)

    class Event:
        def __init__(self, enable_timing=False):
            pass

        def record(self, stream):
            self.at = len(runs)

        def synchronize(self):
            pass

        def elapsed_time(self, other):      # a later run looks a little faster
            return 1.0 / other.at

    monkeypatch.setattr(erosion, "ErosionState", State)
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: None)
    for plan in (object(), None):
        del runs[:]
        best, table = autotune.tune_erosion(
            lambda c, k: SimpleNamespace(V=12, device="cpu", plan=plan, steps=k, chunk=c),
            heights=torch.zeros(12), path=str(tmp_path / "t.json"), graph_chunks=(8, 16, 32, 64))
        assert {k for *_, k in table} == {8, 16, 32, 64}
        if plan is None:
            assert set(runs) == {8, 16, 32, 64} and best.graph_chunk == 64
        else:
            assert set(runs) == {32} and best.graph_chunk == 32
