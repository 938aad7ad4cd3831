"""Autotuner cache on the host (no GPU): versioned JSON, atomic store,
keys that separate architectures, geometries and flags."""

import json

from nlse_amd import autotune


def test_cache_roundtrip(tmp_path, monkeypatch):
    path = tmp_path / "tune.json"
    monkeypatch.setenv("NLSE_AMD_TUNE_CACHE", str(path))
    assert autotune.load() == {}
    autotune.store("plan|gfx950|a", {"col_width": 8, "graph_chunk": 16})
    autotune.store("plan|gfx950|b", {"col_width": 4, "graph_chunk": 0})
    assert autotune.lookup("plan|gfx950|a")["col_width"] == 8
    assert autotune.lookup("plan|gfx950|b")["graph_chunk"] == 0
    data = json.loads(path.read_text())
    assert data["version"] == autotune.VERSION and len(data["entries"]) == 2
    # another version of the cache format is ignored, not misread
    path.write_text(json.dumps({"version": autotune.VERSION + 1, "entries": {"x": {}}}))
    assert autotune.load() == {}
    path.write_text("not json")
    assert autotune.load() == {}


def test_keys_distinguish_shapes_and_flags(monkeypatch):
    monkeypatch.setattr(autotune, "arch", lambda: "gfx950")
    geo = dict(ndim=2, ny=2048, nx=2048, nt=1, items=1, ncomp=1)
    k0 = autotune.plan_key(geo, False, None)
    assert k0 != autotune.plan_key(geo, True, None)
    assert k0 != autotune.plan_key(geo, False, (25, 25))
    assert k0 != autotune.plan_key(dict(geo, ny=1024), False, None)
    assert k0 != autotune.plan_key(dict(geo, ncomp=2), False, None)
    assert autotune.batch_key([(256, 256), (512, 512)]) == autotune.batch_key([(512, 512), (256, 256)])
    assert autotune.batch_key([(256, 256)]) != autotune.batch_key([(256, 256), (256, 256)])


def test_enabled_flag(monkeypatch):
    monkeypatch.delenv("NLSE_AMD_AUTOTUNE", raising=False)
    assert not autotune.enabled()
    monkeypatch.setenv("NLSE_AMD_AUTOTUNE", "1")
    assert autotune.enabled()


class _Batch:
    """A batch engine whose step takes the time given for its grid."""

    def __init__(self, times):
        self.times, self.grid, self.single, self.seen = times, None, False, []

    def set_grid(self, rb, cb):
        assert rb >= 1 and cb >= 1  # refused by the library
        self.grid = (rb, cb)

    def default_grid(self):
        self.grid = autotune.DEFAULT_GRID

    def set_single_launch(self, on):
        self.single = on

    def run(self, A, n, precision):
        pass


def _tune(monkeypatch, times):
    eng = _Batch(times)

    def time_run(run, A0, nsteps, reps=2):
        eng.seen.append((eng.single, eng.grid))
        return times.get(eng.grid, 2.0) + (0.5 if eng.single else 0.0)

    monkeypatch.setattr(autotune, "_time_run", time_run)
    return eng, autotune.tune_batch(eng, None, 0)


def test_batch_tuner_times_the_default_grid(monkeypatch):
    """The engine's own grid is a candidate, in both launch structures, and is
    what the engine and the cache entry hold when it is the fastest."""
    eng, res = _tune(monkeypatch, {autotune.DEFAULT_GRID: 1.0})
    assert {(False, autotune.DEFAULT_GRID), (True, autotune.DEFAULT_GRID)} <= set(eng.seen)
    assert eng.grid == autotune.DEFAULT_GRID and eng.single is False
    assert (res["row_blocks_per_cu"], res["col_blocks_per_cu"]) == autotune.DEFAULT_GRID
    fresh = _Batch({})
    autotune.apply_grid(fresh, [res["row_blocks_per_cu"], res["col_blocks_per_cu"]])
    assert fresh.grid == autotune.DEFAULT_GRID
    eng, res = _tune(monkeypatch, {(8, 4): 1.0})
    assert eng.grid == (8, 4) and (res["row_blocks_per_cu"], res["col_blocks_per_cu"]) == (8, 4)


def test_entries_of_earlier_kernels_are_not_read(tmp_path, monkeypatch):
    """Choices timed before the small-field plans, the 4-column tiles and the
    block-per-pass grids (version 2) would override those defaults."""
    path = tmp_path / "tune.json"
    monkeypatch.setenv("NLSE_AMD_TUNE_CACHE", str(path))
    path.write_text(json.dumps({"version": 2, "entries": {"plan|gfx950|a": {"col_width": 8, "row_points": 16,
                                                                             "graph_chunk": 16}}}))
    assert autotune.lookup("plan|gfx950|a") is None
    autotune.store("plan|gfx950|b", {"col_width": 4, "graph_chunk": 0})
    assert set(autotune.load()) == {"plan|gfx950|b"}
    monkeypatch.delenv("NLSE_AMD_TUNE_CACHE")
    assert "tune-v2" not in autotune.cache_path()
