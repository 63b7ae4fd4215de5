"""Launch-shape parameters: the C ABI's names, ranges and per-box override,
and the shipped tuning table's shape (no GPU: the context entry points
need a device, so only the table and the host helpers run here)."""
import json

from emclarity_amd import autotune


def test_shipped_table_lists_candidates_it_chose():
    t = autotune.load_table()
    if not t:
        return                      # no table shipped: library defaults apply
    for table, by_n in t["params"].items():
        assert table in ("c64", "f16")
        for n, p in by_n.items():
            assert int(n) in (64, 96, 128)
            for name, v in p.items():
                assert v in autotune.CANDIDATES[name]
                times = t["timings_ms"][table][n][name]
                assert float(times[str(v)]) == min(float(x) for x in times.values())


def test_params_for_and_empty_override(tmp_path):
    p = tmp_path / "t.json"
    p.write_text(json.dumps({"params": {"c64": {"64": {"search_tile": 8}}}}))
    t = autotune.load_table(p)
    assert autotune.params_for(64, "c64", t) == {"search_tile": 8}
    assert autotune.params_for(96, "c64", t) == {} and autotune.params_for(64, "f16", t) == {}


def test_search_shapes_are_timed_where_the_column_passes_run(monkeypatch):
    """No call timed for the search's shapes takes the strips, which read none of
    them (fp16 table, 64^3, 0.6 x the support would)."""
    import numpy as np

    from emclarity_amd import batched, device, workload
    timed = []

    class Aligner:
        peak_radius = 6

        def __init__(self, n, ref, bp, table, ctx, tuning):
            self.support, self.table = n / 2 - 1.01, table

        def set_particles(self, *a):
            self.count = len(a[0])

        def search(self, grid, radius):
            timed.append((radius, self.table, self.peak_radius, self.count * len(grid)))

        def _eval_local(self, R, s):
            pass

    class Array:
        def view(self, *a):
            return self

    monkeypatch.setattr(batched, "BatchAligner", Aligner)
    monkeypatch.setattr(device, "DeviceArray", type("D", (), {"from_numpy": staticmethod(lambda *a, **k: Array())}))
    monkeypatch.setattr(workload, "make_size_class", lambda n: (type("S", (), {"ref": None, "bandpass": None}), None))
    monkeypatch.setattr(autotune, "_timed", lambda ctx, fn, names, reps: fn() or 1.0)
    monkeypatch.setattr(autotune, "apply", lambda *a: None)
    monkeypatch.setattr(np.random, "default_rng", lambda seed: type("G", (), {
        "standard_normal": staticmethod(lambda size, dtype=np.float64: np.ones(4) if size == 4 else np.zeros(1))}))
    autotune.tune(None, counts=((64, 1000), (96, 600)))
    assert timed and not any(batched.search_uses_strips(*t) for t in timed)
    assert any(r < 0.7 * 30.99 for r, table, _, _ in timed if table == "c64")
    assert batched.search_uses_strips(0.6 * 30.99, "f16", 6, 28000)
    assert not batched.search_uses_strips(0.6 * 30.99, "f16", 6, 2000)
    assert not batched.search_uses_strips(0.6 * 30.99, "c64", 6, 28000)
