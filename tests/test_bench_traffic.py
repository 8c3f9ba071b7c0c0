"""bench.py pairs measured HBM traffic only with the kernels and launches that
it was measured on."""
import json
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402

ACC = dict(extend_queries=52_000, extend_launches=52, extend_ms=52.0, shadow_queries=26_000, shadow_launches=52,
           shadow_ms=26.0, shade_ms=13.0, splat_ms=0.0, shadow_ramps=26_000, shadow_contributions=26_000,
           segments=52_000, rays=10_000, trace_ms=100.0)
IST = dict(node_visits_closest=1, tri_tests_closest=1, extend_queries=1, node_visits_shadow=1, tri_tests_shadow=1,
           shadow_queries=1)


def _traffic(tmp_path, **kw):
    """k_extend_f's traffic in the bench's output with a file of `kw` beside
    launches of 1000 queries."""
    with open(os.path.join(tmp_path, "traffic_k_extend_f_hall200k.json"), "w") as f:
        json.dump(dict(bytes_per_launch=123_000_000, **kw), f)
    return bench.kernel_rooflines(ACC, IST, {"node_bytes": 64}, str(tmp_path), 1)[0]["k_extend_f"]


def test_traffic_of_another_build_or_length_is_not_used(tmp_path):
    for kw in (dict(), dict(kernel_source="0" * 16, units_per_launch=1000.0),
               dict(kernel_source=bench.kernel_source_id(), units_per_launch=1100.0),
               dict(kernel_source=bench.kernel_source_id())):
        r = _traffic(tmp_path, **kw)
        assert r["traffic"] is None and r["measured_frac"] is None
    r = _traffic(tmp_path, kernel_source=bench.kernel_source_id(), units_per_launch=1001.0)
    assert r["traffic"] == 123_000_000
    assert r["measured_frac"] == pytest.approx(123e6 / 1e-3 / 8e12, abs=1e-4)


def test_source_id_passes_over_comments(tmp_path, monkeypatch):
    csrc = tmp_path / "ear_amd" / "csrc"
    csrc.mkdir(parents=True)
    for n in ("ear_internal.hpp", "ear_math.hpp", "lbvh.hip", "tracer.hip"):
        (csrc / n).write_text("int a;  // one\n")
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    one = bench.kernel_source_id()
    (csrc / "tracer.hip").write_text("// two\nint  a;\n")
    assert bench.kernel_source_id() == one
    (csrc / "tracer.hip").write_text("int b;\n")
    assert bench.kernel_source_id() != one
