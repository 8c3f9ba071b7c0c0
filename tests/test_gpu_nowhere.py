"""Rays whose origin is no number: they miss, at no more than the root's cost
(a source of NaNs must not walk the whole tree with every ray)."""
import numpy as np
import pytest

from ear_amd import api, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [2, 4])
def test_a_source_that_is_nowhere_visits_no_more_than_the_root(gpu_ctx, width):
    s = scenes.hall(target_tris=5000)
    with api.Scene(gpu_ctx, s["tris"], s["mat"], s["materials"], width=width) as sc:
        r = api.render(gpu_ctx, sc, recorders=s["recorders"], n_rays=200, src_pos=(np.nan,) * 3, air=s["air"],
                       max_bounces=20, cutoff=1e-6, n_bins=4096, instrument=True)
    assert r.stats["segments"] == 600
    assert r.stats["node_visits_closest"] <= 600 and r.stats["tri_tests_closest"] == 0
    assert not r.raw.any()


@pytest.mark.parametrize("width", [2, 4])
def test_queries_from_nowhere_miss_and_leave_the_others_alone(gpu_ctx, width):
    s = scenes.hall(target_tris=5000)
    rng = np.random.default_rng(3)
    o = np.tile(np.float32(s["src"]), (256, 1))
    d = rng.normal(size=(256, 3)).astype(np.float32)
    q = rng.uniform(s["tris"].reshape(-1, 3).min(0), s["tris"].reshape(-1, 3).max(0), (256, 3)).astype(np.float32)
    bad = o.copy()
    bad[::3] = np.nan
    with api.Scene(gpu_ctx, s["tris"], s["mat"], s["materials"], width=width) as sc:
        t0, i0 = sc.query_closest(o, d)
        t1, i1 = sc.query_closest(bad, d)
        v0, v1 = sc.query_occluded(o, q), sc.query_occluded(bad, q)
    ok = np.ones(256, bool)
    ok[::3] = False
    assert (i0 >= 0).any() and v0.any()
    assert (i1[~ok] == -1).all() and not v1[~ok].any()
    np.testing.assert_array_equal(i1[ok], i0[ok])
    np.testing.assert_array_equal(t1[ok], t0[ok])
    np.testing.assert_array_equal(v1[ok], v0[ok])
