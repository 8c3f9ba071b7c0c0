"""The walk kernels at the edges of their work split: queue lengths around a
wave and around the grid's lanes (where claiming begins), and rays from
outside the scene (where the folded box planes lose the most bits)."""
import numpy as np
import pytest

from ear_amd import api, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rays", [1, 63, 64, 65, 16383, 16384, 16385, 70001])
def test_queue_lengths_around_a_wave_and_the_grid(gpu_ctx, n_rays):
    """One wave per CU holds 16384 lanes on 256 CUs: shorter queues are handed
    out without claims, longer ones by claims from one or many segments.
    Every split walks the same rays: the sums equal those of one ray per
    lane."""
    s = scenes.hall(target_tris=2_000)
    kw = dict(recorders=s["recorders"], n_rays=n_rays, src_pos=s["src"], air=s["air"], bands=(1,), max_bounces=6,
              cutoff=1e-8, n_bins=22050)
    with api.Scene(gpu_ctx, s["tris"], s["mat"], s["materials"]) as sc:
        res = []
        for trav, segs, chunk in [(1, 0, 0), (3, 0, 0), (3, 1, 0), (3, 64, 5)]:
            gpu_ctx.set_tuning(traversal=trav, waves_per_cu=1, tail_rays=1, fetch_segments=segs, fetch_chunk=chunk)
            res.append(api.render(gpu_ctx, sc, **kw))
        gpu_ctx.set_tuning()
    for r in res[1:]:
        np.testing.assert_array_equal(res[0].raw, r.raw)
        np.testing.assert_array_equal(res[0].abs_raw, r.abs_raw)
        for k in ("segments", "shadow_rays", "contributions"):
            assert res[0].stats[k] == r.stats[k]


@pytest.mark.parametrize("away", [0.0, 1.0, 8.0])
@pytest.mark.parametrize("leaf", [1, 2, 3, 5])
def test_walks_from_outside_the_scene(gpu_ctx, oracle, away, leaf):
    """Origins up to 8 scene extents away: a folded plane moves by a few 2^-24
    of that distance (2e-6 extents), within the boxes' padding (1e-5), so
    every hit is the scan's, bit for bit.  Odd leaf sizes test the triangle
    pairs' remainder."""
    rng = np.random.default_rng(int(away) * 10 + leaf)
    s = scenes.hall(target_tris=1_500)
    tris = s["tris"]
    lo, hi = tris.reshape(-1, 3).min(0), tris.reshape(-1, 3).max(0)
    n = 600
    u = rng.normal(size=(n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    o = rng.uniform(lo, hi, (n, 3)) + u * away * np.max(hi - lo)
    tgt = tris[rng.integers(0, len(tris), n)].mean(axis=1)
    d = tgt - o
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    o, q = o.astype(np.float32), tgt.astype(np.float32)
    with api.Scene(gpu_ctx, tris, s["mat"], s["materials"], leaf_size=leaf) as sc:
        t, idx = sc.query_closest(o, d)
        occ = sc.query_occluded(o, q)
    osc = oracle.OracleScene(tris, s["mat"], s["materials"])
    hits = 0
    for i in range(n):
        ot, oi = osc.closest_hit(o[i], d[i])
        assert idx[i] == oi, (i, idx[i], oi)
        if oi >= 0:
            hits += 1
            assert np.float32(t[i]) == np.float32(ot)
        assert occ[i] == osc.any_hit(o[i], q[i])
    assert hits > n // 2
