"""Queue appends of the wavefront loop: connections to any number of recorders
and the continuing rays from one counter, and rays that are emitted dead."""
import numpy as np
import pytest

from ear_amd import api, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rec", [1, 2, 3, 5, 16])
@pytest.mark.parametrize("n_rays", [1, 255, 257, 5000])
def test_connections_to_many_recorders(gpu_ctx, n_rec, n_rays):
    """The loop's shading (tail_rays 1: to the end) against the tail launch,
    which connects recorder by recorder without queues: same sums."""
    s = scenes.shoebox(tess=(3, 3, 3))
    rng = np.random.default_rng(n_rec)
    recs = [scenes.stereo_recorder(rng.uniform((1, 1, 1), (9, 7, 3))) if i % 3 == 1 else
            dict(kind=0, pos=tuple(rng.uniform((1, 1, 1), (9, 7, 3)))) for i in range(n_rec)]
    kw = dict(recorders=recs, n_rays=n_rays, src_pos=s["src"], air=s["air"], max_bounces=30, cutoff=1e-8, n_bins=22050)
    with api.Scene(gpu_ctx, s["tris"], s["mat"], s["materials"]) as sc:
        gpu_ctx.set_tuning(tail_rays=1)
        a = api.render(gpu_ctx, sc, **kw)
        gpu_ctx.set_tuning()
        b = api.render(gpu_ctx, sc, **kw)
    np.testing.assert_array_equal(a.raw, b.raw)
    np.testing.assert_array_equal(a.abs_raw, b.abs_raw)
    for k in ("segments", "shadow_rays", "contributions", "rays"):
        assert a.stats[k] == b.stats[k]


def test_a_batch_with_items_whose_rays_are_emitted_dead(gpu_ctx):
    """An item with no bounces and one with a cut-off above the source's
    intensity among live ones: every item as alone, all rays counted."""
    s = scenes.room(seed=3, target_tris=300)
    kw = dict(recorders=s["recorders"], src_pos=s["src"], air=s["air"], n_bins=22050)
    opts = [dict(max_bounces=40, cutoff=1e-8), dict(max_bounces=0, cutoff=1e-8), dict(max_bounces=40, cutoff=2.0),
            dict(max_bounces=40, cutoff=1e-6)]
    with api.Scene(gpu_ctx, s["tris"], s["mat"], s["materials"]) as sc:
        items = [(sc, dict(kw, n_rays=700 + i, instance=i, **o)) for i, o in enumerate(opts)]
        res, stats, _ = api.render_batch(gpu_ctx, items)
        alone = [api.render(gpu_ctx, sc, **k) for _, k in items]
    assert stats["rays"] == sum(3 * (700 + i) for i in range(4)) == sum(a.stats["rays"] for a in alone)
    assert stats["segments"] == sum(a.stats["segments"] for a in alone)
    for r, a in zip(res, alone):
        np.testing.assert_array_equal(r.raw, a.raw)
        np.testing.assert_array_equal(r.value, a.value)
