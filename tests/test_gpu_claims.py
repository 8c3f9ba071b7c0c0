"""Queue claims of the largest chunk: no counter wraps, so no entry is handed
out twice (8192 waves' last claims of 2^20 entries each pass 2^32)."""
import numpy as np
import pytest

from ear_amd import api, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("segments", [1, 16, 64])
def test_largest_chunk_hands_every_entry_out_once(gpu_ctx, segments):
    s = scenes.hall(target_tris=2000)
    kw = dict(recorders=s["recorders"], n_rays=1_000_000, src_pos=s["src"], air=s["air"], max_bounces=3, cutoff=1e-6,
              n_bins=22_050)
    try:
        with api.Scene(gpu_ctx, s["tris"], s["mat"], s["materials"]) as sc:
            ref = api.render(gpu_ctx, sc, **kw)
            gpu_ctx.set_tuning(fetch_chunk=1 << 20, fetch_segments=segments, tail_rays=1)
            big = api.render(gpu_ctx, sc, **kw)
    finally:
        gpu_ctx.set_tuning()
    assert big.stats["shadow_rays"] == ref.stats["shadow_rays"]
    np.testing.assert_array_equal(big.raw, ref.raw)
    np.testing.assert_array_equal(big.abs_raw, ref.abs_raw)
