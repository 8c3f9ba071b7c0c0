"""Raw sums returned to the caller: no more device memory than the same render
without them, however few rays and long rows, in whatever pieces, and outside
the render's device time."""
import numpy as np
import pytest

from ear_amd import api, scenes

pytestmark = pytest.mark.gpu

BINS = 1 << 19


def _kw(s, **kw):
    return dict(dict(recorders=s["recorders"], n_rays=1000, src_pos=s["src"], air=s["air"], max_bounces=50,
                     cutoff=1e-6, n_bins=BINS), **kw)


def test_raw_sums_fit_a_cap_that_the_finished_tracks_fit(gpu_ctx):
    """The finished tracks take device memory of their own (8 bytes a bin);
    raw sums do not, so a cap that holds the one render holds the other."""
    s = scenes.shoebox()
    with api.Scene(gpu_ctx, s["tris"], s["mat"], s["materials"]) as sc:
        ref = api.render(gpu_ctx, sc, **_kw(s))
        lo, hi = 0, 1 << 30  # MiB steps: refused, accepted
        try:
            while hi - lo > 1 << 20:
                mid = (lo + hi) // 2
                gpu_ctx.set_memory_cap(mid)
                try:
                    api.render(gpu_ctx, sc, **_kw(s, want_raw=False))
                    hi = mid
                except api.EarError as e:
                    assert e.status_name == "EAR_ERR_OUT_OF_MEMORY"
                    lo = mid
            gpu_ctx.set_memory_cap(hi)
            raw = api.render(gpu_ctx, sc, **_kw(s, want_value=False))
        finally:
            gpu_ctx.set_memory_cap(0)
    np.testing.assert_array_equal(raw.raw, ref.raw)
    np.testing.assert_array_equal(raw.abs_raw, ref.abs_raw)


@pytest.mark.parametrize("abs_hist", [True, False])
def test_rows_longer_than_the_staging_memory(gpu_ctx, abs_hist):
    """One wave per CU leaves a few MB of stacks: a row of 2^19 bins is staged
    in several pieces (one without the small grid)."""
    s = scenes.shoebox(stereo=True)
    with api.Scene(gpu_ctx, s["tris"], s["mat"], s["materials"]) as sc:
        ref = api.render(gpu_ctx, sc, **_kw(s, abs_hist=abs_hist))
        gpu_ctx.set_tuning(waves_per_cu=1)
        try:
            few = api.render(gpu_ctx, sc, **_kw(s, abs_hist=abs_hist))
        finally:
            gpu_ctx.set_tuning()
    assert np.count_nonzero(ref.raw) > 0
    np.testing.assert_array_equal(few.raw, ref.raw)
    np.testing.assert_array_equal(few.value, ref.value)
    if abs_hist:
        np.testing.assert_array_equal(few.abs_raw, ref.abs_raw)
        np.testing.assert_array_equal(few.abs_value, ref.abs_value)


@pytest.mark.parametrize("waves_per_cu", [0, 1])
def test_device_time_leaves_the_copies_of_raw_sums_out(gpu_ctx, waves_per_cu):
    """trace_ms is the device time of the render: the copies of 100 MB of raw
    sums (10 ms at 10 GB/s) are no part of it."""
    s = scenes.shoebox()
    gpu_ctx.set_tuning(waves_per_cu=waves_per_cu)
    try:
        with api.Scene(gpu_ctx, s["tris"], s["mat"], s["materials"]) as sc:
            ms = {raw: min(api.render(gpu_ctx, sc, **_kw(s, n_bins=2 * BINS, want_raw=raw)).stats["trace_ms"]
                           for _ in range(5)) for raw in (False, True)}
    finally:
        gpu_ctx.set_tuning()
    assert ms[True] < 1.5 * ms[False] + 1.0
