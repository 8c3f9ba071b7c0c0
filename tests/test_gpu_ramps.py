"""Ramps kept as one point each (their slope, by the parity of the width) and,
where a head is too wide for that, as second differences: the sums against
the oracle on both sides of the line, near the first bin and cut at the last."""
import numpy as np
import pytest

from ear_amd import api, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_bins", [257, 4000, 44100])
@pytest.mark.parametrize("head,ear", [(0.17, (0.0, 1.0, 0.0)), (0.48, (0.0, 1.0, 0.0)), (0.49, (0.0, 1.0, 0.0)),
                                      (0.17, (0.0, 2.7, 0.0)), (0.17, (2.0, 2.7, 0.0)), (3.0, (0.6, 0.8, 0.0))])
def test_ramps_of_narrow_and_wide_heads(gpu_ctx, oracle, head, ear, n_bins):
    """A mono recorder half a metre from the source (ramps from the first
    bins) beside a stereo one whose delay, head times |ear|, lies on either
    side of the half metre that one point per ramp allows.  The gate is the
    oracle suite's: 1e-5 of the bin's unsigned sum, plus a quantum per
    contribution."""
    s = scenes.shoebox(3.0, 2.5, 2.2, src=(0.6, 0.7, 1.0), rec=(0.9, 1.0, 1.2), spec=0.3)
    recs = [dict(kind=0, pos=(0.9, 1.0, 1.2)), scenes.stereo_recorder((1.9, 1.1, 1.3), right_ear=ear, head_size=head)]
    n_rays, bounces = 800, 60
    kw = dict(recorders=recs, n_rays=n_rays, src_pos=s["src"], max_bounces=bounces, cutoff=1e-8, n_bins=n_bins)
    with api.Scene(gpu_ctx, s["tris"], s["mat"], s["materials"]) as sc:
        res = []
        for splat, abs_hist in [(0, True), (2, True), (0, False), (2, False)]:
            gpu_ctx.set_tuning(splat=splat, tail_rays=1 if splat == 2 else 0)
            res.append(api.render(gpu_ctx, sc, air=s["air"], bands=(1,), abs_hist=abs_hist, **kw))
        gpu_ctx.set_tuning()
        na = api.render_noalloc(gpu_ctx, sc, air=s["air"], bands=(1,), want_raw=False, **kw)
    osc = oracle.OracleScene(s["tris"], s["mat"], s["materials"])
    o = oracle.render(osc, band=1, air=s["air"][1], **kw)
    tol = 1e-5 * o["hist_abs"] + n_rays * (bounces + 1) * 2.0 ** -80
    assert np.any(o["hist_abs"])
    assert np.all(np.abs(api.raw_to_float(res[0].raw[1]) - o["hist_signed"]) <= tol)
    assert np.all(np.abs(api.raw_to_float(res[0].abs_raw[1]) - o["hist_abs"]) <= tol)
    for r in res[1:]:
        np.testing.assert_array_equal(res[0].raw, r.raw)
        np.testing.assert_array_equal(res[0].value, r.value)
    np.testing.assert_array_equal(res[0].abs_raw, res[1].abs_raw)
    np.testing.assert_array_equal(res[0].value, na.value)
    np.testing.assert_array_equal(res[0].abs_value, na.abs_value)
