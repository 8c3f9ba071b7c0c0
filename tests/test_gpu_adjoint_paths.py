"""The vertex forms of the adjoint carry each path to its end in one launch: ray
counts around a wave, a launch's lanes and a chunk; several materials, recorders
and bands; a continuation's main path taken up again."""
import numpy as np
import pytest

from ear_amd import api, scenes

pytestmark = pytest.mark.gpu

NB = 4096


def _room(n_rec):
    r = scenes.room(seed=31, target_tris=400, kind="L")
    recs = list(r["recorders"])
    while len(recs) < n_rec:
        recs.append(dict(recs[0], pos=tuple(c + 0.25 * len(recs) for c in recs[0]["pos"])))
    kw = dict(recorders=recs, src_pos=r["src"], air=r["air"], max_bounces=120, cutoff=1e-8, n_bins=NB, abs_hist=True)
    rng = np.random.default_rng(5)
    n_ch = n_rec
    return r, kw, rng.standard_normal((3, n_ch, NB)), rng.standard_normal((3, n_ch, NB))


@pytest.mark.parametrize("form", ["score", "local"])
@pytest.mark.parametrize("n_rays,chunk,n_rec,width", [(1, 0, 1, 4), (21, 0, 2, 4), (64, 63, 1, 2), (4097, 1000, 2, 2),
                                                      (4097, 1000, 2, 4), (70_001, 65_536, 1, 4)])
def test_chunks_and_bands_sum_to_the_whole(gpu_ctx, form, n_rays, chunk, n_rec, width):
    """All bands at once in one chunk, against each band by itself in chunks:
    the paths and their float weights are the same, so the gradients differ by
    the order of binary64 sums.  A sum of M terms of size up to the largest
    entry is off by at most M 2^-53 of it; with fewer than 1e7 connections
    1e-9 of the largest entry covers that."""
    r, kw, a_v, a_a = _room(n_rec)
    with api.Scene(gpu_ctx, r["tris"], r["mat"], r["materials"], width=width) as sc:
        print(form, n_rays, chunk, n_rec, width, flush=True)
        flags = {form: True}
        w_r, w_s = api.render_backward(gpu_ctx, sc, adj_value=a_v, adj_abs=a_a, n_rays=n_rays, **kw, **flags)
        gpu_ctx.set_tuning(ray_chunk=chunk)
        try:
            for b in range(3):
                g_r, g_s = api.render_backward(gpu_ctx, sc, adj_value=a_v, adj_abs=a_a, n_rays=n_rays, bands=(b,),
                                               **kw, **flags)
                for g, w in ((g_r, w_r), (g_s, w_s)):
                    np.testing.assert_allclose(g[:, b], w[:, b], rtol=0, atol=1e-9 * np.abs(w).max())
                    assert np.all(np.delete(g, b, axis=1) == 0)
        finally:
            gpu_ctx.set_tuning()
    assert n_rays < 64 or (np.any(w_r != 0) and np.any(w_s != 0))
