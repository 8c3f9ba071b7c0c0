"""Performance cases: what a program that uses this framework has it do.

Every case goes through the public Python front end (ear_amd.api), on scenes
of ear_amd.scenes, at sizes of the repository's tests and benchmark.  A case
is a plain dict; its "do" names one of these:

  render    one ear_render of a room or the hall (the band contexts of a source)
  noalloc   one ear_render_noalloc (a serving loop that must not allocate)
  batch     one ear_render_batch of many rooms
  frames    one ear_render_batch of a moving source's keyframes in one hall
  open      a scene uploaded (its tree built) and previewed with few rays
  backward  one ear_render_backward of a fitting step
  backrooms one ear_render_backward_batch of a fitting step of many rooms
  query     closest-hit and occlusion queries of a host tool
  convolve  one ear_convolve, with or without the keyframe cross-fade

Renders are Monte-Carlo sums over paths whose turns depend on how binary32
results round, so a render, its gradients and a query of a big scene have no
64-bit value of their own here (exact gives None); the convolution and the
small queries do.
"""
from __future__ import annotations

import math

import numpy as np

from ear_amd import api, fit, scenes

_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = api.Context(0)
    return _ctx


class _State:
    """What a program holds between calls; its scenes go with it."""

    def __init__(self, case):
        self.case = case
        self.scenes = []

    def upload(self, s, materials=None):
        sc = api.Scene(_context(), s["tris"], s["mat"], materials or s["materials"])
        self.scenes.append(sc)
        return sc

    def __del__(self):
        for sc in self.scenes:
            sc.close()


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest render: one band of the 12-triangle box, as an interactive
        # change of a wall is previewed; launches, allocations and the host count
        dict(name="preview_box", do="render", scene="box", tris=12, rays=20_000, bands=1, bins=44_100, bounces=100,
             recorders=1, raw=True, spec=0.5),
        # the shoebox room in full: 1M rays a band, every path in the tail launch
        dict(name="render_box_1m", do="render", scene="box", tris=12, rays=1_000_000, bands=3, bins=45_056,
             bounces=999, recorders=1, raw=False, spec=0.3),
        # an ordinary room with furniture-sized triangles, an emitting mesh and
        # two receivers (mono and stereo), a ragged ray count, exact sums returned
        dict(name="render_room_mesh", do="render", scene="room", tris=6_000, rays=333_333, bands=3, bins=66_150,
             bounces=999, recorders=2, raw=True, spec=0.0, mesh=True),
        # receiver spheres in a room with transmitting walls: the other estimator
        dict(name="render_room_sphere", do="render", scene="room", tris=1_500, rays=250_000, bands=2, bins=44_100,
             bounces=400, recorders=2, raw=False, spec=0.0, sphere=True, refr=0.2),
        # the headline: a 200k-triangle concert hall, stereo, 10M rays a band
        dict(name="render_hall_10m", do="render", scene="hall", tris=200_000, rays=10_000_000, bands=3, bins=132_300,
             bounces=100, recorders=1, raw=False, spec=0.0),
        # a serving loop's render in a 20k-triangle hall without device allocation
        dict(name="noalloc_hall", do="noalloc", scene="hall", tris=20_000, rays=150_001, bands=3, bins=66_150,
             bounces=100, recorders=1, raw=False, spec=0.0),
        # many rooms of mixed size in one call
        dict(name="batch_rooms", do="batch", rooms=32, tris=20_000, rays=300_000, bins=44_100, bounces=999),
        # a source that moves through a hall, a keyframe an item
        dict(name="frames_hall", do="frames", scene="hall", tris=100_000, frames=12, rays=200_000, bands=3,
             bins=88_200, bounces=100),
        # a scene opened (uploaded, its tree built) and heard once
        dict(name="open_hall", do="open", scene="hall", tris=200_000, rays=10_000, bands=3, bins=44_100, bounces=100,
             recorders=1, raw=False, spec=0.0),
        # the gradient of a fitting step of one room, the form that fitting uses
        dict(name="backward_box", do="backward", rays=1_000_000, form="score", bins=45_056, bounces=999),
        # the gradients of a fitting step of several rooms together
        dict(name="backward_rooms", do="backrooms", rooms=8, tris=20_000, rays=150_000, form="score", bins=45_056,
             bounces=999),
        # three seconds of response and ten of sound, faded between two keyframes
        dict(name="convolve_fade", do="convolve", n_ir=132_300, n_sig=441_000, fade=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    do = rng.choice(["render", "render", "render", "noalloc", "batch", "frames", "open", "backward", "backrooms",
                     "query", "convolve"])
    if do == "convolve":
        return dict(do=do, n_ir=_log(rng, 1_000, 200_000), n_sig=_log(rng, 1_000, 2_000_000), fade=rng.random() < 0.5)
    if do == "query":
        return dict(do=do, scene=rng.choice(["box", "room", "hall"]), tris=_log(rng, 500, 200_000),
                    n=_log(rng, 500, 1_000_000))
    if do == "backward":
        return dict(do=do, rays=_log(rng, 20_000, 1_000_000), form=rng.choice(["score", "score", "local"]),
                    bins=4096 * rng.randint(6, 16), bounces=rng.choice([100, 999]))
    if do == "backrooms":
        return dict(do=do, rooms=rng.randint(2, 12), tris=_log(rng, 200, 20_000), rays=_log(rng, 10_000, 150_000),
                    form=rng.choice(["score", "score", "local"]), bins=45_056, bounces=999)
    if do == "batch":
        return dict(do=do, rooms=rng.randint(2, 48), tris=_log(rng, 1_000, 50_000), rays=_log(rng, 20_000, 300_000),
                    bins=rng.choice([44_100, 66_150]), bounces=999)
    if do == "frames":
        return dict(do=do, scene="hall", tris=_log(rng, 5_000, 200_000), frames=rng.randint(2, 24),
                    rays=_log(rng, 10_000, 200_000), bands=rng.choice([1, 3]), bins=rng.choice([44_100, 88_200]),
                    bounces=100)
    c = dict(do=do, scene=rng.choice(["box", "room", "hall"]), tris=_log(rng, 500, 200_000),
             rays=_log(rng, 5_000, 3_000_000), bands=rng.choice([1, 2, 3]),
             bins=rng.choice([22_050, 44_100, 66_150, 88_201, 132_300]), bounces=rng.choice([50, 100, 999]),
             recorders=rng.choice([1, 1, 2, 3]), raw=rng.random() < 0.3, spec=rng.choice([0.0, 0.0, 0.3, 0.5]))
    if c["scene"] == "box":
        c["tris"] = 12
    if do == "render" and rng.random() < 0.25:
        c["mesh"] = True
    elif do == "render" and rng.random() < 0.2:
        c["sphere"] = True
    if rng.random() < 0.2:
        c["refr"] = 0.2
    if do == "noalloc":
        c["bins"] = min(c["bins"], 66_150)  # the region holds the histograms of about that
        c["recorders"] = min(c["recorders"], 2)
    if do == "open":
        c["rays"] = min(c["rays"], 30_000)
    return c


# ---------------------------------------------------------------------------
# scenes
# ---------------------------------------------------------------------------
def _scene(case, seed):
    """A scene of the case's kind, its materials with the case's options."""
    rng = np.random.default_rng(seed)
    spec = case.get("spec", 0.0)
    if case["scene"] == "box":
        s = scenes.shoebox(rng.uniform(8, 13), rng.uniform(6, 9), rng.uniform(3, 5), seed=seed, spec=spec)
    elif case["scene"] == "room":
        s = scenes.room(seed=seed, target_tris=case["tris"])
    else:
        s = scenes.hall(seed=seed, target_tris=case["tris"])
    if case["scene"] != "box" and (spec or case.get("refr")):
        s["materials"] = scenes.absorption_materials(s["alpha"], spec=[spec] * len(s["alpha"]))
    if case.get("refr"):
        f = float(case["refr"])
        s["materials"] = [([x * (1.0 - f) for x in r], [x * f for x in r], sp) for r, _, sp in s["materials"]]
    return s


def _recorders(case, s, rng):
    """The scene's own recorder, then more of both kinds near it."""
    recs = list(s["recorders"])
    p = np.asarray(recs[0]["pos"], np.float64)
    for i in range(1, case.get("recorders", 1)):
        q = tuple(float(x) for x in p + rng.uniform(-0.3, 0.3, 3))
        recs.append(scenes.stereo_recorder(q) if i % 2 else dict(kind=0, pos=q))
    if case.get("sphere"):
        recs = [dict(r, radius=0.25) for r in recs]
    return recs


def _emitter(s):
    """A small emitting quad at the source's place (3SRC with a mesh)."""
    x, y, z = s["src"]
    q = [(x - 0.1, y - 0.1, z), (x + 0.1, y - 0.1, z), (x + 0.1, y + 0.1, z), (x - 0.1, y + 0.1, z)]
    return np.asarray([[q[0], q[1], q[2]], [q[0], q[2], q[3]]], np.float32)


def _render_kw(case, s, seed):
    rng = np.random.default_rng([seed, 1])
    kw = dict(recorders=_recorders(case, s, rng), n_rays=case["rays"], bands=tuple(range(case.get("bands", 3))),
              src_pos=s["src"], air=s["air"], max_bounces=case["bounces"], cutoff=1e-8, n_bins=case["bins"],
              seed=seed, abs_hist=True, want_raw=bool(case.get("raw")))
    if case.get("mesh"):
        kw["src_tris"] = _emitter(s)
    if case.get("sphere"):
        kw["estimator"] = 1
    return kw


def _rooms(case, seed):
    """Box and L rooms of log-uniform size and ray count, up to the case's."""
    return scenes.batch_rooms(case["rooms"], seed=seed, tris=(12, case["tris"]),
                              rays=(max(1_000, case["rays"] // 30), case["rays"]))


def _fit_room(s, seed):
    """Materials a fitting run starts from: the scene's, up to 20% off."""
    rng = np.random.default_rng([seed, 2])
    n = len(s["materials"])
    return (fit.materials(s["alpha"], np.full(n, 0.3)),
            fit.materials(np.clip(s["alpha"] * rng.uniform(0.8, 1.2, s["alpha"].shape), 0.01, 0.95),
                          0.3 * rng.uniform(0.8, 1.2, n)))


def prepare(case, seed):
    seed = int(seed) & 0x7FFFFFFF
    rng = np.random.default_rng([seed, 3])
    st = _State(case)
    do = case["do"]
    if do in ("render", "noalloc"):
        s = _scene(case, seed)
        st.scene, st.kw = st.upload(s), _render_kw(case, s, seed)
    elif do == "open":
        s = _scene(case, seed)
        st.soup, st.kw = s, _render_kw(case, s, seed)
        _context()
    elif do == "batch":
        st.items = []
        for i, (s, rays) in enumerate(_rooms(case, seed)):
            st.items.append((st.upload(s), dict(recorders=s["recorders"], src_pos=s["src"], air=s["air"], n_rays=rays,
                                                max_bounces=case["bounces"], cutoff=1e-8, n_bins=case["bins"],
                                                instance=i, seed=seed, abs_hist=False, want_raw=False)))
    elif do == "frames":
        s = _scene(case, seed)
        sc = st.upload(s)
        st.items = [(sc, dict(recorders=s["recorders"], src_pos=p, air=s["air"], n_rays=case["rays"], keyframe=k,
                              bands=tuple(range(case["bands"])), max_bounces=case["bounces"], cutoff=1e-8,
                              n_bins=case["bins"], seed=seed, abs_hist=False, want_raw=False))
                    for k, p in enumerate(scenes.stage_path(case["frames"]))]
    elif do in ("backward", "backrooms"):
        if do == "backward":
            # the fitting benchmark's room: 12 x 9 x 5 m, six walls
            rooms = [(scenes.shoebox(12.0, 9.0, 5.0, seed=seed, spec=0.3, alpha_range=(0.1, 0.3), src=(3.0, 4.0, 2.0),
                                     rec=(8.0, 5.0, 1.7)), case["rays"])]
        else:
            rooms = _rooms(case, seed)
        st.items = []
        for s, rays in rooms:
            aim, now = _fit_room(s, seed)
            sc = st.upload(s, aim)
            kw = dict(recorders=s["recorders"], src_pos=s["src"], air=s["air"], n_rays=rays,
                      max_bounces=case["bounces"], cutoff=1e-8, n_bins=case["bins"], seed=seed, abs_hist=True,
                      want_raw=False)
            # the step's adjoint: the log decay curve's distance from the target's
            few = dict(kw, n_rays=min(rays, 50_000))
            target = fit.log_edc(fit.coarse_bins(api.render(_context(), sc, **few).abs_value))
            sc.set_materials(now)
            _, adj = fit.log_edc_loss(api.render(_context(), sc, **few).abs_value, target, fit.decay_mask(target))
            st.items.append((sc, dict(kw, adj_abs=adj, **{case["form"]: True})))
    elif do == "query":
        s = _scene(case, seed)
        st.scene = st.upload(s)
        st.o, st.d, st.q = _query_rays(case, s, rng)
    elif do == "convolve":
        st.ir, st.ir2, st.sig = _tracks(case, rng)
        _context()
    return st


def _query_rays(case, s, rng):
    """Origins inside the scene's box, unit directions, other points inside."""
    lo, hi = s["tris"].reshape(-1, 3).min(0), s["tris"].reshape(-1, 3).max(0)
    o = rng.uniform(lo, hi, (case["n"], 3)).astype(np.float32)
    d = rng.normal(size=(case["n"], 3))
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    return o, d, rng.uniform(lo, hi, (case["n"], 3)).astype(np.float32)


def _tracks(case, rng):
    """Decaying noise (an impulse response, sparse at first) and a sound."""
    def ir():
        t = np.arange(case["n_ir"])
        x = rng.normal(size=case["n_ir"]) * np.exp(-6.9 * t / case["n_ir"])
        return (x * (rng.random(case["n_ir"]) < np.minimum(1.0, 0.01 + t / (0.1 * case["n_ir"])))).astype(np.float32)

    sig = np.clip(0.2 * rng.normal(size=case["n_sig"]), -1.0, 1.0).astype(np.float32)
    return ir(), ir() if case["fade"] else None, sig


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _out(r):
    out = dict(value=r.value, abs_value=r.abs_value, segments=int(r.stats["segments"]))
    if r.raw is not None:
        out.update(raw=r.raw, abs_raw=r.abs_raw)
    return out


def run(state):
    do = state.case["do"]
    ctx = _context()
    if do == "render":
        return _out(api.render(ctx, state.scene, **state.kw))
    if do == "noalloc":
        return _out(api.render_noalloc(ctx, state.scene, **state.kw))
    if do == "open":
        s = state.soup
        with api.Scene(ctx, s["tris"], s["mat"], s["materials"]) as sc:
            return _out(api.render(ctx, sc, **state.kw))
    if do in ("batch", "frames"):
        res, stats, _ = api.render_batch(ctx, state.items)
        return dict(values=[r.value for r in res], segments=int(stats["segments"]))
    if do == "backward":
        sc, kw = state.items[0]
        g_refl, g_spec = api.render_backward(ctx, sc, **kw)
        return dict(refl=g_refl, spec=g_spec)
    if do == "backrooms":
        grads = api.render_backward_batch(ctx, state.items)
        return dict(refl=[g for g, _ in grads], spec=[g for _, g in grads])
    if do == "query":
        t, tri = state.scene.query_closest(state.o, state.d)
        return dict(t=t, tri=tri, occluded=state.scene.query_occluded(state.o, state.q))
    return api.convolve(ctx, state.ir, state.sig, state.ir2)


# ---------------------------------------------------------------------------
# the work of a pass, and 64-bit results
# ---------------------------------------------------------------------------
def _paths(case, tris, rays, bands):
    """Segments of a render: a path loses about 0.5 of its log energy per
    segment to walls and air, down to the cut-off; and the operations of a
    segment: two walks (the next hit, the receiver's sight) of about two box
    pairs per level of a binary tree and two triangles, and the surface."""
    seg = rays * bands * min(case["bounces"], 18.4 / 0.5)
    levels = max(1.0, math.log2(tris / 2.0))
    return seg * (2.0 * (levels * 2 * 24.0 + 2 * 45.0) + 200.0)


def work(case):
    do = case["do"]
    if do == "convolve":
        n = max(1, case["n_ir"] + case["n_sig"])
        k = 2 if case["fade"] else 1
        # 2 k forward transforms and one inverse, 2.5 n log2 n each (real input)
        return {"bytes": 4.0 * (k * case["n_ir"] + case["n_sig"] + n),
                "flops": (2 * k + 1) * 2.5 * n * math.log2(n) + 8.0 * k * n}
    if do == "query":
        return {"bytes": case["n"] * (12.0 * 4 + 9.0) + 38.0 * case["tris"],
                "flops": case["n"] * 2.0 * (math.log2(case["tris"]) * 48.0 + 90.0)}
    if do in ("batch", "backrooms"):
        # log-uniform sizes: the mean of a log-uniform in [lo, hi]
        hi, lo = case["rays"], max(1_000, case["rays"] // 30)
        rays = case["rooms"] * (hi - lo) / math.log(hi / lo)
        tris = (case["tris"] - 12) / math.log(case["tris"] / 12.0)
        one = 3 * case["bins"] * 8.0  # histograms out, or adjoints in
        flops = _paths(case, tris, rays, 3)
        return {"bytes": case["rooms"] * (38.0 * tris + one),
                "flops": flops * (2.0 if do == "backrooms" else 1.0)}  # a gradient's weights about double a path's
    if do == "backward":
        return {"bytes": 12 * 38.0 + 3 * case["bins"] * 8.0, "flops": 2.0 * _paths(case, 12, case["rays"], 3)}
    if do == "frames":
        return {"bytes": 38.0 * case["tris"] + case["frames"] * case["bands"] * 2 * case["bins"] * 8.0,
                "flops": _paths(case, case["tris"], case["frames"] * case["rays"], case["bands"])}
    ch = (2 if case["scene"] == "hall" else 1) + sum(2 if i % 2 else 1 for i in range(1, case.get("recorders", 1)))
    per = 48.0 if case.get("raw") else 16.0  # a bin's value and |value|, and the exact sums of both
    flops = _paths(case, case["tris"], case["rays"], case["bands"])
    if do == "open":
        flops += case["tris"] * math.log2(case["tris"]) * 60.0  # the tree's splits
    return {"bytes": 38.0 * case["tris"] + case["bands"] * ch * case["bins"] * per, "flops": flops}


def _closest64(tris, o, d):
    """Mesh::RayIntersection's nearest hit by a scan of all triangles."""
    v0 = tris[:, 0].astype(np.float64)
    e1 = tris[:, 1].astype(np.float64) - v0
    e2 = tris[:, 2].astype(np.float64) - v0
    t = np.zeros(len(o))
    for i in range(len(o)):
        p = np.cross(d[i], e2)
        det = np.einsum("ij,ij->i", e1, p)
        ok = np.abs(det) >= 1e-5
        inv = 1.0 / np.where(ok, det, 1.0)
        s = o[i] - v0
        u = np.einsum("ij,ij->i", s, p) * inv
        q = np.cross(s, e1)
        v = (q @ d[i]) * inv
        tt = np.einsum("ij,ij->i", e2, q) * inv
        ok &= (u >= 0) & (u <= 1) & (v >= 0) & (u + v <= 1) & (tt > 0.001) & (tt < 1e6)
        if ok.any():
            t[i] = tt[ok].min()
    return t


def exact(case, seed):
    seed = int(seed) & 0x7FFFFFFF
    rng = np.random.default_rng([seed, 3])
    if case["do"] == "query" and case["n"] * (case["tris"] + 300.0) < 2e8:
        s = _scene(case, seed)
        o, d, _ = _query_rays(case, s, rng)
        return dict(t=_closest64(s["tris"], o.astype(np.float64), d.astype(np.float64)), tri=None, occluded=None)
    if case["do"] != "convolve":
        return None
    ir, ir2, sig = _tracks(case, rng)
    n_out = case["n_ir"] + case["n_sig"] + 1
    n = 1 << (n_out - 1).bit_length()

    def conv(a, b):
        return np.fft.irfft(np.fft.rfft(a.astype(np.float64), n) * np.fft.rfft(b.astype(np.float64), n), n)[:n_out]

    if ir2 is None:
        return conv(ir, sig)
    # the reference's fades are running binary32 sums (src/Recorder.cpp:172-181)
    df = np.float32(1.0) / np.float32(max(1, len(sig)))
    step = np.full(len(sig), df, np.float32)
    down, up = -step, step.copy()
    down[0], up[0] = 1.0, 0.0
    fade = lambda f: sig * np.cumsum(f, dtype=np.float32)  # noqa: E731  (binary32 products, as the signal itself is)
    return conv(ir, fade(down)) + conv(ir2, fade(up))
