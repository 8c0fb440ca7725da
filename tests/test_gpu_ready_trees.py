"""GPU: the tree that the walks take is brought up to date by the first call that
needs it after a vertex update, whichever call that is: each entry point straight
after an update gives, bit for bit, what it gives on a context that has rendered
since, with a walk tree, and where an infinite vertex leaves the scene to the
Morton trees and their 4-wide form.  An update alone does not build it.
"""
import numpy as np
import pytest

from tests.scene_util import DeviceArray, camera, cornell, random_rays

pytestmark = pytest.mark.gpu

W, H = 48, 40


def _same(a, b):
    return a.shape == b.shape and a.tobytes() == b.tobytes()


def _calls(capi, p):
    px = np.arange(0, W * H, 3, dtype=np.int32)
    O, D = random_rays(4096, seed=2)

    def batch(c, form):
        b = capi.Batch([c], [p()])
        b.set_config(64, 1, form, 0)
        b.render()
        out = b.accum(0)
        b.close()
        return out

    def cached(c, flags, frames):
        cache = capi.Cache(0, seed=1)
        cp = capi.cache_frame_params(prefix_bounces=2, train_paths=3000, train_bounces=6, train_steps=2, seed=5,
                                     flags=flags, nee_loops=2 if flags & capi.CACHE_EMISSION else 1)
        for f in range(frames):
            capi.render_cached(c, cache, p(subframe=f), cp)
        out = np.concatenate([c.copy_accum(W * H).reshape(-1), cache.weights()])
        cache.close()
        return out

    def queries(c, flags):
        q = capi.cache_trace_queries(c, p(), capi.cache_frame_params(prefix_bounces=2, flags=flags), px)
        return np.concatenate([q["accum"].reshape(-1), q["att"].reshape(-1)])

    return {
        "plain": lambda c: c.render(p())[0],
        "fp64": lambda c: c.render(p(flags=capi.FLAG_FP64_ACCUM))[0],
        "persistent": lambda c: c.render(p(flags=capi.FLAG_PERSISTENT))[0],
        "wavefront": lambda c: c.render(p(flags=capi.FLAG_WAVEFRONT))[0],
        "progressive": lambda c: c.render_progressive(p(), 3),
        "batch 0": lambda c: batch(c, 0), "batch 1": lambda c: batch(c, 1), "batch 2": lambda c: batch(c, 2),
        "queries": lambda c: queries(c, 0), "queries emit": lambda c: queries(c, capi.CACHE_EMISSION),
        "rows": lambda c: capi.cache_trace_rows(c, p(), px)["tgt"],
        "cached": lambda c: cached(c, capi.CACHE_EMISSION, 2),
        "cached serial": lambda c: cached(c, capi.CACHE_SERIAL, 1),
        "cached persistent": lambda c: cached(c, capi.CACHE_PERSISTENT, 1),
        "rays": lambda c: np.stack([x.view(np.uint32) for x in c.trace_rays(O, D)]),
    }


@pytest.mark.parametrize("inf", [False, True])
def test_first_call_after_an_update(capi, inf):
    sc = cornell(64, 32, W, H, 2, 6)
    U, V, Wv = camera(sc, capi)
    p = lambda **k: capi.render_params(W, H, 2, 6, sc["camera"]["eye"], U, V, Wv, **k)  # noqa: E731
    calls = _calls(capi, p)
    rs = np.random.default_rng(4)
    with capi.Context(0) as ctx, capi.Context(0) as ref:
        for c in (ctx, ref):
            c.set_wide_threshold(0)
            c.set_scene(sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"])
            c.render(p())
        for i, (name, call) in enumerate(calls.items()):
            v = (sc["verts"] + rs.normal(scale=0.05, size=sc["verts"].shape)).astype(np.float32)
            if inf:
                v[7, 4] = np.inf
            if i % 2:
                d = DeviceArray(v)
                try:
                    ctx.update_vertices_noalloc(d.ptr)
                finally:
                    d.free()
            else:
                ctx.update_vertices(v)
            ref.update_vertices(v)
            a, _ = ref.render(p())
            b, _ = ref.render(p(flags=capi.FLAG_COUNT))
            assert _same(a, b), name
            assert _same(call(ctx), call(ref)), name


def test_an_update_alone_clusters_nothing(capi):
    """The clustering took three fifths of an update's device time."""
    sc = cornell(256, 128, W, H, 1, 3)
    d = DeviceArray(sc["verts"])
    try:
        with capi.Context(0) as ctx:
            ctx.set_scene(sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"])
            U, V, Wv = camera(sc, capi)
            p = capi.render_params(W, H, 1, 3, sc["camera"]["eye"], U, V, Wv)
            up, after, again = [], [], []
            for _ in range(5):
                ctx.update_vertices_noalloc(d.ptr)
                up.append(ctx.stats()["bvh_build_ms"])
                for to in (after, again):
                    ctx.render(p)
                    to.append(ctx.stats()["render_ms"])
            print(min(up), min(after), min(again), flush=True)
            assert min(up) < min(after) - min(again)
    finally:
        d.free()
