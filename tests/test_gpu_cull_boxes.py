"""GPU: NEE tries culled by the boxes of the emitters' tree (nee_scan with
SceneView::cull) or by none, where a scene's one cull box lies loosely about its
emitters.  Bar: the counting build's image, which culls each try by the one box,
bit for bit, through every form of the plain render and in batches; cache
queries and training rows equal the oracle's; and no slower than that build,
whose rounds it saves.
"""
import numpy as np
import pytest

from tests.scene_util import camera, cornell
from tests.test_gpu_nee_tries import _quad

pytestmark = pytest.mark.gpu


def _lights(name):
    rs = np.random.default_rng(12)
    if name == "corners":
        return [_quad((-0.45, -0.45, -0.45), 0.01, 1), _quad((0.45, 0.45, 0.45), 0.01, 1)]
    if name == "touching":  # at the walls, one of them in the room's corner
        return [_quad((0.5, 0.0, 0.0), 0.02, 0), _quad((-0.5, -0.5, -0.5), 0.03, 2), _quad((0, -0.5, 0.3), 0.01, 1)]
    if name == "lamps":
        return [_quad((x, 0.48, z), 0.03, 1) for x in (-0.4, 0, 0.4) for z in (-0.4, 0, 0.4)]
    if name == "far":
        return [_quad((0.0, 0.47, 0.0), 0.1, 1), _quad((0.0, 1e5, 0.0), 5e3, 1)]
    if name == "slivers":
        a = rs.uniform(-0.45, 0.45, (6, 3))
        return [np.concatenate([p, p + rs.normal(size=3) * 0.05, p + 1e-4])[None] for p in a]
    if name == "nan":
        q = [_quad(rs.uniform(-0.45, 0.45, 3), 0.02, k % 3) for k in range(5)]
        q[2][0, 4] = np.nan
        return q
    if name == "sun and sphere":  # a batch scene's: the one box serves better, or a box each
        from lisa_amd import scenes
        return [_quad((0.0, 0.49, 0.0), 0.3, 1),
                scenes.displaced_icosphere(2)["verts"].reshape(-1, 9) * np.float32(0.1) + np.float32([0.2, -0.2, 0.1] * 3)]
    if name == "none":
        return []
    return [_quad(rs.uniform(-0.45, 0.45, 3), 0.02, int(rs.integers(3))) for _ in range(int(name))]


def _scene(name, seg=16, rings=8, W=40, spp=6, bounces=6):
    sc = dict(cornell(seg, rings, W, W, spp, bounces))
    keep = sc["mat_idx"] != 4  # without the box's own light
    q = _lights(name)
    lv = np.concatenate(q).astype(np.float32) if q else np.zeros((0, 9), np.float32)
    sc["verts"] = np.concatenate([sc["verts"][keep], lv])
    sc["normals"] = np.concatenate([sc["normals"][keep], np.tile(np.float32([0, -1, 0]), (len(lv), 3))])
    sc["mat_idx"] = np.concatenate([sc["mat_idx"][keep], np.full(len(lv), 4, np.int32)])
    return sc


def _same(a, b):
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


# 4, 8 and 9 lights: as many triangles as kCullBoxes and half of it, and one pair more
@pytest.mark.parametrize("name", ["corners", "touching", "lamps", "far", "slivers", "nan", "none", "sun and sphere",
                                  "1", "2", "4", "8", "9", "40"])
def test_image_of_the_counting_build(capi, name):
    sc = _scene(name)
    U, V, W = camera(sc, capi)
    p = lambda **k: capi.render_params(40, 40, 6, 6, sc["camera"]["eye"], U, V, W, **k)  # noqa: E731
    with capi.Context(0) as ctx, capi.Context(0) as plain:
        ctx.set_scene(sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"])
        want, _ = ctx.render(p(flags=capi.FLAG_COUNT))
        assert (want[:, :3] > 0).any() == (name != "none")
        for flags in (0, capi.FLAG_PERSISTENT, capi.FLAG_WAVEFRONT):
            assert _same(ctx.render(p(flags=flags))[0], want), flags
        d, _ = ctx.render(p(flags=capi.FLAG_FP64_ACCUM))
        assert _same(d, ctx.render(p(flags=capi.FLAG_FP64_ACCUM | capi.FLAG_COUNT))[0])
        own = cornell(16, 8, 40, 40, 6, 6)  # a scene that one box serves, in the same batch
        plain.set_scene(own["verts"], own["normals"], own["mat_idx"], own["materials"])
        other, _ = plain.render(p(flags=capi.FLAG_COUNT))
        for form in (0, 1, 2):
            b = capi.Batch([plain, ctx], [p(), p()])
            b.set_config(64, 1, form, 1)
            for _ in range(2):
                b.render()
                assert _same(b.accum(0), other) and _same(b.accum(1), want), form
            b.close()


@pytest.mark.parametrize("name", ["corners", "lamps", "none"])
def test_cache_paths_match_oracle(capi, oracle_mod, name):
    sc = _scene(name, W=64)
    U, V, W = camera(sc, capi)
    eye = sc["camera"]["eye"]
    o = oracle_mod.Scene(sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"])
    px = np.arange(0, 64 * 64, 5, dtype=np.int32)
    with capi.Context(0) as ctx:
        ctx.set_scene(sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"])
        p = capi.render_params(64, 64, 2, 3, eye, U, V, W, subframe=4)
        for emit in (False, True):
            loops = 3 if emit else 1
            cp = capi.cache_frame_params(prefix_bounces=2, flags=capi.CACHE_EMISSION if emit else 0, nee_loops=loops)
            g = capi.cache_trace_queries(ctx, p, cp, px)
            r = o.cache_queries(64, 64, 2, 2, eye, U, V, W, px, subframe=4, threads=8, emit_expect=emit,
                                nee_loops=loops, nee_loops_deep=loops)
            assert g["n"] == r["n"] > 0
            assert np.array_equal(g["item"], r["item"]) and np.array_equal(g["att"], r["att"])


@pytest.mark.parametrize("name", ["corners", "none"])
def test_loose_boxes_cost_no_rounds(capi, name):
    """No longer than the counting build, whose every try's emitter query stays in the
    loop of the tries."""
    sc = _scene(name, 32, 16, W=320, spp=4)
    U, V, W = camera(sc, capi)
    with capi.Context(0) as ctx:
        ctx.set_scene(sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"])
        ms = {}
        for flags in (0, capi.FLAG_COUNT):
            for _ in range(4):
                ctx.render(capi.render_params(320, 320, 4, 7, sc["camera"]["eye"], U, V, W, flags=flags))
                ms[flags] = min(ms.get(flags, 1e9), ctx.stats()["render_ms"])
        print(ms, flush=True)
        assert ms[0] < 0.8 * ms[capi.FLAG_COUNT]


def test_boxes_follow_vertex_updates(capi):
    """Lights that move apart and together again: each update's own boxes, and a batch
    made after it."""
    sc = _scene("4")
    v2 = sc["verts"].copy()
    lights = sc["mat_idx"] == 4
    v2[lights] = np.float32([[0.0, 0.45, 0.0] * 3]) + 0.2 * (v2[lights] - v2[lights][0])
    U, V, W = camera(sc, capi)
    p = lambda **k: capi.render_params(40, 40, 6, 6, sc["camera"]["eye"], U, V, W, **k)  # noqa: E731
    with capi.Context(0) as ctx:
        ctx.set_scene(sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"])
        for v in (v2, sc["verts"], v2):
            ctx.update_vertices(v)
            want, _ = ctx.render(p(flags=capi.FLAG_COUNT))
            assert _same(ctx.render(p())[0], want)
            b = capi.Batch([ctx], [p()])
            b.render()
            assert _same(b.accum(0), want)
            b.close()
