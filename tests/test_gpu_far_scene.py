"""GPU: scenes whose distance from the origin is far above their size.  The walk
tree's planes and the boxes that cull NEE tries are relative to a point of the
scene, so that their margins do not grow with that distance.  Bar: the counting
build's image and the oracle's hits bit for bit, with the scene set there and
moved there, and less time than the counting render, whose walk has no such
margin.
"""
import numpy as np
import pytest

from tests.scene_util import cornell, random_rays
from tests.test_gpu_cull_boxes import _scene
from tests.test_gpu_walk_tree import _same

pytestmark = pytest.mark.gpu


def _moved(sc, far):
    off = np.float64([far, 0.3 * far, -far])
    v = (sc["verts"].reshape(-1, 3).astype(np.float64) + off).astype(np.float32).reshape(-1, 9)
    return off, v


def _images(capi, ctx, sc, off, W=48, spp=2, repeat=1):
    eye, look = (np.asarray(sc["camera"][k], np.float64) + off for k in ("eye", "look_at"))
    U, V, Wv = capi.camera_uvw(eye, look, sc["camera"]["fov"], 1.0)
    img, ms = {}, {}
    for flags in (0, capi.FLAG_WAVEFRONT, capi.FLAG_COUNT):
        for _ in range(repeat):
            img[flags], _ = ctx.render(capi.render_params(W, W, spp, 6, eye, U, V, Wv, flags=flags))
            ms[flags] = min(ms.get(flags, 1e9), ctx.stats()["render_ms"])
    return img[0], img[capi.FLAG_WAVEFRONT], img[capi.FLAG_COUNT], ms[0], ms[capi.FLAG_COUNT]


@pytest.mark.parametrize("far", [-30.0, 1e3, 1e4, 1e6])
@pytest.mark.parametrize("lights", ["one", "corners", "none"])
def test_images_and_hits(capi, oracle_mod, far, lights):
    sc = dict(cornell(32, 16, 48, 48, 2, 6)) if lights == "one" else _scene(lights, 32, 16, W=48)
    off, v = _moved(sc, far)
    O, D = random_rays(4096, seed=6)
    O = (O.astype(np.float64) + off).astype(np.float32)
    D[:256, 0] = 0.0
    D[256:512, 1:] = 0.0
    o = oracle_mod.Scene(v, sc["normals"], sc["mat_idx"], sc["materials"])
    rp, rt, _ = o.closest_hit(O, D, threads=8)
    with capi.Context(0) as ctx:
        ctx.set_wide_threshold(0)
        ctx.set_scene(v, sc["normals"], sc["mat_idx"], sc["materials"])
        for step in range(2):
            gp, gt = ctx.trace_rays(O, D)
            assert np.array_equal(gp, rp) and _same(gt, rt), step
            a, w, b, _, _ = _images(capi, ctx, sc, off)
            assert _same(a, b) and _same(w, b), step
            if step == 0:  # and moved there from the origin
                ctx.set_scene(sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"])
                ctx.update_vertices(v)


def test_distance_costs_no_boxes(capi):
    sc = cornell(256, 128, 320, 320, 4, 6)
    off, v = _moved(sc, 1000.0)
    with capi.Context(0) as ctx:
        ctx.set_scene(v, sc["normals"], sc["mat_idx"], sc["materials"])
        a, _, b, ms, counted = _images(capi, ctx, sc, off, 320, 4, 3)
        print(ms, counted, flush=True)
        assert _same(a, b) and ms < 0.75 * counted
