"""GPU: the box test of the walk tree (closest_walk) where its margin is the
question: scenes whose span is far above the geometry's size, directions and
limits that lisa_trace_rays takes but no path makes.  Bar: the oracle's hits
bit for bit, and no render slower than the counting one, which walks the
Morton tree.
"""
import numpy as np
import pytest

from tests.scene_util import camera, cornell, random_rays
from tests.test_gpu_walk_tree import _same

pytestmark = pytest.mark.gpu


def _far_quad(sc, d):
    """The scene and an emitting quad d above it."""
    s = 0.05 * d
    q = np.float32([[-s, d, -s, s, d, -s, s, d, s], [-s, d, -s, s, d, s, -s, d, s]])
    mats = list(sc["materials"])
    m = np.concatenate([sc["mat_idx"], np.full(2, len(mats))]).astype(np.int32)
    mats.append({"diffuse": (0, 0, 0), "alpha": 1.0, "emit": True, "emission": (3.0, 3.0, 3.0)})
    return np.concatenate([sc["verts"], q]), np.concatenate([sc["normals"], np.tile(np.float32([0, -1, 0]), (2, 3))]), \
        m, mats


@pytest.mark.parametrize("d", [1e3, 1e5, 1e6])
def test_hits_with_a_far_quad(capi, oracle_mod, d):
    sc = cornell(32, 16, 16, 16, 1, 1)
    v, n, m, mats = _far_quad(sc, d)
    o = oracle_mod.Scene(v, n, m, mats)
    O, D = random_rays(6144, seed=int(d) % 97)
    D[:512, 0] = 0.0
    D[512:1024, 1:] = 0.0
    D[1024:1536, 2] = 1e-30
    O[256:768] = np.round(O[256:768] * 8) / 8  # the walls' and boxes' planes among them
    O[:128, 0] = 0.0
    D[2048:3072] = (np.float32([0, d, 0]) - O[2048:3072]) / np.float32(d)  # at the quad
    O[3072:4096] += np.float32([0, d, 0]) * np.float32(0.999)  # from under the quad
    D[3584:4096] = O[:512] - O[3584:4096]  # back at the box, long directions
    with capi.Context(0) as ctx:
        ctx.set_wide_threshold(0)
        ctx.set_scene(v, n, m, mats)
        gp, gt = ctx.trace_rays(O, D)
        rp, rt, _ = o.closest_hit(O, D, threads=8)
        assert (rp >= 0).mean() > 0.5
        assert np.array_equal(gp, rp) and _same(gt, rt)


def test_a_far_quad_costs_no_boxes(capi):
    """A margin of the scene's span made every box near a ray pass (26 times the
    time of the counting render)."""
    sc = cornell(256, 128, 256, 256, 2, 5)
    v, n, m, mats = _far_quad(sc, 1e5)
    U, V, W = camera(sc, capi)
    with capi.Context(0) as ctx:
        ctx.set_scene(v, n, m, mats)
        ms, img = {}, {}
        for flags in (0, capi.FLAG_COUNT):
            p = capi.render_params(256, 256, 2, 5, sc["camera"]["eye"], U, V, W, flags=flags)
            for _ in range(3):
                img[flags], _ = ctx.render(p)
                ms[flags] = min(ms.get(flags, 1e9), ctx.stats()["render_ms"])
        print(ms, flush=True)
        assert _same(img[0], img[capi.FLAG_COUNT])
        assert ms[0] < 1.5 * ms[capi.FLAG_COUNT]


@pytest.mark.parametrize("scale,tmin", [(1e-9, 1e-4), (1e-25, 1e-4), (1e-33, 1e-4), (1e-36, 1.0), (1e30, 1e-34), (1.0, -1.0),
                                        (1.0, 0.0)])
def test_directions_and_limits_no_path_makes(capi, oracle_mod, scale, tmin):
    sc = cornell(32, 16, 16, 16, 1, 1)
    o = oracle_mod.Scene(sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"])
    O, D = random_rays(2048, seed=8)
    D = (D * np.float32(scale)).astype(np.float32)
    with capi.Context(0) as ctx:
        ctx.set_wide_threshold(0)
        ctx.set_scene(sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"])
        gp, gt = ctx.trace_rays(O, D, tmin=tmin, tmax=3e38)
        ctx.set_wide_threshold(1 << 62)
        ctx.set_scene(sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"])
        bp, bt = ctx.trace_rays(O, D, tmin=tmin, tmax=3e38)
        rp, rt, _ = o.closest_hit(O, D, tmin=tmin, tmax=3e38, threads=8)
        assert np.array_equal(bp, rp) and _same(bt, rt)
        assert (rp >= 0).mean() > 0.5
        assert np.array_equal(gp, rp) and _same(gt, rt)
