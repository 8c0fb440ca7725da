"""GPU: the agglomerated 4-wide tree that the path kernels walk.

Bar: hit ids and t of lisa_trace_rays (which walks it from
the wide threshold on) equal the oracle's brute-force loop bit for bit, and a render equals
the counting build's, which walks the Morton tree, bit for bit -- at triangle
counts around the clustering's workgroup sizes, with equal boxes, NaN and
infinite vertices, rays along axes and from far away, and after both kinds of
vertex update.
"""
import numpy as np
import pytest

from lisa_amd import scenes
from tests.scene_util import DeviceArray, camera, cornell, random_rays

pytestmark = pytest.mark.gpu

MATS = [{"diffuse": (0.7, 0.6, 0.5), "alpha": 1.0, "roughness": 1.0},
        {"diffuse": (0, 0, 0), "alpha": 1.0, "emit": True, "emission": (3.0, 3.0, 3.0)}]


def _same(a, b):
    return np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32))


def _soup(T, seed):
    """T triangles of sizes over three orders of magnitude in the unit box; every
    fifth emits."""
    rs = np.random.default_rng(seed)
    c = rs.uniform(-0.5, 0.5, (T, 1, 3))
    v = c + rs.normal(size=(T, 3, 3)) * 10.0 ** rs.uniform(-3, 0, (T, 1, 1)) * 0.3
    n = np.tile(np.float32([0, 1, 0]), (T, 3))
    return v.astype(np.float32).reshape(T, 9), n, (np.arange(T) % 5 == 4).astype(np.int32)


def _both(capi, ctx, W=40, H=32, spp=2, bounces=5, eye=(0.0, 0.1, 1.6)):
    U, V, Wv = capi.camera_uvw(eye, (0.0, 0.0, 0.0), 50.0, W / H)
    a, _ = ctx.render(capi.render_params(W, H, spp, bounces, eye, U, V, Wv))
    b, _ = ctx.render(capi.render_params(W, H, spp, bounces, eye, U, V, Wv, flags=capi.FLAG_COUNT))
    return a, b


# one workgroup's 1024 clusters, its 64 outputs, a second and a third pass
@pytest.mark.parametrize("T", [1, 2, 3, 5, 63, 64, 65, 1023, 1024, 1025, 2049, 16384, 16385])
def test_triangle_counts(capi, oracle_mod, T):
    v, n, m = _soup(T, T)
    o = oracle_mod.Scene(v, n, m, MATS)
    O, D = random_rays(1024, seed=T)
    with capi.Context(0) as ctx:
        ctx.set_wide_threshold(0)
        ctx.set_scene(v, n, m, MATS)
        assert ctx.stats()["wide_tree"]
        gp, gt = ctx.trace_rays(O, D)
        rp, rt, _ = o.closest_hit(O, D, brute=True)
        assert np.array_equal(gp, rp) and _same(gt, rt)
        assert _same(*_both(capi, ctx))


def test_equal_boxes_and_slivers(capi, oracle_mod):
    """3000 copies of one triangle, a row of equal ones and long slivers among
    them: ties of every neighbour, and boxes that span the scene."""
    rs = np.random.default_rng(1)
    one = np.tile(np.float32([[0, 0, 0, 0.1, 0, 0, 0, 0.1, 0.02]]), (3000, 1))
    row = np.tile(np.float32([[0, 0, 0, 0.01, 0, 0, 0, 0.01, 0]]), (2000, 1))
    row[:, [0, 3, 6]] += (np.arange(2000, dtype=np.float32) * 2.0 ** -11)[:, None]
    ends = rs.uniform(-0.5, 0.5, (300, 2, 3))
    sliver = np.concatenate([ends[:, 0], ends[:, 1], ends[:, 1] + 1e-3], 1).astype(np.float32)
    v = np.concatenate([one, row, sliver])
    n, m = np.tile(np.float32([0, 0, 1]), (len(v), 3)), (np.arange(len(v)) % 50 == 0).astype(np.int32)
    o = oracle_mod.Scene(v, n, m, MATS)
    O, D = random_rays(2048, seed=3)
    with capi.Context(0) as ctx:
        ctx.set_wide_threshold(0)
        ctx.set_scene(v, n, m, MATS)
        gp, gt = ctx.trace_rays(O, D)
        rp, rt, _ = o.closest_hit(O, D, brute=True)
        assert (rp >= 0).any() and np.array_equal(gp, rp) and _same(gt, rt)
        assert _same(*_both(capi, ctx))


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_non_finite_vertices(capi, oracle_mod, bad):
    """Non-finite vertices: never hit, and the others' hits stay (an infinite
    box leaves the scene to the Morton tree)."""
    v, n, m = _soup(1500, 9)
    v[::37, 4] = bad
    o = oracle_mod.Scene(v, n, m, MATS)
    O, D = random_rays(1024, seed=9)
    with capi.Context(0) as ctx:
        ctx.set_wide_threshold(0)
        ctx.set_scene(v, n, m, MATS)
        gp, gt = ctx.trace_rays(O, D)
        rp, rt, _ = o.closest_hit(O, D, threads=8)
        assert np.array_equal(gp, rp) and _same(gt, rt)
        assert _same(*_both(capi, ctx))


@pytest.mark.parametrize("scale,shift", [(1.0, 0.0), (1e-4, 0.0), (1e4, 3e4), (1.0, 50.0)])
def test_axis_rays_and_far_origins(capi, oracle_mod, scale, shift):
    """Rays with zero components, origins on box faces and far outside the
    scene, and scenes away from the origin (where the fused box test's margin
    is largest against the boxes)."""
    sc = cornell(32, 16, 16, 16, 1, 1)
    v = (sc["verts"].astype(np.float64) * scale + shift).astype(np.float32)
    o = oracle_mod.Scene(v, sc["normals"], sc["mat_idx"], sc["materials"])
    O, D = random_rays(4096, seed=5)
    D[:512, 0] = 0.0
    D[512:1024, 1:] = 0.0
    D[1024:1536, 2] = 1e-30
    O[256:768] = np.round(O[256:768] * 8) / 8  # grid points: the walls' and boxes' planes among them
    O[1536:2560] = O[1536:2560] - 1000.0 * D[1536:2560]
    D[2560:3072] *= 1e-3
    O = (O.astype(np.float64) * scale + shift).astype(np.float32)
    with capi.Context(0) as ctx:
        ctx.set_wide_threshold(0)
        ctx.set_scene(v, sc["normals"], sc["mat_idx"], sc["materials"])
        gp, gt = ctx.trace_rays(O, D)
        rp, rt, _ = o.closest_hit(O, D, brute=True)
        assert (rp >= 0).mean() > 0.3
        assert np.array_equal(gp, rp) and _same(gt, rt)


@pytest.mark.parametrize("name", ["island", "icosphere", "batch"])
def test_renders_equal_the_morton_walk(capi, name):
    sc = {"island": lambda: scenes.island(n=96, width=64, height=40, bounces=8),
          "icosphere": lambda: scenes.displaced_icosphere(level=5, width=64, height=40, bounces=12),
          "batch": lambda: scenes.batch_scene(2)}[name]()
    with capi.Context(0) as ctx:
        ctx.set_wide_threshold(0)
        ctx.set_scene(sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"])
        U, V, Wv = camera(sc, capi)
        for flags in (0, capi.FLAG_FP64_ACCUM):
            p = capi.render_params(64, 40, 4, sc["bounces"], sc["camera"]["eye"], U, V, Wv, flags=flags)
            a, _ = ctx.render(p)
            p.flags |= capi.FLAG_COUNT
            b, _ = ctx.render(p)
            assert _same(a, b), flags


@pytest.mark.parametrize("T", [1, 1025, 20000])
def test_follows_vertex_updates(capi, oracle_mod, T):
    v, n, m = _soup(T, T + 1)
    w, _, _ = _soup(T, T + 2)
    O, D = random_rays(1024, seed=T)
    with capi.Context(0) as ctx:
        ctx.set_wide_threshold(0)
        ctx.set_scene(v, n, m, MATS)
        for verts, device in ((w, False), (v, True)):
            if device:
                d = DeviceArray(verts)
                try:
                    ctx.update_vertices_noalloc(d.ptr)
                finally:
                    d.free()
            else:
                ctx.update_vertices(verts)
            o = oracle_mod.Scene(verts, n, m, MATS)
            gp, gt = ctx.trace_rays(O, D)
            rp, rt, _ = o.closest_hit(O, D, brute=True)
            assert np.array_equal(gp, rp) and _same(gt, rt)
            assert _same(*_both(capi, ctx))


def test_hits_at_the_edge_of_the_leaf_box(capi, oracle_mod):
    """Rays whose rounded hit lies just past tmin, or just inside a triangle's
    edge, while the Morton walk's test of the leaf's own box fails (or just
    passes): the Morton walk's answer.  Large flat quads among small ones give t
    a relative error near 1e-3."""
    rs = np.random.default_rng(7)
    q = np.float32([[-1.6, 0, -1.6, -1.6, 0, 1.6, 1.6, 0, 1.6], [-1.6, 0, -1.6, 1.6, 0, 1.6, 1.6, 0, -1.6]])
    small, n, _ = _soup(400, 7)
    v = np.concatenate([q, small * 0.1 + np.float32([0.0, -1.5, 0.0] * 3)])
    n, m = np.tile(np.float32([0, 1, 0]), (len(v), 3)), np.zeros(len(v), np.int32)
    k = 1 << 20
    D = rs.normal(size=(k, 3))
    D /= np.linalg.norm(D, axis=1, keepdims=True)
    D[:, 1] = np.abs(D[:, 1]) + 0.01
    O = rs.uniform(-1.5, 1.5, (k, 3))
    O[:, 1] = -D[:, 1] * 1e-4 * (1.0 + rs.uniform(-2e-3, 2e-3, k))  # t near tmin
    h = k // 2  # the quads' outer edges, from a distance
    P = rs.uniform(-1.6, 1.6, (h, 3))
    P[:, 0] = np.where(rs.random(h) < 0.5, 1.0, -1.0) * np.float64(np.float32(1.6)) * (1 + rs.uniform(-2e-7, 2e-7, h))
    P[:, 1] = 0.0
    O[:h] = P - D[:h] * rs.uniform(0.5, 3.0, (h, 1))
    O, D = O.astype(np.float32), D.astype(np.float32)
    o = oracle_mod.Scene(v, n, m, MATS)
    with capi.Context(0) as ctx:
        ctx.set_wide_threshold(0)
        ctx.set_scene(v, n, m, MATS)
        gp, gt = ctx.trace_rays(O, D)
        rp, rt, _ = o.closest_hit(O, D, threads=16)
        near = (rt > 0) & (rt < 1.1e-4)
        assert near.any() and (~near[h:]).any() and (rp[:h] < 0).any()
        bp, _, _ = o.closest_hit(O[h:h + 8192], D[h:h + 8192], brute=True)
        assert (bp != rp[h:h + 8192]).any()  # the box does decide some of these
        assert np.array_equal(gp, rp) and _same(gt, rt)
