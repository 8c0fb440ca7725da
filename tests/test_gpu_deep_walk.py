"""GPU: walks that need more stack than a lane has in LDS.  Triangles in random
order whose Morton codes a far quad puts into one cell make a tree of boxes that
all overlap: the paused walk's stack goes to private memory and comes back.  Bar:
the counting build's image and the oracle's hits bit for bit, and less time than
the counting render (started over in the Morton tree, such walks took up to four times
as long)."""
import numpy as np
import pytest

from lisa_amd import scenes
from tests.scene_util import camera, random_rays
from tests.test_gpu_walk_margin import _far_quad
from tests.test_gpu_walk_tree import _same

pytestmark = pytest.mark.gpu


def _shuffled(seg, rings):
    sc = scenes.cornell(seg, rings, 96, 96, 1, 5)
    v, n, m, mats = _far_quad(sc, 1e4)
    o = np.random.default_rng(3).permutation(len(v))
    return sc, v[o], n[o], m[o], mats


@pytest.mark.parametrize("seg,rings", [(16, 8), (64, 32), (256, 128)])
def test_deep_walks(capi, oracle_mod, seg, rings):
    sc, v, n, m, mats = _shuffled(seg, rings)
    U, V, W = camera(sc, capi)
    with capi.Context(0) as ctx:
        ctx.set_wide_threshold(0)
        ctx.set_scene(v, n, m, mats)
        ms, img = {}, {}
        for flags in (0, capi.FLAG_PERSISTENT, capi.FLAG_COUNT):
            p = capi.render_params(96, 96, 1, 5, sc["camera"]["eye"], U, V, W, flags=flags)
            for _ in range(2):
                img[flags], _ = ctx.render(p)
                ms[flags] = min(ms.get(flags, 1e9), ctx.stats()["render_ms"])
        print(len(v), ms, flush=True)
        assert _same(img[0], img[capi.FLAG_COUNT]) and _same(img[capi.FLAG_PERSISTENT], img[capi.FLAG_COUNT])
        if seg == 256:
            assert ms[0] < ms[capi.FLAG_COUNT]
        O, D = random_rays(2048, seed=seg)
        gp, gt = ctx.trace_rays(O, D)
        rp, rt, _ = oracle_mod.Scene(v, n, m, mats).closest_hit(O, D, threads=16)
        assert (rp >= 0).mean() > 0.8 and np.array_equal(gp, rp) and _same(gt, rt)
