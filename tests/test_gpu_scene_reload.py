"""GPU: scenes set and moved one after the other on one context, whose memory
goes from each to the next, against contexts that see only one of them."""
import numpy as np
import pytest

from tests.test_gpu_walk_tree import MATS, _both, _same, _soup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(20000, 500, 20000, 1, 60000, 59000), (1, 0, 3000, 3001, 2999)])
def test_one_context_many_scenes(capi, sizes):
    with capi.Context(0) as ctx:
        for i, T in enumerate(sizes):
            v, n, m = _soup(max(T, 1), i)
            v, n, m = v[:T], n[:T], m[:T]
            ctx.set_scene(v, n, m, MATS)
            got, counted = _both(capi, ctx)
            with capi.Context(0) as fresh:
                fresh.set_scene(v, n, m, MATS)
                want, _ = _both(capi, fresh)
                assert _same(got, want) and _same(counted, want), T
                assert ctx.stats()["device_bytes"] == fresh.stats()["device_bytes"]
                if T:
                    a, b = ctx.bvh(), fresh.bvh()
                    assert all(np.array_equal(a[k], b[k]) for k in ("morton", "prim", "refs"))
                    assert _same(a["boxes"], b["boxes"])
                    w, _, _ = _soup(T, 100 + i)
                    for c in (ctx, fresh):
                        c.update_vertices(w, n)
                    assert _same(_both(capi, ctx)[0], _both(capi, fresh)[0])
