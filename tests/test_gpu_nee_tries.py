"""GPU: the NEE tries of the uncounted path kernels, which skip culled tries in
next_try, against the counting build's, which sees each try -- the same image
bit for bit where the emitters are small, large, behind the vertices, around
them, flat on an axis, missing or non-finite, and through every form of the
plain render (the ray-level wavefront form keeps the try-by-try loop)."""
import numpy as np
import pytest

from tests.scene_util import camera, cornell

pytestmark = pytest.mark.gpu


def _quad(c, s, flat):
    """Two triangles of half size s about c, spanning the axes other than `flat`."""
    a, b = [k for k in range(3) if k != flat]
    p = np.tile(np.asarray(c, np.float32), (4, 1))
    for i, (x, y) in enumerate(((-s, -s), (s, -s), (s, s), (-s, s))):
        p[i, a] += x
        p[i, b] += y
    return np.stack([p[[0, 1, 2]], p[[0, 2, 3]]]).reshape(2, 9)


LIGHTS = {"tiny": [((0.1, 0.3, 0.1), 1e-3, 1)], "wall": [((0.0, 0.499, 0.0), 0.5, 1)],
          "two": [((-0.45, 0.2, 0.0), 0.1, 0), ((0.3, -0.45, 0.4), 0.05, 1)],
          "behind": [((0.0, 0.0, 3.0), 0.3, 2)], "around": [((0.0, 1.0, 0.0), 30.0, 1)], "none": []}


@pytest.mark.parametrize("name", sorted(LIGHTS) + ["nan"])
def test_scanned_tries_equal_single_tries(capi, name):
    sc = cornell(16, 8, 40, 40, 8, 6)
    keep = sc["mat_idx"] != 4  # without the box's own light
    lights = LIGHTS.get(name, LIGHTS["two"])
    lv = np.concatenate([_quad(*q) for q in lights]).astype(np.float32) if lights else np.zeros((0, 9), np.float32)
    if name == "nan":
        lv[0, 0] = np.nan
    v = np.concatenate([sc["verts"][keep], lv])
    n = np.concatenate([sc["normals"][keep], np.tile(np.float32([0, -1, 0]), (len(lv), 3))])
    m = np.concatenate([sc["mat_idx"][keep], np.full(len(lv), 4, np.int32)])
    U, V, Wv = camera(sc, capi)
    with capi.Context(0) as ctx:
        ctx.set_scene(v, n, m, sc["materials"])
        p = capi.render_params(40, 40, 8, 6, sc["camera"]["eye"], U, V, Wv, flags=capi.FLAG_COUNT)
        want, _ = ctx.render(p)
        assert name in ("none", "behind") or (want[:, :3] > 0).any()
        for flags in (0, capi.FLAG_PERSISTENT, capi.FLAG_WAVEFRONT):
            p.flags = flags
            got, _ = ctx.render(p)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), flags
