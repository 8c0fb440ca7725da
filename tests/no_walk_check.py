"""Every form of the path loop on small scenes, as arrays (run as a script by
tests/test_gpu_no_walk.py with LISA_LIBRARY pointing at the build that gives no
scene a walk tree, which is how scenes past the walk tree's node limit render;
the test itself takes the same arrays from the normal build).  Writes them to
the .npz named by the second argument and prints OK."""
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import numpy as np  # noqa: E402

from lisa_amd import capi  # noqa: E402
from tests.scene_util import camera, cornell, random_rays  # noqa: E402

MATS = [{"diffuse": (0.7, 0.6, 0.5), "alpha": 1.0, "roughness": 1.0},
        {"diffuse": (0, 0, 0), "alpha": 1.0, "emit": True, "emission": (3.0, 3.0, 3.0)}]


def _scenes():
    """Name, vertices, normals, material ids, materials, eye, U, V, W: a Cornell
    box with its two light triangles, and a soup whose every fifth triangle
    emits.  In neither is triangle 0 an emitter."""
    sc = cornell(32, 16, 40, 32, 2, 5)
    U, V, W = camera(sc, capi)
    yield "cornell", sc["verts"], sc["normals"], sc["mat_idx"], sc["materials"], sc["camera"]["eye"], U, V, W
    rs = np.random.default_rng(3)
    T = 1500
    c = rs.uniform(-0.5, 0.5, (T, 1, 3))
    v = c + rs.normal(size=(T, 3, 3)) * 10.0 ** rs.uniform(-3, 0, (T, 1, 1)) * 0.3
    eye = (0.0, 0.1, 1.6)
    U, V, W = capi.camera_uvw(eye, (0.0, 0.0, 0.0), 50.0, 40 / 32)
    yield ("soup", v.astype(np.float32).reshape(T, 9), np.tile(np.float32([0, 1, 0]), (T, 3)),
           (np.arange(T) % 5 == 4).astype(np.int32), MATS, eye, U, V, W)


def results(wide):
    """name -> array for each scene and each entry point that walks it; `wide`: with
    the 4-wide form of the Morton tree.  "<scene> counted" is the counting build's
    image, which walks the binary Morton tree in every library."""
    out = {}
    threshold = 0 if wide else 1 << 62
    O, D = random_rays(4096, seed=11)
    for name, v, n, m, mats, eye, U, V, W in _scenes():
        p = lambda spp=2, b=5, **k: capi.render_params(40, 32, spp, b, eye, U, V, W, **k)  # noqa: E731
        with capi.Context(0) as ctx, capi.Context(0) as other:
            for c in (ctx, other):
                c.set_wide_threshold(threshold)
                c.set_scene(v, n, m, mats)
                assert c.stats()["wide_tree"] == wide
            out[name + " counted"] = ctx.render(p(flags=capi.FLAG_COUNT))[0]
            for key, fl in (("plain", 0), ("fp64", capi.FLAG_FP64_ACCUM), ("persistent", capi.FLAG_PERSISTENT),
                            ("wavefront", capi.FLAG_WAVEFRONT)):
                out[f"{name} {key}"] = ctx.render(p(flags=fl))[0]
            out[name + " progressive"] = ctx.render_progressive(p(), 3)
            out[name + " progressive fp64"] = ctx.render_progressive(p(flags=capi.FLAG_FP64_ACCUM), 2)
            prim, t = ctx.trace_rays(O, D)
            out[name + " prim"], out[name + " t"] = prim, t
            for form in (0, 1, 2):
                b = capi.Batch([ctx, other], [p(), p()])
                b.set_config(64, 1, form, 0)
                b.render()
                out[f"{name} batch {form}"] = np.stack([b.accum(0), b.accum(1)])
                b.close()
            px = np.arange(0, 40 * 32, 3, dtype=np.int32)
            for emit in (False, True):
                cp = capi.cache_frame_params(prefix_bounces=2, flags=capi.CACHE_EMISSION if emit else 0,
                                             nee_loops=3 if emit else 1, nee_loops_deep=2 if emit else 1)
                q = capi.cache_trace_queries(ctx, p(2, 3), cp, px)
                for k in ("accum", "feat", "att", "item"):
                    out[f"{name} queries {emit} {k}"] = q[k]
            r = capi.cache_trace_rows(ctx, p(), px)
            out[name + " rows feat"], out[name + " rows target"] = r["feat"], r["tgt"]
            for fl in (capi.CACHE_EMISSION, capi.CACHE_EMISSION | capi.CACHE_PERSISTENT):
                cache = capi.Cache(0, seed=1)
                for f in range(3):
                    cp = capi.cache_frame_params(prefix_bounces=2, train_paths=2000, train_bounces=5, train_steps=2,
                                                 seed=5, flags=fl, nee_loops=4,
                                                 fallback_loss=1e-9 if f == 2 else 0.0)
                    capi.render_cached(ctx, cache, p(subframe=f), cp)
                    out[f"{name} cached {fl} {f}"] = ctx.copy_accum(40 * 32)
                cache.close()
        print(name, "wide" if wide else "binary", "done", flush=True)
    return out


def main():
    assert os.path.samefile(capi.LIB_PATH, sys.argv[1]), capi.LIB_PATH
    np.savez(sys.argv[2], **{f"{w} {k}": a for w in (False, True) for k, a in results(w).items()})
    print("OK", flush=True)


if __name__ == "__main__":
    main()
