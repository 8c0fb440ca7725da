"""Performance cases: the calls that programs on this path tracer spend their time in.

Each case is one pass through the public interface (`lisa_amd.capi`): plain
renders from a preview subframe to the benchmark frames, progressive runs,
geometry that is set or moved before its frame, several scenes in one batched
launch, frames of the learned radiance cache, and the cache's own inference
and training calls.  Scene sizes, resolutions, sample and bounce counts are
those of the scenes in `lisa_amd.scenes`, of `bench.py` and of the tests, with
ragged image sizes among them.

A case's seed moves the camera, tints the materials and displaces the mesh by
a smooth field, so every seed is another scene of the same size.
"""
import functools
import math

import numpy as np
import torch  # noqa: F401  (its HIP runtime is the process's one; load it first)

from lisa_amd import capi, scenes

# Samples (pixels x spp) that a drawn case may ask for, and its scene sizes.
MAX_SAMPLES = 48 << 20
PARAMS, INPUTS = capi.CACHE_PARAMS, capi.CACHE_INPUTS
_OUT_DIM, _IN_DIM = (64, 64, 64, 64, 16), (160, 64, 64, 64, 64)
_OFFSET = (0, 10240, 14336, 18432, 22528, 23552)
_REAL_IN, _REAL_OUT = (144, 64, 64, 64, 64), (64, 64, 64, 64, 3)


def _case(kind, scene, size, width, height, spp, bounces, **more):
    c = {"kind": kind, "scene": scene, "size": size, "width": width, "height": height,
         "spp": spp, "bounces": bounces, "fp64": False, "rgba8": False, "frames": 1}
    c.update(more)
    return c


def listed():
    def named(name, case):
        return dict(case, name=name)
    return [
        # The display loop (`lisa -d`) on a small window: one subframe of one
        # sample blended into the running mean, shown as bytes.  The smallest
        # call; launch and latency count.
        named("preview_256_1spp", _case("subframe", "cornell", 32, 256, 256, 1, 7, rgba8=True)),
        # `lisa -s scene.rto` on the small Cornell box: the whole image, as
        # the bytes of its PPM.
        named("cornell_small_16spp", _case("render", "cornell", 32, 256, 256, 16, 7, rgba8=True)),
        # The headline benchmark: 65k triangles, 1024^2, 256 samples.
        named("cornell_65k_256spp", _case("render", "cornell", 256, 1024, 1024, 256, 7)),
        # The large-scene benchmark: 5.24M triangles of glass at 1080p.
        named("icosphere_5m_64spp", _case("render", "icosphere", 9, 1920, 1080, 64, 12)),
        # A reference render in FP64 sums over an open landscape (2.1M
        # triangles): one of its many subframes.
        named("island_fp64_subframe", _case("subframe", "island", 1024, 1920, 1080, 8, 12, fp64=True)),
        # An image refined offline: a run of subframes in one graph launch,
        # at an odd size.
        named("progressive_24x2spp", _case("progressive", "icosphere", 6, 513, 389, 2, 12, frames=24)),
        # Animation: new vertex positions every frame, then a noisy frame.
        named("animate_82k_4spp", _case("update", "icosphere", 6, 641, 359, 4, 8)),
        # A scene is loaded and its first image drawn.
        named("load_292k_4spp", _case("load", "batch", 0, 384, 384, 4, 8)),
        # Many small scenes in one launch (thumbnails, a render service).
        named("batch_12_scenes", _case("batch", "batch", 12, 0, 0, 16, 8)),
        # The learned cache's frames on the island, trained as they go.
        named("island_cached_4_frames", _case("cached", "island", 1024, 1920, 1080, 4, 12, frames=4)),
        # The cache's network by itself: radiance queries of other renderers,
        # and an online training step on a frame's rows.
        named("cache_infer_262k", {"kind": "infer", "rows": 262144}),
        named("cache_train_65k", {"kind": "train", "rows": 65536}),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["render", "render", "render", "subframe", "progressive", "update", "load",
                       "batch", "cached", "infer", "train"])
    if kind == "infer":
        return {"kind": kind, "rows": _log(rng, 1000, 1000000)}
    if kind == "train":
        return {"kind": kind, "rows": _log(rng, 1000, 65536)}
    scene = rng.choice(["cornell", "icosphere", "island", "batch"])
    if kind == "batch":
        return _case(kind, "batch", rng.randint(2, 12), 0, 0, _log(rng, 1, 16), rng.randint(2, 12))
    if kind == "cached":
        scene = "island"
    size = {"cornell": lambda: _log(rng, 16, 256), "icosphere": lambda: rng.randint(3, 8),
            "island": lambda: _log(rng, 96, 1024), "batch": lambda: rng.randint(0, 11)}[scene]()
    w = _log(rng, 64, 1920)
    h = max(48, min(1080, int(w * rng.uniform(0.5, 1.2))))
    frames = {"progressive": rng.randint(2, 32), "cached": rng.randint(1, 4)}.get(kind, 1)
    most = {"cached": 8, "update": 16, "load": 16, "progressive": 8, "subframe": 16}.get(kind, 256)
    spp = _log(rng, 1, max(1, min(most, MAX_SAMPLES // (w * h * frames))))
    return _case(kind, scene, size, w, h, spp, rng.randint(3, 12), frames=frames,
                 fp64=kind in ("subframe", "progressive") and rng.random() < 0.3,
                 rgba8=kind in ("render", "subframe") and rng.random() < 0.3)


@functools.lru_cache(maxsize=None)
def _base(scene, size):
    if scene == "cornell":
        return scenes.cornell(size, max(size // 2, 3))
    if scene == "icosphere":
        return scenes.displaced_icosphere(size)
    if scene == "island":
        return scenes.island(size)
    return scenes.batch_scene(size)


def _moved(base, rs):
    """The scene's vertices under a smooth seeded displacement; its light and its
    largest (flat) triangles stay where they are."""
    v = base["verts"].reshape(-1, 3, 3)
    lo, hi = v.reshape(-1, 3).min(0), v.reshape(-1, 3).max(0)
    extent = v.max(1) - v.min(1)
    small = (extent.max(1) < 0.1 * float((hi - lo).max())).astype(np.float32)
    f = rs.uniform(2.0, 5.0, 2).astype(np.float32)
    ph = np.float32(rs.uniform(0.0, 2.0 * np.pi))
    a = np.float32(0.01 * (hi[1] - lo[1]))
    out = v.copy()
    out[:, :, 1] += a * small[:, None] * np.sin(f[0] * v[:, :, 0] + f[1] * v[:, :, 2] + ph)
    return out.reshape(-1, 9)


def _tinted(base, rs):
    mats = []
    for m in base["materials"]:
        m = dict(m)
        k = rs.uniform(0.8, 1.0, 3)
        key = "emission" if m.get("emit") else "diffuse"
        m[key] = tuple(float(x * y) for x, y in zip(m[key], k))
        mats.append(m)
    return mats


def _view(base, rs, width, height, spp, bounces, subframe=0, flags=0):
    cam = base["camera"]
    eye = np.asarray(cam["eye"], np.float64) + rs.uniform(-0.05, 0.05, 3)
    look = np.asarray(cam["look_at"], np.float64) + rs.uniform(-0.02, 0.02, 3)
    U, V, W = capi.camera_uvw(eye, look, cam["fov"], width / height)
    return capi.render_params(width, height, spp, bounces, eye, U, V, W, subframe=subframe, flags=flags)


def _scene_context(base, rs):
    verts, mats = _moved(base, rs), _tinted(base, rs)
    ctx = capi.Context(0)
    ctx.set_scene(verts, base["normals"], base["mat_idx"], mats)
    return ctx


def _weights(rs):
    """He-uniform weights in the packed layout of the cache's network."""
    w = np.zeros(PARAMS, np.float32)
    for l in range(5):
        a = math.sqrt(6.0 / _REAL_IN[l])
        m = w[_OFFSET[l]:_OFFSET[l + 1]].reshape(_OUT_DIM[l], _IN_DIM[l])
        m[:_REAL_OUT[l], :_REAL_IN[l]] = rs.uniform(-a, a, (_REAL_OUT[l], _REAL_IN[l]))
    return w


def _rows(rs, n):
    """Surface-hit features: positions, directions, normals, albedo, roughness, and one
    hit in eight on glass."""
    f = rs.random((n, INPUTS), dtype=np.float32)
    glass = rs.random(n) < 0.125
    f[:, 10] = np.where(glass, 0.0, 1.0)
    f[:, 11] = glass
    return f


def _targets(rs, f):
    """Radiance that follows the features, with a path tracer's noise about it."""
    base = 0.3 + 0.25 * np.sin(6.0 * f[:, 0:1] + 4.0 * f[:, 2:3]) + 0.3 * f[:, 7:10]
    noise = np.exp(0.5 * rs.standard_normal((f.shape[0], 3)) - 0.125)
    return np.maximum(base * noise, 0.0).astype(np.float32)


def _cache_inputs(case, seed):
    rs = np.random.default_rng([seed, 77])
    w = _weights(rs)
    f = _rows(rs, case["rows"])
    return w, f, _targets(rs, f)


def prepare(case, seed):
    rs = np.random.default_rng([seed, 11])
    kind = case["kind"]
    st = {"case": case, "frame": 0}
    if kind in ("infer", "train"):
        w, f, t = _cache_inputs(case, seed)
        st["cache"] = capi.Cache(0, seed=1)
        st["cache"].set_weights(w)
        st["feat"], st["target"] = f, t
        return st
    spp, bounces = case["spp"], case["bounces"]
    if kind == "batch":
        ctxs, params = [], []
        for i in range(case["size"]):
            base = _base("batch", i)
            ctxs.append(_scene_context(base, rs))
            params.append(_view(base, rs, base["width"], base["height"], spp, bounces))
        st["ctxs"] = ctxs
        st["batch"] = capi.Batch(ctxs, params)
        return st
    base = _base(case["scene"], case["size"])
    flags = capi.FLAG_FP64_ACCUM if case["fp64"] else 0
    if kind == "load":
        st["mesh"] = (_moved(base, rs), base["normals"], base["mat_idx"], _tinted(base, rs))
        st["ctx"] = capi.Context(0)
    else:
        st["ctx"] = _scene_context(base, rs)
        if kind == "update":
            st["verts"] = [_moved(base, rs) for _ in range(2)]
    st["view"] = _view(base, rs, case["width"], case["height"], spp, bounces, flags=flags)
    if kind == "subframe":  # the image's first subframe is there already
        st["ctx"].render(st["view"], want_accum=False)
        st["frame"] = 1
    if kind == "cached":
        st["cache"] = capi.Cache(0, seed=1)
        st["cparams"] = capi.cache_frame_params(
            prefix_bounces=2, train_paths=262144, train_bounces=bounces, train_max=1 << 16, train_steps=8,
            seed=3, flags=capi.CACHE_EMISSION, nee_loops=8, nee_loops_deep=1)
    return st


def run(st):
    case, kind = st["case"], st["case"]["kind"]
    if kind == "infer":
        return st["cache"].infer(st["feat"])
    if kind == "train":
        loss = st["cache"].train(st["feat"], st["target"])
        return {"loss": loss, "weights": st["cache"].weights()}
    if kind == "batch":
        st["batch"].render()
        return [st["batch"].accum(i) for i in range(case["size"])]
    ctx, view = st["ctx"], st["view"]
    if kind == "render":
        return _image(ctx.render(view, want_rgba8=case["rgba8"]))
    if kind == "subframe":
        view.subframe = st["frame"]
        st["frame"] += 1
        return _image(ctx.render(view, want_rgba8=case["rgba8"]))
    if kind == "progressive":
        view.subframe = 0
        return ctx.render_progressive(view, case["frames"])
    if kind == "update":
        ctx.update_vertices(st["verts"][st["frame"] % 2])
        st["frame"] += 1
        return _image(ctx.render(view))
    if kind == "load":
        ctx.set_scene(*st["mesh"])
        return _image(ctx.render(view))
    for _ in range(case["frames"]):  # cached
        view.subframe = st["frame"]
        st["frame"] += 1
        capi.render_cached(ctx, st["cache"], view, st["cparams"])
    return ctx.copy_accum(case["width"] * case["height"])


def _image(out):
    acc, rgb = out
    return {"accum": acc} if rgb is None else {"accum": acc, "rgba8": rgb}


# Operations of one sample that no scheme of this path tracer does without,
# as an estimate: about four radiance rays, each a walk of log2(triangles)
# box tests (about 20 operations) to its hit and one triangle test and shading
# (about 150), and at each of two diffuse hits the reference's up to thirty
# hemisphere draws against the emitters (about 20 each).
def _sample_flops(tris):
    return 4.0 * (20.0 * math.log2(max(tris, 2)) + 150.0) + 2 * 30 * 20.0


_NET_FLOPS = 2.0 * 21696  # one forward pass of the network


def work(case):
    kind = case["kind"]
    if kind == "infer":
        return {"bytes": case["rows"] * 4.0 * (INPUTS + 3), "flops": case["rows"] * _NET_FLOPS}
    if kind == "train":
        return {"bytes": case["rows"] * 4.0 * (INPUTS + 3) + 7 * 4.0 * PARAMS,
                "flops": case["rows"] * 3 * _NET_FLOPS}
    if kind == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        for i in range(case["size"]):
            base = _base("batch", i)
            tris, px = base["verts"].shape[0], base["width"] * base["height"]
            total["bytes"] += tris * 76.0 + px * 16.0
            total["flops"] += px * case["spp"] * _sample_flops(tris)
        return total
    tris = _base(case["scene"], case["size"])["verts"].shape[0]
    px = case["width"] * case["height"]
    samples = px * case["spp"] * case["frames"]
    flops = samples * _sample_flops(tris)
    if kind == "cached":  # 62k rows x 8 steps, and a query for every fourth sample
        flops += case["frames"] * 62000 * 8 * 3 * _NET_FLOPS + 0.25 * samples * _NET_FLOPS
    image = 16.0 + (4.0 if case["rgba8"] else 0.0) + (16.0 if kind == "subframe" else 0.0) \
        + (64.0 if case["fp64"] else 0.0)
    return {"bytes": tris * 76.0 + px * image, "flops": flops}


# ---------------------------------------------------------------------------
# 64-bit values.  A path-traced image has none: its value is defined by the
# FP32 operations and the random stream of every path, and is held to the
# images of the code itself.
# ---------------------------------------------------------------------------
def _forward(w, feat):
    p = feat.astype(np.float64)
    ang = np.pi * p[:, :, None] * (2.0 ** np.arange(6))
    h = np.zeros((p.shape[0], 160))
    h[:, :144] = np.stack([np.sin(ang), np.cos(ang)], -1).reshape(p.shape[0], 144)
    acts = [h]
    for l in range(4):
        W = w[_OFFSET[l]:_OFFSET[l + 1]].reshape(_OUT_DIM[l], _IN_DIM[l])
        h = np.maximum(h @ W.T, 0.0)
        acts.append(h)
    W = w[_OFFSET[4]:_OFFSET[5]].reshape(_OUT_DIM[4], _IN_DIM[4])
    return (h @ W.T)[:, :3], acts


def exact(case, seed):
    if case["kind"] not in ("infer", "train"):
        return None
    w, f, t = _cache_inputs(case, seed)
    w = w.astype(np.float64)
    if case["kind"] == "infer":
        return np.concatenate([_forward(w, f[i:i + 65536])[0] for i in range(0, f.shape[0], 65536)])
    y, acts = _forward(w, f)
    n = y.shape[0]
    den = y * y + 0.01
    loss = float((((y - t) ** 2) / den).sum() / (3 * n))
    dz = np.zeros((n, 16))
    dz[:, :3] = 2.0 * (y - t) / den / (3.0 * n)
    new = w.copy()
    for l in range(4, -1, -1):
        sl = slice(_OFFSET[l], _OFFSET[l + 1])
        W = w[sl].reshape(_OUT_DIM[l], _IN_DIM[l])
        g = np.zeros_like(W)
        g[:_REAL_OUT[l], :_REAL_IN[l]] = (dz.T @ acts[l])[:_REAL_OUT[l], :_REAL_IN[l]]
        # Adam's first step: both moments bias-corrected to g and g^2
        new[sl] = (W - 1e-3 * g / (np.abs(g) + 1e-8)).reshape(-1)
        if l > 0:
            dz = (dz @ W) * (acts[l] > 0)
    return {"loss": loss, "weights": new}
