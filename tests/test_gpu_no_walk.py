"""GPU: scenes without a walk tree (more than 2^25 walk nodes: about 31 million
triangles, or half of that if all emit).  The library built with no room for
walk nodes (lisa_amd/_build/nowalk, made by __graft_entry__.build) renders small
scenes as the normal one renders those: the Morton trees answer every query,
with and without the 4-wide form.  Each form of the path loop gives the normal
build's results bit for bit, and its images equal the counting build's.
"""
import os
import subprocess
import sys

import numpy as np
import pytest

from lisa_amd import build as lb

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def no_walk(tmp_path_factory):
    lib = os.path.join(lb.NO_WALK, "liblisa.so")
    assert os.path.exists(lib), "build the no-walk library first (__graft_entry__.build)"
    to = str(tmp_path_factory.mktemp("nowalk") / "out.npz")
    res = subprocess.run([sys.executable, "-u", os.path.join(HERE, "no_walk_check.py"), lib, to],
                         env=dict(os.environ, LISA_LIBRARY=lib), capture_output=True, text=True, timeout=300)
    print(res.stdout, res.stderr[-3000:], flush=True)
    assert res.returncode == 0 and res.stdout.strip().endswith("OK")
    with np.load(to) as z:
        return {k: z[k] for k in z.files}


def _same(a, b):
    return a.shape == b.shape and a.tobytes() == b.tobytes()


@pytest.mark.parametrize("wide", [False, True])
def test_every_form_without_a_walk_tree(capi, no_walk, wide):
    from tests.no_walk_check import results
    want = results(wide)
    got = {k.split(" ", 1)[1]: a for k, a in no_walk.items() if k.startswith(f"{wide} ")}
    assert sorted(got) == sorted(want)
    assert [k for k in want if not _same(got[k], want[k])] == []
    for name in ("cornell", "soup"):
        counted = got[name + " counted"]
        assert (counted[:, :3] > 0).any()
        for form in ("plain", "persistent", "wavefront"):
            assert _same(got[f"{name} {form}"], counted), (name, form)


def test_hits_without_a_walk_tree(capi, oracle_mod, no_walk):
    """lisa_trace_rays from the binary and from the 4-wide Morton walk."""
    from tests import no_walk_check as c
    from tests.scene_util import random_rays
    O, D = random_rays(4096, seed=11)
    for name, v, n, m, mats, *_ in c._scenes():
        rp, rt, _ = oracle_mod.Scene(v, n, m, mats).closest_hit(O, D, brute=True)
        for wide in (False, True):
            assert _same(no_walk[f"{wide} {name} prim"], rp) and _same(no_walk[f"{wide} {name} t"], rt)


def test_an_infinite_vertex_costs_no_rounds(capi):
    """A scene that loses its walk tree to an infinite vertex, and with it the cull of
    NEE tries: the render takes no longer than the counting one, which walks the
    same trees (left to the round's walk, each try's emitter query made it take four
    times as long)."""
    from lisa_amd import scenes
    from tests.scene_util import camera
    sc = scenes.cornell_65k()
    v = np.array(sc["verts"], np.float32)
    v[1000, 4] = np.inf
    with capi.Context(0) as ctx:
        ctx.set_scene(v, sc["normals"], sc["mat_idx"], sc["materials"])
        U, V, W = camera(sc, capi)
        ms, img = {}, {}
        for flags in (0, capi.FLAG_COUNT):
            p = capi.render_params(320, 320, 4, 7, sc["camera"]["eye"], U, V, W, flags=flags)
            for _ in range(3):
                img[flags], _ = ctx.render(p)
                ms[flags] = min(ms.get(flags, 1e9), ctx.stats()["render_ms"])
        print(ms, flush=True)
        assert _same(img[0], img[capi.FLAG_COUNT])
        assert ms[0] < 1.5 * ms[capi.FLAG_COUNT]
