"""The image bytes of lisa_render (quantised on the device by a table of steps)
against lisa_srgb_quantize."""
import numpy as np
import pytest


def _bytes(capi, x):
    """lisa_srgb_quantize of single channels."""
    x = np.asarray(x, np.float32)
    n = -(-len(x) // 3)
    rgba = np.zeros((n, 4), np.float32)
    flat = np.zeros(3 * n, np.float32)
    flat[: len(x)] = x
    rgba[:, :3] = flat.reshape(n, 3)
    return capi.srgb_quantize(rgba)[:, :3].reshape(-1)[: len(x)]


def test_bytes_never_fall(capi):
    """A channel's byte never falls from one float to the next, over every float
    from 2^-9 (below the curve's linear part's end, 0.0031308) to 1: a byte is
    then the number of steps at or below the float.  Below, the product of a
    constant cannot fall."""
    lo, hi, step = 0x3B000000, 0x3F800000, 1 << 22
    last = 0
    for a in range(lo, hi + 1, step):
        b = _bytes(capi, np.arange(a, min(a + step, hi + 1), dtype=np.uint32).view(np.float32)).astype(np.int16)
        assert b[0] >= last and (np.diff(b) >= 0).all()
        last = b[-1]
    assert last == 255


@pytest.mark.gpu
def test_device_bytes_at_every_step(capi):
    """A camera inside an emitter: every pixel is its emission.  The step of each
    byte, the floats beside it, and values outside [0, 1]."""
    bits = np.zeros(255, np.int64)
    hi = np.full(255, 0x3F800000, np.int64)
    while (bits < hi).any():  # the steps by bisection
        mid = (bits + hi) // 2
        up = _bytes(capi, mid.astype(np.uint32).view(np.float32)) >= np.arange(1, 256)
        hi = np.where(up, mid, hi)
        bits = np.where(up, bits, mid + 1)
    t = bits.astype(np.uint32).view(np.float32)
    values = [(np.nextafter(v, np.float32(0)), v, np.nextafter(v, np.float32(2))) for v in t]
    values += [(np.float32(0), np.float32(1), np.float32(2)), (np.float32(np.inf), np.float32(-1), np.float32(1e-40))]
    v = np.float32([[-9, -9, -1, 9, -9, -1, 0, 9, -1]])
    n = np.tile(np.float32([0, 0, 1]), (1, 3))
    U, V, W = capi.camera_uvw((0, 0, 1), (0, 0, 0), 40.0, 11 / 7)
    with capi.Context(0) as ctx:
        for e in values:
            ctx.set_scene(v, n, [0], [{"emit": True, "emission": e}])
            acc, rgb = ctx.render(capi.render_params(11, 7, 1, 2, (0, 0, 1), U, V, W), want_rgba8=True)
            assert np.array_equal(acc[0, :3], np.float32(e))
            assert np.array_equal(rgb, capi.srgb_quantize(acc)), e
            _, alone = ctx.render(capi.render_params(11, 7, 1, 2, (0, 0, 1), U, V, W), want_accum=False,
                                  want_rgba8=True)
            assert np.array_equal(alone, rgb)
