"""Every tile of an image is cast once, whatever order the queue takes: one
tile, ragged tiles, fewer and more tiles than the queue's eight ranges, both
sides of the costly-first rule (few_items), a camera that misses the volume
(no tile has a cost), rays along an axis, a perspective lens, and images of
several sizes in one launch.  The order must not change a value: persistent
batches with one and several tiles per item, render_noalloc and plain
launches give the same images bit for bit.
"""

import numpy as np
import pytest

from yt_amd import _lib, render

from .helpers import c0_params, uniform_lognormal, vr_tf_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def volume(ctx):
    ds = uniform_lognormal(20, seed=91, psize=(2, 1, 1))
    vol = render.ResidentVolume(ctx, ds, proj_fields="density", vr_field="density")
    yield vol, _lib.TF.from_tf_obj(vr_tf_for(ds, nbins=32))
    vol.free()


CAMERAS = {
    "one_tile": dict(res=(5, 3)),
    "five_tiles": dict(res=(8, 33)),
    "ragged": dict(res=(203, 61), width=1.7),
    "axis": dict(res=(70, 70), normal=(0.0, 0.0, 1.0), width=1.4),
    "miss": dict(res=(64, 40), center=(5.0, 0.5, 0.5), width=0.3),
    "many": dict(res=(1300, 1031), width=2.5),
}


def _request(volume, name, kind):
    vol, tf = volume
    p = c0_params(**CAMERAS[name])
    return vol.projection_request(p) if kind == "proj" else vol.vr_request(p, tf)


def _batch(ctx, specs, flags=_lib.BATCH_PERSISTENT, **kw):
    b = _lib.Batch(ctx, specs, flags, **kw)
    try:
        b.run()
        return [b.read_image(i) for i in range(len(specs))]
    finally:
        b.close()


@pytest.mark.parametrize("kind", ["proj", "vr"])
@pytest.mark.parametrize("name", sorted(CAMERAS))
def test_order_leaves_images_alone(ctx, volume, name, kind):
    spec = _request(volume, name, kind)
    want = _batch(ctx, [spec], _lib.BATCH_PLAIN)[0]
    assert (np.abs(want).max() > 0) == (name != "miss")
    for kw in ({}, {"item_tiles": 2}, {"item_tiles": 8}, {"tile": (4, 16)}):
        assert np.array_equal(_batch(ctx, [spec], **kw)[0], want), kw
    assert np.array_equal(ctx.render_noalloc(spec), want)


def test_sizes_mixed(ctx, volume):
    specs = [_request(volume, n, k) for n in sorted(CAMERAS) for k in ("vr", "proj")]
    for spec, img in zip(specs, _batch(ctx, specs)):
        assert np.array_equal(img, _batch(ctx, [spec], _lib.BATCH_PLAIN)[0])


def test_perspective(ctx, volume):
    vol, tf = volume
    p = render.perspective_params((0.5, 0.4, 2.2), (0.5, 0.5, 0.5), (1.6, 1.6, 1.7), (77, 130))
    spec = vol.vr_request(p, tf)
    want = _batch(ctx, [spec], _lib.BATCH_PLAIN)[0]
    assert np.array_equal(_batch(ctx, [spec])[0], want)
    assert np.array_equal(ctx.render_noalloc(spec), want)
