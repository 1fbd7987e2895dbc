"""walk_iproj_fast (interpolated projections of one field, no record) against
the FP64 oracle, at the bar of test_gpu_iproj.py: rel-L2 <= 1e-5, and values
that are not finite at the same pixels.

Bricks of 2 cells and of sides that end inside a vertex block, rays of one
visit and of many, axes that rays never step, z-buffers that end a ray inside
a cell, one and many sub-samples.
"""

import numpy as np
import pytest

from oracle import oracle
from yt_amd import _lib, data, render

from .conftest import rel_l2
from .helpers import oracle_vr_bricks

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _images(ctx, spec):
    out = [ctx.render_noalloc(spec)]
    for flags in (_lib.BATCH_PERSISTENT, _lib.BATCH_PLAIN):
        b = _lib.Batch(ctx, [spec], flags)
        b.run()
        out.append(b.read_image(0))
        b.close()
    return out


def _check(ctx, vol, p, n_samples=10, zbuffer=None):
    spec = vol.interpolated_projection_request(p, n_samples=n_samples, zbuffer=zbuffer)
    kw = {} if zbuffer is None else dict(zbuffer=zbuffer)
    want = oracle.cast(2, p, oracle_vr_bricks(vol), order=spec.order, n_samples=n_samples, **kw)[..., 0]
    ok = np.isfinite(want)
    assert np.any(want[ok] != 0)
    for im in _images(ctx, spec):
        assert np.array_equal(np.isfinite(im[..., 0]), ok)
        assert rel_l2(im[..., 0][ok], want[ok]) <= TOL
        assert np.all(im[..., 1:] == 0.0)
    return ok


@pytest.mark.parametrize("n_samples", [1, 2, 10, 37])
@pytest.mark.parametrize("dims,split", [((2, 2, 2), 1), ((5, 3, 9), 1), ((16, 16, 16), 4), ((33, 40, 17), 1)])
def test_images(ctx, dims, split, n_samples):
    rng = np.random.default_rng(sum(dims) + n_samples)
    ds = data.load_uniform_grid({"density": rng.uniform(0.5, 2.0, size=dims)},
                                psize=(split,) * 3 if split > 1 else None)
    vol = render.ResidentVolume(ctx, ds, vr_field="density", log_field=False)
    try:
        for normal, width, nv in [((0.3, -0.5, 0.8), 1.3, (37, 41)), ((0.0, 0.0, 1.0), 1.0, (16, 64)),
                                  ((0.0, -0.6, 0.8), 0.4, (9, 7))]:
            print(f"iproj: {dims} {split} {n_samples} {normal}", flush=True)
            north = (0.0, 1.0, 0.0) if normal[2] == 1.0 else (0.1, 0.2, 1.0)
            p = render.camera_params((0.5, 0.5, 0.5), normal, width, nv, north)
            _check(ctx, vol, p, n_samples)
            _check(ctx, vol, p, n_samples, zbuffer=rng.uniform(0.4, 1.0, size=nv))
        p = render.perspective_params((0.5, -1.4, 0.6), (0.5, 0.5, 0.5), (1.2, 1.2, 1.5), (25, 18), (0.0, 0.1, 1.0))
        _check(ctx, vol, p, n_samples)
    finally:
        vol.free()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_values_that_are_not_finite(ctx, bad):
    a = np.ones((9, 9, 9))
    a[4, 4, 4] = bad
    ds = data.load_uniform_grid({"density": a})
    vol = render.ResidentVolume(ctx, ds, vr_field="density", log_field=False)
    try:
        p = render.camera_params((0.5, 0.5, 0.5), (0.3, -0.5, 0.8), 1.0, (40, 40), (0.0, 0.0, 1.0))
        assert not _check(ctx, vol, p).all()
    finally:
        vol.free()
