"""Which volume renders take four waves to a tile (k_split), and that the
cameras of the tests that compare it with one wave a tile do take them; the
edge geometry of the timed kernels' oracle test in both; and a brick that
k_split's fast walk refuses (strides beyond 24 bits), which it walks visit by
visit.  Bar: the same image bit for bit."""

import numpy as np
import pytest

from yt_amd import _lib, render
from yt_amd.transfer_functions import gaussian_ctf

from .helpers import c0_params, small_amr, uniform_lognormal, vr_tf_for
from .test_gpu_fast_walks import CAMERAS as EDGE_CAMERAS
from .test_gpu_fast_walks import _dataset
from .test_gpu_split import CAMERAS

pytestmark = pytest.mark.gpu


def _both(ctx, spec, waves=4):
    """The image with as many waves to a tile as the rule gives (which are
    `waves`) and with one."""
    b = _lib.Batch(ctx, [spec], _lib.BATCH_PERSISTENT)
    one = _lib.Batch(ctx, [spec], _lib.BATCH_PERSISTENT)
    try:
        assert b.tile_waves(0) == waves
        one.set_launch(2, 0)
        assert one.tile_waves(0) == 1
        b.run()
        one.run()
        got, want = b.read_image(0), one.read_image(0)
        assert np.array_equal(got, want)
        return got
    finally:
        b.close()
        one.close()


def test_small_images_take_four_waves(ctx):
    for ds in (uniform_lognormal(24, seed=511), uniform_lognormal(24, seed=511, nprocs=8), small_amr(16, 2)):
        tf = vr_tf_for(ds, nbins=64)
        vol = render.ResidentVolume(ctx, ds, vr_field="density")
        try:
            for normal, width, nv in CAMERAS:
                north = (0.0, 1.0, 0.0) if normal[2] == 1.0 else (0.1, 0.2, 1.0)
                p = render.camera_params((0.5, 0.5, 0.5), normal, width, nv, north)
                print(f"split rule: {len(vol.leaves)} bricks, {nv}", flush=True)
                _both(ctx, vol.vr_request(p, tf))
            p = render.perspective_params((0.5, -1.4, 0.6), (0.5, 0.5, 0.5), (1.2, 1.2, 1.5), (33, 50), (0.0, 0.1, 1.0))
            _both(ctx, vol.vr_request(p, tf))
            # 16384 tiles, most of them full: one wave each
            _both(ctx, vol.vr_request(c0_params(1024, width=0.8), tf), waves=1)
        finally:
            vol.free()


@pytest.mark.parametrize("dname", ["uniform37", "amr", "long512", "long600"])
def test_edge_geometry(ctx, dname):
    ds, _ = _dataset(dname)
    tf = vr_tf_for(ds, nbins=128)
    vol = render.ResidentVolume(ctx, ds, vr_field="density")
    try:
        for name, normal, width in EDGE_CAMERAS:
            print(f"split rule: {dname} {name}", flush=True)
            assert np.any(_both(ctx, vol.vr_request(c0_params(40, normal=normal, width=width), tf)) != 0)
    finally:
        vol.free()


def test_brick_that_the_fast_walk_refuses(ctx):
    # 32775 vertex blocks along the last axis: 2^24 bytes and more a row
    n = (2, 2, 131098)
    rng = np.random.default_rng(581)
    ds = ctx.upload([((0.0, 0.0, 0.0), (1.0, 1.0, 1.0), n, True)], [[rng.uniform(-1.0, 1.0, [x + 1 for x in n])]])
    try:
        tf = _lib.TF.from_tf_obj(gaussian_ctf((-1.0, 1.0), n_gauss=4, nbins=64))
        for normal, width in (((1.0, 0.0, 0.0), 1.1), ((0.8, 0.6, 0.0), 1.6), ((0.6, 0.8, 1e-3), 0.9)):
            print(f"split rule: refused brick {normal}", flush=True)
            p = render.camera_params((0.5, 0.5, 0.5), normal, width, (21, 40), (0.0, 0.1, 1.0))
            assert np.any(_both(ctx, _lib.RequestSpec(_lib.VOLUME_RENDER, p, ds, [0], tf=tf)) != 0)
    finally:
        ctx.free(ds)

