"""The transfer-function tables beside which four waves to a tile (k_split)
still fit a workgroup's LDS: the largest bin count that takes them and the
next one, which has to go to one wave a tile.

Bar: both render, in a batch and in ytrc_render_noalloc, and equal the two
waves a workgroup of one wave a tile bit for bit.
"""

import numpy as np
import pytest

from yt_amd import _lib, render

from .helpers import c0_params, uniform_lognormal, vr_tf_for

pytestmark = pytest.mark.gpu


def _waves(ctx, spec):
    b = _lib.Batch(ctx, [spec], _lib.BATCH_PERSISTENT)
    try:
        return b.tile_waves(0)
    finally:
        b.close()


def test_tables_at_the_lds_limit(ctx):
    ds = uniform_lognormal(24, seed=531)
    vol = render.ResidentVolume(ctx, ds, vr_field="density")
    p = c0_params(40)
    try:
        # the bin count up to which a small image takes four waves a tile
        lo, hi = 64, ctx.max_lds // 48 - 2
        assert _waves(ctx, vol.vr_request(p, vr_tf_for(ds, nbins=lo))) == 4
        assert _waves(ctx, vol.vr_request(p, vr_tf_for(ds, nbins=hi))) == 1
        while hi - lo > 1:
            mid = (lo + hi) // 2
            if _waves(ctx, vol.vr_request(p, vr_tf_for(ds, nbins=mid))) == 4:
                lo = mid
            else:
                hi = mid
        # (48 bytes a bin: not a bin of room is left unused)
        for nbins, waves in ((lo, 4), (hi, 1)):
            spec = vol.vr_request(p, vr_tf_for(ds, nbins=nbins))
            print(f"split LDS: {nbins} bins, {waves} waves a tile", flush=True)
            b = _lib.Batch(ctx, [spec], _lib.BATCH_PERSISTENT)
            one = _lib.Batch(ctx, [spec], _lib.BATCH_PERSISTENT)
            try:
                assert b.tile_waves(0) == waves
                one.set_launch(2, 0)
                assert one.tile_waves(0) == 1
                b.run()
                one.run()
                want = one.read_image(0)
                assert np.any(want != 0)
                assert np.array_equal(b.read_image(0), want)
                assert np.array_equal(ctx.render_noalloc(spec), want)
            finally:
                b.close()
                one.close()
    finally:
        vol.free()
