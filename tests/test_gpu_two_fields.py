"""Weighted projections in launches of few and of many tiles, which run
different builds of one kernel.  Bar: the same image bit for bit, alone, in a
batch with large images, through the server and render_noalloc."""

import numpy as np
import pytest

from yt_amd import _lib, render

from .helpers import c0_params, uniform_lognormal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nprocs", [1, 8])
def test_small_and_large_launches_agree(ctx, nprocs):
    ds = uniform_lognormal(24, seed=551, nprocs=nprocs, with_temperature=True)
    vol = render.ResidentVolume(ctx, ds, proj_fields="temperature", weight="density")
    srv = _lib.Server(ctx, max_requests=8, budget_bytes=256 << 20, chunk_tiles=1 << 16)
    try:
        small = [vol.projection_request(c0_params(nv, width=1.4)) for nv in ((8, 8), (41, 63), (1, 200), (104, 104))]
        # 34000 tiles: more than 36 for each of 256 CUs
        large = [vol.projection_request(c0_params((1475, 1475)))]
        print(f"two fields: {nprocs} bricks", flush=True)
        few = _lib.Batch(ctx, small, _lib.BATCH_PERSISTENT)
        many = _lib.Batch(ctx, small + large, _lib.BATCH_PERSISTENT)
        few.run()
        many.run()
        ids = [srv.submit(s) for s in large + small]
        left = set(ids)
        while left:
            left -= set(srv.wait())
        served = [srv.read(i) for i in ids]
        for i, spec in enumerate(small):
            want = few.read_image(i)
            assert want.shape == spec.nv + (4,)
            assert np.array_equal(many.read_image(i), want)
            assert np.array_equal(served[1 + i], want)
            assert np.array_equal(ctx.render_noalloc(spec), want)
        assert np.any(few.read_image(1)[..., :2] != 0)
        assert np.array_equal(many.read_image(len(small)), served[0])
        few.close()
        many.close()
    finally:
        srv.close()
        vol.free()
