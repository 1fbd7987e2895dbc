"""Background pixels that are not finite, in volume renders of few tiles.

Four waves share a tile of such a render (k_split) and take every visit of
the tile's rays through each pixel's transmittance, also for the pixels whose
own ray takes no part in the visit: outside the data, past its end, a masked
cell, a value with no logarithm.  Those have to keep an infinite transmittance
as it is.  Bar: the image of one wave a tile bit for bit, and the caller's own
value where the pixel's ray meets no data.
"""

import numpy as np
import pytest

from yt_amd import _lib, data, render

from .helpers import small_amr, uniform_lognormal, vr_tf_for

pytestmark = pytest.mark.gpu

SPECIAL = (np.inf, -np.inf, 1e39, -1e39, np.nan, -0.0, 3e38)


def _render(ctx, spec, waves):
    b = _lib.Batch(ctx, [spec], _lib.BATCH_PERSISTENT)
    try:
        b.set_launch(waves, 0)
        b.run()
        return b.read_image(0)
    finally:
        b.close()


def _volume(name):
    if name == "amr":
        return small_amr(root_n=16, levels=2)
    if name == "zeros":
        rho = data.lognormal_density(24, seed=521)
        rho[np.random.default_rng(522).random(rho.shape) < 0.05] = 0.0
        return data.load_uniform_grid({"density": rho})
    return uniform_lognormal(24, seed=523, nprocs=8 if name == "8 bricks" else 1)


@pytest.mark.parametrize("lens", ["parallel", "perspective"])
@pytest.mark.parametrize("name", ["1 brick", "8 bricks", "amr", "zeros"])
def test_infinite_background(ctx, name, lens):
    ds = _volume(name)
    tf = vr_tf_for(uniform_lognormal(24, seed=523), nbins=64)
    vol = render.ResidentVolume(ctx, ds, vr_field="density")
    nv = (61, 90)
    try:
        if lens == "parallel":
            p = render.camera_params((0.5, 0.5, 0.5), (0.3, -0.5, 0.8), 2.2, nv, (0.1, 0.2, 1.0))
        else:
            p = render.perspective_params((0.5, -1.4, 0.6), (0.5, 0.5, 0.5), (2.2, 2.2, 1.5), nv, (0.0, 0.1, 1.0))
        clear = vol.vr_request(p, tf)
        clear.image_in = np.zeros(nv + (4,))
        hit = np.any(_render(ctx, clear, 2)[..., :3] != 0, axis=-1)
        rng = np.random.default_rng(524)
        spec = vol.vr_request(p, tf)
        spec.image_in = np.where(rng.random(nv + (4,)) < 0.5, rng.choice(SPECIAL, size=nv + (4,)),
                                 rng.uniform(0.0, 0.5, size=nv + (4,)))
        print(f"split, infinite background: {name} {lens}", flush=True)
        want = _render(ctx, spec, 2)
        for got in (_render(ctx, spec, 4), ctx.render_noalloc(spec)):
            assert np.array_equal(got, want, equal_nan=True)
        # rays that miss the volume, and their neighbours that meet it, share tiles
        corner = np.zeros(nv, dtype=bool)
        corner[:4] = corner[-4:] = corner[:, :4] = corner[:, -4:] = True
        assert np.any(hit) and not np.any(hit & corner)
        assert np.array_equal(want[corner], spec.image_in[corner], equal_nan=True)
    finally:
        vol.free()
