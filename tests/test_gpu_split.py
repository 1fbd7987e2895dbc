"""k_split (four waves to a tile) against k_persist (one), which a batch of
two waves a workgroup runs.  Bar: the same image bit for bit."""

import numpy as np
import pytest

from yt_amd import _lib, data, render

from .helpers import small_amr, uniform_lognormal, vr_tf_for

pytestmark = pytest.mark.gpu


def _same(ctx, specs):
    b = _lib.Batch(ctx, specs, _lib.BATCH_PERSISTENT | _lib.BATCH_GRAPH)
    one = _lib.Batch(ctx, specs, _lib.BATCH_PERSISTENT)
    try:
        one.set_launch(2, 0)
        one.run()
        for _ in range(2):
            b.run()
            for i, spec in enumerate(specs):
                want = one.read_image(i)
                assert np.array_equal(b.read_image(i), want)
                assert np.array_equal(ctx.render_noalloc(spec), want)
        return want
    finally:
        b.close()
        one.close()


CAMERAS = [((0.3, -0.5, 0.8), 1.4, (41, 63)), ((0.0, 0.0, 1.0), 1.0, (8, 8)), ((0.0, -0.6, 0.8), 0.35, (9, 200)),
           ((-0.7, 0.1, -0.2), 2.5, (130, 17))]


@pytest.mark.parametrize("volume", ["2x2x2", "2x3x2", "24", "24 in 8", "amr"])
def test_same_image_as_one_wave_a_tile(ctx, volume):
    if volume == "amr":
        ds = small_amr(root_n=16, levels=2)
    elif volume.startswith("24"):
        ds = uniform_lognormal(24, seed=511, nprocs=8 if "8" in volume else 1)
    else:
        dims = tuple(int(x) for x in volume.split("x"))
        ds = data.load_uniform_grid({"density": np.random.default_rng(512).lognormal(size=dims)})
    tf = vr_tf_for(ds, nbins=64)
    vol = render.ResidentVolume(ctx, ds, vr_field="density")
    rng = np.random.default_rng(513)
    try:
        for n_samples in (10, 3):
            for normal, width, nv in CAMERAS:
                print(f"split: {volume} {n_samples} {normal}", flush=True)
                north = (0.0, 1.0, 0.0) if normal[2] == 1.0 else (0.1, 0.2, 1.0)
                p = render.camera_params((0.5, 0.5, 0.5), normal, width, nv, north)
                specs = [vol.vr_request(p, tf, n_samples=n_samples),
                         vol.vr_request(p, tf, n_samples=n_samples, zbuffer=rng.uniform(0.1, 1.0, size=nv)),
                         vol.vr_request(p, tf, n_samples=n_samples)]
                specs[2].image_in = rng.uniform(0.0, 0.5, size=nv + (4,))
                assert np.any(_same(ctx, specs) != 0)
            p = render.perspective_params((0.5, -1.4, 0.6), (0.5, 0.5, 0.5), (1.2, 1.2, 1.5), (33, 50), (0.0, 0.1, 1.0))
            assert np.any(_same(ctx, [vol.vr_request(p, tf, n_samples=n_samples)]) != 0)
    finally:
        vol.free()

