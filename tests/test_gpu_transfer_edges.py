"""Images at the sizes where the way they travel changes: one thread's copy
and the pinned transfer (by pixels and channels), the transfer's parts (256 KiB
to a quarter of an image, five where the count is no multiple of 16) and its 12
MiB window, and render_noalloc's 4 MiB of output in pinned memory.  Bar: every
value bit for bit.
"""

import numpy as np
import pytest

from yt_amd import _lib, render

from .helpers import c0_params, uniform_lognormal, vr_tf_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def volume(ctx):
    ds = uniform_lognormal(12, seed=561)
    vol = render.ResidentVolume(ctx, ds, proj_fields="density", vr_field="density")
    yield ds, vol
    vol.free()


def _read(ctx, spec):
    """The image, the planes and the image of render_noalloc."""
    b = _lib.Batch(ctx, [spec], _lib.BATCH_PERSISTENT)
    b.run()
    image = b.read_image(0)
    b.close()
    srv = _lib.Server(ctx, max_requests=4, budget_bytes=512 << 20)
    ids = [srv.submit(spec), srv.submit(spec)]
    left = set(ids)
    while left:
        left -= set(srv.wait())
    planes = srv.read_planar(ids[0])
    served = srv.read(ids[1])
    srv.close()
    return image, planes, served, ctx.render_noalloc(spec)


# pixels (as a row of 1, so that every count is met) at which one thread's
# copy ends for 1, 3 and 4 channels and 3 and 4 with an input image, the
# planes' one copy ends, a part reaches 256 KiB, render_noalloc's output 4 MiB
# and the window 12 MiB
COUNTS = {
    1: (50000, 65536, 240000, 1048576, 3145728),
    3: (12500, 20000, 20000, 21844, 25000, 80000, 349525, 1048576),
    4: (11111, 15000, 20000, 60000, 262144, 786432),
}


@pytest.mark.parametrize("kind,nch,n", [(k, c, n) for k, c in (("projection", 1), ("render", 3), ("grey", 4))
                                        for n in COUNTS[c]])
def test_images_at_the_edges(ctx, volume, kind, nch, n):
    ds, vol = volume
    tf = vr_tf_for(ds, nbins=16)
    tf.grey_opacity = kind == "grey"
    rng = np.random.default_rng(n)
    for count in (n - 1, n, n + 1):
        print(f"transfer edge: {kind} {count}", flush=True)
        nv = (2, (count + 1) // 2) if count % 2 == 0 else (1, count)
        p = c0_params(nv, center=(40.0, 40.0, 40.0))  # no ray meets the volume: the input image comes back
        spec = vol.projection_request(p) if kind == "projection" else vol.vr_request(p, tf)
        spec.image_in = rng.uniform(0.1, 0.9, size=nv + (4,))
        image, planes, served, direct = _read(ctx, spec)
        for got in (image, served, direct):
            assert np.array_equal(got, spec.image_in)
        assert planes.shape[0] == nch
        assert np.array_equal(planes, np.moveaxis(spec.image_in[..., :nch], -1, 0).astype(np.float32))
        if count == n:
            # without an input image: every pixel is written
            p = c0_params(nv, width=0.2)
            spec = vol.projection_request(p) if kind == "projection" else vol.vr_request(p, tf)
            image, planes, served, direct = _read(ctx, spec)
            assert nv[0] == 1 or np.any(image != 0)
            assert np.array_equal(served, image) and np.array_equal(direct, image)
            assert np.array_equal(planes, np.moveaxis(image[..., :nch], -1, 0).astype(np.float32))
