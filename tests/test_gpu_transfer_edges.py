"""Images at the sizes where the way they travel changes: one thread's copy
and the pinned transfer (by pixels and channels), the transfer's parts (256 KiB
to a quarter of an image, five where the count is no multiple of 16) and its 12
MiB window, and render_noalloc's 4 MiB of output in pinned memory; and uploads
on either side of the rule that copies them as they are or through the pinned
windows.  Bar: every value bit for bit.
"""

import numpy as np
import pytest

from yt_amd import _lib, render

from .helpers import c0_params, uniform_lognormal, vr_tf_for
from .test_gpu_transfer import _blocked

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


# one piece on either side of 16 and 48 KiB and of 3 MiB, two pieces below, at and above 128 KiB
# and 3 MiB in all, three pieces
@pytest.mark.parametrize("dims,nf,dtype", [
    ([(1, 3, 5)], 1, np.float64),
    ([(16, 16, 15)], 1, np.float32),
    ([(16, 16, 16)], 1, np.float32),
    ([(16, 16, 24)], 1, np.float64),
    ([(16, 17, 24)], 1, np.float64),
    ([(96, 64, 127)], 1, np.float32),
    ([(96, 64, 128)], 1, np.float32),
    ([(3, 65536, 2)], 1, np.float64),
    ([(96, 64, 129)], 1, np.float32),
    ([(32, 32, 16)], 2, np.float32),
    ([(16, 32, 16), (16, 32, 16)], 1, np.float64),
    ([(32, 32, 16), (32, 33, 16)], 1, np.float32),
    ([(64, 64, 47), (64, 64, 48)], 1, np.float64),
    ([(64, 64, 48), (64, 64, 48)], 1, np.float64),
    ([(64, 64, 49), (64, 64, 49)], 1, np.float64),
    ([(31, 17, 9)], 3, np.float64),
])
def test_uploads_at_the_edges(ctx, dims, nf, dtype):
    print(f"upload edge: {dims} {nf} {dtype.__name__}", flush=True)
    rng = np.random.default_rng(nf)
    bricks = [((k, 0.0, 0.0), (k + 1.0, 1.0, 1.0), d, False) for k, d in enumerate(dims)]
    fields = [[rng.standard_normal(d).astype(dtype) for _ in range(nf)] for d in dims]
    for _ in range(2):
        ds = ctx.upload(bricks, fields)
        try:
            for b in range(len(dims)):
                assert np.array_equal(ctx.read_points(ds, b), _blocked(fields[b])), b
        finally:
            ctx.free(ds)
