"""Images and fields through the pinned transfer buffers.

Read-back moves planes through a 12 MiB buffer, in quarters; uploads move
windows of at most 4 MiB, and fields are staged up to 32 MiB at a time.  Sizes
from one pixel and one cell to more than those; the exact edges are
test_gpu_transfer_edges.py's.  Bar: every value bit for bit.

* An image that no ray of a volume render touches comes back as the input
  image: the device holds its float32 values, and a pixel whose value went
  anywhere else would differ from (float32) of its own input.
* Without an input image the result is that of an input image of zeros.
* Stored points are float32 of the uploaded values, in blocks.
"""

import numpy as np
import pytest

from yt_amd import _lib, render

from .helpers import c0_params, uniform_lognormal, vr_tf_for

pytestmark = pytest.mark.gpu

SIZES = [(2, 5), (63, 65), (64, 64), (17, 241), (590, 591), (1024, 1024), (1025, 1025), (1303, 1201)]


@pytest.fixture(scope="module")
def volume(ctx):
    ds = uniform_lognormal(12, seed=411)
    vol = render.ResidentVolume(ctx, ds, proj_fields="density", vr_field="density")
    yield ds, vol
    vol.free()


def _read_all(ctx, spec):
    """The image through every call that returns one."""
    out = [ctx.render_noalloc(spec)]
    b = _lib.Batch(ctx, [spec], _lib.BATCH_PERSISTENT)
    b.run()
    out += [b.read_image(0), b.read_image(0)]
    b.close()
    srv = _lib.Server(ctx, max_requests=4, budget_bytes=256 << 20)
    rids = [srv.submit(spec), srv.submit(spec)]
    left = set(rids)
    while left:
        left -= set(srv.wait())
    out.append(srv.read(rids[0]))
    planes = srv.read_planar(rids[1])
    srv.close()
    return out, planes


@pytest.mark.parametrize("nv", SIZES)
def test_untouched_image_comes_back(ctx, volume, nv):
    ds, vol = volume
    print(f"transfer: untouched {nv}", flush=True)
    p = c0_params(nv, center=(40.0, 40.0, 40.0))
    spec = vol.vr_request(p, vr_tf_for(ds, nbins=32))
    rng = np.random.default_rng(nv[0])
    spec.image_in = rng.uniform(0.1, 0.9, size=nv + (4,))
    images, planes = _read_all(ctx, spec)
    for im in images:
        assert np.array_equal(im, spec.image_in)
    n = planes.shape[0]
    assert np.array_equal(planes, np.moveaxis(spec.image_in[..., :n], -1, 0).astype(np.float32))


@pytest.mark.parametrize("nv", [(63, 65), (1024, 1024), (1031, 1023)])
@pytest.mark.parametrize("kind", ["projection", "render", "grey"])
def test_image_without_input(ctx, volume, nv, kind):
    ds, vol = volume
    print(f"transfer: {kind} {nv}", flush=True)
    p = c0_params(nv)
    tf = vr_tf_for(ds, nbins=32)
    tf.grey_opacity = kind == "grey"

    def request():
        return vol.projection_request(p) if kind == "projection" else vol.vr_request(p, tf)

    spec = request()
    images, planes = _read_all(ctx, spec)
    spec0 = request()
    spec0.image_in = np.zeros(nv + (4,))
    want, wplanes = _read_all(ctx, spec0)
    assert np.any(images[0] != 0)
    for im in images + want:
        assert np.array_equal(im, images[0])
    assert np.array_equal(planes, wplanes)
    n = planes.shape[0]
    assert np.array_equal(planes, np.moveaxis(images[0][..., :n], -1, 0).astype(np.float32))


def _blocked(fields):
    """Cell-centred storage: 4^3 blocks in C order, fields interleaved."""
    d = fields[0].shape
    nb = [(x + 3) // 4 for x in d]
    nfp = {1: 1, 2: 2, 3: 4, 4: 4}[len(fields)]
    out = np.zeros([4 * x for x in nb] + [nfp], dtype=np.float32)
    for f, a in enumerate(fields):
        out[: d[0], : d[1], : d[2], f] = a
    out = out.reshape(nb[0], 4, nb[1], 4, nb[2], 4, nfp).transpose(0, 2, 4, 1, 3, 5, 6)
    return out.reshape(-1)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dims,nf", [
    ([(1, 1, 1)], 1),
    ([(5, 3, 7), (1, 2, 1), (64, 64, 64), (33, 17, 9)], 3),
    ([(128, 128, 64)], 2),
    ([(7, 5, 3)] * 300, 1),
    ([(150, 131, 140), (150, 131, 140), (9, 9, 9)], 2),  # more than one staging of 32 MiB in float64
    ([(210, 200, 205), (3, 3, 3)], 1),  # a field of more than 32 MiB
])
def test_upload_stores_every_value(ctx, dims, nf, dtype):
    print(f"transfer: upload {dims[:3]} {nf} {dtype.__name__}", flush=True)
    rng = np.random.default_rng(len(dims) + nf)
    bricks, fields = [], []
    for k, d in enumerate(dims):
        bricks.append(((k, 0.0, 0.0), (k + 1.0, 1.0, 1.0), d, False))
        fields.append([rng.standard_normal(d).astype(dtype) for _ in range(nf)])
    for _ in range(2):
        ds = ctx.upload(bricks, fields)
        try:
            for b in sorted({0, len(dims) // 2, len(dims) - 1}):
                assert np.array_equal(ctx.read_points(ds, b), _blocked(fields[b])), b
        finally:
            ctx.free(ds)
