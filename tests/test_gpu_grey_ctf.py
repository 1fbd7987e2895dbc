"""The grey-opacity ColorTransferFunction kernels (ctf_visit_grey) against
the FP64 oracle: unrolled and counted sub-samples, parallel and perspective
rays, cells without a value, masked AMR bricks, an input image, and a table
so opaque that dt * alpha exceeds 1 (the reference's clamp acts, so the
general tables run).  A field held at either bound of the table lies outside
FIT_get_value's open range (field_interpolation_tables.pxd:63-82): black.  Bar, per channel: rel-L2 and max-abs/max <= 1e-5, the bar of the
other samplers' FP32 lookups.
"""

import numpy as np
import pytest

from oracle import oracle
from yt_amd import _lib, data, render
from yt_amd.transfer_functions import ColorTransferFunction

from .helpers import c0_params, oracle_vr_bricks, small_amr, tf_dict, uniform_lognormal

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _grey_tf(lo, hi, nbins, opacity):
    tf = ColorTransferFunction((lo, hi), nbins=nbins, grey_opacity=True)
    w = 0.02 * (hi - lo) ** 2
    # the first Gaussian sits on the lower bound: a value there that is taken
    # for inside the table emits
    for at, rgb in ((0.0, (0.9, 0.2, 0.1)), (0.45, (0.2, 0.9, 0.3)), (0.8, (0.1, 0.4, 0.9))):
        tf.add_gaussian(lo + at * (hi - lo), w, [*rgb, opacity * (0.3 + at)])
    return tf


def _dataset(name):
    if name == "amr":
        return small_amr(root_n=24, levels=2, seed=71)
    if name == "ragged":
        return uniform_lognormal(37, seed=72, psize=(3, 2, 5))
    rho = data.lognormal_density(29, seed=73)
    rho[5:9, 3:20, 11:13] = 0.0  # cells without a value
    return data.load_uniform_grid({"density": rho})


@pytest.mark.parametrize("dname,n_samples,nbins,opacity", [
    ("ragged", 10, 64, 1.0), ("ragged", 7, 2, 40.0), ("ragged", 1, 256, 20.0),
    ("holes", 10, 33, 5.0), ("amr", 10, 256, 30.0), ("amr", 3, 128, 3000.0)])
def test_grey_ctf(ctx, dname, n_samples, nbins, opacity):
    ds = _dataset(dname)
    vals = np.concatenate([np.asarray(g["density"], dtype="f8").ravel() for g in ds.grids])
    vals = vals[vals > 0]
    lo, hi = float(np.log10(vals.min())), float(np.log10(vals.max()))
    tf = _grey_tf(lo, hi, nbins, opacity)
    vol = render.ResidentVolume(ctx, ds, vr_field="density")
    try:
        p1 = c0_params(37, width=1.3)
        p2 = render.perspective_params((0.5, 0.4, 2.2), (0.5, 0.5, 0.5), (1.6, 1.6, 1.7), (29, 41))
        specs = [vol.vr_request(p1, tf, n_samples=n_samples), vol.vr_request(p2, tf, n_samples=n_samples)]
        start = np.random.default_rng(74).random((37, 37, 4))
        specs.append(_lib.RequestSpec(_lib.VOLUME_RENDER, p1, vol.vr_ds_id, specs[0].order,
                                      n_samples=n_samples, tf=specs[0].tf, image_in=start))
        b = _lib.Batch(ctx, specs, _lib.BATCH_PERSISTENT | _lib.BATCH_GRAPH)
        try:
            b.run()
            imgs = [b.read_image(i) for i in range(3)]
        finally:
            b.close()
        bricks = oracle_vr_bricks(vol)
        for k, (p, kw) in enumerate([(p1, {}), (p2, {}), (p1, {"image": start})]):
            want = oracle.cast(1, p, bricks, order=specs[k].order, tf=tf_dict(tf), n_samples=n_samples, **kw)
            assert np.abs(want).max() > 0
            for c in range(4):
                d = imgs[k][..., c] - want[..., c]
                e = np.linalg.norm(d) / np.linalg.norm(want[..., c])
                m = np.abs(d).max() / np.abs(want[..., c]).max()
                print(f"{dname} ns={n_samples} request {k} ch{c}: rel-L2 {e:.2e} max-abs/max {m:.2e}", flush=True)
                assert e <= TOL and m <= TOL, (k, c, e, m)
    finally:
        vol.free()


@pytest.mark.parametrize("at", [0, 1])
def test_grey_flat_field_on_a_bound(ctx, at):
    ds = data.load_uniform_grid({"density": np.full((9, 9, 9), 0.5)})
    v = float(np.log10(0.5))
    lo, hi = (v, v + 2.0) if at == 0 else (v - 2.0, v)
    tf = ColorTransferFunction((lo, hi), nbins=64, grey_opacity=True)
    tf.add_gaussian(v, 0.3, [0.9, 0.5, 0.2, 5.0])
    vol = render.ResidentVolume(ctx, ds, vr_field="density")
    try:
        img = ctx.render_noalloc(vol.vr_request(c0_params(24), tf))
        assert np.all(img == 0.0)
    finally:
        vol.free()
