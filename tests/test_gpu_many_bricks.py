"""The tile's brick list (64 extents tested per ballot in render_tile) at its
edges: orders of 1, 63, 64, 65 and 130 bricks, an order that names a brick
more than once and one that leaves bricks out, front to back for early ray
termination, against the FP64 oracle.  Bars: rel-L2 <= 1e-5 per channel, and
2e-4 for early termination (rays stop below a transmittance of 1e-4).
"""

import numpy as np
import pytest

from oracle import oracle
from yt_amd import _lib, data, render

from .helpers import c0_params, oracle_proj_bricks, oracle_vr_bricks, tf_dict, vr_tf_for

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 130])
def test_orders_of_n_bricks(ctx, n):
    rho = np.random.default_rng(n).lognormal(0.0, 1.0, size=(2 * n, 9, 11))
    ds = data.load_uniform_grid({"density": rho}, psize=(n, 1, 1))
    vol = render.ResidentVolume(ctx, ds, proj_fields="density", vr_field="density")
    try:
        tf = vr_tf_for(ds, nbins=64)
        p = c0_params(44, normal=(0.8, 0.5, 0.3), width=1.4)
        rng = np.random.default_rng(n + 1)
        full = vol.projection_request(p)
        some = rng.permutation(n)[: (n + 1) // 2].astype(np.int32)
        orders = [full.order, np.concatenate([full.order, some]), some]
        specs = [_lib.RequestSpec(_lib.PROJECTION, p, vol.proj_ds_id, o) for o in orders]
        specs += [vol.vr_request(p, tf), vol.vr_request(p, tf, ert=True)]
        b = _lib.Batch(ctx, specs, _lib.BATCH_PERSISTENT)
        try:
            b.run()
            imgs = [b.read_image(i) for i in range(len(specs))]
        finally:
            b.close()
        pb, vb = oracle_proj_bricks(ds, ["density"]), oracle_vr_bricks(vol)
        for img, o in zip(imgs, orders):
            assert _rel(img[..., 0], oracle.cast(0, p, pb, order=o)[..., 0]) <= 1e-5
        want = oracle.cast(1, p, vb, order=specs[3].order, tf=tf_dict(tf), n_samples=10)
        for c in range(3):
            assert _rel(imgs[3][..., c], want[..., c]) <= 1e-5
            assert _rel(imgs[4][..., c], want[..., c]) <= 2e-4
    finally:
        vol.free()
