"""Several threads that read images of one context and upload fields to it at
once: some through the pinned transfer, the others by themselves.  Bar: every
value as when one thread does it alone."""

import threading

import numpy as np
import pytest

from yt_amd import _lib, render

from .helpers import c0_params, uniform_lognormal, vr_tf_for

pytestmark = pytest.mark.gpu


def test_threads_read_and_upload_at_once(ctx):
    ds = uniform_lognormal(12, seed=571)
    vol = render.ResidentVolume(ctx, ds, proj_fields="density", vr_field="density")
    tf = vr_tf_for(ds, nbins=16)
    jobs, errors = [], []
    for k, side in enumerate((40, 300, 500, 700, 260, 512)):
        p = c0_params(side, width=0.8)
        spec = vol.projection_request(p) if k % 2 else vol.vr_request(p, tf)
        b = _lib.Batch(ctx, [spec], _lib.BATCH_PERSISTENT)
        b.run()
        jobs.append((b, b.read_image(0), spec))

    def read(b, want, spec, direct):
        try:
            for _ in range(12):
                got = ctx.render_noalloc(spec) if direct else b.read_image(0)
                assert np.array_equal(got, want)
        except Exception as e:  # handed to the test's own thread
            errors.append(e)

    def upload(seed):
        try:
            rng = np.random.default_rng(seed)
            for n in (9, 40, 70, 110):
                f = rng.standard_normal((n, n, n))
                d = ctx.upload([((0, 0, 0), (1, 1, 1), (n, n, n), False)], [[f]])
                got = ctx.read_points(d, 0)
                assert np.array_equal(np.sort(got[got != 0]), np.sort(f.astype(np.float32).ravel()))
                ctx.free(d)
        except Exception as e:
            errors.append(e)

    try:
        threads = [threading.Thread(target=read, args=(*j, k == 2)) for k, j in enumerate(jobs)]
        threads += [threading.Thread(target=upload, args=(s,)) for s in (1, 2)]
        print("transfer threads", flush=True)
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors[0]
        assert all(np.any(want != 0) for _, want, _ in jobs)
    finally:
        for b, _, _ in jobs:
            b.close()
        vol.free()
