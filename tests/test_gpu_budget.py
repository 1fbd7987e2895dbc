"""A context with a budget: what it accepts and refuses depends on what is in
use alone, whatever it held before."""

import numpy as np
import pytest

from yt_amd import _lib, render

from .helpers import c0_params, uniform_lognormal

pytestmark = pytest.mark.gpu


def test_budget_after_frees_of_other_sizes():
    def bricks(n):
        return [((0, 0, 0), (1, 1, 1), (n, n, n), False)], [[np.random.default_rng(n).random((n, n, n))]]

    free = _lib.Context(0)
    try:
        sizes = {n: 0 for n in (60, 64, 72, 80)}
        for n in sizes:
            ds = free.upload(*bricks(n))
            sizes[n] = free.dataset_bytes(ds)
            free.free(ds)
    finally:
        free.close()
    budget = sizes[80]
    c = _lib.Context(0, budget_bytes=budget)
    try:
        for n in (60, 64, 72, 80, 80, 60, 80):
            print(f"budget: {n}", flush=True)
            ds = c.upload(*bricks(n))
            assert c.used_bytes()[0] == sizes[n]
            got = c.read_points(ds, 0)
            assert got.dtype == np.float32 and np.array_equal(np.sort(got[got != 0]), np.sort(
                bricks(n)[1][0][0].astype(np.float32).ravel()))
            if n == 80:
                with pytest.raises(_lib.YtrcBudgetError):
                    c.upload(*bricks(8))
            c.free(ds)
            assert c.used_bytes()[0] == 0
        with pytest.raises(_lib.YtrcBudgetError):
            c.upload(*bricks(84))
        # a batch, then the largest dataset again
        vol = render.ResidentVolume(c, uniform_lognormal(16, seed=541), proj_fields="density")
        b = _lib.Batch(c, [vol.projection_request(c0_params(64))], _lib.BATCH_PERSISTENT)
        b.run()
        assert np.any(b.read_image(0) != 0)
        b.close()
        vol.free()
        assert c.used_bytes()[0] == 0
        c.free(c.upload(*bricks(80)))
    finally:
        c.close()
