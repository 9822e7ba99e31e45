"""The plain FP64 form with 16, 32 and 64 lanes of a wave in use: frames whose pixel counts lie at the
edges of the three, against a batch of their pixels, which takes 16.  A pixel's sums are the same bit
for bit, whichever lanes work on it."""
import numpy as np
import pytest

import tinypt_amd as T
from tinypt_amd import scenes

from parity_scenes import PARITY_CASES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(64, 128), (8193, 1), (127, 129), (113, 145), (223, 220), (49153, 1)])
@pytest.mark.parametrize("deep", [False, True])
def test_lanes_in_use_keep_the_samples(gpu_ctx, deep, w, h):
    if deep:
        ds = T.DeviceScene(scenes.mesh_scene(w, h, subdivisions=4, env=scenes.synthetic_env(32, 16, seed=2)), gpu_ctx)
    else:
        ds = T.DeviceScene(PARITY_CASES["cornell"][0](), gpu_ctx)
    cfg = T.RenderConfig(width=w, height=h, spp=2, max_bounces=4, rr_start=2, seed=9, precision=T.FP64_PLAIN)
    full = T.render(ds, cfg)
    assert (full.acc_w == 2).all()
    # the first and last pixels of waves of all three forms, and some others
    pix = np.unique(np.concatenate([np.arange(70), np.arange(w * h - 70, w * h),
                                    np.random.default_rng(w).choice(w * h, 1500, replace=False)])).astype(np.int32)
    s, sw, sq, _ = T.render_pixels(ds, cfg, pix, want_sq=True)
    assert np.array_equal(s, full.acc.reshape(-1, 3)[pix]) and np.array_equal(sq, full.acc_sq.reshape(-1, 3)[pix])
    assert (sw == 2).all()
