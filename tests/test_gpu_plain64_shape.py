"""The plain FP64 form gives a pixel one lane or four, and few or many lanes of a wave, by the image's
size and the depth of the scene's trees.  A pixel's samples must not depend on it: frames large
enough for one lane per pixel, and for four in full waves, against batches of their pixels small
enough for four lanes in part of a wave, bit for bit."""
import numpy as np
import pytest

import tinypt_amd as T

from parity_scenes import PARITY_CASES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", sorted(PARITY_CASES))
@pytest.mark.parametrize("w,h", [(500, 400), (211, 197)])
def test_lanes_per_pixel_keep_the_samples(gpu_ctx, case, w, h):
    build, _, _, _, mb, rr, seed = PARITY_CASES[case]
    ds = T.DeviceScene(build(), gpu_ctx)
    cfg = T.RenderConfig(width=w, height=h, spp=2, max_bounces=mb, rr_start=rr, seed=seed, precision=T.FP64_PLAIN)
    full = T.render(ds, cfg)
    assert (full.acc_w == 2).all()
    for n in (1, 5, 3001):
        pix = np.random.default_rng(n).choice(w * h, n, replace=False).astype(np.int32)
        s, sw, sq, _ = T.render_pixels(ds, cfg, pix, want_sq=True)
        assert np.array_equal(s, full.acc.reshape(-1, 3)[pix]) and np.array_equal(sq, full.acc_sq.reshape(-1, 3)[pix])
        assert (sw == 2).all()


def test_adaptive_over_several_launches(gpu_ctx):
    """Samples split over launches (100 spp, at most 64 a launch) with a stop rule that some pixels
    meet: the state carried between launches gives the sums of the pixels alone."""
    build, _, _, _, mb, rr, seed = PARITY_CASES["cornell"]
    ds = T.DeviceScene(build(), gpu_ctx)
    cfg = T.RenderConfig(width=64, height=48, spp=100, max_bounces=mb, rr_start=rr, seed=seed, precision=T.FP64_PLAIN,
                         adaptive_enabled=True, adaptive_min_spp=16, adaptive_threshold=0.1)
    full = T.render(ds, cfg)
    assert full.acc_w.min() < 100 and full.acc_w.max() > 64
    pix = np.arange(1500, 1533, dtype=np.int32)
    s, sw, _, _ = T.render_pixels(ds, cfg, pix)
    assert np.array_equal(s, full.acc.reshape(-1, 3)[pix]) and np.array_equal(sw, full.acc_w.reshape(-1)[pix])
