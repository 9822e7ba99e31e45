"""A pass of few paths, and the last paths of a large pass, are walked to their ends by one kernel
(one lane per path) instead of bounce by bounce through queues.  A path's radiance must not depend
on which of the two took it: a frame of 307,200 paths, which starts bounce by bounce and ends in
that kernel, against the same frame in two batches of 153,600 paths, which the kernel takes whole --
every pixel's sums bit for bit, and the same numbers of rays and light samples.  The scenes cover
both stack forms, scenes with and without environment light, area lights and all materials."""
import numpy as np
import pytest

import tinypt_amd as T

from parity_scenes import PARITY_CASES

pytestmark = pytest.mark.gpu

COUNTS = ("paths", "rays_extension", "rays_shadow", "light_samples", "light_self_occluded")


@pytest.mark.parametrize("case", sorted(PARITY_CASES))
def test_whole_paths_equal_bounce_by_bounce(gpu_ctx, case):
    build, _, _, _, mb, rr, seed = PARITY_CASES[case]
    ds = T.DeviceScene(build(), gpu_ctx)
    w, h = 640, 480
    cfg = T.RenderConfig(width=w, height=h, spp=1, max_bounces=mb, rr_start=rr, seed=seed)
    full = T.render(ds, cfg)
    half = w * h // 2
    parts = [T.render_pixels(ds, cfg, np.arange(p0, p0 + half), want_sq=True) for p0 in (0, half)]
    assert np.array_equal(np.concatenate([p[0] for p in parts]), full.acc.reshape(-1, 3))
    assert np.array_equal(np.concatenate([p[2] for p in parts]), full.acc_sq.reshape(-1, 3))
    for k in COUNTS:
        assert sum(p[3][k] for p in parts) == full.stats[k], k
    assert full.stats["trace_launches"] > 0 and all(p[3]["trace_launches"] == 0 for p in parts)


@pytest.mark.parametrize("n", [1, 7, 8, 63, 65, 2049, 20_000])
def test_few_paths(gpu_ctx, n):
    """Batches from one path to more than the kernel's waves at eight lanes each."""
    build, _, _, _, mb, rr, seed = PARITY_CASES["material_zoo"]
    ds = T.DeviceScene(build(), gpu_ctx)
    w, h = 640, 480
    cfg = T.RenderConfig(width=w, height=h, spp=1, max_bounces=mb, rr_start=rr, seed=seed)
    full = T.render(ds, cfg).acc.reshape(-1, 3)
    pix = np.random.default_rng(n).choice(w * h, n, replace=False).astype(np.int32)
    s, sw, _, _ = T.render_pixels(ds, cfg, pix)
    assert np.array_equal(s, full[pix]) and (sw == 1).all()
