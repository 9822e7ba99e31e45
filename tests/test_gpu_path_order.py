"""The order in which a pass numbers its paths (pixel groups, samples inside a group) must not
change what each pixel sums: renders whose pixel counts leave a partial last group, in one pass
in passes of other sample counts and through the adaptive sampler's active lists (a threshold of
zero never stops a pixel), against one sample per pass, where each pixel has one path."""
import numpy as np
import pytest

import tinypt_amd as T
from tinypt_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(1, 1), (2, 1), (3, 1), (37, 23), (64, 2)])
def test_path_order_keeps_each_pixels_samples(gpu_ctx, w, h):
    ds = T.DeviceScene(scenes.cornell_box(w, h), gpu_ctx)
    spp = 21
    kw = dict(width=w, height=h, spp=spp, max_bounces=6, rr_start=3, seed=17)
    one = T.render(ds, T.RenderConfig(samples_per_pass=1, **kw))
    others = [T.render(ds, T.RenderConfig(samples_per_pass=k, **kw)) for k in (2, 5, spp)]
    others += [T.render(ds, T.RenderConfig(adaptive_enabled=True, adaptive_min_spp=m, adaptive_threshold=0.0, **kw))
               for m in (1, 5)]
    for o in others:
        assert (o.acc_w == spp).all()
        # FP64 sums of 21 non-negative terms, grouped differently: a few FP64 ulps
        np.testing.assert_allclose(o.acc, one.acc, rtol=1e-13, atol=0)
        np.testing.assert_allclose(o.acc_sq, one.acc_sq, rtol=1e-13, atol=0)
