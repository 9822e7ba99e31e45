"""Gradients stay the sums they were.  The waves of a block add their gradient terms in FP32 in the
order in which they come to them, so how lanes are scheduled through the traversal shows in the last
bits: single renders lie up to 4.5e-8 (2-norm, relative) from the mean of many, and that mean moved
by 0.7e-7 to 1.3e-7 when the adjoint's traversal took the vote of the forward kernels.  Here the mean
of 32 renders is held to the recorded mean of 24 (tests/golden/adjoint_sums.json; its thirds differ by
at most 1e-8) within half of FP32's rounding unit: 2^-25.  Meshes of 81,922 and 20,482
triangles under an environment light, paths with one replay (6 bounces) and with two (12)."""
import json
import os

import numpy as np
import pytest

import tinypt_amd as T
from tinypt_amd import scenes

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "adjoint_sums.json")


@pytest.mark.parametrize("w,h,spp,bounces,subdivisions", [(80, 81, 8, 6, 6), (111, 112, 15, 6, 5), (61, 45, 5, 12, 5)])
def test_mean_gradient_is_the_recorded_one(gpu_ctx, w, h, spp, bounces, subdivisions):
    with open(GOLDEN) as f:
        want = np.array(json.load(f)["%d_%d_%d_%d_%d" % (w, h, spp, bounces, subdivisions)])
    sc = scenes.mesh_scene(w, h, subdivisions=subdivisions, env=scenes.synthetic_env(64, 32, seed=4))
    ds = T.DeviceScene(sc, gpu_ctx)
    dl = np.random.default_rng(11).standard_normal((h, w, 3)).astype(np.float32) / (h * w)
    cfg = T.RenderConfig(width=w, height=h, spp=spp, max_bounces=bounces, rr_start=3, seed=11)
    got = np.mean([np.asarray(T.render_adjoint(ds, cfg, dl)[0]) for _ in range(32)], axis=0)
    assert np.linalg.norm(got - want) <= 2.0 ** -25 * np.linalg.norm(want)
