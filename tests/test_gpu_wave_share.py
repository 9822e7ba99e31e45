"""Persistent traversal on device memory (each wave takes rays from its own share, a lane's next ray
held ahead) against one ray per lane: the sums are equal bit for bit at every number of lanes that
may go idle, for passes that leave waves with a partial share or none, with and without the
stack's overflow area.  Passes of more than 2^18 paths, so that the queued kernels run."""
import numpy as np
import pytest

import tinypt_amd as T
from parity_scenes import PARITY_CASES
from tinypt_amd import scenes

pytestmark = pytest.mark.gpu

SCENES = {
    "mesh_1280": lambda: scenes.mesh_scene(64, 64, subdivisions=3, env=scenes.synthetic_env(32, 16, seed=2)),
    "mesh_20480": lambda: scenes.mesh_scene(64, 64, subdivisions=5, env=scenes.synthetic_env(32, 16, seed=2)),
    "zoo": PARITY_CASES["material_zoo"][0],
    "instances": PARITY_CASES["instanced_small"][0],
}


@pytest.mark.parametrize("name", list(SCENES))
@pytest.mark.parametrize("w,h,spp", [(67, 61, 131), (257, 129, 8)])
def test_wave_shares_keep_the_image(gpu_ctx, name, w, h, spp):
    ds = T.DeviceScene(SCENES[name](), gpu_ctx)
    kw = dict(width=w, height=h, spp=spp, max_bounces=6, rr_start=4, seed=13)
    ref = T.render(ds, T.RenderConfig(traversal_refill=-1, **kw))
    for lanes in (0, 1, 48, 63):
        out = T.render(ds, T.RenderConfig(traversal_refill=lanes, **kw))
        for f in ("acc", "acc_w", "acc_sq"):
            np.testing.assert_array_equal(getattr(out, f), getattr(ref, f), err_msg=f"{f} {lanes}")
        for k in ("rays_extension", "rays_shadow", "light_samples", "light_self_occluded"):
            assert out.stats[k] == ref.stats[k], (k, lanes)
