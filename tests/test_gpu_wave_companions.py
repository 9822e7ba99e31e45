"""The traversal schedules a wave's lanes together (a lane may wait at an inner node or at a leaf for
the others), so a ray's hit must not depend on the rays that share its wave: every ray of a batch
again in a wave of its own (each ray 64 times), in batches that leave partial waves, and shuffled.
Hits are compared bit for bit: a ray's own sequence of tests is the same in all of them."""
import numpy as np
import pytest

import tinypt_amd as T
from parity_scenes import PARITY_CASES
from trace_checks import path_rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["cornell", "material_zoo", "mesh_small", "instanced_small"])
def test_hits_do_not_depend_on_the_wave(gpu_ctx, name):
    sc = PARITY_CASES[name][0]()
    rng = np.random.default_rng(23)
    rays = path_rays(sc, rng, 4096)
    rays = rays[rng.permutation(len(rays))][:1500]
    ds = T.DeviceScene(sc, gpu_ctx)
    ref = ds.trace_closest(rays)
    one = ds.trace_closest(np.repeat(rays, 64, axis=0))
    perm = rng.permutation(len(rays))
    mixed = ds.trace_closest(rays[perm])
    for key, v in ref.items():
        np.testing.assert_array_equal(one[key].reshape(len(rays), 64), np.repeat(v[:, None], 64, axis=1), err_msg=key)
        np.testing.assert_array_equal(mixed[key], v[perm], err_msg=key)
        for n in (1, 2, 63, 64, 65, 257):
            np.testing.assert_array_equal(ds.trace_closest(rays[:n])[key], v[:n], err_msg=f"{key} {n}")
