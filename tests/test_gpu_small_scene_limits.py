"""Scenes on both sides of the limits of the small-scene kernels: 32 KB of trees (meshes of 340 to 432
triangles cross it) and 20 stack entries (chains of spheres of growing size).  The image is the
same bit for bit from the kernels that the scene's shape selects, from one ray per lane and from
persistent waves, whose extension and shadow kernels are all different ones; so is that of a scene
with nothing in it."""
import numpy as np
import pytest

import tinypt_amd as T
from tinypt_amd import scenes
from tinypt_amd.scene import Camera, DiffuseLight, EnvMap, Lambert, Transform

pytestmark = pytest.mark.gpu

ENV = scenes.synthetic_env(32, 16, seed=2)


def _cloud(n):
    rng = np.random.default_rng(1)
    b = scenes.SceneBuilder()
    b.mesh_instance(rng.uniform(-1, 1, (n, 1, 3)) + rng.uniform(-0.15, 0.15, (n, 3, 3)), Transform.identity(),
                    Lambert((0.6, 0.5, 0.4)))
    b.sphere((0.0, 2.0, 1.0), 0.4, DiffuseLight((5.0, 5.0, 5.0)))
    return b.build(Camera.look_at((0, 0, 3.5), (0, 0, 0), (0, 1, 0), 50, 1.0), ENV)


def _chain(n):
    b = scenes.SceneBuilder()
    for k in range(n):
        x = 1.6 ** k * 1e-3
        b.sphere((x, 0.0, 0.0), 0.2 * x, Lambert((0.5, 0.6, 0.7)))
    b.sphere((0.0, 3.0, 2.0), 0.4, DiffuseLight((5.0, 5.0, 5.0)))
    return b.build(Camera.look_at((0, 0, 5), (0, 0, 0), (0, 1, 0), 40, 1.0), ENV)


def _same_image(ds):
    kw = dict(width=65, height=63, spp=67, max_bounces=4, rr_start=4, seed=31)  # more than 2^18 paths
    a, *rest = [T.render(ds, T.RenderConfig(traversal_refill=r, **kw)) for r in (0, -1, 48)]
    assert (a.acc_w == 67).all() and a.acc.max() > 0
    for b in rest:
        np.testing.assert_array_equal(a.acc, b.acc)
        np.testing.assert_array_equal(a.acc_sq, b.acc_sq)
        for k in ("rays_extension", "rays_shadow", "light_samples", "light_self_occluded"):
            assert a.stats[k] == b.stats[k], k


@pytest.mark.parametrize("n", range(340, 433, 4))
def test_byte_limit(gpu_ctx, n):
    _same_image(T.DeviceScene(_cloud(n), gpu_ctx))


@pytest.mark.parametrize("stack", [18, 19, 20, 21, 22])
def test_stack_limit(gpu_ctx, stack):
    n = next(n for n in range(12, 40) if T.HostScene(_chain(n)).info()["traversal_stack"] >= stack)
    _same_image(T.DeviceScene(_chain(n), gpu_ctx))


def test_nothing_to_hit(gpu_ctx):
    b = scenes.SceneBuilder()
    _same_image(T.DeviceScene(b.build(Camera.look_at((0, 0, 5), (0, 0, 0), (0, 1, 0), 40, 1.0), ENV), gpu_ctx))
