"""Traversal kernels for small scenes (trees in LDS, rays handed to idle lanes from each wave's own
share) against the one-ray-per-lane kernels on device memory (traversal_refill = -1): each ray's
sequence of tests is the same, so the sums are equal bit for bit.  Scenes: a flattened tree alone
(also one whose root is a leaf), spheres alone, both, a single triangle, nothing, the largest that
fits the LDS and the smallest that does not.  Passes of more than 2^18 paths, since a smaller one
goes to the kernel that walks whole paths; path counts that are no multiple of a wave."""
import numpy as np
import pytest

import tinypt_amd as T
from parity_scenes import PARITY_CASES, floorlight
from tinypt_amd import scenes
from tinypt_amd.scene import DiffuseLight, Instance, Mesh, Transform

pytestmark = pytest.mark.gpu


def _mesh(subdivisions):
    return scenes.mesh_scene(64, 64, subdivisions=subdivisions, env=scenes.synthetic_env(32, 16, seed=2))


def _without(sc, n_instances):
    sc.world.instances = sc.world.instances[:n_instances]
    return sc


SCENES = {
    "cornell": lambda: scenes.cornell_box(64, 64),
    "spheres": lambda: scenes.default_scene(64, 64, "sky"),
    "spheres_in_box": lambda: scenes.inverse_scene(scenes.inverse_params(3, 16), 64, 64, 16),
    "zoo": PARITY_CASES["material_zoo"][0],
    "root_is_a_leaf": floorlight,
    "empty": lambda: _without(floorlight(), 0),
    "80_triangles": lambda: _mesh(1),
    "320_triangles": lambda: _mesh(2),
    "1280_triangles": lambda: _mesh(3),
}


@pytest.mark.parametrize("name", list(SCENES))
@pytest.mark.parametrize("w,h,spp", [(67, 61, 131), (64, 64, 65)])
def test_small_scene_kernels_keep_the_image(gpu_ctx, name, w, h, spp):
    ds = T.DeviceScene(SCENES[name](), gpu_ctx)
    kw = dict(width=w, height=h, spp=spp, max_bounces=6, rr_start=4, seed=31)
    a, b = (T.render(ds, T.RenderConfig(traversal_refill=r, **kw)) for r in (0, -1))
    for f in ("acc", "acc_w", "acc_sq"):
        np.testing.assert_array_equal(getattr(a, f), getattr(b, f), err_msg=f)
    for k in ("rays_extension", "rays_shadow", "light_samples", "light_self_occluded"):
        assert a.stats[k] == b.stats[k], k


@pytest.mark.parametrize("name", ["cornell", "1280_triangles"])
@pytest.mark.parametrize("w,h,spp", [(513, 1, 512), (1, 300, 1024), (640, 360, 3), (1023, 513, 1)])
def test_camera_rays_are_each_traced_once(gpu_ctx, name, w, h, spp):
    """The order in which blocks take the camera rays, at widths and path counts around multiples of
    a block and of the grid: every path is counted and traced once, and one pass sums what passes
    of single samples (which go to the kernel that walks whole paths) sum."""
    ds = T.DeviceScene(SCENES[name](), gpu_ctx)
    kw = dict(width=w, height=h, spp=spp, max_bounces=3, rr_start=4, seed=3)
    a = T.render(ds, T.RenderConfig(**kw))
    b = T.render(ds, T.RenderConfig(samples_per_pass=min(spp, 512 if w == 1 else 1 if w < 1000 else spp),
                                    traversal_refill=-1, **kw))
    assert a.stats["paths"] == b.stats["paths"] == w * h * spp
    assert a.stats["rays_extension"] == b.stats["rays_extension"]
    np.testing.assert_allclose(a.acc, b.acc, rtol=1e-12, atol=0)  # FP64 sums of up to 1024 terms, grouped differently


@pytest.mark.parametrize("bounces", [6, 12])
@pytest.mark.parametrize("name", ["cornell", "spheres", "spheres_in_box", "zoo", "root_is_a_leaf", "80_triangles"])
def test_short_passes_and_gradients_of_small_scenes(gpu_ctx, name, bounces):
    """The kernel that walks whole paths and the adjoint read the trees from LDS too: the sums of a
    short pass equal those of the device-memory form bit for bit, and the gradient that of the same
    scene with 5120 triangles added far away, which make it a large one.  Both sum the same path
    terms, a block at a time in FP32 and in another order: n = 1536 terms of a block give
    sqrt(n) 2^-24 = 2.3e-6 of the sum of their magnitudes, 1e-4 of the largest gradient where a
    fortieth of that sum is left; roughness differences cancel further, 1e-3."""
    kw = dict(width=41, height=29, spp=12, max_bounces=bounces, rr_start=4, seed=5)
    ds = T.DeviceScene(SCENES[name](), gpu_ctx)
    few, plain = (T.render(ds, T.RenderConfig(traversal_refill=r, **kw)) for r in (0, -1))
    for f in ("acc", "acc_w", "acc_sq"):
        np.testing.assert_array_equal(getattr(few, f), getattr(plain, f), err_msg=f)
    big = SCENES[name]()
    speck = 1e-3 * scenes.displaced_icosphere(4)[0] + np.array([3e3, -9e3, 5e3])
    dark = next(k for k, m in enumerate(big.mats) if m.kind != DiffuseLight((1, 1, 1)).kind)
    big.world.meshes.append(Mesh(speck, dark))
    big.world.instances.append(Instance(len(big.world.meshes) - 1, Transform.identity(), None))
    dl = np.ones((29, 41, 3), np.float32)
    g, _ = T.render_adjoint(ds, T.RenderConfig(**kw), dl)
    h, _ = T.render_adjoint(T.DeviceScene(big, gpu_ctx), T.RenderConfig(**kw), dl)
    g, h = np.asarray(g), np.asarray(h)
    scale = np.abs(h).max()
    np.testing.assert_allclose(g[:, :3], h[:, :3], rtol=0, atol=1e-4 * scale)
    np.testing.assert_allclose(g[:, 3], h[:, 3], rtol=0, atol=1e-3 * scale)
