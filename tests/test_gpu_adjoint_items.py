"""Roughness gradients of paths too long to log their vertices: the wave gathers its paths' (path, GGX
material) items and replays them two lanes an item.  A closed box of GGX walls around GGX spheres,
without Russian roulette, gives every path several items -- more than one filling of the wave's item
list -- and an image of 37 x 5 pixels at 3 spp leaves partial waves and a partial block.  The
gradient is the central difference of the render's own loss with the same seeds (h = 1e-3), to the
1% at which the render's FP32 sums resolve it."""
import numpy as np
import pytest

import tinypt_amd as T
from tinypt_amd import _abi, scenes
from tinypt_amd.scene import Camera, DiffuseLight, EnvMap, Ggx, Transform

pytestmark = pytest.mark.gpu

H = 1e-3


def ggx_box():
    b = scenes.SceneBuilder()
    R, S, Tr = Transform.rotate, Transform.scale, Transform.translate
    rect = scenes.unit_rectangle_tris()
    walls = [((0, -1, 0), (1, 0, 0), -90), ((0, 1, 0), (1, 0, 0), 90), ((-1, 0, 0), (0, 1, 0), 90),
             ((1, 0, 0), (0, 1, 0), -90), ((0, 0, -1), (0, 1, 0), 0), ((0, 0, 1), (0, 1, 0), 180)]
    for k, (t, axis, deg) in enumerate(walls):
        b.mesh_instance(rect, scenes.compose_ops([Tr(t), R(axis, float(deg)), S((1.0, 1.0, 1.0))]),
                        Ggx((0.7, 0.8, 0.9), 0.25 + 0.05 * k))
    for k in range(6):
        b.sphere((-0.5 + 0.2 * k, -0.4 + 0.15 * (k % 3), -0.3 + 0.2 * (k % 2)), 0.12, Ggx((0.9, 0.8, 0.7), 0.2 + 0.04 * k))
    b.sphere((0.0, 0.6, 0.1), 0.15, DiffuseLight((6.0, 5.0, 4.0)))
    return b.build(Camera.look_at((0, 0, 0.9), (0, 0, 0), (0, 1, 0), 70, 37 / 5), EnvMap.constant((0, 0, 0)))


@pytest.mark.parametrize("w,h,spp", [(37, 5, 3), (64, 32, 16)])
def test_roughness_of_many_materials_per_path(gpu_ctx, w, h, spp):
    sc = ggx_box()
    ds = T.DeviceScene(sc, gpu_ctx)
    base = np.array([m.param for m in sc.mats], dtype=np.float64)
    dl = np.random.default_rng(17).uniform(0.0, 1.0, (h, w, 3)).astype(np.float32)
    cfg = T.RenderConfig(width=w, height=h, spp=spp, max_bounces=12, rr_start=12, seed=21)
    g, st = T.render_adjoint(ds, cfg, dl)
    assert st["paths"] == w * h * spp

    def loss(params):
        ds.update_materials(params)
        return float((dl.astype(np.float64) * (T.render(ds, cfg, want_sq=False).acc / spp)).sum())

    ggx = [i for i, m in enumerate(sc.mats) if m.kind == _abi.MAT_GGX]
    fd = []
    for i in ggx:
        p = base.copy()
        p[i, 3] += H
        up = loss(p)
        p[i, 3] -= 2 * H
        fd.append((up - loss(p)) / (2 * H))
    ds.update_materials(base)
    fd, ad = np.array(fd), g[ggx, 3]
    sig = np.abs(fd) > 1e-3 * np.abs(fd).max()
    assert sig.sum() >= 4  # few paths of the small image meet the spheres
    assert (np.abs(ad - fd)[sig] / np.abs(fd)[sig]).max() < 0.01, (ad, fd)
