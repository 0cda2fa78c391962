"""Depths at which a slab is less than an ulp of t (between half of one, where a ray still advances, and a
whole one): the marching wavefronts of the tile kernels against the per-ray slab stepper, which
``packet=False`` selects."""

import numpy as np
import pytest
import torch

from ray_gauss_amd import scenes
from ray_gauss_amd.cameras import look_at_camera
from ray_gauss_amd.caster import TuneConfig

from gpu_helpers import max_rel, prepared_caster

pytestmark = pytest.mark.gpu

# About 1600 rounds add to a Gaussian's sums one after the other in FP32 (6e-8 of the partial sum each, at
# worst all in one direction: 1e-4), and the moments along the ray cancel up to tenfold.
TOL = 1e-3


@pytest.mark.parametrize("words", [0, 64, 8192])
@pytest.mark.parametrize("w,h", [(16, 8), (200, 200)])
@pytest.mark.parametrize("f", [1.0, 4.0])
def test_slabs_below_an_ulp(gpu_device, f, w, h, words):
    """A thin scene at t = 3e5 (slabs of 0.02, an ulp is 0.03125) and 1.2e6 (0.08 and 0.125): every round
    takes its laggard along, so the march ends; images, hits and gradients are the stepper's."""
    depth, n = 3e5 * f, 24
    assert 0.5 < 8 * 0.0025 * f / float(np.spacing(np.float32(depth))) < 2.0 / 3.0
    sc = scenes.scene_uniform(n, seed=1)
    sc.positions[:] = (sc.positions * 20.0 * f + np.array([0.0, depth, 0.0])).astype(np.float32)
    sc.scales[:] = np.array([300.0, 3.0, 300.0], np.float32) * f
    sc.quats[:] = np.array([1.0, 0.0, 0.0, 0.0], np.float32)
    sc.densities[:] = 0.11 + 0.01 * np.arange(n, dtype=np.float32) / n
    prm = scenes.RenderParams(dt=0.0025 * f, t_eps=1e-4)
    cam = look_at_camera(np.zeros(3), target=(0.0, 1.0, 0.0), width=w, height=h, fovx_deg=0.005).launch_record()
    gen = torch.Generator(device=gpu_device).manual_seed(3)
    dL = torch.rand((w * h, 3), generator=gen, device=gpu_device)
    out = {}
    for packet in (False, True):
        rc, _ = prepared_caster(sc, prm, [cam], gpu_device, TuneConfig(packet=packet, replay_words=words))
        img = rc.forward(0, None, depth=True, opacity=True)
        st = rc.stats()
        rc.backward(0, None, img[0], dL, rc.last_token)
        assert rc.stats()["dropped"] == 0
        out[packet] = (img, st, {k: v.cpu().numpy() for k, v in rc.finish_grads().items() if v is not None})
    a, b = out[False], out[True]
    for i in range(3):
        assert torch.equal(a[0][i], b[0][i]), i
    assert a[1]["slab_hits"] == b[1]["slab_hits"] > 300 * w * h and a[1]["pairs"] == b[1]["pairs"]
    for k, v in a[2].items():
        assert max_rel(b[2][k], v) <= TOL, k
