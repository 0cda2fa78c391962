"""The LBVH build (radix sort, refit) and the users of its sort at the sizes where their blocks end: a
refit block spans 256 leaves, a climb 16 blocks (4096, 65536, 1048576 leaves), a sort tile 2048 keys;
past 4096 tiles (8.4M keys) the sort scans its histogram in one block.  The tree check compares every
internal box with the exact union of its children's and every leaf with its Gaussian's, and the links,
which a wrongly sorted order breaks.  After a refit over moved Gaussians the check holds again."""

import numpy as np
import pytest
import torch

from oracle import densify_oracle as D
from oracle import loss_oracle as LO
from ray_gauss_amd import densify as G
from ray_gauss_amd import scenes
from ray_gauss_amd.caster import RayCaster, TuneConfig
from ray_gauss_amd.loss import l1_ssim_forward

pytestmark = pytest.mark.gpu


def _gaussians(n, dev, duplicates):
    g = torch.Generator(device=dev).manual_seed(n)
    pos = torch.rand((n, 3), generator=g, device=dev) * 2 - 1
    if duplicates:  # runs of equal Morton codes, longer than a block of leaves
        pos[: n // 2] = pos[0]
    q = torch.randn((n, 4), generator=g, device=dev)
    return {"positions": pos, "scales": 0.01 + 0.02 * torch.rand((n, 3), generator=g, device=dev),
            "quats": q / q.norm(dim=1, keepdim=True), "densities": torch.rand((n,), generator=g, device=dev),
            "sh": torch.zeros((n, 3, 1), device=dev)}


@pytest.mark.parametrize("duplicates", [False, True])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 512, 2047, 2049, 4095, 4096, 4097, 65535, 65536, 65537, 1048577,
                               4096 * 2048 + 1])
def test_build_and_refit_sizes(gpu_device, n, duplicates):
    t = _gaussians(n, gpu_device, duplicates)
    rc = RayCaster(scenes.RenderParams(), TuneConfig())
    rc.prepare(*t.values(), rebuild=True)
    assert rc.check_bvh() == 0
    cost = rc.tree_cost()
    t["positions"] += 0.05 * torch.randn((n, 3), generator=torch.Generator(device=gpu_device).manual_seed(1),
                                         device=gpu_device)
    for _ in range(3):  # a refit leaves nothing behind for the next
        rc.prepare(*t.values(), rebuild=False)
        assert rc.check_bvh() == 0
    assert n < 3 or rc.tree_cost() != cost


@pytest.mark.parametrize("n", [15, 16, 17, 1025, 4111])
def test_nearest_neighbours_at_wavefront_edges(gpu_device, n):
    """Sixteen queries per wavefront, buckets of 64: counts beside those, with an outlier whose search
    reaches every bucket and one point that is no number (it is nobody's neighbour)."""
    p = np.random.default_rng(n).normal(size=(n, 3)).astype(np.float32)
    p[n // 2] = 1000.0
    ref = D.knn3_mean_dist(p)
    got = G.distCUDA2(torch.from_numpy(p).to(gpu_device)).cpu().numpy()
    assert (np.abs(got - ref) <= 1e-5 * ref).all()
    nan = np.concatenate([p, np.full((1, 3), np.nan, np.float32)])
    got = G.distCUDA2(torch.from_numpy(nan).to(gpu_device)).cpu().numpy()
    assert (np.abs(got[:n] - ref) <= 1e-5 * ref).all()


@pytest.mark.parametrize("W,H,f", [(1, 1, 1), (32, 16, 1), (31, 15, 2), (33, 17, 1), (6, 5, 3), (70, 49, 1)])
def test_loss_at_tile_edges(gpu_device, W, H, f):
    """Images beside a 32x16 tile and smaller than the window: tolerances of the loss tests."""
    rng = np.random.default_rng(W + H)
    rays = rng.uniform(0, 1, (H * f * W * f, 3)).astype(np.float32)
    target = rng.uniform(0, 1, (3, H, W)).astype(np.float32)
    L, g, l1, s = LO.loss(rays.astype(np.float64), target.astype(np.float64), W, H, f, f)
    loss, parts, grad = l1_ssim_forward(torch.from_numpy(rays).to(gpu_device), torch.from_numpy(target).to(gpu_device),
                                        W, H, (f, f))
    assert abs(float(loss) - L) <= 2e-6 * max(1.0, abs(L))
    assert abs(float(parts[0]) - l1) <= 2e-6 and abs(float(parts[1]) - s) <= 2e-6
    assert np.abs(grad.cpu().numpy() - g).max() <= 1e-4 * np.abs(g).max()
