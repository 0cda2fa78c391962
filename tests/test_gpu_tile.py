"""Tiles (wavefronts of rays marching as one beam) against the per-ray slab stepper, which
``packet=False`` selects: the images are bit-identical (the same hits in the same order) and the
gradients equal up to the order of atomic sums, with replayed records, records that end early and
none, over the shapes where the two could part: ragged tiles, several views in a wavefront, beams
too wide for a tile, rounds with more candidates than the list holds, a camera inside the scene."""

import numpy as np
import pytest
import torch

from ray_gauss_amd import scenes
from ray_gauss_amd.batch import tile_order_pixels
from ray_gauss_amd.cameras import look_at_camera, orbit_eye
from ray_gauss_amd.caster import TuneConfig

from gpu_helpers import max_rel, prepared_caster

pytestmark = pytest.mark.gpu


def _compare(scene, params, cams, dev, rv, rp, words):
    rv = torch.as_tensor(np.asarray(rv, np.int32)).to(dev)
    rp = torch.as_tensor(np.asarray(rp, np.int32)).to(dev)
    gen = torch.Generator(device=dev).manual_seed(3)
    dL = torch.randn((rv.shape[0], 3), generator=gen, device=dev)
    out = {}
    for packet in (False, True):
        rc, _ = prepared_caster(scene, params, cams, dev, TuneConfig(packet=packet, replay_words=words))
        rgb, depth, opac = rc.forward_batch(rv, rp, depth=True, opacity=True)
        st = rc.stats()
        rc.backward_batch(rv, rp, rgb, dL, rc.last_token)
        assert rc.stats()["dropped"] == 0
        g = {k: v.cpu().numpy() for k, v in rc.finish_grads().items() if v is not None}
        out[packet] = (rgb, depth, opac, st, g)
    a, b = out[False], out[True]
    for i in range(3):
        assert torch.equal(a[i], b[i]), i
    assert a[3]["slab_hits"] == b[3]["slab_hits"] and a[3]["pairs"] == b[3]["pairs"]
    for k, v in a[4].items():
        assert max_rel(b[4][k], v) <= 1e-5, k
    return b[3]


def _view(w, h, radius=3.0, fov=40.0, az=30.0):
    return look_at_camera(orbit_eye(radius, az, 20.0), width=w, height=h, fovx_deg=fov).launch_record()


@pytest.mark.parametrize("words", [0, 8, 1536])
@pytest.mark.parametrize("w,h", [(1, 1), (7, 9), (64, 1), (65, 17)])
def test_ragged_tiles(gpu_device, w, h, words):
    sc = scenes.scene_uniform(3000, seed=w + h)
    prm = scenes.RenderParams(dt=0.01, t_eps=1e-4, white_background=True)
    cam = _view(w, h)
    st = _compare(sc, prm, [cam], gpu_device, np.zeros(w * h), np.arange(w * h), words)
    assert st["slab_hits"] > 0


@pytest.mark.parametrize("views,fov", [(3, 2.0), (6, 2.0), (2, 120.0)])
def test_wavefronts_of_several_views_and_wide_beams(gpu_device, views, fov):
    """Rays of three narrow views in turn march as three beams of one wavefront; six views, or views
    whose 64 rays spread over 120 degrees, go to the slab stepper."""
    sc = scenes.scene_uniform(3000, seed=views)
    prm = scenes.RenderParams(dt=0.01, t_eps=1e-4)
    cams = [_view(16, 16, fov=fov, az=50.0 * v) for v in range(views)]
    i = np.arange(16 * 16 * views)
    st = _compare(sc, prm, cams, gpu_device, i % views, np.random.default_rng(0).permutation(256)[i // views], 64)
    assert st["slab_hits"] > 0


@pytest.mark.parametrize("words", [0, 16, 1536])
def test_wavefronts_across_rows_of_tiles(gpu_device, words):
    """A large list of 8x8 tiles of a view whose width is no multiple of eight: wavefronts of 64 rays
    that hold the end of a row of tiles and the start of the next march as two beams of one view."""
    sc = scenes.scene_uniform(2000, seed=4)
    prm = scenes.RenderParams(dt=0.02, t_eps=1e-4)
    cam = _view(611, 401)
    rp = tile_order_pixels(611, 401)
    st = _compare(sc, prm, [cam], gpu_device, np.zeros(len(rp)), rp, words)
    assert st["slab_hits"] > 0


@pytest.mark.parametrize("words", [0, 64, 4096])
def test_rounds_with_more_candidates_than_the_list(gpu_device, words):
    """Large overlapping Gaussians: single slabs hold more candidates than a tile's list, so their
    rounds go on with further lists (in a backward without records, walk the tree) and have more
    events than one batch."""
    sc = scenes.scene_uniform(1200, seed=5, log_scale_mean=-1.2)
    sc.densities[:] = 0.11 + 0.002 * np.arange(1200, dtype=np.float32) / 1200
    sc.scales[:] *= 4.0
    prm = scenes.RenderParams(dt=0.02, t_eps=1e-4)
    st = _compare(sc, prm, [_view(9, 9)], gpu_device, np.zeros(81), np.arange(81), words)
    assert st["fallback_slabs"] > 0 and st["slab_hits"] > 300 * 64


@pytest.mark.parametrize("t_near", [0.0, 0.7, -0.5])
def test_camera_inside_the_scene(gpu_device, t_near):
    """Rays that start inside the scene (and inside ellipsoids); depths below zero are left to the
    slab stepper."""
    sc = scenes.scene_uniform(3000, seed=11, log_scale_mean=-2.5)
    prm = scenes.RenderParams(dt=0.01, t_eps=1e-4, t_near=t_near, t_far=2.5)
    st = _compare(sc, prm, [_view(24, 16, radius=0.3)], gpu_device, np.zeros(384), np.arange(384), 512)
    assert st["slab_hits"] > 0


@pytest.mark.parametrize("n", [255, 256, 257, 511, 513])
def test_lists_around_their_capacity(gpu_device, n):
    """Every Gaussian is a candidate of the rounds at the centre: lists of all, or split between leaves."""
    sc = scenes.scene_uniform(n, seed=n)
    sc.positions[:] *= 0.01
    sc.scales[:] = 0.3
    sc.densities[:] = 0.11 + 0.002 * np.arange(n, dtype=np.float32) / n
    prm = scenes.RenderParams(dt=0.02, t_eps=1e-4)
    st = _compare(sc, prm, [_view(16, 8)], gpu_device, np.zeros(128), np.arange(128), 4096)
    assert st["slab_hits"] >= n


@pytest.mark.parametrize("power", [-34, -29, 0, 29, 34])
def test_scales_beyond_the_range_of_the_fast_terms(gpu_device, power):
    """A scene scaled by powers of two: squared lengths in ellipsoid space from 2^-70 to 2^80, inside and
    outside the range in which the predicate's terms take the short square root."""
    f = 2.0 ** power
    sc = scenes.scene_uniform(600, seed=2)
    sc.positions[:] *= f
    sc.scales[:] *= f
    prm = scenes.RenderParams(dt=0.01 * f, t_eps=1e-4, t_far=10.0 * f)
    cam = look_at_camera(orbit_eye(3.0, 30.0, 20.0) * f, target=(0.0, 0.0, 0.0), width=24, height=16,
                         fovx_deg=40.0).launch_record()
    st = _compare(sc, prm, [cam], gpu_device, np.zeros(384), np.arange(384), 512)
    assert st["slab_hits"] > 0


@pytest.mark.parametrize("words", [0, 64, 2048])
@pytest.mark.parametrize("w,h", [(264, 520), (447, 455)])
def test_split_wavefronts(gpu_device, w, h, words):
    """Whole views with a dense spot: the dear wavefronts (of 32 rays and of 64, with ragged edges) march
    in quarters, forward and backward; a backward of another view does not take their records."""
    sc = scenes.scene_uniform(6000, seed=7)
    sc.positions[:5000] = 0.08 * sc.positions[:5000] + 0.3
    sc.scales[:5000] *= 0.2
    prm = scenes.RenderParams(dt=0.01, t_eps=1e-4, white_background=True)
    cams = [_view(w, h), _view(w, h, az=75.0)]
    gen = torch.Generator(device=gpu_device).manual_seed(3)
    dL = torch.randn((w * h, 3), generator=gen, device=gpu_device)
    out = {}
    for packet in (False, True):
        rc, _ = prepared_caster(sc, prm, cams, gpu_device, TuneConfig(packet=packet, replay_words=words))
        img = [rc.forward(v, None, depth=True, opacity=True) for v in (1, 0)]
        st = rc.stats()
        grads = []
        for v in (0, 1):
            rc.backward(v, None, img[1 - v][0], dL, rc.last_token)
            assert rc.stats()["dropped"] == 0
            grads.append({k: t.cpu().numpy() for k, t in rc.finish_grads().items() if t is not None})
        out[packet] = (img, st, grads)
    a, b = out[False], out[True]
    for v in range(2):
        for i in range(3):
            assert torch.equal(a[0][v][i], b[0][v][i]), (v, i)
        for k, t in a[2][v].items():
            assert max_rel(b[2][v][k], t) <= 1e-5, (v, k)
    assert a[1]["slab_hits"] == b[1]["slab_hits"] > 0 and a[1]["pairs"] == b[1]["pairs"]


@pytest.mark.parametrize("rnd", [0, 1, 2])
@pytest.mark.parametrize("spb", [3, 8, 11])
def test_samples_across_lanes(gpu_device, spb, rnd):
    """Small jobs hold a ray in eight lanes, one sample each (with more than eight per slab they take the
    other form), with every placement of the samples."""
    sc = scenes.scene_uniform(2000, seed=spb)
    prm = scenes.RenderParams(dt=0.02, samples_per_slab=spb, t_eps=1e-3, jitter=rnd & 1, rnd_sample=rnd, iteration=7,
                              white_background=True)
    st = _compare(sc, prm, [_view(29, 19)], gpu_device, np.zeros(551), np.arange(551), 512)
    assert st["slab_hits"] > 0


def _blocks(size, block, groups, seed):
    """Rays in groups of 64, random pixels of a block each, of a view size x size."""
    rng = np.random.default_rng(seed)
    x, y = (rng.integers(0, size - block + 1, groups)[:, None] + rng.integers(0, block, (groups, 64)) for _ in range(2))
    return (y * size + x).reshape(-1)


@pytest.mark.parametrize("words", [0, 512])
@pytest.mark.parametrize("block,groups", [(96, 600), (256, 600), (512, 600), (256, 3200), (512, 3200)])
def test_random_rays_of_blocks(gpu_device, block, groups, words):
    """Wavefronts of 16 and 64 random rays of wide blocks beside ordinary tiles: some are beams, the others
    are left to the stepper in parts; where many are left, beams are held to half the width."""
    sc = scenes.scene_uniform(3000, seed=block)
    prm = scenes.RenderParams(dt=0.02, t_eps=1e-4, white_background=True)
    px = np.concatenate([_blocks(1024, block, groups, 1), tile_order_pixels(1024, 1024)[: 64 * 100]])
    st = _compare(sc, prm, [_view(1024, 1024)], gpu_device, np.zeros(len(px)), px, words)
    assert st["slab_hits"] > 0


@pytest.mark.parametrize("words", [0, 64, 4096])
def test_wide_beams_in_dense_stretches(gpu_device, words):
    """Wide beams whose rounds hold more candidates than the list: they are walked, and the rounds after
    them too, a growing number before the next gather."""
    sc = scenes.scene_uniform(1200, seed=5, log_scale_mean=-1.2)
    sc.densities[:] = 0.11 + 0.002 * np.arange(1200, dtype=np.float32) / 1200
    sc.scales[:] *= 3.0
    prm = scenes.RenderParams(dt=0.02, t_eps=1e-4)
    px = _blocks(128, 16, 4, 2)
    st = _compare(sc, prm, [_view(128, 128)], gpu_device, np.zeros(len(px)), px, words)
    assert st["fallback_slabs"] > 0 and st["slab_hits"] > 300 * 256
