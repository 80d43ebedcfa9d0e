"""The march over a world's grid of bytes against the general march, bit for
bit: the general march serves traced updates and several rays per lane."""
import numpy as np
import pytest

from lum_amd import synth
from lum_amd.api import Batch, Model, World, camera_default, placement, radiance_params
from lum_amd._lib import RADIANCE_BF16, RADIANCE_F16, RADIANCE_F32

pytestmark = pytest.mark.gpu


def sparse_palette(rng, n):
    """Slots from empty over single voxels and octants to full."""
    pal = np.zeros((n, 16, 16, 16), np.uint8)
    for k in range(1, n):
        fill = (0.0, 0.0005, 0.01, 0.3, 1.0)[k % 5]
        pal[k] = np.where(rng.random((16, 16, 16)) < fill, rng.integers(1, 256, (16, 16, 16)), 0)
        if k % 3 == 0:  # some octants only
            z, y, x = rng.integers(0, 2, 3) * 8
            keep = np.zeros((16, 16, 16), bool)
            keep[z:z + 8, y:y + 8, x:x + 8] = True
            pal[k] = np.where(keep, pal[k], 0)
    return pal


def make_world(ctx, size, rng, fmt, pal, density):
    wx, wy, wz = size
    blocks = synth.make_world(size, rng, 32)
    loose = rng.random((wz, wy, wx)) < density
    blocks = np.where(loose, rng.integers(1, 32, (wz, wy, wx)), blocks).astype(np.int16)
    w = World(ctx, size, static_blocks=32, radiance_format=fmt)
    w.set_blocks(blocks)
    w.set_palette(pal)
    w.set_materials(synth.make_materials(rng))
    w.write_radiance(synth.make_field(size, rng))
    w.upload_blocks()
    return w


def assert_same(w, params, requests=None):
    """One update by the grid march, and the same one by the general march."""
    import torch
    start = w.read_radiance()
    w.radiance_update(requests, params)
    torch.cuda.synchronize()
    got = w.read_radiance()
    w.write_radiance(start)
    w.radiance_update(requests, params, traced=True)
    torch.cuda.synchronize()
    ref = w.read_radiance()
    if requests is None or requests.shape[0] >= params.size:  # a list shorter than the stride dispatches nothing
        assert not np.array_equal(start, ref)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("size,rays,fmt,max_dist,max_steps", [
    ((1, 1, 1), 64, RADIANCE_F32, 128.0, 0),       # the padded grid does not fit
    ((5, 5, 3), 128, RADIANCE_F32, 128.0, 0),
    ((33, 17, 9), 16, RADIANCE_F16, 128.0, 0),     # tiles with remainders
    ((32, 16, 8), 64, RADIANCE_BF16, 128.0, 40),
    ((31, 19, 12), 192, RADIANCE_F32, 128.0, 1),
    ((70, 9, 6), 256, RADIANCE_F16, 128.0, 64),
    ((20, 20, 20), 64, RADIANCE_F32, 37.25, 0),
    ((20, 20, 20), 64, RADIANCE_F32, 128.25, 0),   # beyond the grid's reach
    ((600, 4, 3), 32, RADIANCE_F32, 128.0, 0),     # no octants: an axis beyond 512 blocks
])
def test_grid_march_bit_exact(gpu_ctx, size, rays, fmt, max_dist, max_steps):
    import torch
    rng = np.random.default_rng([rays, *size])
    w = make_world(gpu_ctx, size, rng, fmt, sparse_palette(rng, 32), 0.05)
    try:
        params = radiance_params(rays=rays, time_seed=5, alpha=0.3, max_dist=max_dist, max_steps=max_steps)
        assert_same(w, params)
        n = size[0] * size[1] * size[2]
        flat = rng.permutation(n)[: max(2, n // 3)]
        req = np.stack([flat % size[0], flat // size[0] % size[1], flat // (size[0] * size[1]), 0 * flat], 1)
        req = torch.from_numpy(req.astype(np.int32)).cuda()
        assert_same(w, radiance_params(rays=rays, time_seed=6, alpha=0.3, max_dist=max_dist, max_steps=max_steps,
                                       size=2, shift=1), req)
    finally:
        w.close()


def test_grid_follows_blocks_palette_maps_and_residency(gpu_ctx):
    rng = np.random.default_rng(3)
    size = (24, 20, 12)
    w = make_world(gpu_ctx, size, rng, RADIANCE_F32, sparse_palette(rng, 32), 0.02)
    voxels, quats, shifts = synth.make_models(rng, n=5, lo=9, hi=40, fill=0.05, world_size=size)
    models = [Model(gpu_ctx, v) for v in voxels]
    places = [placement(q, s, m.size) for q, s, m in zip(quats, shifts, models)]
    params = radiance_params(rays=64, time_seed=8, alpha=0.3)
    batch = Batch(gpu_ctx, [w])
    try:
        w.map_models_device(models, places)
        assert_same(w, params)
        w.evict()
        w.restore()
        assert_same(w, params)
        w.set_palette(sparse_palette(rng, 32))     # other octants under the same blocks
        assert_same(w, params)
        w.map_models_placed(models[:3], places[:3])
        assert_same(w, params)
        batch.map_models([models], [places])
        assert_same(w, params)
        w.map_models_device([], [])
        assert_same(w, params)
        w.set_blocks(synth.make_world(size, rng, 32))
        w.upload_blocks()
        assert_same(w, params)
        solid0 = sparse_palette(rng, 32)
        solid0[0, 3, 4, 5] = 7                     # slot 0 is not air
        w.set_palette(solid0)
        assert_same(w, params)
    finally:
        batch.close()
        for m in models:
            m.close()
        w.close()


@pytest.mark.parametrize("size,fmt,width,height,max_dist,max_steps", [
    ((24, 20, 12), RADIANCE_F32, 97, 61, 128.0, 0),
    ((24, 20, 12), RADIANCE_F16, 33, 17, 1024.0, 64),
    ((24, 20, 12), RADIANCE_F16, 33, 17, 1025.0, 64),  # the general march
    ((5, 5, 3), RADIANCE_BF16, 16, 16, 0.25, 1),
    ((1, 1, 1), RADIANCE_F32, 1, 1, 128.0, 0),
])
def test_glossy_grid_march_bit_exact(gpu_ctx, size, fmt, width, height, max_dist, max_steps):
    """Origins in, around and far outside the world; NaN and infinite depths;
    unnormalized view directions on both sides of the grid's limit."""
    import torch
    rng = np.random.default_rng([width, *size])
    w = make_world(gpu_ctx, size, rng, fmt, sparse_palette(rng, 32), 0.1)
    try:
        matnorm = rng.integers(0, 256, (height, width, 4)).astype(np.uint8)
        depth = rng.uniform(-0.1, 0.4, (height, width)).astype(np.float32)
        odd = rng.random((height, width))
        depth[odd < 0.02] = np.nan
        depth[(odd >= 0.02) & (odd < 0.04)] = np.inf
        depth[(odd >= 0.04) & (odd < 0.06)] = -1e30
        mn, dp = torch.from_numpy(matnorm).cuda(), torch.from_numpy(depth).cuda()
        for scale in (1.0, 7.0, 40.0):
            cam = camera_default(width, height)
            for k in range(3):
                cam.campos[k] = 8.0 * size[k]
                cam.camdir[k] *= scale
            for frame in ((float(width), float(height)), (0.5, 3e5)):
                cam.frame_size[0], cam.frame_size[1] = frame
                got = w.glossy(mn, dp, cam, max_dist, max_steps)
                ref, _ = w.glossy(mn, dp, cam, max_dist, max_steps, traced=True)
                torch.cuda.synchronize()
                assert np.array_equal(got.cpu().numpy().view(np.uint32), ref.cpu().numpy().view(np.uint32))
    finally:
        w.close()
