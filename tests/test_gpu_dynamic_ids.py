"""Origin worlds that name dynamic slots themselves: models are written into
those slots too, so every march and every residency change has to see them,
wherever they lie relative to the palette counter."""
import numpy as np
import pytest

from lum_amd import synth
from lum_amd.api import Batch, Model, World, camera_default, placement, radiance_params
from lum_amd._lib import RADIANCE_F32

pytestmark = pytest.mark.gpu

SIZE = (24, 20, 12)
STATIC, SLOTS = 32, 512
VARIANTS = [dict(variant=0), dict(variant=0, rays_per_lane=2), dict(variant=2),
            dict(variant=1, threads=256, probes_per_batch=4, lds_block_bits=1, lds_palette_bits=1),
            dict(variant=3, probes_per_batch=2)]


def dynamic_world(ctx, low, high):
    rng = np.random.default_rng([low, high])
    blocks = synth.make_world(SIZE, rng, STATIC)
    ids = rng.integers(low, high, (3, 10, 10))
    blocks[6:9, 6:16, 6:16] = np.where(rng.random(ids.shape) < 0.3, ids, 0)
    w = World(ctx, SIZE, STATIC, SLOTS, RADIANCE_F32)
    w.set_blocks(blocks)
    w.set_palette(synth.make_palette(rng, STATIC))
    w.set_materials(synth.make_materials(rng))
    w.write_radiance(synth.make_field(SIZE, rng))
    w.upload_blocks()
    voxels = np.where(rng.random((40, 100, 100)) < 0.2, rng.integers(1, 256, (40, 100, 100)), 0).astype(np.uint8)
    m = Model(ctx, voxels)
    return w, m, placement([1.0, 0.0, 0.0, 0.0], [110.0, 110.0, 100.0], m.size)


def update(w, start, traced=False, **tune):
    import torch
    w.write_radiance(start)
    w.set_tuning(**tune)
    w.radiance_update(None, radiance_params(rays=64, time_seed=5, alpha=0.3), traced=traced)
    torch.cuda.synchronize()
    w.set_tuning(variant=0, rays_per_lane=0)
    return w.read_radiance()


@pytest.mark.parametrize("how", ["placed", "batch", "device"])
@pytest.mark.parametrize("low,high", [(40, 50), (40, 400), (511, 512)])  # below, around and above the counter
def test_marches_see_dynamic_origin_slots(gpu_ctx, how, low, high):
    import torch
    w, m, place = dynamic_world(gpu_ctx, low, high)
    batch = Batch(gpu_ctx, [w])
    rng = np.random.default_rng(2)
    try:
        for round_ in range(2):
            if how == "placed":
                w.map_models_placed([m], [place])
            elif how == "batch":
                batch.map_models([[m]], [[place]])
            else:
                w.map_models_device([m], [place])
            start = w.read_radiance()
            ref = update(w, start, traced=True)
            for tune in VARIANTS:
                assert np.array_equal(update(w, start, **tune), ref), tune
            w.write_radiance(start)
            batch.radiance([radiance_params(rays=64, time_seed=5, alpha=0.3)])
            torch.cuda.synchronize()
            assert np.array_equal(w.read_radiance(), ref)
            mn = torch.from_numpy(rng.integers(0, 256, (61, 97, 4)).astype(np.uint8)).cuda()
            dp = torch.from_numpy(rng.uniform(-0.1, 0.4, (61, 97)).astype(np.float32)).cuda()
            cam = camera_default(97, 61)
            for k in range(3):
                cam.campos[k] = 8.0 * SIZE[k]
            got = w.glossy(mn, dp, cam)
            want, _ = w.glossy(mn, dp, cam, traced=True)
            torch.cuda.synchronize()
            assert torch.equal(got.view(torch.int32), want.view(torch.int32))
            # Eviction keeps those slots' voxels.
            palette = w.get_palette(0, SLOTS)
            assert palette[low:high].any()
            w.evict()
            w.restore()
            assert np.array_equal(w.get_palette(0, SLOTS), palette)
            for tune in VARIANTS:
                assert np.array_equal(update(w, start, **tune), ref), tune
            w.write_radiance(start)
    finally:
        batch.close()
        m.close()
        w.close()


def test_slots_of_an_earlier_origin_world(gpu_ctx):
    """A slot that no block names for a while keeps its voxels, as nothing
    clears it: also over an eviction, and for the block that names it again."""
    w, m, place = dynamic_world(gpu_ctx, 400, 410)
    blocks = w.get_blocks(False)
    try:
        w.map_models_placed([m], [place])
        w.set_blocks(np.where(blocks >= STATIC, 0, blocks))
        w.upload_blocks()
        palette = w.get_palette(0, SLOTS)
        assert palette[400:410].any()
        w.evict()
        w.restore()
        assert np.array_equal(w.get_palette(0, SLOTS), palette)
        w.set_blocks(blocks)
        w.upload_blocks()
        start = w.read_radiance()
        ref = update(w, start, traced=True)
        for tune in VARIANTS:
            assert np.array_equal(update(w, start, **tune), ref), tune
    finally:
        m.close()
        w.close()
