"""Updates of more than 2^31 rays: the ray index of a launch takes 32 bits."""
import numpy as np
import pytest

from lum_amd import synth
from lum_amd.api import World, radiance_params
from lum_amd._lib import LumxError, RADIANCE_F16

pytestmark = pytest.mark.gpu


def big_world(ctx, size):
    rng = np.random.default_rng(1)
    w = World(ctx, size, static_blocks=32, palette_slots=32, radiance_format=RADIANCE_F16)
    w.set_blocks(synth.make_world(size, rng, 32))
    w.set_palette(synth.make_palette(rng, 32))
    w.set_materials(synth.make_materials(rng))
    w.upload_blocks()
    return w


def test_more_than_2_pow_31_rays(gpu_ctx):
    """One ray per lane (2^31 + 2^26 threads) against four (2^29 + 2^24)."""
    import torch
    w = big_world(gpu_ctx, (256, 256, 33))
    try:
        start = np.ones((33, 256, 256, 4), np.float32)
        params = radiance_params(rays=1024, time_seed=2, alpha=0.5, max_steps=8)
        out = []
        for per_lane in (1, 4):
            w.write_radiance(start)
            w.set_tuning(variant=0, rays_per_lane=per_lane)
            w.radiance_update(None, params)
            torch.cuda.synchronize()
            out.append(w.read_radiance())
        # A probe that was left out would keep the other buffer's texel.  (A probe
        # with a NaN ray stores 0: nine of them here.)
        assert (out[0][..., :3] >= 0.5).all(-1).sum() > 0.999 * out[0].size / 4
        assert np.array_equal(out[0], out[1])
    finally:
        w.close()


def test_more_than_2_pow_32_rays_are_refused(gpu_ctx):
    w = big_world(gpu_ctx, (256, 256, 65))
    try:
        params = radiance_params(rays=1024)
        for tune in (dict(variant=0, rays_per_lane=1), dict(variant=2)):
            w.set_tuning(**tune)
            with pytest.raises(LumxError):
                w.radiance_update(None, params)
        # In two parts, 2^31 + 2^25 rays each: accepted.
        w.set_tuning(variant=0, rays_per_lane=1)
        for shift in range(2):
            w.radiance_update(None, radiance_params(rays=1024, size=2, shift=shift, max_steps=8))
    finally:
        w.close()
