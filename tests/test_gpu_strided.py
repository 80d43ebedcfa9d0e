"""A strided update without a request list takes every size-th probe of the
x-fastest order, from the shift-th, on every launch shape."""
import numpy as np
import pytest

from lum_amd.api import Batch, radiance_params
import tests._oracle as orc
from tests.test_gpu_parity import full_palette, gpu_world, make_case

pytestmark = pytest.mark.gpu

SHAPES = {
    "lane": dict(variant=0, compact=-1),
    "compact": dict(variant=0, compact=1),
    "four_rays": dict(variant=0, compact=-1, rays_per_lane=4),
    "tiled": dict(variant=1, threads=256, probes_per_batch=4),
    "bits": dict(variant=2, compact=-1),
    "refill": dict(variant=3, probes_per_batch=2),
    "traced": None,
    "batch": None,
}


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("size,stride,shift,rays", [((16, 16, 32), 4, 2, 64), ((9, 7, 5), 3, 0, 64)])
def test_strided_update_without_a_list(gpu_ctx, shape, size, stride, shift, rays):
    blocks, pal, mats, field = make_case(size, 311)
    w = gpu_world(gpu_ctx, blocks, pal, mats, field)
    full = full_palette(w, pal)
    params = radiance_params(rays=rays, time_seed=31, size=stride, shift=shift, alpha=0.3)
    batch = Batch(gpu_ctx, [w])
    try:
        if SHAPES[shape]:
            w.set_tuning(**SHAPES[shape])
        if shape == "batch":
            batch.radiance([params])
        else:
            w.radiance_update(None, params, traced=shape == "traced")
        got = w.read_radiance()
    finally:
        batch.close()
        w.close()
    wd = orc.WorldData(blocks, full, mats)
    ref = orc.radiance_update(wd, field, rays=rays, time_seed=31, size=stride, shift=shift, alpha=0.3)
    assert np.array_equal(got, ref)
