"""A map that is refused leaves the world as it was: the march grid too, whose
place the device map's claims take while it runs."""
import numpy as np
import pytest

from lum_amd import synth
from lum_amd.api import Batch, Model, World, placement, radiance_params
from lum_amd._lib import LumxError, RADIANCE_F16

pytestmark = pytest.mark.gpu

SIZE = (24, 20, 12)


def oversized(model, count):
    """Dispatch boxes of 2.56e8 workgroup tiles, side by side; a single one of
    6.9e10."""
    out = []
    for i in range(count):
        p = placement([1.0, 0.0, 0.0, 0.0], [110.0, 110.0, 100.0], model.size)
        for a in range(3):
            p.groups[a] = 1600 if count > 1 else 16384
        p.shift[0] += 6400 * i
        out.append(p)
    return out


@pytest.mark.parametrize("how", ["map_models_placed", "map_models_device", "map_models_device_noalloc", "batch"])
@pytest.mark.parametrize("count", [1, 9])  # one dispatch, and the launch of all, too large
def test_refused_map_changes_nothing(gpu_ctx, how, count):
    import torch
    rng = np.random.default_rng(count)
    w = World(gpu_ctx, SIZE, static_blocks=32, radiance_format=RADIANCE_F16)
    m = Model(gpu_ctx, rng.integers(0, 2, (20, 20, 20)).astype(np.uint8))
    good = placement([1.0, 0.0, 0.0, 0.0], [70.0, 70.0, 60.0], m.size)
    batch = Batch(gpu_ctx, [w])
    params = radiance_params(rays=64, time_seed=3, alpha=0.3)

    def update(traced=False):
        w.write_radiance(start)
        w.radiance_update(None, params, traced=traced)
        torch.cuda.synchronize()
        return w.read_radiance()

    try:
        w.set_blocks(synth.make_world(SIZE, rng, 32))
        w.set_palette(synth.make_palette(rng, 32))
        w.set_materials(synth.make_materials(rng))
        w.write_radiance(synth.make_field(SIZE, rng))
        w.map_models_device([m], [good])
        start = w.read_radiance()
        before = update()
        blocks, counter = w.get_blocks(), w.palette_counter()
        bad = oversized(m, count)
        with pytest.raises(LumxError):
            if how == "batch":
                batch.map_models([[m] * count], [bad])
            else:
                getattr(w, how)([m] * count, bad)
        assert np.array_equal(update(), before)
        assert np.array_equal(update(traced=True), before)
        assert np.array_equal(w.get_blocks(), blocks) and w.palette_counter() == counter
        w.map_models_placed([m], [good])
        assert np.array_equal(update(), before)
    finally:
        batch.close()
        m.close()
        w.close()
