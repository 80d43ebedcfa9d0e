"""Device blockify on both sides of the number of tiles from which the tile
offsets get a launch of their own (2048 tiles of 2048 elements), against the
host path."""
import numpy as np
import pytest

from lum_amd import synth
from lum_amd.api import Model, World, placement
from lum_amd._lib import RADIANCE_F16

pytestmark = pytest.mark.gpu

SIZE = (128, 128, 64)
STATIC = 8


@pytest.mark.parametrize("extra", [0, 1, 2048])  # elements above 4 * 2^20: 2048, 2049 and 2049 tiles
def test_blockify_tiles(gpu_ctx, extra):
    rng = np.random.default_rng(extra)
    shape = SIZE[::-1]
    # A block in a hundred can be allocated; the others name a dynamic slot.
    blocks = np.where(rng.random(shape) < 0.01, rng.integers(0, STATIC, shape), 9).astype(np.int16)
    m = Model(gpu_ctx, np.ones((4, 4, 4), np.uint8))
    worlds = [World(gpu_ctx, SIZE, STATIC, radiance_format=RADIANCE_F16) for _ in range(2)]
    places = []
    for k in range(4 + (extra > 0)):
        p = placement([1.0, 0.0, 0.0, 0.0], [100.0, 100.0, 100.0], m.size)
        box = SIZE if k < 4 else (1, 1, 1) if extra == 1 else (32, 16, 4)
        for a in range(3):
            p.groups[a] = 0  # its box alone
            p.aabb_min[a] = 1.0
            p.aabb_max[a] = 16.0 * box[a] - 2.0
        places.insert(0, p)  # the small box first: its claims win
    try:
        for w in worlds:
            w.set_blocks(blocks)
            w.set_palette(synth.make_palette(rng, STATIC) if w is worlds[0] else worlds[0].get_palette(0, STATIC))
        for _ in range(2):  # the second map finds the first one's counters
            worlds[0].map_models_device([m] * len(places), places)
            worlds[1].map_models_placed([m] * len(places), places)
            n = worlds[1].palette_counter()
            assert worlds[0].palette_counter() == n and n == STATIC + (blocks < STATIC).sum()
            assert np.array_equal(worlds[0].get_blocks(), worlds[1].get_blocks())
            assert np.array_equal(worlds[0].get_palette(0, n), worlds[1].get_palette(0, n))
    finally:
        m.close()
        for w in worlds:
            w.close()
