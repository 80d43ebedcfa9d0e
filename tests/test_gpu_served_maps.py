"""Worlds whose last map ran on the device, served under an HBM budget: the
palette they are evicted and restored with is that map's."""
import numpy as np
import pytest

from lum_amd import synth
from lum_amd.api import Model, Server, World, placement, radiance_params, radiance_request
from lum_amd._lib import RADIANCE_F16

pytestmark = pytest.mark.gpu

SIZE = (16, 16, 8)


def mapped_worlds(ctx, n, how):
    out = []
    for i in range(n):
        rng = np.random.default_rng(i)
        w = World(ctx, SIZE, static_blocks=32, palette_slots=512, radiance_format=RADIANCE_F16)
        w.set_blocks(synth.make_world(SIZE, rng, 32))
        w.set_palette(synth.make_palette(rng, 32))
        w.set_materials(synth.make_materials(rng))
        w.write_radiance(synth.make_field(SIZE, rng))
        m = Model(ctx, np.where(rng.random((30, 40, 50)) < 0.2, rng.integers(1, 256, (30, 40, 50)), 0).astype(np.uint8))
        # Two models over each other: the boxes hold more blocks than the map allocates.
        getattr(w, how)([m, m], [placement([1.0, 0.0, 0.0, 0.0], [90.0 + 9.0 * k, 90.0, 50.0], m.size)
                                 for k in range(2)])
        out.append((w, m))
    return out


@pytest.mark.parametrize("how", ["map_models_device", "map_models_placed"])
def test_mapped_worlds_served_under_a_budget(gpu_ctx, how):
    import torch
    n, frames = 4, 3
    alone = mapped_worlds(gpu_ctx, n, how)
    served = mapped_worlds(gpu_ctx, n, how)
    params = [[radiance_params(rays=64, time_seed=10 * f + i, alpha=0.3) for i in range(n)] for f in range(frames)]
    server = Server(gpu_ctx, [w for w, _ in served], hbm_budget=2 * served[0][0].resident()[1] + 4096, max_batch=2)
    try:
        for f in range(frames):
            tickets = [server.submit(radiance_request(i, params[f][i])) for i in range(n)]
            for t in tickets:
                server.wait(t)
            for i in range(n):
                alone[i][0].radiance_update(None, params[f][i])
        torch.cuda.synchronize()
    finally:
        server.close()
    try:
        for (a, _), (b, _) in zip(alone, served):
            if not b.resident()[0]:
                b.restore()
            assert np.array_equal(a.read_radiance(), b.read_radiance())
            assert np.array_equal(a.get_palette(0, 512), b.get_palette(0, 512))
            assert a.palette_counter() == b.palette_counter()
    finally:
        for w, m in alone + served:
            m.close()
            w.close()
