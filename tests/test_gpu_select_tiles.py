"""Device probe selection on both sides of the number of tiles from which the
tile offsets get a launch of their own (2048 tiles of 2048 probes)."""
import numpy as np
import pytest

from lum_amd import synth
from lum_amd.api import World
from lum_amd._lib import RADIANCE_F16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(5, 4, 3), (64, 32, 1), (64, 33, 1), (256, 128, 128), (256, 128, 129)])
def test_select_tiles(gpu_ctx, size):
    import torch
    wx, wy, wz = size
    rng = np.random.default_rng(wx * wy * wz)
    blocks = np.where(rng.random((wz, wy, wx)) < 0.02, 1, 0).astype(np.int16)
    w = World(gpu_ctx, size, static_blocks=2, palette_slots=2, radiance_format=RADIANCE_F16)
    try:
        w.set_blocks(blocks)
        w.set_palette(synth.make_palette(rng, 2))
        w.upload_blocks()
        pad = np.pad(blocks != 0, 1, mode="edge")
        near = np.zeros_like(pad[1:-1, 1:-1, 1:-1])
        for dz in range(3):
            for dy in range(3):
                for dx in range(3):
                    near |= pad[dz:dz + wz, dy:dy + wy, dx:dx + wx]
        z, y, x = np.nonzero(near)
        want = np.stack([x, y, z, 0 * x], 1)
        special = np.stack([rng.integers(-1, s + 1, 40) for s in size] + [np.arange(40)], 1)
        keep = [(0 <= q[:3]).all() and (q[:3] < size).all() and not near[q[2], q[1], q[0]] for q in special]
        want = np.concatenate([want, special[keep]])[: wx * wy * wz].astype(np.int32)
        got, count = w.select_probes_device(torch.from_numpy(special.astype(np.int32)).cuda())
        torch.cuda.synchronize()
        n = int(count.cpu()[0])
        assert n == len(want)
        assert np.array_equal(got[:n].cpu().numpy(), want)
    finally:
        w.close()
