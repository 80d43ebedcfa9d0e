"""The grid march of the default radiance and glossy passes (lum_amd/csrc/
march_grid.hpp), compiled for the host, against the general march ray by ray:
sparse octants, rays that start in the padding around the world, axis-parallel
and long directions, caps on the distance and on the samples."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def mg(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("march_grid_host") / "libmarch_grid_host.so")
    subprocess.run([hipcc, "-x", "hip", "--cuda-host-only", "-O2", "-std=c++17", "-fPIC", "-shared",
                    "-ffp-contract=off", os.path.join(HERE, "march_grid_host.cpp"), "-o", out],
                   check=True, capture_output=True)
    return C.CDLL(out)


def _p(a):
    return a.ctypes.data_as(C.c_void_p)


def make_world(rng, size, slots):
    wx, wy, wz = size
    pal = np.zeros((slots, 16, 16, 16), np.uint8)
    for k in range(1, slots):
        fill = (0.001, 0.02, 0.3, 1.0, 0.0)[k % 5]
        pal[k] = np.where(rng.random((16, 16, 16)) < fill, rng.integers(1, 256, (16, 16, 16)), 0)
        if k % 3 == 0:  # one octant only
            z, y, x = rng.integers(0, 2, 3) * 8
            keep = np.zeros((16, 16, 16), bool)
            keep[z:z + 8, y:y + 8, x:x + 8] = True
            pal[k] = np.where(keep, pal[k], 0)
    blocks = np.where(rng.random((wz, wy, wx)) < 0.15, rng.integers(1, slots, (wz, wy, wx)), 0).astype(np.int16)
    octants = (pal.reshape(slots, 2, 8, 2, 8, 2, 8) != 0).any((2, 4, 6)).reshape(slots, 8)  # [z][y][x]
    mask = np.maximum((octants << np.arange(8)).sum(1), 1).astype(np.uint8)
    grid = np.full((wz + 2, wy + 2, wx + 2), 0xff, np.uint8)
    grid[1:-1, 1:-1, 1:-1] = np.where(blocks == 0, 0, mask[blocks])
    return pal, blocks, grid


def make_rays(rng, size, n):
    """Rays whose first sample lies in the world or in the block around it, no
    axis of a direction longer than 16."""
    ext = 16.0 * np.array(size)
    first = rng.uniform(-16.0, ext + 16.0, (n, 3))
    first[: n // 2] = rng.uniform(0.0, ext, (n // 2, 3))
    first[-n // 8:] = rng.uniform(-16.0, 0.0, (n - (n - n // 8), 3))  # the corner below 0
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    kind = rng.integers(0, 5, n)
    d = np.where((kind == 1)[:, None], d * rng.uniform(0.05, 16.0, (n, 1)), d)
    d = np.where((kind == 2)[:, None], rng.choice([-16.0, 16.0], (n, 3)), d)
    axis = rng.integers(0, 3, n)
    d[np.arange(n)[kind == 3], axis[kind == 3]] *= 1e-4
    d[np.arange(n)[kind == 4], axis[kind == 4]] = 0.0
    d = d.astype(np.float32)
    o = (first - 0.5 * d).astype(np.float32)
    p = o + d * np.float32(0.5)
    ok = ((p > -16.0) & (p < ext + 16.0)).all(1)
    return np.ascontiguousarray(o[ok]), np.ascontiguousarray(d[ok])


@pytest.mark.parametrize("size,max_dist,max_steps", [
    ((5, 4, 3), 128.0, 0), ((24, 20, 12), 128.0, 0), ((24, 20, 12), 1024.0, 0), ((40, 3, 7), 37.25, 0),
    ((16, 16, 8), 128.0, 1), ((16, 16, 8), 128.0, 2), ((16, 16, 8), 128.0, 7), ((16, 16, 8), 1024.0, 64),
])
def test_grid_march_equals_general_march(mg, size, max_dist, max_steps):
    rng = np.random.default_rng([*size, int(max_dist), max_steps])
    slots = 48
    pal, blocks, grid = make_world(rng, size, slots)
    o, d = make_rays(rng, size, 40000)
    n = len(o)
    hit, voxel = np.zeros((n, 2), np.int32), np.zeros((n, 2), np.int32)
    fn = np.zeros((n, 2, 4), np.float32)
    mg.mg_cast(_p(blocks), _p(pal), *size, slots, _p(grid), n, _p(o), _p(d), C.c_float(max_dist), max_steps, _p(hit),
               _p(voxel), _p(fn))
    assert np.array_equal(hit[:, 0], hit[:, 1]) and np.array_equal(voxel[:, 0], voxel[:, 1])
    # (Without a refinement step the fraction is a zero of either sign: origin + fraction * d is the origin.)
    assert np.array_equal(fn[:, 0], fn[:, 1], equal_nan=True)
    if max_steps == 0:
        assert 0.05 * n < hit[:, 0].sum() < n


def test_any_grid_leads_no_read_out_of_it(mg):
    """Bytes of a grid that is being rewritten: whatever they say, the march
    reads inside the grid, the blocks and the palette, and ends."""
    rng = np.random.default_rng(5)
    size, slots = (9, 7, 5), 48
    pal, blocks, grid = make_world(rng, size, slots)
    o, d = make_rays(rng, size, 40000)
    n = len(o)
    hit, voxel = np.zeros((n, 2), np.int32), np.zeros((n, 2), np.int32)
    fn = np.zeros((n, 2, 4), np.float32)
    for zeros in (0.0, 0.5, 1.0):
        junk = np.where(rng.random(grid.shape) < zeros, 0, rng.integers(0, 256, grid.shape)).astype(np.uint8)
        mg.mg_cast(_p(blocks), _p(pal), *size, slots, _p(junk), n, _p(o), _p(d), C.c_float(128.0), 0, _p(hit),
                   _p(voxel), _p(fn))
