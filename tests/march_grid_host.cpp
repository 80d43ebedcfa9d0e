// march_grid_host.cpp - the march over a world's grid of bytes compiled for
// the host (tests/test_march_grid_cpu.py), against cast_ray on the same rays.
#include "../lum_amd/csrc/march_grid.hpp"

using namespace lumx;

namespace {
struct HostArgs {
    WorldView world;
    const uint8_t* grid;
    float max_dist;
    int max_steps;
};
}  // namespace

extern "C" {

// hit[2 i + k], voxel[2 i + k], fn[8 i + 4 k ..] = {fraction, normal} of ray i
// by cast_ray (k = 0) and cast_ray_grid (k = 1).
void mg_cast(const int16_t* blocks, const uint8_t* palette, int wx, int wy, int wz, int slots, const uint8_t* grid,
             int n, const float* o, const float* d, float max_dist, int max_steps, int* hit, int* voxel, float* fn) {
    HostArgs a{};
    a.world.blocks = blocks;
    a.world.palette = palette;
    a.world.wx = wx;
    a.world.wy = wy;
    a.world.wz = wz;
    a.world.palette_slots = slots;
    a.world.block0_empty = 1;
    a.grid = grid;
    a.max_dist = max_dist;
    a.max_steps = max_steps;
    for (int i = 0; i < n; ++i) {
        const f3 oo = {o[3 * i], o[3 * i + 1], o[3 * i + 2]}, dd = {d[3 * i], d[3 * i + 1], d[3 * i + 2]};
        for (int k = 0; k < 2; ++k) {
            const RayHit h = k ? cast_ray_grid(a, oo, dd) : cast_ray(a.world, oo, dd, max_dist, max_steps);
            hit[2 * i + k] = h.hit;
            if (!h.hit) continue;
            voxel[2 * i + k] = h.voxel;
            float* f = fn + 8 * i + 4 * k;
            f[0] = h.fraction;
            f[1] = h.normal.x;
            f[2] = h.normal.y;
            f[3] = h.normal.z;
        }
    }
}

}  // extern "C"
