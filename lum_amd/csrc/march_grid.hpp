// march_grid.hpp - the march over a world's grid of bytes (GridArgs in
// lumx_internal.hpp), shared by the probe and the glossy kernels, and what
// their batched launches share.
#pragma once

#include "march.hpp"
#include "lumx_internal.hpp"

namespace lumx {

// The refinement of refine_hit after a coarse hit in the block of grid key
// `key` (its id `id`), for a ray in div_range and a start no lower than -8.
// Voxels of one block in a row cost one load each: the block id is fetched
// only when the block changes.
template <class Args>
LUMX_HD RayHit refine_grid(const Args& a, const MarchRay& m, f3 bh, int key, int id) {
    const WorldView& w = a.world;
    const int kx = w.wx + 2, kxy = kx * (w.wy + 2);
    const f3 d = m.d, inv = m.inv;
    // Voxel coordinates as floats (exact integers): truncation towards zero.
    f3 v = {truncf(bh.x), truncf(bh.y), truncf(bh.z)};
    auto fetch = [&]() {
        const int ix = (int)v.x, iy = (int)v.y, iz = (int)v.z;
        // Block 0 also holds -15 .. -1 (the shader's truncating division).
        const int bx = block_axis(ix), by = block_axis(iy), bz = block_axis(iz);
        const int k = bx + (int)(mul24((unsigned)by, (unsigned)kx) + mul24((unsigned)bz, (unsigned)kxy));
        if (k != key) {
            key = k;
            id = 0;
            if (bx < w.wx && by < w.wy && bz < w.wz) id = block_id(w, bx, by, bz);
            if (id >= w.palette_slots) id = 0;
        }
        int cv = 0;
        if (id != 0) cv = gld(w.palette, ((uint32_t)id << 12) | voxel_offset(ix, iy, iz));
        return cv;
    };
    RayHit r;
    r.hit = 1;
    int cv = fetch();
    f3 st = {0.0f, 0.0f, 0.0f}, tf = st;
    const f3 s = {__builtin_copysignf(1.0f, d.x), __builtin_copysignf(1.0f, d.y), __builtin_copysignf(1.0f, d.z)};
    if (cv == 0) {
        const f3 fl = {floorf(bh.x), floorf(bh.y), floorf(bh.z)};
        const f3 q = fl - bh;
        f3 c1 = {div_rn(q.x, d.x, inv.x), div_rn(q.y, d.y, inv.y), div_rn(q.z, d.z, inv.z)};
        if (!div_range(bh)) c1 = {q.x / d.x, q.y / d.y, q.z / d.z};
        const f3 c2 = c1 + inv;
        f3 t = {fmaxf(c1.x, c2.x), fmaxf(c1.y, c2.y), fmaxf(c1.z, c2.z)};
        const f3 dt = {fabsf(inv.x), fabsf(inv.y), fabsf(inv.z)};
        int left = 5;
        do {
            // Every axis at the minimum steps (ties step together).
            const float tm = fminf(t.x, fminf(t.y, t.z));
            st = {t.x == tm ? 1.0f : 0.0f, t.y == tm ? 1.0f : 0.0f, t.z == tm ? 1.0f : 0.0f};
            // Products with 0 or 1 are exact: one rounding, as t + dt * st.
            v = {fmaf(s.x, st.x, v.x), fmaf(s.y, st.y, v.y), fmaf(s.z, st.z, v.z)};
            t = {fmaf(dt.x, st.x, t.x), fmaf(dt.y, st.y, t.y), fmaf(dt.z, st.z, t.z)};
            cv = fetch();
        } while (--left > 0 && cv == 0);
        tf = t - dt;
    }
    r.normal = -(s * st);
    r.fraction = dot3(tf, st);
    r.voxel = cv;
    return r;
}

// A float index into the grid, within it whatever its value (v_med3_f32).
LUMX_HD unsigned clamp_index(float index, float last) {
#if defined(__HIP_DEVICE_COMPILE__)
    return (unsigned)__builtin_amdgcn_fmed3f(index, 0.0f, last);
#else
    return (unsigned)fminf(fmaxf(index, 0.0f), last);
#endif
}

// cast_ray over the world's march grid (a.grid, which takes slot 0 as air).
// The ray's first sample lies in the world or in the block around it, and no
// axis of d is longer than 16: then no sample lies further out, the next one
// after a sample in the world being half a voxel's step past its block.
//
// The fractions of a ray's samples do not depend on what it reads as long as
// it stays in plain air, so two samples are taken at a time: the second's grid
// byte is on its way before the first's arrives, and counts only if the first
// was air.  (A second sample after a first outside the world may lie further
// out: indices are clamped at both ends, so that not even a grid that is being
// rewritten by an unordered map leads a read out of it.)  Grid indices are
// formed in floats, exact below 2^24: six 2-cycle operations and a conversion
// instead of three conversions and two 4-cycle multiply-adds.
//
// In a block that holds something, samples lie half a voxel apart.  The grid
// byte tells its empty octants: n samples in one are passed by at once.
//   - Positions: an axis is monotone in the fraction, so samples between the
//     current one and one short of the octant's far face stay inside it.
//     Rounding moves a position by under 2^-9 (worlds up to 512 blocks an
//     axis), the face is taken 2^-8 early.
//   - The fraction: adding 1/2 is exact but where the result enters the next
//     binade, and it does so once (n + 1 samples at most double it); rounding
//     there commutes with adding multiples of 1/2.
// Elsewhere the next kAhead samples are loaded together.  A world with 32 models
// (48 x 48 x 16 blocks, 64 rays, map and glossy query included) took 320 us
// with 1, 288 with 2 and 303 with 4, which is past 64 registers (measured
// before the air loop counted its samples per wave and before the selection
// and blockify passes were cut; the same frame takes 236 us now, with 2).
template <class Args>
LUMX_HD RayHit cast_ray_grid(const Args& a, f3 o, f3 d) {
    const WorldView& w = a.world;
    const MarchRay m = march_ray(o, d);
    const int kx = w.wx + 2, kxy = kx * (w.wy + 2);
    float fx = (float)kx, fxy = (float)kxy, corner = (float)(1 + kx + kxy), last = (float)(kxy * (w.wz + 2) - 1);
    struct Sample {
        float fraction, next;  // here, and past the block if it is air
        float index;
    };
    auto sample = [&](float from) {
        Sample q;
        q.fraction = from + 0.5f;
        const f3 pos = m.o + m.d * q.fraction;
        const f3 ps = pos * 0.0625f;
        // The truncating block coordinate for p >= 0; the padding below 0.
        const f3 cell = {floorf(ps.x), floorf(ps.y), floorf(ps.z)};
        q.index = fmaf(cell.y, fx, fmaf(cell.z, fxy, corner)) + cell.x;
        const f3 box = {fmaf(cell.x, 16.0f, m.corner.x), fmaf(cell.y, 16.0f, m.corner.y),
                        fmaf(cell.z, 16.0f, m.corner.z)};
        const f3 tmp = (-pos) * m.inv;
        const f3 bc = box * m.inv + tmp;
        q.next = q.fraction + fmaxf(fminf(bc.x, fminf(bc.y, bc.z)), 0.01f);
        return q;
    };
    float fraction = 0.0f;
    constexpr int kAhead = 2;
    constexpr float kMargin = 0.00390625f;
    const f3 near = {d.x > 0.0f ? 8.0f - kMargin : kMargin, d.y > 0.0f ? 8.0f - kMargin : kMargin,
                     d.z > 0.0f ? 8.0f - kMargin : kMargin};
    int left = a.max_steps > 0 ? a.max_steps : 1 << 20;  // samples
    int state = 0, id = 0, key = 0;
    while (state == 0) {
        // Lanes that go on take two samples each turn, so `taken` is the wave's:
        // a count in every lane, with and without a cap, cost a fifth of the
        // turn's 87 vector instructions (72 now).
        unsigned b0, b1;
        bool second, on;
        Sample s0, s1;
        int taken = 0;
        do {
            s0 = sample(fraction);
            b0 = gld(a.grid, clamp_index(s0.index, last));
            s1 = sample(s0.next);
            b1 = gld(a.grid, clamp_index(s1.index, last));
            second = b0 == 0 && s0.next < a.max_dist && left > taken + 1;
            on = second && b1 == 0 && s1.next < a.max_dist && left > taken + 2;
            fraction = s1.next;
            taken += 2;
        } while (on);
        left -= second ? taken : taken - 1;
        fraction = second ? s1.fraction : s0.fraction;
        const unsigned mask = second ? b1 : b0;
        if (mask == 0) {
            state = -1;  // air to the end of the ray or of its samples
        } else {
            // A block that is not empty, or a sample outside the world, in
            // coarse_sample's order of tests; then the samples half a voxel
            // apart that stay in that block.
            f3 pos = m.o + m.d * fraction;
            int ix = (int)pos.x, iy = (int)pos.y, iz = (int)pos.z;
            const int bx = block_axis(ix), by = block_axis(iy), bz = block_axis(iz);
            id = 0;
            if (block_axis_in(ix, w.wx) && block_axis_in(iy, w.wy) && block_axis_in(iz, w.wz))
                id = block_id(w, bx, by, bz);
            if (mask == 0xffu && id == 0) state = -1;  // outside, or air below 0
            const uint32_t slot = (uint32_t)id << 12;
            const bool voxels = (unsigned)(id - 1) < (unsigned)(w.palette_slots - 1);
            auto leaves = [&]() {
                return fminf(pos.x, fminf(pos.y, pos.z)) < 0.0f || fraction >= a.max_dist || left == 0;
            };
            key = bx + (int)(mul24((unsigned)by, (unsigned)kx) + mul24((unsigned)bz, (unsigned)kxy));
            if (voxels && gld(w.palette, slot | voxel_offset(ix, iy, iz)) != 0) state = 1;
            else if (leaves()) state = -1;
            bool same = true;
            while (state == 0 && same) {
                const unsigned oct = ((ix >> 3) & 1) | ((iy >> 2) & 2) | ((iz >> 1) & 4);
                if (!((mask >> oct) & 1)) {
                    // Straight on to the last sample in this empty octant.
                    const f3 end = {(float)(ix & ~7) + near.x, (float)(iy & ~7) + near.y, (float)(iz & ~7) + near.z};
                    const f3 t = (end - m.o) * m.inv;
                    const float stop = fminf(fminf(t.x, fminf(t.y, t.z)), fminf(a.max_dist, 2.0f * fraction) - 0.5f);
                    const float n = fminf(truncf((stop - fraction) * 2.0f), (float)(left - 1));
                    if (n > 0.0f) {
                        fraction = fmaf(n, 0.5f, fraction);
                        left -= (int)n;
                    }
                }
                // The next kAhead samples at once.
                float f[kAhead];
                f3 p[kAhead];
                int q[3][kAhead];
                uint8_t v[kAhead];
#pragma unroll
                for (int k = 0; k < kAhead; ++k) {
                    f[k] = (k ? f[k - 1] : fraction) + 0.5f;
                    p[k] = m.o + m.d * f[k];
                    q[0][k] = (int)p[k].x;
                    q[1][k] = (int)p[k].y;
                    q[2][k] = (int)p[k].z;
                    v[k] = 0;
                    if (voxels) v[k] = gld(w.palette, slot | voxel_offset(q[0][k], q[1][k], q[2][k]));
                }
#pragma unroll
                for (int k = 0; k < kAhead; ++k) {
                    same = same && (unsigned)((q[0][k] ^ ix) | (q[1][k] ^ iy) | (q[2][k] ^ iz)) < 16u;
                    if (state == 0 && same) {  // else the grid takes it from the last sample in the block
                        fraction = f[k];
                        pos = p[k];
                        --left;
                        if (v[k] != 0) state = 1;
                        else if (leaves()) state = -1;
                    }
                }
                ix = (int)pos.x;
                iy = (int)pos.y;
                iz = (int)pos.z;
            }
        }
    }
    RayHit h;
    h.hit = 0;
    if (state > 0) {
        const f3 bh = m.o + m.d * (fraction - 1.5f);
        if (div_range(m.d) && fminf(bh.x, fminf(bh.y, bh.z)) >= -8.0f) h = refine_grid(a, m, bh, key, id);
        else h = refine_hit(w, m, fraction);
    }
    return h;
}

// Batched launches: the last item that begins at or before workgroup or thread
// b (uniform), 64 items a step, one a lane.  (A scalar binary search is a
// chain of loads, 1% of a radiance launch.)
__device__ __forceinline__ int last_begin(const int* begin, int n, int b) {
    int lo = -1;
    for (int i0 = 0; i0 < n; i0 += 64) {
        const int i = i0 + (int)(threadIdx.x & 63);
        const int in = __popcll(__ballot(i < n && begin[i] <= b));
        lo += in;
        if (in < 64) break;
    }
    return lo;
}

// An item's arguments as constants (no thread writes them).
template <class Args>
__device__ __forceinline__ const Args* constant_args(const Args* p) {
    return (const Args*)(const __attribute__((address_space(4))) Args*)(uintptr_t)p;
}

}  // namespace lumx
