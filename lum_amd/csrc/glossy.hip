// glossy.hip - per-pixel glossy reflection march (gfx950).
//
// Restates shaders/glossy.frag:444-493 (main) with get_origin_from_depth
// (:43-49), ProcessHit (:312-326), trace_glossy_ray (:328-360), load_norm /
// load_mat / load_depth (:367-382) and the stencil mask of
// shaders/fillStencilGlossy.frag:29-35 (roughness > 0.5 -> pixel untouched).
// The output is the fragment's pre-blend value vec4(L / 8, 1 - roughness).
// Launch: 16 x 16 pixel tiles, one thread per pixel.
//
// Bound by the gather path (its unit is busy 73% of the time) and by vector
// issue together: every pixel reads eight texels of its own at the surface and
// eight at the hit.  So the march reads the world's byte grid, the material
// table sits in LDS, and the surface's light is computed after the march,
// which then fits 64 registers and eight waves a SIMD.  1920 x 1080 pixels
// with a normal and depth each: 72.6 -> 65.8 us; 638 x 359 in flat patches:
// 14.6 -> 13.3 us; 24 frames of 640 x 360 in a batch 205 -> 182 us.
#include "lumx_internal.hpp"
#include "march_grid.hpp"

namespace lumx {

__device__ __forceinline__ f3 unpack_normal(uchar4 mn) {
    const float r255 = 1.0f / 255.0f;
    return {div_rn((float)mn.y, 255.0f, r255) * 2.0f - 1.0f, div_rn((float)mn.z, 255.0f, r255) * 2.0f - 1.0f,
            div_rn((float)mn.w, 255.0f, r255) * 2.0f - 1.0f};
}

// The material table in LDS: 256 rows of a pixel's own choice are the widest
// gathers of the pass, and the gather path is what bounds it.
__device__ __forceinline__ void load_materials(const WorldView& w, float* mats) {
    for (int i = threadIdx.x; i < 256 * 6 / 4; i += 256) ((float4*)mats)[i] = gld((const float4*)w.mats, i);
    __syncthreads();
}
__device__ __forceinline__ MatF lds_mat(const float* mats, int i) {
    const float* r = mats + i * 6;
    return {f3{r[0], r[1], r[2]}, r[4], r[5]};
}

template <int STORE, bool TRACED>
__device__ __forceinline__ void glossy_pixel(const GlossyArgs& a, const float* mats, const int px, const int py) {
    unsigned pi = (unsigned)py * (unsigned)a.width + (unsigned)px;
    const WorldView& w = a.world;
    if (TRACED) a.keys[pi] = 0;
    uchar4 mn = a.matnorm[pi];
    if (lds_mat(mats, mn.x).rough > 0.5f) return;

    const float fx = (float)px + 0.5f, fy = (float)py + 0.5f;
    const float cx = (a.inv_w != 0.0f ? div_rn(fx, a.frame_w, a.inv_w) : fx / a.frame_w) * 2.0f - 1.0f;
    const float cy = (a.inv_h != 0.0f ? div_rn(fy, a.frame_h, a.inv_h) : fy / a.frame_h) * 2.0f - 1.0f;
    const float dep = a.depth[pi] * 1000.0f;
    const f3 campos = {a.campos[0], a.campos[1], a.campos[2]};
    const f3 camdir = {a.camdir[0], a.camdir[1], a.camdir[2]};
    const f3 horiz = {a.horiz[0], a.horiz[1], a.horiz[2]};
    const f3 verti = {a.verti[0], a.verti[1], a.verti[2]};
    f3 origin = campos + horiz * cx + verti * cy + camdir * dep;
    f3 dir = camdir;
    // ProcessHit at the surface with fraction 0: the reflection first.
    origin = origin + 0.0f * dir;
    const f3 normal = unpack_normal(mn);
    const float dn = dot3(normal, dir);
    dir = dir - (2.0f * dn) * normal;

    RayHit h;
    h.hit = 0;
    bool general = true;
    if (!TRACED && a.grid) {
        // A ray whose first sample lies outside the padded world ends there;
        // NaN and directions too long for the grid take the general march.
        const f3 p = origin + dir * 0.5f;
        const bool inside = fminf(p.x, fminf(p.y, p.z)) > -16.0f && p.x < (float)(16 * w.wx + 16) &&
                            p.y < (float)(16 * w.wy + 16) && p.z < (float)(16 * w.wz + 16);
        general = !(fabsf(p.x) + fabsf(p.y) + fabsf(p.z) < kHuge &&
                    fmaxf(fabsf(dir.x), fmaxf(fabsf(dir.y), fabsf(dir.z))) <= 16.0f);
        if (inside && !general) h = cast_ray_grid(a, origin, dir);
    }
    if (general) h = cast_ray(w, origin, dir, a.max_dist, a.max_steps);

    // The surface's own light.  Its inputs are read again: kept over the
    // march, they cost it a fifth of its registers.
    asm volatile("" : "+v"(pi));
    mn = a.matnorm[pi];
    const MatF mat = lds_mat(mats, mn.x);
    f3 L = {0.0f, 0.0f, 0.0f}, R = {1.0f, 1.0f, 1.0f};
    const f3 diff = sample_radiance<STORE>(a.field, w.wx, w.wy, w.wz, origin, unpack_normal(mn));
    R = R * mat.color;
    L = L + R * (f3{mat.emit, mat.emit, mat.emit} + diff);
    if (h.hit) {
        const MatF hm = lds_mat(mats, h.voxel);
        f3 o2 = origin + h.fraction * dir;
        f3 d2 = sample_radiance<STORE>(a.field, w.wx, w.wy, w.wz, o2, h.normal);
        R = R * hm.color;
        L = L + R * (f3{hm.emit, hm.emit, hm.emit} + d2);
        if (TRACED) a.keys[pi] = h.key;
    } else {
        const f3 gl = {a.light[0], a.light[1], a.light[2]};
        float s = -dot3(dir, gl);
        if (s > 0.9f) {
            f3 sun = f3{0.9f, 0.9f, 0.6f} * 0.5f;
            L = L + ((sun * R) * (s - 0.9f)) * 10.0f;
        }
        f3 sky = f3{0.53f, 0.81f, 0.92f} * 0.1f;
        L = L + sky * R;
    }
    a.out[pi] = make_float4(L.x / 8.0f, L.y / 8.0f, L.z / 8.0f, 1.0f - mat.rough);
}

template <int STORE, bool TRACED>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_num_sgpr(80), amdgpu_waves_per_eu(8))) glossy_kernel(GlossyArgs a) {
    __shared__ __attribute__((aligned(16))) float mats[256 * 6];
    load_materials(a.world, mats);
    const int px = blockIdx.x * 16 + (threadIdx.x & 15);
    const int py = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (px >= a.width || py >= a.height) return;
    glossy_pixel<STORE, TRACED>(a, mats, px, py);
}

// Many frames in one launch: frame w owns workgroups [begin[w], begin[w + 1]),
// one 16 x 16 pixel tile each, tiles row-major (the single-frame kernel's
// tiling, so a wave's reflection rays start from a 16 x 4 patch).
template <int STORE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_num_sgpr(80), amdgpu_waves_per_eu(8))) glossy_batch_kernel(const GlossyArgs* args, const int* begin, int n) {
    const int b = (int)blockIdx.x;
    const int lo = last_begin(begin, n, b);
    const GlossyArgs& a = *constant_args(args + lo);
    __shared__ __attribute__((aligned(16))) float mats[256 * 6];
    load_materials(a.world, mats);
    const int t = b - begin[lo];
    const int tiles_x = (a.width + 15) >> 4;
    const int ty = t / tiles_x;
    const int px = (t - ty * tiles_x) * 16 + (int)(threadIdx.x & 15);
    const int py = ty * 16 + (int)(threadIdx.x >> 4);
    if (px >= a.width || py >= a.height) return;
    glossy_pixel<STORE, false>(a, mats, px, py);
}

hipError_t launch_glossy_batch(const GlossyArgs* args_dev, const int* begin_dev, int n, int total_tiles, int store,
                               hipStream_t stream) {
    if (n <= 0 || total_tiles <= 0) return hipSuccess;
    const int grid = total_tiles;
    switch (store) {
        case STORE_F16:
            hipLaunchKernelGGL(glossy_batch_kernel<STORE_F16>, dim3(grid), dim3(256), 0, stream, args_dev, begin_dev, n);
            break;
        case STORE_BF16:
            hipLaunchKernelGGL(glossy_batch_kernel<STORE_BF16>, dim3(grid), dim3(256), 0, stream, args_dev, begin_dev, n);
            break;
        default:
            hipLaunchKernelGGL(glossy_batch_kernel<STORE_F32>, dim3(grid), dim3(256), 0, stream, args_dev, begin_dev, n);
            break;
    }
    return hipGetLastError();
}

template <int STORE, bool TRACED>
static hipError_t launch_g(const GlossyArgs& a, hipStream_t stream) {
    dim3 grid((a.width + 15) / 16, (a.height + 15) / 16);
    if (grid.x == 0 || grid.y == 0) return hipSuccess;
    hipLaunchKernelGGL((glossy_kernel<STORE, TRACED>), grid, dim3(256), 0, stream, a);
    return hipGetLastError();
}

hipError_t launch_glossy(const GlossyArgs& a, int store, bool traced, hipStream_t stream) {
    if (traced) {
        switch (store) {
            case STORE_F16: return launch_g<STORE_F16, true>(a, stream);
            case STORE_BF16: return launch_g<STORE_BF16, true>(a, stream);
            default: return launch_g<STORE_F32, true>(a, stream);
        }
    }
    switch (store) {
        case STORE_F16: return launch_g<STORE_F16, false>(a, stream);
        case STORE_BF16: return launch_g<STORE_BF16, false>(a, stream);
        default: return launch_g<STORE_F32, false>(a, stream);
    }
}

}  // namespace lumx
