// Visibility-buffer shading resolve and display transform (gfx950).
//
//   k_resolve   render_geometry main()   src/shaders/render_geometry.comp:70-266
//               CalcFullBary / interpolate  src/shaders/common/vbuffer.glsl:11-119
//               BRDF + Filament terms    src/shaders/common/pbr.glsl:1-96
//   k_tonemap   display_transform        src/shaders/display_transform.comp:5-81
//
// One thread per pixel, 8x8 tiles (the reference's workgroup shape).  The
// per-pixel dependent chain key -> meshlet table -> instance -> mesh info ->
// meshlet -> micro indices -> remap -> vertices is the reference's; the key
// carries a stable meshlet id, resolved through the scene's meshlet table.
// Differences from the reference, all documented in the build's design notes:
// factors for roughness / metallic and a vec3 sun intensity (identity defaults
// reproduce the reference), a constant sky in place of the absent skybox,
// isotropic trilinear filtering in place of 16x anisotropy, and the absent
// tony-mc-mapface LUT replaced by its own x/(x+1) pre-encoding.
//
// A batch flattens the 8x8 tiles of all its views into one grid (per-view
// tile offsets planned on the host), so views of very different sizes share
// one launch without idle blocks.
#include "kernels.h"
#include "shading.h"

using namespace lhd;

namespace {

LH_DEV void resolve_tile(const lh_scene& s, const lh_view& v, uint32_t tx, uint32_t ty, const lh_resolve_params& p) {
    const uint32_t x = tx * 8 + (threadIdx.x & 7), y = ty * 8 + (threadIdx.x >> 3);
    if (x >= v.width || y >= v.height) return;
    const f3 c = shading::resolve_pixel(s, v, x, y, p);
    const size_t o = size_t(y) * v.width + x;
    reinterpret_cast<float4*>(v.radiance)[o] = make_float4(c.x, c.y, c.z, 1.0f);
    if (v.ldr) v.ldr[o] = shading::display_pixel(v, x, y, c);
}

}  // namespace

// Bound by VALU issue (61% of the time) and by the gathers' addresses (the
// texture-address unit is busy for half of it), with four waves per SIMD to
// hide their latency; five or six waves spill (3840x2160: 388, 502, 626 us at
// 4, 5, 6).  The shadow footprint in four 16-byte loads and shared blends, the
// texel pairs in 8-byte loads and one copy of the block decoders took the 4K
// field from 440 to 388 us (2,170 -> 1,910 VALU and 100 -> 86 load
// instructions per covered wave), 1080p from 114 to 98.
__global__ void __launch_bounds__(64) LH_RESOLVE_OCCUPANCY k_resolve(lh_scene s, OneView vs, lh_resolve_params p) {
    resolve_tile(s, vs.v, blockIdx.x, blockIdx.y, p);
}

// Four waves per SIMD: without the target the batch variant's view lookup
// takes it one register past 128 (three waves).
__global__ void __launch_bounds__(64) LH_WAVES_ATTR(4) k_resolve_batch(lh_scene s, ViewTable vs, lh_resolve_params p) {
    const uint32_t g = blockIdx.x;
    uint32_t lo = 0, hi = vs.n;  // last view with tile_offsets[view] <= g
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (vs.tile_offsets[mid] <= g)
            lo = mid;
        else
            hi = mid;
    }
    const lh_view& v = vs.get(lo);
    const uint32_t local = g - vs.tile_offsets[lo], tiles_x = (v.width + 7) / 8;
    resolve_tile(s, v, local % tiles_x, local / tiles_x, p);
}

template <class VS>
__global__ void __launch_bounds__(256) k_tonemap(VS vs) {
    const lh_view& v = vs.get(blockIdx.z);
    const uint64_t n = uint64_t(v.width) * v.height;
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x) {
        float4 c = reinterpret_cast<const float4*>(v.radiance)[i];
        v.ldr[i] = shading::display_pixel(v, uint32_t(i % v.width), uint32_t(i / v.width), f3{c.x, c.y, c.z});
    }
}

namespace lhk {

template <>
hipError_t resolve<OneView>(const lh_scene& s, const OneView& vs, uint32_t, const lh_resolve_params& p,
                            hipStream_t st) {
    dim3 grid((vs.v.width + 7) / 8, (vs.v.height + 7) / 8);
    mark("resolve", st);
    hipLaunchKernelGGL(k_resolve, grid, dim3(64), 0, st, s, vs, p);
    return hipGetLastError();
}

template <>
hipError_t resolve<ViewTable>(const lh_scene& s, const ViewTable& vs, uint32_t total_tiles,
                              const lh_resolve_params& p, hipStream_t st) {
    mark("resolve", st);
    hipLaunchKernelGGL(k_resolve_batch, dim3(std::max(total_tiles, 1u)), dim3(64), 0, st, s, vs, p);
    return hipGetLastError();
}

template <class VS>
hipError_t tonemap(const VS& vs, uint64_t max_pixels, hipStream_t st) {
    uint32_t blocks = uint32_t(std::min<uint64_t>((max_pixels + 255) / 256, 4096));
    mark("tonemap", st);
    hipLaunchKernelGGL(k_tonemap<VS>, dim3(std::max(blocks, 1u), 1, vs.count()), dim3(256), 0, st, vs);
    return hipGetLastError();
}

template hipError_t tonemap<OneView>(const OneView&, uint64_t, hipStream_t);
template hipError_t tonemap<ViewTable>(const ViewTable&, uint64_t, hipStream_t);

}  // namespace lhk
