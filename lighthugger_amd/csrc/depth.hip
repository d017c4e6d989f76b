// Depth bounds and cascade fitting (gfx950).
//
//   k_depth_bounds   read_depth                src/shaders/compute/read_depth.glsl:3-83
//   k_fit_cascades   generate_shadow_matrices  src/shaders/compute/generate_shadow_matrices.glsl:15-110
//
// The reference gathers 4x4 texels of the D32 depth buffer per thread and
// reduces with subgroupMin / subgroupMax; here the depth bits come from the
// visibility-buffer keys (depth.h).  min ignores zero (sky) exactly like
// min_if_not_zero (read_depth.glsl:3-18).
#include "cascade.h"
#include "depth.h"
#include "kernels.h"

using namespace lhd;

template <class VS>
__global__ void __launch_bounds__(256) k_depth_bounds(VS vs) {
    __shared__ uint32_t smin[4], smax[4];
    const lh_view& v = vs.get(blockIdx.z);
    depth::block_bounds(v, smin, smax);
}

// One lane per cascade, one block per view.
template <class VS>
__global__ void __launch_bounds__(64) k_fit_cascades(VS vs) {
    const lh_view& v = vs.get(blockIdx.z);
    const uint32_t c = threadIdx.x;
    const uint32_t min_bits = v.misc->min_depth, max_bits = v.misc->max_depth;
    if (c == 0 && min_bits == 0xFFFFFFFFu) atomicOr(&v.counters[LH_CNT_FLAGS], LH_FLAG_EMPTY_VIEW);
    if (c >= LH_NUM_CASCADES) return;
    cascade::store(*v.misc, c, cascade::fit(*v.uniforms, min_bits, max_bits, c));
}

namespace lhk {

template <class VS>
hipError_t depth_bounds(const VS& vs, uint64_t max_pixels, hipStream_t st) {
    const uint32_t blocks = depth::blocks(max_pixels);
    mark("depth_bounds", st);
    hipLaunchKernelGGL(k_depth_bounds<VS>, dim3(blocks, 1, vs.count()), dim3(256), 0, st, vs);
    return hipGetLastError();
}

template <class VS>
hipError_t fit_cascades(const VS& vs, hipStream_t st) {
    mark("fit_cascades", st);
    hipLaunchKernelGGL(k_fit_cascades<VS>, dim3(1, 1, vs.count()), dim3(64), 0, st, vs);
    return hipGetLastError();
}

template hipError_t depth_bounds<OneView>(const OneView&, uint64_t, hipStream_t);
template hipError_t depth_bounds<ViewTable>(const ViewTable&, uint64_t, hipStream_t);
template hipError_t fit_cascades<OneView>(const OneView&, hipStream_t);
template hipError_t fit_cascades<ViewTable>(const ViewTable&, hipStream_t);

}  // namespace lhk
