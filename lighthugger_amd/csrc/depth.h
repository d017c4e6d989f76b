// Depth-bounds reduction of one 256-thread block (device code) and its grid.
//
// read_depth (src/shaders/compute/read_depth.glsl:3-83): min over non-zero and
// max of the depth bits, which come straight from the visibility-buffer keys
// (depth = ~(key >> 32)).
#pragma once

#include <algorithm>

#include "lh_device.h"

namespace depth {

using namespace lhd;

// ~16 keys per thread, at most one block per CU and view (their pairs of
// atomics go to two addresses).
inline uint32_t blocks(uint64_t pixels) { return uint32_t(std::max<uint64_t>(std::min<uint64_t>((pixels + 4095) / 4096, 256), 1)); }

// Thread x of block blockIdx.x streams its slice with 16-byte loads, the block
// reduces, and one atomic pair lands in MiscStorage.
LH_DEV void block_bounds(const lh_view& v, uint32_t* smin /* LDS [4] */, uint32_t* smax /* LDS [4] */) {
    const uint64_t n = uint64_t(v.width) * v.height;
    uint32_t mn = 0xFFFFFFFFu, mx = 0u;
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x * 2;
    uint64_t i = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) * 2;
    for (; i + 1 < n; i += stride) {
        ulonglong2 k = *reinterpret_cast<const ulonglong2*>(v.visbuffer + i);
        uint32_t a = ~uint32_t(k.x >> 32), b = ~uint32_t(k.y >> 32);
        if (a) mn = min(mn, a);
        if (b) mn = min(mn, b);
        mx = max(mx, max(a, b));
    }
    if (i < n) {
        uint32_t a = ~uint32_t(v.visbuffer[i] >> 32);
        if (a) mn = min(mn, a);
        mx = max(mx, a);
    }
    mn = wave_min_u32(mn);
    mx = wave_max_u32(mx);
    const uint32_t w = threadIdx.x >> 6;
    if (lane_id() == 0) {
        smin[w] = mn;
        smax[w] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        mn = min(min(smin[0], smin[1]), min(smin[2], smin[3]));
        mx = max(max(smax[0], smax[1]), max(smax[2], smax[3]));
        if (mn != 0xFFFFFFFFu) atomicMin(&v.misc->min_depth, mn);
        atomicMax(&v.misc->max_depth, mx);
    }
}

}  // namespace depth
