// Two-phase occlusion culling of the main view (LH_VIEW_HIZ), kernels.
//
//   k_hiz_build  one wave per 8x8 pixel tile: the tile's minimum depth
//                (reverse-Z: the farthest) from the phase-1 visibility buffer,
//                0 where a pixel is still empty.  Stored in the view's
//                radiance buffer, which the resolve overwrites later.  Also
//                records the phase-1 draw count and empties the view's
//                clip / big-triangle queues for phase 2.
//   k_hiz_cull   one lane per candidate meshlet (staged in draws[1]): its
//                conservative screen rectangle and nearest depth against the
//                tiles it touches; survivors are appended to draws[0] after
//                the phase-1 draws.
// The raster then runs again over draws[0][phase-1 count, total).
#include "hiz.h"
#include "kernels.h"

using namespace lhd;

namespace {

__global__ void __launch_bounds__(64) k_hiz_build(OneView vs, uint32_t history_words) {
    const lh_view& v = vs.v;
    // the view's cull has read the last frame's history: empty it for this one's
    if (v.history) {
        const uint32_t threads = gridDim.x * gridDim.y * 64;
        for (uint32_t i = (blockIdx.y * gridDim.x + blockIdx.x) * 64 + threadIdx.x; i < history_words; i += threads)
            v.history[i] = 0u;
    }
    const uint32_t tiles_x = (v.width + hiz::kTile - 1) / hiz::kTile;
    const uint32_t tx = blockIdx.x, ty = blockIdx.y;
    const uint32_t x = tx * hiz::kTile + (threadIdx.x & 7), y = ty * hiz::kTile + (threadIdx.x >> 3);
    uint32_t d = 0xFFFFFFFFu;  // pixels outside the image do not count
    if (x < v.width && y < v.height) d = ~uint32_t(v.visbuffer[size_t(y) * v.width + x] >> 32);  // empty -> 0.0
    d = wave_min_u32(d);  // non-negative floats order as their bits
    if (threadIdx.x == 0) v.radiance[size_t(ty) * tiles_x + tx] = __uint_as_float(d);
    if (tx == 0 && ty == 0 && threadIdx.x == 0) {
        v.counters[LH_CNT_HIZ_PHASE1] = min(v.counters[LH_CNT_DRAWS], v.draw_capacity);
        v.counters[LH_CNT_CLIP] = 0;
        v.counters[LH_CNT_BIG] = 0;
    }
}

__global__ void __launch_bounds__(256) k_hiz_cull(lh_scene s, OneView vs) {
    const lh_view& v = vs.v;
    const uint32_t n = min(v.counters[LH_CNT_HIZ_CANDIDATES], v.draw_capacity);
    const MeshletReference* cand = v.draws + size_t(v.draw_capacity);
    MeshletReference* out = v.draws;
    const uint32_t tiles_x = (v.width + hiz::kTile - 1) / hiz::kTile;
    const float* tiles = v.radiance;
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += stride) {
        const uint32_t i = base + threadIdx.x;
        bool draw = false;
        MeshletReference ref{0, 0};
        if (i < n) {
            ref = cand[i];
            const Instance& in = s.instances[ref.instance_index];
            const MeshInfo& mi = mesh_info_at(in.mesh_info_address);
            const Meshlet& ml = ptr<Meshlet>(mi.meshlets)[ref.meshlet_index];
            f3 c;
            float r;
            world_sphere(in, ml.bounding_sphere, c, r);
            const hiz::ScreenBound b =
                hiz::sphere_bound(v.uniforms->combined_perspective_view, c, r, v.width, v.height);
            draw = !b.valid;
            if (b.valid && b.x0 <= b.x1 && b.y0 <= b.y1) {
                const uint32_t tx0 = uint32_t(b.x0) / hiz::kTile, tx1 = uint32_t(b.x1) / hiz::kTile;
                const uint32_t ty0 = uint32_t(b.y0) / hiz::kTile, ty1 = uint32_t(b.y1) / hiz::kTile;
                float farthest = 3.0e38f;
                for (uint32_t ty = ty0; ty <= ty1; ty++)
                    for (uint32_t tx = tx0; tx <= tx1; tx++) farthest = fminf(farthest, tiles[size_t(ty) * tiles_x + tx]);
                draw = !(b.zmax * (1.0f + hiz::kDepthMargin) < farthest);
            }
        }
        const uint32_t slot = wave_append(&v.counters[LH_CNT_DRAWS], draw);
        if (draw) {
            if (slot < v.draw_capacity)
                out[slot] = ref;
            else
                atomicOr(&v.counters[LH_CNT_OVERFLOW], LH_OVERFLOW_DRAWS);
        }
    }
}

// Visibility history of the frame just rasterized: one bit per meshlet that
// owns a pixel (k_hiz_build has cleared it).  Device atomics on one cache line
// run one after another, and the line of a near instance collects the bits of
// a large part of the screen: a block of 64x32 pixels first gathers its bits in
// a small table in LDS, by history word, and sends each word once.  A word
// whose slot is taken by another goes straight to memory.  1080p: 64 us when
// every wave merged its own lanes' bits.
constexpr uint32_t kHistorySlots = 512, kHistoryRows = 32;

__global__ void __launch_bounds__(256) k_history_mark(OneView vs, uint32_t total_meshlets) {
    __shared__ uint32_t word[kHistorySlots], bits[kHistorySlots];
    const lh_view& v = vs.v;
    for (uint32_t i = threadIdx.x; i < kHistorySlots; i += 256) {
        word[i] = ~0u;
        bits[i] = 0u;
    }
    __syncthreads();
    const uint32_t x = blockIdx.x * 64 + lane_id();
    const uint32_t y0 = blockIdx.y * kHistoryRows + (threadIdx.x >> 6);
    uint64_t key[kHistoryRows / 4];
#pragma unroll
    for (uint32_t r = 0; r < kHistoryRows / 4; r++) {
        const uint32_t y = y0 + r * 4;
        key[r] = x < v.width && y < v.height ? v.visbuffer[uint64_t(y) * v.width + x] : LH_VISBUFFER_CLEAR;
    }
#pragma unroll
    for (uint32_t r = 0; r < kHistoryRows / 4; r++) {
        const uint32_t id = uint32_t(key[r] >> LH_KEY_TRI_BITS) & (LH_MAX_SCENE_MESHLETS - 1);
        const uint32_t mid = key[r] != LH_VISBUFFER_CLEAR && id < total_meshlets ? id : ~0u;
        const uint32_t before = __shfl_up(mid, 1, 64);
        if (mid != ~0u && (lane_id() == 0 || mid != before)) {
            const uint32_t w = mid >> 5, bit = 1u << (mid & 31), slot = w & (kHistorySlots - 1);
            const uint32_t had = atomicCAS(word + slot, ~0u, w);
            if (had == ~0u || had == w)
                atomicOr(bits + slot, bit);
            else
                atomicOr(v.history + w, bit);
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kHistorySlots; i += 256)
        if (bits[i]) atomicOr(v.history + word[i], bits[i]);
}

}  // namespace

namespace lhk {

hipError_t update_history(const lh_scene& s, const OneView& vs, hipStream_t st) {
    const lh_view& v = vs.v;
    if (!v.history) return hipSuccess;
    mark("history_update", st);
    hipLaunchKernelGGL(k_history_mark, dim3((v.width + 63) / 64, (v.height + kHistoryRows - 1) / kHistoryRows),
                       dim3(256), 0, st, vs, s.total_meshlets);
    return hipGetLastError();
}

hipError_t hiz_cull(const lh_scene& s, const OneView& vs, uint32_t blocks, hipStream_t st) {
    const lh_view& v = vs.v;
    const dim3 tiles((v.width + hiz::kTile - 1) / hiz::kTile, (v.height + hiz::kTile - 1) / hiz::kTile);
    mark("hiz_build", st);
    hipLaunchKernelGGL(k_hiz_build, tiles, dim3(64), 0, st, vs, (s.total_meshlets + 31) / 32);
    mark("hiz_cull", st);
    hipLaunchKernelGGL(k_hiz_cull, dim3(std::max(blocks, 1u)), dim3(256), 0, st, s, vs);
    return hipGetLastError();
}

}  // namespace lhk
