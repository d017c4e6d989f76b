// Internal launcher interface between the C ABI (capi.hip, batch.hip) and the
// kernels.  Launchers are templated on the view source (lhd::OneView for one
// view, lhd::ViewTable for a batch) and instantiated for both.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "lh/lh.h"
#include "lh_device.h"

namespace lhk {

// Raster tunables (chosen by the autotuner; output is independent of them).
// The values here hold until a program sets others; the autotuner's file, which
// the Python loader applies, is faster (1920x1080 field 361 us a frame for 457).
struct RasterTuning {
    uint32_t small_extent_px = 4;   // kept as set: the least medium extent
    uint32_t medium_extent_px = 64; // larger triangles go to the large-triangle queue
    uint32_t meshlet_blocks = 8192; // persistent grid of the per-meshlet kernel (64-thread blocks)
    uint32_t big_blocks = 2048;     // persistent grid of the large-triangle kernel (256-thread blocks)
    uint32_t clip_blocks = 256;     // kept as set: clipped triangles run on the large-triangle grid
    uint32_t tile_item_entries = 64; // tiled main-view raster: binned meshlets per work item (>= 8)
    uint32_t tile_blocks = 1024;    // tiled main-view raster: persistent grid (512-thread blocks)
    uint32_t tile_raster = 1;       // main view through the tiled raster (when bin_capacity > 0)
    uint32_t shadow_small_extent_px = 0;  // the cascades' least medium extent (0: the same)
    uint32_t shadow_medium_extent_px = 0; // the cascades' medium_extent_px (0: the same)
    bool short_queues = false;      // a batch with a view whose queues are short
};

// Queues below the least of the Python defaults.  A low medium extent queues
// many times the triangles (12 px in place of 16 at 1920x1080: 80 k for 33 k),
// and one over 120 px that finds the large-triangle queue full needs a place in
// the clip queue.  Where neither is ample their owner sized them, and raster()
// keeps the extents at which they were found long enough.
inline bool short_queues(const lh_view& v) { return v.big_capacity < 1u << 18 && v.clip_capacity < 1u << 16; }

struct Tuning {
    RasterTuning raster;
    uint32_t cull_blocks = 1024;    // persistent grid of the meshlet cull (256-thread blocks)
};

// Optional per-kernel timing: when a Profiler is installed, every launcher
// records an event on the launch stream right before each kernel, so the
// interval between consecutive events is that kernel's device time.
struct Profiler {
    static constexpr int kMax = 2048;
    hipEvent_t ev[kMax];
    const char* name[kMax];
    int n = 0;
    bool created = false;
};
extern Profiler* g_profiler;
inline void mark(const char* name, hipStream_t st) {
    Profiler* p = g_profiler;
    if (p && p->n < Profiler::kMax) {
        (void)hipEventRecord(p->ev[p->n], st);  // a failed record shows up as a failed elapsed-time query
        p->name[p->n++] = name;
    }
}

template <class VS>
hipError_t view_reset(const VS& vs, hipStream_t st);
// Clears visibility buffers and shadow maps; max_pixels = largest W*H of the views.
template <class VS>
hipError_t clear_targets(const VS& vs, uint64_t max_pixels, hipStream_t st);
template <class VS>
hipError_t cull_instances(const lh_scene& s, const VS& vs, bool shadow, hipStream_t st);
// Small scenes: view reset + main-view instance cull in one block, and depth
// bounds + cascade fit + shadow instance cull in one launch.
constexpr uint32_t kSmallReset = 1024, kSmallFit = 256;  // instances
hipError_t reset_cull_instances(const lh_scene& s, const lhd::OneView& vs, hipStream_t st);
hipError_t depth_fit_cull(const lh_scene& s, const lhd::OneView& vs, hipStream_t st);
// generate_shadow_matrices + cull_instances_shadows in one launch.
template <class VS>
hipError_t fit_cull_instances_shadow(const lh_scene& s, const VS& vs, hipStream_t st);
// Render targets a meshlet-cull launch clears after its culling (the frame's
// clears, moved into the latency-bound cull launches that precede the
// rasters writing those targets).
constexpr uint32_t kClearVisbuffer = 1, kClearShadowMaps = 2, kClearBins = 4;  // kClearBins: the tile counts
template <class VS>
hipError_t cull_meshlets(const lh_scene& s, const VS& vs, uint32_t pass0, uint32_t npasses, uint32_t blocks,
                         hipStream_t st, uint32_t clear = 0);
// Rasterizes passes [pass0, pass0 + npasses) in one set of launches (the main
// view alone, or any run of cascades).
template <class VS>
hipError_t raster(const lh_scene& s, const VS& vs, uint32_t pass0, uint32_t npasses, const RasterTuning& t,
                  hipStream_t st, bool phase2 = false, bool bins_clear = false);
// LH_VIEW_HIZ: depth pyramid of the phase-1 raster and the occlusion test of
// the staged candidates (appended to draws[0] for the phase-2 raster).
hipError_t hiz_cull(const lh_scene& s, const lhd::OneView& vs, uint32_t blocks, hipStream_t st);
// LH_VIEW_HIZ: rewrites the view's visibility history from its visibility buffer.
hipError_t update_history(const lh_scene& s, const lhd::OneView& vs, hipStream_t st);
// The main-view raster of one view: phase 1, and with LH_VIEW_HIZ the
// pyramid, the occlusion test and phase 2.
// bins_clear: the meshlet cull before it zeroed the tile counts (kClearBins).
hipError_t raster_main(const lh_scene& s, const lhd::OneView& vs, const Tuning& t, hipStream_t st,
                       bool bins_clear = false);
template <class VS>
hipError_t depth_bounds(const VS& vs, uint64_t max_pixels, hipStream_t st);
template <class VS>
hipError_t fit_cascades(const VS& vs, hipStream_t st);
// total_tiles: 8x8 tiles over all views of a batch (ignored for one view);
// params: the differentiable-parameter overrides (all NULL = scene values).
template <class VS>
hipError_t resolve(const lh_scene& s, const VS& vs, uint32_t total_tiles, const lh_resolve_params& params,
                   hipStream_t st);
// Adjoint of the single-view resolve (lh_resolve_backward); uses the first
// kBackwardScratchBytes of the view's scratch for per-block partial sums.
constexpr uint32_t kBackwardBlocks = 2048;
constexpr uint64_t kBackwardScratchBytes = uint64_t(kBackwardBlocks) * 8 * sizeof(double);
hipError_t resolve_backward(const lh_scene& s, const lhd::OneView& vs, const lh_resolve_params& params,
                            const float* grad_radiance, const lh_resolve_grads& grads, hipStream_t st);
template <class VS>
hipError_t tonemap(const VS& vs, uint64_t max_pixels, hipStream_t st);

// Batch plan: exclusive scan of the per-(view, pass) surviving meshlet counts.
hipError_t plan_segments(const lhd::ViewTable& vt, uint32_t pass0, uint32_t npasses, hipStream_t st);

}  // namespace lhk
