// Software rasterizer of the GPU-driven frame (gfx950, wave64).
//
// Replaces the reference's fixed-function raster of its meshlet draws:
//   visbuffer_opaque_vertex/pixel   src/shaders/rasterization.glsl:38-58
//   shadowmap_opaque_vertex         src/shaders/rasterization.glsl:101-111
//   pipeline state                  src/pipelines.cpp:10-77 (cull back / front,
//                                   depth GREATER / LESS, CCW front faces)
//   draws                           src/rendering.cpp:235-242, :405-412
// with the Vulkan rasterization rules restated for software:
//   - clip to 0 <= z <= w and to the guard band |x|,|y| <= 4w
//     (Sutherland-Hodgman, intersections computed from the inside vertex);
//   - x_f = (W/2) x/w + W/2 (same for y), snapped to 8 subpixel bits (rint);
//   - pixel centres (x + 0.5, y + 0.5); exact integer edge functions;
//     top-left fill rule in y-down framebuffer coordinates;
//   - depth = z0 + l1 (z1 - z0) + l2 (z2 - z0), l_i = E_i / area, clamped to [0, 1].
// Main view: 64-bit atomicMin of ~bits(z) << 32 | meshlet << 7 | tri (nearest
// wins under reverse-Z); shadows: 32-bit atomicMin of bits(z).
//
// One launch covers a pass set - the main view, or all four cascades - whose
// draw lists are concatenated into one index space, so the persistent grid is
// balanced across cascades of very different load.  Work split:
//   k_raster_meshlets  one-wave blocks over the surviving meshlets: a wave
//                      loads the heads of its next 64 draws together, requests
//                      a meshlet's indices, corners and positions while the
//                      one before is in hand, transforms its <= 64 vertices
//                      (one per lane) into LDS and sets up its <= 124 triangles
//                      (two per lane).  Triangles within `medium_extent` that
//                      cover a pixel centre's row and column go to the wave's
//                      triangle queue, rasterized 64 at a time (raster_queue);
//                      larger ones go to the big queue, clip-crossing ones to
//                      the clip queue (one atomic per wave, tagged with the
//                      pass).  k_raster_alpha: the same for alpha-clip draws.
//   k_raster_clip      clips queued triangles and queues the fan pieces.
//   k_raster_big       queued triangles, one wave each (whole block for
//                      boxes over kWaveBoxPx pixels).
#include "raster.h"

using namespace lhd;
using namespace lhr;

namespace {

// Occupancy target of the meshlet raster (waves per SIMD).  It is bound by
// VALU issue (about 320 instructions a meshlet, most of them the transform and
// the setup of triangles that cover nothing) and, before the heads and the
// fetches were pipelined, by the chain of dependent loads.  Four cascades of
// the 20,000-instance field (2.0 M meshlets), per launch: 1.99 ms with one
// meshlet at a time and each round's few survivors in their own lanes; 2.06,
// 1.53, 1.49, 1.48 ms at 8, 7, 6, 5 waves with the pipeline and the queue (at
// 8 the 64 VGPRs spill); 1.41 ms with the spans of raster_queue.
#ifndef LH_MESHLET_WAVES
#define LH_MESHLET_WAVES 6
#endif

// Queues of the clip and large-triangle kernels.
LH_DEV void queue_clip(const lh_view& v, uint32_t pass0, bool pred, uint32_t d, uint32_t t, uint32_t pi, bool alpha) {
    if (ballot(pred) == 0) return;
    const uint32_t slot = wave_append(&v.counters[LH_CNT_CLIP + pass0], pred);
    if (!pred) return;
    if (slot < v.clip_capacity)
        queues(v).clip[slot] = make_uint2((d << LH_KEY_TRI_BITS) | t, pi | (alpha ? kClipAlpha : 0u));
    else
        atomicOr(&v.counters[LH_CNT_OVERFLOW], LH_OVERFLOW_CLIP);
}

// ALPHA selects the draws of alpha-clip mesh infos (double-sided, alpha test
// per sample); the opaque instantiation skips them.  The alpha instantiation
// returns at once when the culls counted no alpha-clip draw in its passes.
template <int KIND, class VS, bool ST, bool ALPHA>
LH_DEV void raster_meshlets(const lh_scene& s, const VS& vs, const PassSet& ps) {
    __shared__ WaveVerts wv;
    __shared__ TriQueue queue;
    const uint32_t lane = threadIdx.x;
    if constexpr (ALPHA) {
        uint32_t n = 0;
        for (uint32_t k = lane; k < vs.count() * ps.n; k += 64)
            n += vs.get(k / ps.n).counters[LH_CNT_ALPHA_DRAWS + ps.pass0 + k % ps.n];
        if (wave_sum_u32(n) == 0) return;
    }
    const Segments<VS> seg(vs, ps);
    uint32_t total = seg.total();
    const uint32_t* list = nullptr;
    if constexpr (std::is_same<VS, OneView>::value) {
        if (ps.direct) {  // the draws the tiled raster left to this kernel
            const lh_view& v = vs.get(0);
            const lhs::ScratchLayout L = lhs::scratch_layout(v);
            list = reinterpret_cast<const uint32_t*>(static_cast<const char*>(v.scratch) + L.direct);
            total = min(v.counters[LH_CNT_TILE_DIRECT], L.direct_capacity);
        }
    }
    Tally<ST> tally;
    uint32_t held = 0;            // triangles in the queue
    uint32_t at = ~0u;            // view << 3 | pass within the set that they belong to
    Pass p{};
    LhMat4 M{};
    auto flush = [&]() {
        if (held) raster_queue<KIND, ST, ALPHA>(s, M, p, queue, 0, held, lane, tally);
        held = 0;
        if (at != ~0u) tally.flush(vs.get(at >> 3), p.pass);
    };
    for (uint32_t k0 = 0;; k0 += 64) {
        // the heads of the wave's next 64 draws, one per lane
        const uint32_t g = seg.draw(k0 + lane);
        const uint64_t some = ballot(g < total);
        if (some == 0) break;
        DrawHead head{};
        uint32_t where = 0, draw = 0;
        bool clip_queued = false;
        if (g < total) {
            const uint32_t e = list ? list[g] : g;
            uint32_t view, pi;
            seg.find(e & ~(list ? lhs::kBinDirect : 0u), view, pi, draw);
            clip_queued = list && (e & lhs::kBinDirect) != 0;
            where = view << 3 | pi;
            const lh_view& v = vs.get(view);
            head = load_head(s, v.draws[size_t(ps.pass0 + pi) * v.draw_capacity + draw]);
        }
        uint64_t todo = ballot(g < total && (((head.info >> 16) & MESH_INFO_FLAGS_ALPHA_CLIP) != 0) == ALPHA);
        const uint64_t clip_done = ballot(clip_queued);
        if (todo == 0) continue;
        MeshletFetch next;
        DrawHead h = head_of_lane(head, first_lane(todo));
        next.request(h, lane);
        next.request_position(h, lane);
        while (todo) {
            const uint32_t l = first_lane(todo);
            todo &= todo - 1;
            const DrawHead cur = h;
            MeshletFetch f = next;
            if (todo) {  // the next draw's indices and corners travel while this one is transformed
                h = head_of_lane(head, first_lane(todo));
                next.request(h, lane);
            }
            const uint32_t here = readlane_u32(where, l), d = readlane_u32(draw, l), pi = here & 7u;
            const lh_view& v = vs.get(here >> 3);
            if (here != at) {  // wave-uniform: another view or pass than the queue's
                flush();
                at = here;
                p = make_pass(v, ps.pass0 + pi);
                M = load_mat4(reinterpret_cast<uint64_t>(&view_matrix<KIND>(v, p.pass)));
            }
            const LhMat4 T = load_mat4(reinterpret_cast<uint64_t>(&s.instances[cur.instance].transform));
            SV sv;
            lds_order();
            const bool clean = transform_vertices(cur, f, T, M, p.W, p.H, lane, wv, sv);
            lds_order();
            if (todo) next.request_position(h, lane);
            const uint32_t ntri = cur.triangles();
            for (uint32_t round = 0; round * 64 < ntri; round++) {
                const uint32_t t = lane + 64 * round;
                const TriSetup ts = triangle_setup<KIND>(wv, f.corners(cur, lane, round), t < ntri, clean, ALPHA, p.W, p.H);
                if (!clean && !((clip_done >> l) & 1)) queue_clip(v, ps.pass0, ts.clip, d, t, pi, ALPHA);
                const bool big = ts.inside && ts.extent > ps.medium_extent, push = ts.inside && !big;
                const uint32_t id = (cur.mid << LH_KEY_TRI_BITS) | t;
                if (ballot(big)) {
                    const uint32_t slot = wave_append(&v.counters[LH_CNT_BIG + ps.pass0], big);
                    if (big) {
                        const SV v0{ts.a.x, ts.a.y, wv.Z[ts.i0]}, v1{ts.b.x, ts.b.y, wv.Z[ts.i1]},
                            v2{ts.c.x, ts.c.y, wv.Z[ts.i2]};
                        if (slot < v.big_capacity)
                            store_big(queues(v).big + slot, v0, ts.swapped ? v2 : v1, ts.swapped ? v1 : v2, id, ts.xlo,
                                      ts.xhi, ts.ylo, ts.yhi, pi, ALPHA);
                        else
                            atomicOr(&v.counters[LH_CNT_OVERFLOW], LH_OVERFLOW_BIG);
                    }
                }
                const uint64_t pm = ballot(push);
                if (pm == 0) continue;
                if (push) {
                    const uint32_t slot = held + lanes_below(pm);
                    const int32_t X0 = ts.xlo * 256, Y0 = ts.ylo * 256;
                    const uint32_t va = pack_xy(ts.a.x - X0, ts.a.y - Y0), vb = pack_xy(ts.b.x - X0, ts.b.y - Y0),
                                   vc = pack_xy(ts.c.x - X0, ts.c.y - Y0);
                    const uint32_t za = __float_as_uint(wv.Z[ts.i0]), zb = __float_as_uint(wv.Z[ts.i1]),
                                   zc = __float_as_uint(wv.Z[ts.i2]);
                    queue.box[slot] = make_uint4(uint32_t(ts.xlo) | uint32_t(ts.ylo) << 16, va, ts.swapped ? vc : vb,
                                                 ts.swapped ? vb : vc);
                    queue.att[slot] = make_uint4(za, ts.swapped ? zc : zb, ts.swapped ? zb : zc, id);
                }
                held += uint32_t(__popcll(pm));
                if (held >= 64) {  // the last 64 entries: nothing moves
                    held -= 64;
                    raster_queue<KIND, ST, ALPHA>(s, M, p, queue, held, 64, lane, tally);
                    lds_order();
                }
            }
        }
    }
    flush();
}

template <int KIND, class VS, bool ST>
__global__ void __launch_bounds__(64) LH_WAVES_ATTR(LH_MESHLET_WAVES) k_raster_meshlets(lh_scene s, VS vs, PassSet ps) {
    raster_meshlets<KIND, VS, ST, false>(s, vs, ps);
}
// The alpha test's texture fetch needs twice the registers.
template <int KIND, class VS, bool ST>
__global__ void __launch_bounds__(64) LH_WAVES_ATTR(4) k_raster_alpha(lh_scene s, VS vs, PassSet ps) {
    raster_meshlets<KIND, VS, ST, true>(s, vs, ps);
}

// Clip polygon in homogeneous coordinates (Sutherland-Hodgman).
LH_DEV f4 clip_point(f4 a, f4 b, float da, float db) {
    float t = da / (da - db);
    return {a.x + (b.x - a.x) * t, a.y + (b.y - a.y) * t, a.z + (b.z - a.z) * t, a.w + (b.w - a.w) * t};
}

// View blockIdx.z; grid-stride over that view's clip queue.
template <int KIND, class VS>
__global__ void __launch_bounds__(64) k_raster_clip(lh_scene s, VS vs, PassSet ps) {
    const lh_view& v = vs.get(blockIdx.z);
    const Queues qs = queues(v);
    const uint32_t count = min(v.counters[LH_CNT_CLIP + ps.pass0], v.clip_capacity);
    uint32_t* big_counter = &v.counters[LH_CNT_BIG + ps.pass0];
    for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < count; q += gridDim.x * blockDim.x) {
        const uint2 e = qs.clip[q];
        const uint32_t d = e.x >> LH_KEY_TRI_BITS, t = e.x & ((1u << LH_KEY_TRI_BITS) - 1), pi = e.y & ~kClipAlpha;
        const bool alpha = (e.y & kClipAlpha) != 0;
        const Pass p = make_pass(v, ps.pass0 + pi);
        const LhMat4 M = view_matrix<KIND>(v, p.pass);
        const MeshletReference ref = p.draws[d];
        const Instance& in = s.instances[ref.instance_index];
        const MeshInfo& mi = mesh_info_at(in.mesh_info_address);
        const Meshlet& ml = ptr<Meshlet>(mi.meshlets)[ref.meshlet_index];
        const uint32_t mid = s.instance_meshlet_base[ref.instance_index] + ref.meshlet_index;
        const uint8_t* micro = ptr<uint8_t>(mi.micro_indices) + ml.triangle_offset;
        f4 poly[12], tmp[12];
        for (int j = 0; j < 3; j++) {
            f3 w = mat4_point(in.transform, load_position(mi, load_index(mi, ml.index_offset + micro[3 * t + j])));
            poly[j] = mat4_mul_vec4(M, f4{w.x, w.y, w.z, 1.0f});
        }
        int n = 3;
        for (int k = 0; k < 6 && n >= 3; k++) {
            int m = 0;
            for (int i = 0; i < n; i++) {
                f4 a = poly[i], b = poly[i + 1 == n ? 0 : i + 1];
                float da = plane_dist(a, k), db = plane_dist(b, k);
                bool ia = da >= 0.0f, ib = db >= 0.0f;
                if (ia) tmp[m++] = a;
                if (ia != ib) tmp[m++] = ia ? clip_point(a, b, da, db) : clip_point(b, a, db, da);
            }
            for (int i = 0; i < m; i++) poly[i] = tmp[i];
            n = m;
        }
        if (n < 3) continue;
        SV sv[12];
        bool ok = true;
        for (int i = 0; i < n; i++) ok = ok && project(poly[i], p.W, p.H, sv[i]);
        if (!ok) continue;
        const uint32_t id = (mid << LH_KEY_TRI_BITS) | t;
        for (int i = 1; i + 1 < n; i++) {
            SV a = sv[0], b = sv[i], c = sv[i + 1];
            int64_t area;
            int32_t xlo, xhi, ylo, yhi, ex, ey;
            if (!setup<KIND>(a, b, c, p.W, p.H, area, xlo, xhi, ylo, yhi, ex, ey, alpha)) continue;
            uint32_t slot = atomicAdd(big_counter, 1u);
            if (slot < v.big_capacity)
                store_big(qs.big + slot, a, b, c, id, xlo, xhi, ylo, yhi, pi, alpha);
            else
                atomicOr(&v.counters[LH_CNT_OVERFLOW], LH_OVERFLOW_BIG);
        }
    }
}

// Triangles of the large queue whose pixel box holds at most this many pixels
// are rasterized by one wave alone; larger ones by the whole block.
constexpr int32_t kWaveBoxPx = 4096;

// Rasterizes the pixels of one queued triangle's box that fall on lanes
// first, first + stride, ... of the box's row-major pixel order.  Coverage
// and depth of each pixel are evaluated exactly as in the other paths
// (64-bit edge functions at the pixel centre, top-left rule).
template <int KIND, bool ST, bool ALPHA>
LH_DEV void raster_box(const lh_scene& s, const lh_view& v, const PassSet& ps, const BigTri& b, int32_t first,
                       int32_t stride, Tally<ST>* tally) {
    const uint32_t pi = uint32_t(b.xlo) >> 13;
    const Pass p = make_pass(v, ps.pass0 + pi);
    const int32_t X0 = b.X[0], X1 = b.X[1], X2 = b.X[2], Y0 = b.Y[0], Y1 = b.Y[1], Y2 = b.Y[2];
    const int64_t area = edge64(X0, Y0, X1, Y1, X2, Y2);
    const float inv_area = 1.0f / float(area);
    const float z0 = b.z[0], d10 = b.z[1] - b.z[0], d20 = b.z[2] - b.z[0];
    const bool tl0 = top_left(X1, Y1, X2, Y2), tl1 = top_left(X2, Y2, X0, Y0), tl2 = top_left(X0, Y0, X1, Y1);
    const int32_t xlo = b.xlo & 0x1FFF, xhi = b.xhi, ylo = b.ylo & ~kBigAlpha, yhi = b.yhi;
    const int32_t bw = xhi - xlo + 1, n = bw * (yhi - ylo + 1);
    if (first >= n) return;
    // Step by `stride` pixels in row-major order: sy rows and sx columns,
    // plus one row when the column passes the box's right edge.
    const int32_t sy = stride / bw, sx = stride - sy * bw;
    int32_t py = ylo + first / bw, px = xlo + (first - (first / bw) * bw);
    for (int32_t i = first; i < n; i += stride) {
        const int32_t Px = px * 256 + 128, Py = py * 256 + 128;
        const int64_t e0 = edge64(X1, Y1, X2, Y2, Px, Py);
        const int64_t e1 = edge64(X2, Y2, X0, Y0, Px, Py);
        const int64_t e2 = edge64(X0, Y0, X1, Y1, Px, Py);
        const bool in = (e0 > 0 || (e0 == 0 && tl0)) && (e1 > 0 || (e1 == 0 && tl1)) && (e2 > 0 || (e2 == 0 && tl2));
        if (in && (!ALPHA || alpha_pass<KIND>(s, v, p, b.id, px, py))) {
            const float l1 = float(e1) * inv_area, l2 = float(e2) * inv_area;
            const bool issued = fragment<KIND>(p, px, py, (z0 + l1 * d10) + l2 * d20, b.id);
#pragma unroll
            for (uint32_t q = 0; q < LH_NUM_CASCADES; q++)
                if (q == pi) tally[q].hit(issued);
        }
        px += sx;
        py += sy;
        if (px > xhi) {
            px -= bw;
            py++;
        }
    }
}

// View blockIdx.z.  Each round the block takes four queue entries, one per
// wave.  A wave rasterizes its own triangle when the box is at most
// kWaveBoxPx pixels (most of the queue: slivers just over the medium extent),
// so a 54-pixel box costs one wave pass instead of a 256-thread block; the
// larger boxes of the round are rasterized by all four waves together first.
// ALPHA selects the entries of alpha-clip geometry (alpha test per sample),
// so the opaque instantiation keeps its small register footprint; the alpha
// one returns at once when the view's culls counted no alpha-clip draw.
template <int KIND, class VS, bool ST, bool ALPHA>
__global__ void __launch_bounds__(256) k_raster_big(lh_scene s, VS vs, PassSet ps) {
    const lh_view& v = vs.get(blockIdx.z);
    if constexpr (ALPHA) {
        uint32_t n = 0;
        for (uint32_t k = 0; k < ps.n; k++) n += v.counters[LH_CNT_ALPHA_DRAWS + ps.pass0 + k];
        if (n == 0) return;
    }
    const Queues qs = queues(v);
    const uint32_t count = min(v.counters[LH_CNT_BIG + ps.pass0], v.big_capacity);
    const uint32_t wave = threadIdx.x >> 6;
    // wide[r & 1][w]: wave w's triangle of round r goes to the whole block.
    // Two buffers, because a wave may write round r + 1's flag while another
    // still reads round r's (no wave gets two rounds ahead: each round has a
    // barrier).
    __shared__ uint32_t wide[2][4];
    // Statistics: each lane counts per pass of the set over all of the
    // block's triangles, and the wave adds them to the view's counters once
    // at the end (a flush per triangle also measured wrong depths on the
    // large frame's sliver triangles with statistics on).
    Tally<ST> tally[LH_NUM_CASCADES];
    uint32_t round = 0;
    for (uint32_t e0 = blockIdx.x * 4; e0 < count; e0 += gridDim.x * 4, round ^= 1) {  // block-uniform
        const uint32_t e = e0 + wave;
        bool own = false, shared = false;
        BigTri b;
        if (e < count) {
            b = qs.big[e];
            if (((b.ylo & kBigAlpha) != 0) == ALPHA) {
                const int32_t bw = b.xhi - (b.xlo & 0x1FFF) + 1, bh = b.yhi - (b.ylo & ~kBigAlpha) + 1;
                own = bw * bh <= kWaveBoxPx;
                shared = !own;
            }
        }
        if (lane_id() == 0) wide[round][wave] = shared ? 1u : 0u;
        __syncthreads();
        for (uint32_t w = 0; w < 4; w++)
            if (wide[round][w]) raster_box<KIND, ST, ALPHA>(s, v, ps, qs.big[e0 + w], threadIdx.x, 256, tally);
        if (own) raster_box<KIND, ST, ALPHA>(s, v, ps, b, int32_t(lane_id()), 64, tally);
    }
#pragma unroll
    for (uint32_t q = 0; q < LH_NUM_CASCADES; q++)
        if (q < ps.n) tally[q].flush(v, ps.pass0 + q);
}

// Batch plan: off[k + 1] = off[k] + surviving meshlets of segment k
// (segment = view k / np, pass pass0 + k % np), scanned in LDS by one block.
__global__ void __launch_bounds__(256) k_plan_segments(ViewTable vs, uint32_t pass0, uint32_t np) {
    __shared__ uint32_t cnt[LH_MAX_BATCH_SEGMENTS];
    const uint32_t nseg = vs.n * np;
    for (uint32_t k = threadIdx.x; k < nseg; k += blockDim.x) {
        const lh_view& v = vs.get(k / np);
        cnt[k] = min(v.counters[LH_CNT_DRAWS + pass0 + k % np], v.draw_capacity);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t acc = 0;
        for (uint32_t k = 0; k < nseg; k++) {
            uint32_t c = cnt[k];
            cnt[k] = acc;
            acc += c;
        }
        vs.seg_offsets[nseg] = acc;
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < nseg; k += blockDim.x) vs.seg_offsets[k] = cnt[k];
}

}  // namespace

namespace lhk {

// The per-meshlet raster of a pass set and its queue launches.  A single
// view's main pass with bin_capacity > 0 goes through the tiled raster first
// (tile.hip) when its tuning class asks for it; the per-meshlet kernel then
// covers only the draws it left.
template <int KIND, bool ST, class VS>
hipError_t launch_kernels(const lh_scene& s, const VS& vs, PassSet ps, const RasterTuning& t, uint32_t clip_blocks,
                          uint32_t big_blocks, hipStream_t st) {
    const uint32_t nv = vs.count();
    bool tiled = false;
    if constexpr (std::is_same<VS, OneView>::value)
        tiled = KIND == 0 && vs.v.bin_capacity > 0 && t.tile_raster != 0;
    if (tiled) {
        if constexpr (std::is_same<VS, OneView>::value) {
            hipError_t e = raster_tiles<ST>(s, vs, ps, t, st);
            if (e != hipSuccess) return e;
        }
        ps.direct = 1;
        mark("raster_direct_view", st);
    } else {
        mark(KIND == 0 ? "raster_meshlets_view" : "raster_meshlets_shadow", st);
    }
    hipLaunchKernelGGL((k_raster_meshlets<KIND, VS, ST>), dim3(t.meshlet_blocks), dim3(64), 0, st, s, vs, ps);
    ps.direct = 0;
    const bool alpha = !(s.flags & LH_SCENE_OPAQUE_ONLY);
    if (alpha) {
        mark(KIND == 0 ? "raster_alpha_view" : "raster_alpha_shadow", st);
        hipLaunchKernelGGL((k_raster_alpha<KIND, VS, ST>), dim3(t.meshlet_blocks), dim3(64), 0, st, s, vs,
                           ps);
    }
    mark(KIND == 0 ? "raster_clip_view" : "raster_clip_shadow", st);
    hipLaunchKernelGGL((k_raster_clip<KIND, VS>), dim3(clip_blocks, 1, nv), dim3(64), 0, st, s, vs, ps);
    mark(KIND == 0 ? "raster_big_view" : "raster_big_shadow", st);
    hipLaunchKernelGGL((k_raster_big<KIND, VS, ST, false>), dim3(big_blocks, 1, nv), dim3(256), 0, st, s, vs, ps);
    if (alpha) {
        mark(KIND == 0 ? "raster_big_alpha_view" : "raster_big_alpha_shadow", st);
        hipLaunchKernelGGL((k_raster_big<KIND, VS, ST, true>), dim3(big_blocks, 1, nv), dim3(256), 0, st, s, vs, ps);
    }
    return hipGetLastError();
}

// Statistics are a single-view feature (LH_VIEW_STATISTICS).
template <int KIND>
hipError_t launch_set(const lh_scene& s, const OneView& vs, const PassSet& ps, const RasterTuning& t, uint32_t cb,
                      uint32_t bb, hipStream_t st) {
    if (vs.v.flags & LH_VIEW_STATISTICS) return launch_kernels<KIND, true>(s, vs, ps, t, cb, bb, st);
    return launch_kernels<KIND, false>(s, vs, ps, t, cb, bb, st);
}
template <int KIND>
hipError_t launch_set(const lh_scene& s, const ViewTable& vs, const PassSet& ps, const RasterTuning& t, uint32_t cb,
                      uint32_t bb, hipStream_t st) {
    return launch_kernels<KIND, false>(s, vs, ps, t, cb, bb, st);
}

template <class VS>
hipError_t raster(const lh_scene& s, const VS& vs, uint32_t pass0, uint32_t npasses, const RasterTuning& t,
                  hipStream_t st, bool phase2) {
    if (npasses == 0 || npasses > LH_NUM_CASCADES || pass0 + npasses > LH_NUM_PASSES || (pass0 == 0 && npasses != 1))
        return hipErrorInvalidValue;
    // the cascades may take their own extents (their triangles are smaller
    // and their raster depth-only)
    const bool cascades = pass0 > 0;
    const uint32_t small_sel = cascades && t.shadow_small_extent_px ? t.shadow_small_extent_px : t.small_extent_px;
    const uint32_t medium_sel = cascades && t.shadow_medium_extent_px ? t.shadow_medium_extent_px : t.medium_extent_px;
    const uint32_t small_px = std::min<uint32_t>(std::max<uint32_t>(small_sel, 1), 32);
    const uint32_t medium_px = std::min<uint32_t>(std::max(medium_sel, small_px), 64);
    PassSet ps{pass0, npasses, int32_t(small_px * 256), int32_t(medium_px * 256), phase2 ? 1u : 0u, 0u};
    const uint32_t nv = vs.count();
    // per-view persistent grids of the queue kernels shrink with the batch size
    const uint32_t clip_blocks = nv > 1 ? std::max(t.clip_blocks / 16, 4u) : t.clip_blocks;
    const uint32_t big_blocks = nv > 1 ? std::max(t.big_blocks / 16, 32u) : t.big_blocks;
    if (pass0 == 0) return launch_set<0>(s, vs, ps, t, clip_blocks, big_blocks, st);
    return launch_set<1>(s, vs, ps, t, clip_blocks, big_blocks, st);
}

template hipError_t raster<OneView>(const lh_scene&, const OneView&, uint32_t, uint32_t, const RasterTuning&,
                                    hipStream_t, bool);
template hipError_t raster<ViewTable>(const lh_scene&, const ViewTable&, uint32_t, uint32_t, const RasterTuning&,
                                      hipStream_t, bool);

hipError_t plan_segments(const ViewTable& vt, uint32_t pass0, uint32_t npasses, hipStream_t st) {
    if (vt.n * npasses > LH_MAX_BATCH_SEGMENTS) return hipErrorInvalidValue;
    mark("plan_segments", st);
    hipLaunchKernelGGL(k_plan_segments, dim3(1), dim3(256), 0, st, vt, pass0, npasses);
    return hipGetLastError();
}

}  // namespace lhk
