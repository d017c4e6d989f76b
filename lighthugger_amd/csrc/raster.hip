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
//   k_raster_big       the queued large triangles, up to 64 to a wave, and the
//                      clip-crossing ones, one to a block.
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

// ALPHA selects the draws of alpha-clip mesh infos (double-sided, alpha test
// per sample); the opaque instantiation skips them.  The alpha instantiation
// returns at once when the culls counted no alpha-clip draw in its passes.
template <int KIND, class VS, bool ST, bool ALPHA>
LH_DEV void raster_meshlets(const lh_scene& s, const VS& vs, const PassSet& ps) {
    __shared__ WaveVerts wv;
    __shared__ TriQueue queue;
    __shared__ std::conditional_t<ALPHA, AlphaStore, NoAlpha> alpha;
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
    // The early test pays where it saves an alpha test (statistics count every
    // covered sample and do without); without one it costs: the cascades of
    // the 20,000-instance field 1.17 -> 1.25 ms, its main view 764 -> 620 us,
    // but 1280x720 54 -> 78, 1920x1080 99 -> 116 and 12 cameras 848 -> 967.
    constexpr bool kEarly = ALPHA && !ST;
    uint32_t held = 0;            // triangles in the queue
    uint32_t at = ~0u;            // view << 3 | pass within the set that they belong to
    Pass p{};
    LhMat4 M{};
    auto flush = [&]() {
        if (held) raster_queue<KIND, ST, ALPHA, kEarly>(s, M, p, queue, alpha, 0, held, lane, tally);
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
        bool binned = false;
        if (g < total) {
            const uint32_t e = list ? list[g] : g;
            uint32_t view, pi;
            seg.find(e & ~(list ? lhs::kBinDirect : 0u), view, pi, draw);
            binned = list && (e & lhs::kBinDirect) != 0;
            where = view << 3 | pi;
            const lh_view& v = vs.get(view);
            head = load_head(s, v.draws[size_t(ps.pass0 + pi) * v.draw_capacity + draw]);
        }
        uint64_t todo = ballot(g < total && (((head.info >> 16) & MESH_INFO_FLAGS_ALPHA_CLIP) != 0) == ALPHA);
        const uint64_t queues_done = ballot(binned);
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
            const bool queued = ((queues_done >> l) & 1) != 0;  // by the tiled raster's binning
            for (uint32_t round = 0; round * 64 < ntri; round++) {
                const uint32_t t = lane + 64 * round;
                const TriSetup ts = triangle_setup<KIND>(wv, f.corners(cur, lane, round), t < ntri, clean, ALPHA, p.W, p.H);
                const bool big = ts.inside && ts.extent > ps.medium_extent;
                const uint32_t id = (cur.mid << LH_KEY_TRI_BITS) | t;
                bool push = ts.inside && !big;
                if (!clean || ballot(big && !queued)) {
                    // A full queue: the wave keeps the triangle, or, a wide one, the
                    // clip queue takes it (nothing is cut off then).
                    const bool full = queue_big(v, ps.pass0, big && !queued, wv, ts, id, pi, ALPHA);
                    queue_clip(v, ps.pass0, (ts.clip && !queued) || (full && ts.extent > kNarrow), d, t, pi, ALPHA);
                    push = push || (full && ts.extent <= kNarrow);
                }
                const uint64_t pm = ballot(push);
                if (pm == 0) continue;
                if (push) queue.store(held + lanes_below(pm), wv, ts, id);
                held += uint32_t(__popcll(pm));
                if (held >= 64) {  // the last 64 entries: nothing moves
                    held -= 64;
                    raster_queue<KIND, ST, ALPHA, kEarly>(s, M, p, queue, alpha, held, 64, lane, tally);
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
// Alpha-clipped triangles over this extent go to the large-triangle raster,
// which spreads them over the chip: their samples are far dearer than opaque
// ones, and a wave would keep its meshlet's to itself (1,500 alpha-clipped
// cards at 720p: 1.07, 0.88, 0.71, 0.68, 0.67 ms a frame at 16, 12, 8, 6, 4 px).
constexpr uint32_t kAlphaMediumPx = 6;

// Corners that the clipped polygon may have in LDS.  A convex one has at most
// nine after six planes, but corners that lie on a plane to within rounding may
// alternate about it (ten occur), and each change of side adds a corner: a
// plane makes at most m + floor(m / 2) of m corners, from 3 at most 4, 6, 9,
// 13, 19, 28.
constexpr uint32_t poly_corners(uint32_t planes) {
    const uint32_t m = planes == 0 ? 3 : poly_corners(planes - 1);
    return planes == 0 ? m : m + m / 2;
}
constexpr uint32_t kPolyMax = poly_corners(6);
static_assert(kPolyMax == 28 && kPolyMax <= 64, "one corner per lane");

// Clips a polygon held one corner per lane (lanes 0..n-1) by the six planes
// and returns its number of corners (0 when nothing is left).  Per plane every
// lane emits its own corner if it is inside and the crossing to the next
// corner if the edge crosses; the emissions are ordered by two ballots and
// exchanged through LDS.
LH_DEV uint32_t clip_polygon(f4& v, uint32_t n, uint32_t lane, float4* poly) {
    for (int k = 0; k < 6 && n >= 3; k++) {
        lds_order();
        if (lane < n) poly[lane] = make_float4(v.x, v.y, v.z, v.w);
        lds_order();
        const bool live = lane < n;
        const float4 q = poly[live && lane + 1 < n ? lane + 1 : 0];
        const f4 b{q.x, q.y, q.z, q.w};
        const float da = plane_dist(v, k), db = plane_dist(b, k);
        const bool ia = da >= 0.0f, ib = db >= 0.0f, keep = live && ia, cross = live && ia != ib;
        const uint64_t mk = ballot(keep), mc = ballot(cross);
        const uint32_t at = lanes_below(mk) + lanes_below(mc);
        lds_order();
        if (keep) poly[at] = make_float4(v.x, v.y, v.z, v.w);
        if (cross) {
            const f4 c = ia ? clip_point(v, b, da, db) : clip_point(b, v, db, da);
            poly[at + (keep ? 1u : 0u)] = make_float4(c.x, c.y, c.z, c.w);
        }
        lds_order();
        n = uint32_t(__popcll(mk) + __popcll(mc));
        if (lane < n) {
            const float4 c = poly[lane];
            v = f4{c.x, c.y, c.z, c.w};
        }
    }
    return n >= 3 ? n : 0u;
}

// Triangles over kNarrow whose pixel box holds at most this many pixels are
// rasterized by one wave alone; larger ones by the whole block.
constexpr int32_t kWaveBoxPx = 4096;
constexpr uint32_t kMaxShareLog2 = 3;
constexpr uint32_t kDirectShareLog2 = 4;

// float(e), rounded once, for |e| < 2^53: exact as a double first (four
// instructions; the direct conversion takes a dozen).
LH_DEV float to_float(int64_t e) {
    return float(__builtin_fma(double(int32_t(e >> 32)), 4294967296.0, double(uint32_t(e))));
}

// Rasterizes the pixels of one triangle's box that fall on lanes first,
// first + stride, ... of the box's row-major pixel order.  Coverage and depth
// of each pixel are evaluated exactly as in the other paths (64-bit edge
// functions at the pixel centre, stepped exactly; top-left rule).
template <int KIND, bool ST, bool ALPHA, class A>
LH_DEV void raster_box(const lh_scene& s, const lh_view& v, const Pass& p, const BigTri& b, A& alpha, int32_t first,
                       int32_t stride, Tally<ST>& tally) {
    if constexpr (ALPHA) {
        lds_order();
        if (lane_id() == 0) alpha.store(0, shading::alpha_setup(s, view_matrix<KIND>(v, p.pass), b.id));
        lds_order();
    }
    const int32_t X0 = b.X[0], X1 = b.X[1], X2 = b.X[2], Y0 = b.Y[0], Y1 = b.Y[1], Y2 = b.Y[2];
    const int64_t area = edge64(X0, Y0, X1, Y1, X2, Y2);
    const float inv_area = 1.0f / float(area);
    const float z0 = b.z[0], d10 = b.z[1] - b.z[0], d20 = b.z[2] - b.z[0];
    const int64_t m0 = top_left(X1, Y1, X2, Y2) ? 0 : 1, m1 = top_left(X2, Y2, X0, Y0) ? 0 : 1,
                  m2 = top_left(X0, Y0, X1, Y1) ? 0 : 1;
    const int32_t xlo = b.xlo & 0x1FFF, xhi = b.xhi, ylo = b.ylo & ~kBigAlpha, yhi = b.yhi;
    const int32_t bw = xhi - xlo + 1, n = bw * (yhi - ylo + 1);
    if (first >= n) return;
    // Step by `stride` pixels in row-major order: sy rows and sx columns, and
    // one row on and bw columns back when the column passes the right edge.
    const int32_t sy = stride / bw, sx = stride - sy * bw;
    int32_t py = ylo + first / bw, px = xlo + (first - (first / bw) * bw);
    const int32_t Px = px * 256 + 128, Py = py * 256 + 128;
    int64_t e0 = edge64(X1, Y1, X2, Y2, Px, Py), e1 = edge64(X2, Y2, X0, Y0, Px, Py), e2 = edge64(X0, Y0, X1, Y1, Px, Py);
    const int64_t c0 = -256ll * (Y2 - Y1), r0 = 256ll * (X2 - X1), c1 = -256ll * (Y0 - Y2), r1 = 256ll * (X0 - X2),
                  c2 = -256ll * (Y1 - Y0), r2 = 256ll * (X1 - X0);
    const int64_t a0 = sx * c0 + sy * r0, a1 = sx * c1 + sy * r1, a2 = sx * c2 + sy * r2;
    const int64_t w0 = r0 - bw * c0, w1 = r1 - bw * c1, w2 = r2 - bw * c2;
    for (int32_t i = first; i < n; i += stride) {
        if (e0 >= m0 && e1 >= m1 && e2 >= m2) {
            const float l1 = to_float(e1) * inv_area, l2 = to_float(e2) * inv_area;
            fragment<KIND, ST, !ST>(p, px, py, (z0 + l1 * d10) + l2 * d20, b.id, tally, [&] {
                if constexpr (ALPHA)
                    return shading::alpha_at(s, alpha.load(0), p.W, p.H, px, py);
                else
                    return true;
            });
        }
        px += sx, py += sy;
        e0 += a0, e1 += a1, e2 += a2;
        if (px > xhi) {
            px -= bw, py++;
            e0 += w0, e1 += w1, e2 += w2;
        }
    }
}

// The clip-crossing and the large triangles of view blockIdx.z.
//
// Large triangles: a wave takes up to 64 queue entries at a time.  Those within kNarrow (most of the
// queue: triangles just over the medium extent) go through raster_queue
// together, pass by pass; a wider one is rasterized by its wave alone when its
// box holds at most kWaveBoxPx pixels, and by the block's four waves together
// above.  Clip-crossing triangles: a block takes one at a time (several blocks
// a part each where there are few); its waves all clip it (they need no
// exchange to agree) and share the pieces of the fan: a narrow piece goes to
// one wave, a wide one to the whole block.
//
// ALPHA selects the entries of alpha-clip geometry (alpha test per sample), so
// the opaque instantiation keeps its small register footprint; the alpha one
// returns at once when the view's culls counted no alpha-clip draw.
//
// Bound by the depth atomics (20 M samples of the 4K field in 306 k wave
// instructions) until the target is read first, which leaves a third of them.
// 3840x2160, 220 k queued triangles: 215 us when every triangle walked its box
// alone with 64-bit edges, 556 with four-pixel runs per lane (a wave's atomics
// on 64 rows at once) and contiguous entries, 401 with single pixels, 181 with
// the entries dealt out, 120 with the early test, 111 on 4,096 blocks.
template <int KIND, class VS, bool ST, bool ALPHA>
__global__ void __launch_bounds__(256) LH_WAVES_ATTR(ALPHA ? 4 : 6) k_raster_big(lh_scene s, VS vs, PassSet ps) {
    const lh_view& v = vs.get(blockIdx.z);
    if constexpr (ALPHA) {
        uint32_t n = 0;
        for (uint32_t k = 0; k < ps.n; k++) n += v.counters[LH_CNT_ALPHA_DRAWS + ps.pass0 + k];
        if (n == 0) return;
    }
    const uint32_t count = min(v.counters[LH_CNT_BIG + ps.pass0], v.big_capacity);
    const uint32_t clips = min(v.counters[LH_CNT_CLIP + ps.pass0], v.clip_capacity);
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    __shared__ TriQueueOf<64> queues4[4];
    __shared__ float4 poly4[4][kPolyMax];
    // giant[r & 1][w]: wave w's entries of round r for the whole block.  Two
    // buffers, because a wave may write round r + 1's mask while another still
    // reads round r's (no wave gets two rounds ahead: each has a barrier).
    __shared__ uint64_t giant[2][4];
    TriQueueOf<64>& queue = queues4[wave];
    __shared__ std::conditional_t<ALPHA, AlphaStore, NoAlpha> alphas4[4];
    auto& alpha = alphas4[wave];
    const Queues qs = queues(v);
    // Statistics: each lane counts per pass of the set, and the block adds its
    // counts to the view's once at the end: one pair of same-address atomics a
    // block and pass, where a pair after every batch of triangles took this
    // launch of the 1920x1080 field from 72 to 393 us.  (A form that flushed
    // after every triangle, one to a block, once wrote wrong depths in frames with
    // statistics; the cause was never found, so nothing is flushed between
    // triangles.)
    Tally<ST> tally, sums[LH_NUM_CASCADES];
    auto raster_narrow = [&](uint32_t n, const Pass& p, Share share) {
        LhMat4 M{};
        if constexpr (ALPHA) M = load_mat4(reinterpret_cast<uint64_t>(&view_matrix<KIND>(v, p.pass)));
        raster_queue<KIND, ST, ALPHA, !ST>(s, M, p, queue, alpha, 0, n, lane, tally, share);
        lds_order();
        tally.move_to(sums, p.pass - ps.pass0);
    };
    const uint32_t waves = gridDim.x * 4;
    // The draws that the tiled raster left because of their size (few, over
    // LH_TILE_MAX_RECT tiles each): their triangles within the medium extent;
    // the others are queued already.  A wave alone on one of them ends long
    // after the rest, so up to 2^kDirectShareLog2 waves set up the same draw and
    // take a part of its triangles' rows each.  Medium extent 64, frame of the
    // field at 1920x1080 and 3840x2160: 882 and 1,746 us with one wave a draw,
    // 539 and 1,109 with 4, 483 and 998 with 8, 448 and 959 with 16, 440 and 948
    // with 32 (839 and 1,743 when a launch of its own drew them).
    if constexpr (KIND == 0 && !ALPHA && std::is_same<VS, OneView>::value) {
        if (ps.direct) {  // (skipped whole without it: 8.2 -> 6.3 us of an empty launch)
            __shared__ WaveVerts verts4[4];
            WaveVerts& wv = verts4[wave];
            const lhs::ScratchLayout L = lhs::scratch_layout(v);
            const uint32_t* list = reinterpret_cast<const uint32_t*>(static_cast<const char*>(v.scratch) + L.direct);
            const uint32_t n = min(v.counters[LH_CNT_TILE_DIRECT], L.direct_capacity);
            const Segments<VS> seg(vs, ps);
            const Pass p = make_pass(v, ps.pass0);
            uint32_t lg = 0;
            while (lg < kDirectShareLog2 && n << (lg + 1) <= waves) lg++;
            for (uint32_t i = blockIdx.x * 4 + wave; i < n << lg; i += waves) {
                uint32_t view, pi, d;
                seg.find(uniform_u32(list[i >> lg]) & ~lhs::kBinDirect, view, pi, d);
                const DrawHead h = head_of_lane(load_head(s, p.draws[d]), 0);
                MeshletFetch f;
                f.request(h, lane);
                f.request_position(h, lane);
                const LhMat4 T = load_mat4(reinterpret_cast<uint64_t>(&s.instances[h.instance].transform));
                const LhMat4 M = load_mat4(reinterpret_cast<uint64_t>(&view_matrix<KIND>(v, p.pass)));
                SV sv;
                lds_order();
                const bool clean = transform_vertices(h, f, T, M, p.W, p.H, lane, wv, sv);
                lds_order();
                for (uint32_t r = 0; r * 64 < h.triangles(); r++) {
                    const uint32_t t = lane + 64 * r;
                    const TriSetup ts =
                        triangle_setup<KIND>(wv, f.corners(h, lane, r), t < h.triangles(), clean, false, p.W, p.H);
                    const bool push = ts.inside && ts.extent <= ps.medium_extent;
                    const uint64_t pm = ballot(push);
                    if (pm == 0) continue;
                    if (push) queue.store(lanes_below(pm), wv, ts, (h.mid << LH_KEY_TRI_BITS) | t);
                    raster_narrow(uint32_t(__popcll(pm)), p, Share{i & ((1u << lg) - 1u), lg});
                }
            }
        }
    }
    // Entry of lane l of wave w in the round that starts at b0.  Neighbours in
    // the queue are neighbours on a mesh and of much the same size, so a
    // wave's entries lie apart: a run of large ones is shared out.
    // Where a wave would hold few entries, up to 2^kMaxShareLog2 waves take a
    // part of each instead (their lanes have room for all those entries at
    // once): the last wave to end is the one with the largest triangles, 200 us
    // after the rest when one alone walked 4,096 pixels with an alpha test on
    // each.  Alpha-clipped 1280x720, 33 k to 50 k entries, 197 of them wide:
    // alpha launches 466 + 356 -> 146 + 151 us, the opaque one 56 -> 30; without
    // wide ones 121 + 118 -> 96 + 133.  A limit of 8 or 32 entries a wave
    // in place of 16 measures the same within the noise on opaque fields.
    const uint32_t lg = share_out(count, waves, ALPHA ? 32 : 16, ALPHA ? kShareWavesAlpha : kShareWaves, kMaxShareLog2);
    const uint32_t groups = waves >> lg;
    // Number of the block's wave w.  A block's four waves follow one another,
    // but in a queue with at most an entry for every other block each goes to a
    // block of its own: four triangles over kWaveBoxPx in one block, one after the
    // other and their samples behind a read of the target, outlast all else.
    // 1,500 opaque triangles at 1920x1080, frame: of 150 px 325 -> 254 us (307
    // in a form without the read), of 300 px 556 -> 323, of 20 px 123 -> 124;
    // 4,000 of 60 px, over the limit, 244 (261 apart).  Alpha-clipped ones lose
    // more by it (4,000 of 60 px 433 -> 644: neighbours share texels) than they
    // gain.
    const bool apart = !ALPHA && count << lg <= gridDim.x / 2;
    auto number = [&](uint32_t w) { return apart ? blockIdx.x + w * gridDim.x : blockIdx.x * 4 + w; };
    auto entry = [&](uint32_t b0, uint32_t w, uint32_t l) { return b0 + (number(w) >> lg) + l * groups; };
    auto share = [&](uint32_t w) { return Share{number(w) & ((1u << lg) - 1u), lg}; };
    uint32_t round = 0;
    for (uint32_t b0 = 0; b0 + (number(0) >> lg) < count; b0 += 64 * groups, round ^= 1) {  // block-uniform
        const uint32_t e = entry(b0, wave, lane);
        BigTri b{};
        const bool mine = e < count && number(wave) >> lg < groups;
        if (mine) b = qs.big[e];
        const int32_t xlo = b.xlo & 0x1FFF, ylo = b.ylo & ~kBigAlpha;
        const uint32_t pi = uint32_t(b.xlo) >> 13;
        const int32_t extent = max(max(b.X[0], max(b.X[1], b.X[2])) - min(b.X[0], min(b.X[1], b.X[2])),
                                   max(b.Y[0], max(b.Y[1], b.Y[2])) - min(b.Y[0], min(b.Y[1], b.Y[2])));
        const bool drawn = mine && ((b.ylo & kBigAlpha) != 0) == ALPHA;
        const bool wide = drawn && extent > kNarrow;
        const bool huge = wide && (b.xhi - xlo + 1) * (b.yhi - ylo + 1) > kWaveBoxPx;
        for (uint32_t q = 0; q < ps.n; q++) {
            const bool now = drawn && !wide && pi == q;
            const uint64_t m = ballot(now);
            if (m == 0) continue;
            if (now)
                queue.store(lanes_below(m), xlo, ylo, SV{b.X[0], b.Y[0], b.z[0]}, SV{b.X[1], b.Y[1], b.z[1]},
                            SV{b.X[2], b.Y[2], b.z[2]}, b.id);
            raster_narrow(uint32_t(__popcll(m)), make_pass(v, ps.pass0 + q), share(wave));
        }
        for (uint64_t m = ballot(wide && !huge); m; m &= m - 1) {
            const BigTri t = qs.big[entry(b0, wave, first_lane(m))];
            const Pass p = make_pass(v, ps.pass0 + (uint32_t(t.xlo) >> 13));
            raster_box<KIND, ST, ALPHA>(s, v, p, t, alpha, share(wave).first(lane, 64), 64 << lg, tally);
            tally.move_to(sums, p.pass - ps.pass0);
        }
        const uint64_t hm = ballot(huge);
        if (lane == 0) giant[round][wave] = hm;
        __syncthreads();
        for (uint32_t w = 0; w < 4; w++)
            for (uint64_t m = giant[round][w]; m; m &= m - 1) {
                const BigTri t = qs.big[entry(b0, w, first_lane(m))];
                const Pass p = make_pass(v, ps.pass0 + (uint32_t(t.xlo) >> 13));
                raster_box<KIND, ST, ALPHA>(s, v, p, t, alpha, share(w).first(threadIdx.x, 256), 256 << lg, tally);
                tally.move_to(sums, p.pass - ps.pass0);
            }
    }
    const uint32_t clip_lg = share_out(clips, waves, 1, kShareWaves, kMaxShareLog2);
    for (uint32_t c = blockIdx.x; c < clips << clip_lg; c += gridDim.x) {
        const uint2 e = qs.clip[c >> clip_lg];
        const Share part{c & ((1u << clip_lg) - 1u), clip_lg};
        if (((e.y & kClipAlpha) != 0) != ALPHA) continue;
        const uint32_t d = e.x >> LH_KEY_TRI_BITS, t = e.x & ((1u << LH_KEY_TRI_BITS) - 1), pi = e.y & ~kClipAlpha;
        const Pass p = make_pass(v, ps.pass0 + pi);
        const MeshletReference ref = p.draws[d];
        const Instance& in = s.instances[ref.instance_index];
        const MeshInfo& mi = mesh_info_at(in.mesh_info_address);
        const Meshlet& ml = ptr<Meshlet>(mi.meshlets)[ref.meshlet_index];
        const uint32_t mid = s.instance_meshlet_base[ref.instance_index] + ref.meshlet_index;
        f4 corner{0, 0, 0, 0};
        if (lane < 3) {
            const uint32_t micro = ptr<uint8_t>(mi.micro_indices)[ml.triangle_offset + 3 * t + lane];
            const f3 w = mat4_point(in.transform, load_position(mi, load_index(mi, ml.index_offset + micro)));
            corner = mat4_mul_vec4(view_matrix<KIND>(v, p.pass), f4{w.x, w.y, w.z, 1.0f});
        }
        const uint32_t n = clip_polygon(corner, 3, lane, poly4[wave]);
        SV sv{0, 0, 0.0f};
        const bool ok = lane >= n || project(corner, p.W, p.H, sv);
        if (n == 0 || ballot(!ok) != 0) continue;
        // piece i of the fan (lanes 1..n-2): corners 0, i, i + 1
        const uint32_t after = min(lane + 1, 63u);
        SV v0{__shfl(sv.X, 0, 64), __shfl(sv.Y, 0, 64), __shfl(sv.z, 0, 64)}, v1 = sv,
           v2{__shfl(sv.X, int(after), 64), __shfl(sv.Y, int(after), 64), __shfl(sv.z, int(after), 64)};
        int64_t area;
        int32_t xlo, xhi, ylo, yhi, ex, ey;
        const bool set = setup<KIND>(v0, v1, v2, p.W, p.H, area, xlo, xhi, ylo, yhi, ex, ey, ALPHA);
        const bool piece = set && lane >= 1 && lane + 1 < n;
        const bool wide = piece && max(ex, ey) > kNarrow;
        const uint32_t id = (mid << LH_KEY_TRI_BITS) | t;
        const bool narrow = piece && !wide && (lane & 3u) == wave;
        const uint64_t nm = ballot(narrow);
        if (nm) {
            if (narrow) queue.store(lanes_below(nm), xlo, ylo, v0, v1, v2, id);
            raster_narrow(uint32_t(__popcll(nm)), p, part);
        }
        for (uint64_t m = ballot(wide); m; m &= m - 1) {
            const uint32_t l = first_lane(m);
            BigTri b;
            b.X[0] = readlane(v0.X, l), b.X[1] = readlane(v1.X, l), b.X[2] = readlane(v2.X, l);
            b.Y[0] = readlane(v0.Y, l), b.Y[1] = readlane(v1.Y, l), b.Y[2] = readlane(v2.Y, l);
            b.z[0] = readlane(v0.z, l), b.z[1] = readlane(v1.z, l), b.z[2] = readlane(v2.z, l);
            b.id = id;
            b.xlo = uint16_t(readlane(xlo, l)), b.ylo = uint16_t(readlane(ylo, l));
            b.xhi = uint16_t(readlane(xhi, l)), b.yhi = uint16_t(readlane(yhi, l));
            raster_box<KIND, ST, ALPHA>(s, v, p, b, alpha, part.first(threadIdx.x, 256), 256 << clip_lg, tally);
            tally.move_to(sums, p.pass - ps.pass0);
        }
    }
    if constexpr (ST) {
        __shared__ uint32_t counts[4][2 * LH_NUM_CASCADES];
#pragma unroll
        for (uint32_t q = 0; q < LH_NUM_CASCADES; q++) {
            const uint32_t f = wave_sum_u32(sums[q].frags), a = wave_sum_u32(sums[q].atomics);
            if (lane == 0) counts[wave][2 * q] = f, counts[wave][2 * q + 1] = a;
        }
        __syncthreads();
        const uint32_t q = threadIdx.x >> 1;
        if (q < ps.n) {
            uint32_t n = 0;
            for (uint32_t w = 0; w < 4; w++) n += counts[w][threadIdx.x];
            if (n) atomicAdd(&v.counters[(threadIdx.x & 1 ? LH_CNT_ATOMICS : LH_CNT_FRAGMENTS) + ps.pass0 + q], n);
        }
    }
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
hipError_t launch_kernels(const lh_scene& s, const VS& vs, PassSet ps, const RasterTuning& t, uint32_t big_blocks,
                          int32_t alpha_extent, bool bins_clear, hipStream_t st) {
    const uint32_t nv = vs.count();
    bool tiled = false;
    if constexpr (std::is_same<VS, OneView>::value)
        tiled = KIND == 0 && vs.v.bin_capacity > 0 && t.tile_raster != 0;
    // The draw count is on the device; the scene's meshlets bound what a pass
    // can draw (a block without a draw still costs its launch: 24,576 empty
    // ones 4 us).
    const uint64_t most = uint64_t(std::max(s.total_meshlets, 1u)) * nv;
    const uint32_t blocks = uint32_t(std::min<uint64_t>(t.meshlet_blocks, most));
    bool direct = false;  // the direct list is drawn by the large-triangle launch
    if (tiled) {
        if constexpr (std::is_same<VS, OneView>::value) {
            hipError_t e = raster_tiles<ST>(s, vs, ps, t, bins_clear, st);
            if (e != hipSuccess) return e;
            // every draw can be binned: the list holds only the few that are
            // too large for the bins; else any number beyond the bins
            direct = vs.v.bin_capacity >= std::min(vs.v.draw_capacity, s.total_meshlets);
        }
    }
    if (!tiled || !direct) {
        ps.direct = tiled ? 1u : 0u;
        mark(tiled ? "raster_direct_view" : KIND == 0 ? "raster_meshlets_view" : "raster_meshlets_shadow", st);
        hipLaunchKernelGGL((k_raster_meshlets<KIND, VS, ST>), dim3(blocks), dim3(64), 0, st, s, vs, ps);
        ps.direct = 0;
    }
    const bool alpha = !(s.flags & LH_SCENE_OPAQUE_ONLY);
    if (alpha) {
        mark(KIND == 0 ? "raster_alpha_view" : "raster_alpha_shadow", st);
        PassSet pa = ps;
        pa.medium_extent = alpha_extent;
        hipLaunchKernelGGL((k_raster_alpha<KIND, VS, ST>), dim3(blocks), dim3(64), 0, st, s, vs, pa);
    }
    ps.direct = direct ? 1u : 0u;
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
hipError_t launch_set(const lh_scene& s, const OneView& vs, const PassSet& ps, const RasterTuning& t, uint32_t bb,
                      int32_t alpha_extent, bool bins_clear, hipStream_t st) {
    if (vs.v.flags & LH_VIEW_STATISTICS) return launch_kernels<KIND, true>(s, vs, ps, t, bb, alpha_extent, bins_clear, st);
    return launch_kernels<KIND, false>(s, vs, ps, t, bb, alpha_extent, bins_clear, st);
}
template <int KIND>
hipError_t launch_set(const lh_scene& s, const ViewTable& vs, const PassSet& ps, const RasterTuning& t, uint32_t bb,
                      int32_t alpha_extent, bool bins_clear, hipStream_t st) {
    return launch_kernels<KIND, false>(s, vs, ps, t, bb, alpha_extent, bins_clear, st);
}

template <class VS>
hipError_t raster(const lh_scene& s, const VS& vs, uint32_t pass0, uint32_t npasses, const RasterTuning& t,
                  hipStream_t st, bool phase2, bool bins_clear) {
    if (npasses == 0 || npasses > LH_NUM_CASCADES || pass0 + npasses > LH_NUM_PASSES || (pass0 == 0 && npasses != 1))
        return hipErrorInvalidValue;
    // the cascades may take their own extents (their triangles are smaller
    // and their raster depth-only)
    const bool cascades = pass0 > 0;
    const uint32_t small_sel = cascades && t.shadow_small_extent_px ? t.shadow_small_extent_px : t.small_extent_px;
    const uint32_t medium_sel = cascades && t.shadow_medium_extent_px ? t.shadow_medium_extent_px : t.medium_extent_px;
    const uint32_t small_px = std::min<uint32_t>(std::max<uint32_t>(small_sel, 1), 32);
    // Short queues keep 16 px, 64 px in a batch, and alpha-clipped triangles the
    // same extent as others.
    bool short_q = t.short_queues;
    if constexpr (std::is_same<VS, OneView>::value) short_q = short_queues(vs.v);
    const uint32_t least_px = !short_q ? 1u : std::is_same<VS, OneView>::value ? 16u : 64u;
    const uint32_t medium_px = std::min<uint32_t>(std::max({medium_sel, small_px, least_px}), 64);
    const int32_t alpha_extent = int32_t(256 * (short_q ? medium_px : std::min(medium_px, kAlphaMediumPx)));
    PassSet ps{pass0, npasses, int32_t(medium_px * 256), phase2 ? 1u : 0u, 0u};
    const uint32_t nv = vs.count();
    // the per-view persistent grid of the queue kernel shrinks with the batch size
    const uint32_t big_blocks = nv > 1 ? std::max(t.big_blocks / 16, 32u) : t.big_blocks;
    if (pass0 == 0) return launch_set<0>(s, vs, ps, t, big_blocks, alpha_extent, bins_clear, st);
    return launch_set<1>(s, vs, ps, t, big_blocks, alpha_extent, bins_clear, st);
}

template hipError_t raster<OneView>(const lh_scene&, const OneView&, uint32_t, uint32_t, const RasterTuning&,
                                    hipStream_t, bool, bool);
template hipError_t raster<ViewTable>(const lh_scene&, const ViewTable&, uint32_t, uint32_t, const RasterTuning&,
                                      hipStream_t, bool, bool);

hipError_t plan_segments(const ViewTable& vt, uint32_t pass0, uint32_t npasses, hipStream_t st) {
    if (vt.n * npasses > LH_MAX_BATCH_SEGMENTS) return hipErrorInvalidValue;
    mark("plan_segments", st);
    hipLaunchKernelGGL(k_plan_segments, dim3(1), dim3(256), 0, st, vt, pass0, npasses);
    return hipGetLastError();
}

}  // namespace lhk
