// Device helpers shared by the raster kernels (raster.hip: per-meshlet raster
// with device-scope depth atomics; tile.hip: the LDS-binned screen-tile
// raster): the software restatement of the Vulkan rasterization rules, the
// render targets of a pass, the raster queues inside lh_view.scratch, and the
// flattened draw-index space of a launch.
#pragma once

#include <type_traits>

#include "kernels.h"
#include "lh_device.h"
#include "scratch.h"
#include "shading.h"

namespace lhr {

using namespace lhd;

constexpr float kGuard = 4.0f;
constexpr uint32_t kBadVertex = 64u;  // non-finite, or w <= 0 inside every plane

struct BigTri {
    int32_t X[3];
    int32_t Y[3];
    float z[3];
    uint32_t id;
    uint16_t xlo, ylo, xhi, yhi;  // xlo bits 13..15: pass index within the set; ylo bit 15: alpha clip
};
static_assert(sizeof(BigTri) == LH_BIG_ENTRY_BYTES, "big queue entry");

struct SV {
    int32_t X, Y;
    float z;
};

// One render target of a launch.
struct Pass {
    static constexpr int32_t kLanePx = 4;  // boxes up to this many pixels are walked by one lane
    uint32_t pass, W, H;
    uint64_t* vis;
    uint32_t* depth;
    const MeshletReference* draws;
};

// A launch rasterizes passes [pass0, pass0 + n) of every view of its source;
// the passes of one view share that view's queues, counted at
// LH_CNT_CLIP / LH_CNT_BIG + pass0.
struct PassSet {
    uint32_t pass0, n;
    int32_t medium_extent;  // subpixels: larger triangles go to the large-triangle queue (<= 64 px)
    uint32_t phase2;        // main view, second occlusion phase: draws from LH_CNT_HIZ_PHASE1 on
    uint32_t direct;        // single view: rasterize the draws the tiled raster left on its direct list
                            // (flattened index | kBinDirect when their queue triangles are queued already)
};

template <int KIND>
LH_DEV const LhMat4& view_matrix(const lh_view& v, uint32_t pass) {
    return KIND == 0 ? v.uniforms->combined_perspective_view : v.misc->shadow_matrices[pass - 1];
}

LH_DEV Pass make_pass(const lh_view& v, uint32_t pass) {
    Pass p;
    p.pass = pass;
    if (pass == 0) {
        p.W = v.width;
        p.H = v.height;
        p.vis = v.visbuffer;
        p.depth = nullptr;
    } else {
        p.W = p.H = v.shadow_size;
        p.vis = nullptr;
        p.depth = v.shadow_maps + size_t(pass - 1) * v.shadow_size * v.shadow_size;
    }
    p.draws = v.draws + size_t(pass) * v.draw_capacity;
    return p;
}

// Queue layout inside lh_view.scratch: clip entries {draw << 7 | triangle,
// pass index within the set | alpha clip << 31}, then (256-byte aligned) the
// big-triangle entries.
constexpr uint32_t kClipAlpha = 0x80000000u;
constexpr uint16_t kBigAlpha = 0x8000u;
struct Queues {
    uint2* clip;
    BigTri* big;
};
LH_DEV Queues queues(const lh_view& v) {
    const lhs::ScratchLayout L = lhs::scratch_layout(v);
    return {reinterpret_cast<uint2*>(static_cast<char*>(v.scratch) + L.clip),
            reinterpret_cast<BigTri*>(static_cast<char*>(v.scratch) + L.big)};
}

LH_DEV float plane_dist(f4 v, int k) {
    switch (k) {
        case 0: return v.w - v.z;
        case 1: return v.z;
        case 2: return kGuard * v.w - v.x;
        case 3: return kGuard * v.w + v.x;
        case 4: return kGuard * v.w - v.y;
        default: return kGuard * v.w + v.y;
    }
}
LH_DEV uint32_t outcode(f4 v) {
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < 6; k++)
        if (!(plane_dist(v, k) >= 0.0f)) c |= 1u << k;
    return c;
}
LH_DEV bool finite4(f4 v) { return isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w); }

LH_DEV bool project(f4 c, uint32_t W, uint32_t H, SV& o) {
    if (!(c.w > 0.0f)) return false;
    // x / 1 is x exactly: the orthographic cascades (w == 1 at every vertex)
    // skip the three correctly rounded divisions.
    float xn = c.x, yn = c.y, zn = c.z;
    if (c.w != 1.0f) {
        xn = c.x / c.w;
        yn = c.y / c.w;
        zn = c.z / c.w;
    }
    float hw = 0.5f * float(W), hh = 0.5f * float(H);
    float xf = xn * hw + hw, yf = yn * hh + hh;
    o.X = int32_t(rintf(xf * 256.0f));
    o.Y = int32_t(rintf(yf * 256.0f));
    o.z = zn;
    return true;
}

LH_DEV int64_t edge64(int32_t ax, int32_t ay, int32_t bx, int32_t by, int32_t px, int32_t py) {
    return int64_t(bx - ax) * int64_t(py - ay) - int64_t(by - ay) * int64_t(px - ax);
}
LH_DEV bool top_left(int32_t ax, int32_t ay, int32_t bx, int32_t by) {
    int32_t dx = bx - ax, dy = by - ay;
    return dy < 0 || (dy == 0 && dx > 0);
}

// Culls by facing (alpha-clip geometry is double-sided: only zero area is
// culled, src/pipelines.cpp:22-25), orients to positive area and computes the
// pixel bbox.  Every output is written on every path (the bbox first: it does
// not depend on the vertex order).
template <int KIND>
LH_DEV bool setup(SV& v0, SV& v1, SV& v2, uint32_t W, uint32_t H, int64_t& area, int32_t& xlo, int32_t& xhi,
                  int32_t& ylo, int32_t& yhi, int32_t& extx, int32_t& exty, bool two_sided = false,
                  bool* swapped = nullptr) {
    const int32_t minX = min(v0.X, min(v1.X, v2.X)), maxX = max(v0.X, max(v1.X, v2.X));
    const int32_t minY = min(v0.Y, min(v1.Y, v2.Y)), maxY = max(v0.Y, max(v1.Y, v2.Y));
    xlo = max((minX + 127) >> 8, 0);
    xhi = min((maxX - 128) >> 8, int32_t(W) - 1);
    ylo = max((minY + 127) >> 8, 0);
    yhi = min((maxY - 128) >> 8, int32_t(H) - 1);
    extx = maxX - minX;
    exty = maxY - minY;
    area = edge64(v0.X, v0.Y, v1.X, v1.Y, v2.X, v2.Y);
    if (swapped) *swapped = area < 0;
    if (two_sided ? area == 0 : (KIND == 0 ? area >= 0 : area <= 0)) return false;
    if (area < 0) {
        SV t = v1;
        v1 = v2;
        v2 = t;
        area = -area;
    }
    return xlo <= xhi && ylo <= yhi;
}

// Raster statistics (LH_VIEW_STATISTICS): covered samples and issued depth
// atomics per lane, wave-reduced into the view's counters.  Tally<false>
// compiles to nothing.
template <bool ON>
struct Tally {
    LH_DEV void hit(bool) {}
    LH_DEV void flush(const lh_view&, uint32_t) {}
    LH_DEV void move_to(Tally*, uint32_t) {}
};
template <>
struct Tally<true> {
    uint32_t frags = 0, atomics = 0;
    LH_DEV void hit(bool issued) {
        frags++;
        atomics += issued ? 1u : 0u;
    }
    // Called by the whole wave.
    LH_DEV void flush(const lh_view& v, uint32_t pass) {
        const uint32_t f = wave_sum_u32(frags), a = wave_sum_u32(atomics);
        if (lane_id() == 0 && f != 0) {
            atomicAdd(&v.counters[LH_CNT_FRAGMENTS + pass], f);
            atomicAdd(&v.counters[LH_CNT_ATOMICS + pass], a);
        }
        frags = atomics = 0;
    }
    // Adds the lane's counts to those of pass `pi` of sum[LH_NUM_CASCADES].
    LH_DEV void move_to(Tally* sum, uint32_t pi) {
#pragma unroll
        for (uint32_t q = 0; q < LH_NUM_CASCADES; q++)
            if (q == pi) sum[q].frags += frags, sum[q].atomics += atomics;
        frags = atomics = 0;
    }
};

// Depth test of one covered sample that `visible()` (the alpha test) lets
// pass.  Without EARLY the atomic is issued without reading the target first:
// in the meshlet raster a read-before-atomic early-out saves atomics but makes
// every sample wait for a load.  With EARLY the target is read first, and a
// sample that loses against what it holds costs neither an alpha test nor an
// atomic (the value read may be an old one, which is only larger).
template <int KIND, bool ST, bool EARLY, class F>
LH_DEV void fragment(const Pass& p, int32_t px, int32_t py, float z, uint32_t id, Tally<ST>& tally, F&& visible) {
    z = fminf(fmaxf(z, 0.0f), 1.0f);
    const size_t o = size_t(py) * p.W + uint32_t(px);
    if (KIND == 0) {
        const bool issue = z > 0.0f;  // depth GREATER against the 0.0 clear
        const unsigned long long key = ((unsigned long long)(~__float_as_uint(z)) << 32) | id;
        if (EARLY && (!issue || key >= p.vis[o])) return;
        if (!visible()) return;
        tally.hit(issue);
        if (issue) atomicMin(reinterpret_cast<unsigned long long*>(p.vis + o), key);
    } else {
        if (EARLY && __float_as_uint(z) >= p.depth[o]) return;
        if (!visible()) return;
        tally.hit(true);
        atomicMin(p.depth + o, __float_as_uint(z));
    }
}

LH_DEV int32_t readlane(int32_t v, uint32_t l) { return __builtin_amdgcn_readlane(v, int(l)); }
LH_DEV float readlane(float v, uint32_t l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), int(l))); }

LH_DEV void store_big(BigTri* q, const SV& v0, const SV& v1, const SV& v2, uint32_t id, int32_t xlo, int32_t xhi,
                      int32_t ylo, int32_t yhi, uint32_t pi, bool alpha) {
    BigTri b;
    b.X[0] = v0.X, b.X[1] = v1.X, b.X[2] = v2.X;
    b.Y[0] = v0.Y, b.Y[1] = v1.Y, b.Y[2] = v2.Y;
    b.z[0] = v0.z, b.z[1] = v1.z, b.z[2] = v2.z;
    b.id = id;
    b.xlo = uint16_t(uint32_t(xlo) | (pi << 13)), b.ylo = uint16_t(uint32_t(ylo) | (alpha ? kBigAlpha : 0u));
    b.xhi = uint16_t(xhi), b.yhi = uint16_t(yhi);
    uint4* dst = reinterpret_cast<uint4*>(q);
    const uint4* src = reinterpret_cast<const uint4*>(&b);
    dst[0] = src[0];
    dst[1] = src[1];
    dst[2] = src[2];
}

// Vertex fetch (load_vertex_data, src/shaders/rasterization.glsl:12-34, and
// calculate_world_pos, src/shaders/common/util.glsl:11-16).
LH_DEV uint32_t load_index(const MeshInfo& mi, uint32_t i) {
    if (mi.flags & MESH_INFO_FLAGS_32_BIT_INDICES) return ptr<uint32_t>(mi.indices)[i];
    return ptr<uint16_t>(mi.indices)[i];
}
LH_DEV f3 load_position(const MeshInfo& mi, uint32_t v) {
    if (mi.flags & MESH_INFO_FLAGS_FP32_VERTICES) {
        const float* q = ptr<float>(mi.positions) + 3 * size_t(v);
        return {q[0], q[1], q[2]};
    }
    const uint16_t* q = ptr<uint16_t>(mi.positions) + 3 * size_t(v);
    return {float(q[0]), float(q[1]), float(q[2])};
}

// Memory that no launch of the raster writes (instances, uniforms, cascade
// matrices, a batch's view table), read at wave-uniform addresses through the
// constant address space: scalar loads into scalar registers, instead of the
// vector loads that the compiler must choose in a kernel that also writes.
template <class T>
using ConstPtr = const __attribute__((address_space(4))) T*;
template <class T>
LH_DEV ConstPtr<T> const_ptr(uint64_t addr) {
    const uint32_t lo = uniform_u32(uint32_t(addr)), hi = uniform_u32(uint32_t(addr >> 32));
    return reinterpret_cast<ConstPtr<T>>(uint64_t(lo) | (uint64_t(hi) << 32));
}
LH_DEV LhMat4 load_mat4(uint64_t addr) {
    const ConstPtr<float> q = const_ptr<float>(addr);
    LhMat4 m;
#pragma unroll
    for (int c = 0; c < 4; c++) m.c[c] = LhVec4{q[4 * c], q[4 * c + 1], q[4 * c + 2], q[4 * c + 3]};
    return m;
}

// What a wave needs to know of a draw before it can fetch the meshlet's
// vertices: the end of the dependent chain draw -> instance -> mesh info ->
// meshlet.  A wave loads the heads of its next 64 draws together, one per
// lane, and then broadcasts them one at a time: the chain's four latencies
// are paid once per 64 draws instead of once per draw.
struct DrawHead {
    uint64_t positions, indices, micro;  // remap table and triangle corners: at the meshlet's first
    uint32_t instance, mid, info;        // info: triangles | vertices << 8 | MeshInfo.flags << 16
    LH_DEV uint32_t triangles() const { return info & 255u; }
    LH_DEV uint32_t vertices() const { return (info >> 8) & 255u; }
    LH_DEV bool has(uint32_t flag) const { return (info >> 16 & flag) != 0; }
};
LH_DEV DrawHead load_head(const lh_scene& s, MeshletReference ref) {
    const MeshInfo& mi = mesh_info_at(s.instances[ref.instance_index].mesh_info_address);
    const Meshlet& ml = ptr<Meshlet>(mi.meshlets)[ref.meshlet_index];
    DrawHead h;
    h.positions = mi.positions;
    h.indices = mi.indices + uint64_t(ml.index_offset) * ((mi.flags & MESH_INFO_FLAGS_32_BIT_INDICES) ? 4u : 2u);
    h.micro = mi.micro_indices + ml.triangle_offset;
    h.instance = ref.instance_index;
    h.mid = s.instance_meshlet_base[ref.instance_index] + ref.meshlet_index;
    h.info = uint32_t(ml.triangle_count) | uint32_t(ml.index_count) << 8 | uint32_t(mi.flags) << 16;
    return h;
}
LH_DEV uint32_t readlane_u32(uint32_t v, uint32_t l) { return uint32_t(__builtin_amdgcn_readlane(int(v), int(l))); }
LH_DEV uint64_t readlane_u64(uint64_t v, uint32_t l) {
    return uint64_t(readlane_u32(uint32_t(v), l)) | uint64_t(readlane_u32(uint32_t(v >> 32), l)) << 32;
}
LH_DEV DrawHead head_of_lane(const DrawHead& h, uint32_t l) {
    return {readlane_u64(h.positions, l), readlane_u64(h.indices, l), readlane_u64(h.micro, l),
            readlane_u32(h.instance, l),  readlane_u32(h.mid, l),     readlane_u32(h.info, l)};
}

// The vertex (one per lane) and corner (two triangles per lane) words of one
// meshlet, requested ahead of their use: the remap index and the corners
// first, the position once the index is there.
struct MeshletFetch {
    uint32_t vertex, corner[2];
    f3 pos;
    // Triangle t's three corner bytes come in one unaligned word: the three
    // bytes and the next triangle's first, or, for the last triangle (whose
    // word would end past the table), the byte before and the three.  A
    // single triangle is read byte by byte.
    LH_DEV void request(const DrawHead& h, uint32_t lane) {
        if (lane < h.vertices())
            vertex = h.has(MESH_INFO_FLAGS_32_BIT_INDICES) ? ptr<uint32_t>(h.indices)[lane]
                                                          : uint32_t(ptr<uint16_t>(h.indices)[lane]);
        const uint8_t* micro = ptr<uint8_t>(h.micro);
        const uint32_t ntri = h.triangles();
#pragma unroll
        for (uint32_t r = 0; r < 2; r++) {
            const uint32_t t = lane + 64 * r;
            corner[r] = 0;
            if (ntri == 1) {
                if (t == 0) corner[r] = uint32_t(micro[0]) | uint32_t(micro[1]) << 8 | uint32_t(micro[2]) << 16;
            } else if (t < ntri) {
                __builtin_memcpy(&corner[r], micro + (3 * t - (t + 1 == ntri ? 1u : 0u)), 4);
            }
        }
    }
    LH_DEV void request_position(const DrawHead& h, uint32_t lane) {
        if (lane >= h.vertices()) return;
        if (h.has(MESH_INFO_FLAGS_FP32_VERTICES)) {
            const float* q = ptr<float>(h.positions) + 3 * size_t(vertex);
            pos = {q[0], q[1], q[2]};
        } else {
            const uint16_t* q = ptr<uint16_t>(h.positions) + 3 * size_t(vertex);
            pos = {float(q[0]), float(q[1]), float(q[2])};
        }
    }
    // corners i0 | i1 << 8 | i2 << 16 of triangle lane + 64 r
    LH_DEV uint32_t corners(const DrawHead& h, uint32_t lane, uint32_t r) const {
        const uint32_t ntri = h.triangles();
        const uint32_t c = r == 0 ? corner[0] : corner[1];
        return (ntri > 1 && lane + 64 * r + 1 == ntri ? c >> 8 : c) & 0xFFFFFFu;
    }
};

// Orders a wave's own LDS accesses (one-wave blocks: no barrier, and no wait
// on the global loads that are in flight).
LH_DEV void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Snapped vertices of the meshlet in hand.
struct WaveVerts {
    int2 XY[64];
    float Z[64];
    uint32_t O[64];  // outcode, kBadVertex
};
// Transforms the wave's vertices into `sv`; returns whether every vertex is
// inside the clip volume (their outcodes are written only when one is not).
// Clipped and invalid vertices store zeros, so that the triangle setup may
// read any corner.
LH_DEV bool transform_vertices(const DrawHead& h, const MeshletFetch& f, const LhMat4& T, const LhMat4& M, uint32_t W,
                               uint32_t H, uint32_t lane, WaveVerts& wv, SV& sv) {
    const f3 w = mat4_point(T, f.pos);
    const f4 c = mat4_mul_vec4(M, f4{w.x, w.y, w.z, 1.0f});
    const bool live = lane < h.vertices();
    // Almost every meshlet lies inside the clip volume whole: one test of all
    // its planes, each with plane_dist's own outcome (a difference has the
    // sign of its comparison), without the outcodes.
    const float gw = kGuard * c.w;
    const bool in = fabsf(c.x) <= gw && fabsf(c.y) <= gw && c.z >= 0.0f && c.z <= c.w && c.w > 0.0f && gw < INFINITY;
    const bool clean = ballot(live && !in) == 0;  // wave-uniform
    if (clean) {
        project(c, W, H, sv);
    } else {
        uint32_t oc = finite4(c) ? outcode(c) : kBadVertex;
        sv = SV{0, 0, 0.0f};
        if (oc == 0 && !project(c, W, H, sv)) oc = kBadVertex;
        if (live) wv.O[lane] = oc;
    }
    if (live) {
        wv.XY[lane] = make_int2(sv.X, sv.Y);
        wv.Z[lane] = sv.z;
    }
    return clean;
}

// Class and box of one triangle per lane, from the wave's snapped vertices.
struct TriSetup {
    int2 a, b, c;
    int32_t xlo, ylo, xhi, yhi, extent;
    uint32_t i0, i1, i2;
    bool clip, inside, swapped;  // inside: faces the right way, covers a pixel centre's row and column
};
// Extents (subpixels) up to which the edge functions are evaluated in 32 bits:
// at 120 px a difference has 15 bits and a step 23, so that the 24-bit
// multiplier is exact, and an edge value within two pixels of the box stays
// below 2 x 30720 x 31232 < 2^31; the area stays below 2^30 (rcp_exact).
constexpr int32_t kNarrow = 120 * 256;
static_assert(int64_t(kNarrow) * kNarrow <= 1 << 30, "rcp_exact");
static_assert(2 * int64_t(kNarrow) * (kNarrow + 2 * 256) < int64_t(1) << 31, "edge values");
template <int KIND>
LH_DEV TriSetup triangle_setup(const WaveVerts& wv, uint32_t corners, bool live, bool clean, bool two_sided, uint32_t W,
                               uint32_t H) {
    TriSetup t;
    t.i0 = corners & 255u, t.i1 = (corners >> 8) & 255u, t.i2 = corners >> 16;
    t.a = wv.XY[t.i0], t.b = wv.XY[t.i1], t.c = wv.XY[t.i2];
    bool drawn = live, whole = true;
    if (!clean) {  // wave-uniform; the outcodes of most meshlets are all zero
        const uint32_t o0 = wv.O[t.i0], o1 = wv.O[t.i1], o2 = wv.O[t.i2];
        drawn = live && ((o0 | o1 | o2) & kBadVertex) == 0 && (o0 & o1 & o2) == 0;
        whole = (o0 | o1 | o2) == 0;
    }
    const int32_t minX = min(t.a.x, min(t.b.x, t.c.x)), maxX = max(t.a.x, max(t.b.x, t.c.x));
    const int32_t minY = min(t.a.y, min(t.b.y, t.c.y)), maxY = max(t.a.y, max(t.b.y, t.c.y));
    t.xlo = max((minX + 127) >> 8, 0);
    t.xhi = min((maxX - 128) >> 8, int32_t(W) - 1);
    t.ylo = max((minY + 127) >> 8, 0);
    t.yhi = min((maxY - 128) >> 8, int32_t(H) - 1);
    t.extent = max(maxX - minX, maxY - minY);
    t.clip = drawn && !whole;
    t.inside = drawn && whole && t.xlo <= t.xhi && t.ylo <= t.yhi;
    // Sign of the area.  Within kNarrow the products are exact on the 24-bit
    // multiplier; only a wave with a larger triangle that may be drawn takes
    // the 64-bit ones.
    bool neg, pos;
    if (ballot(t.inside && t.extent > kNarrow) == 0) {
        const int32_t area = __mul24(t.b.x - t.a.x, t.c.y - t.a.y) - __mul24(t.b.y - t.a.y, t.c.x - t.a.x);
        neg = area < 0, pos = area > 0;
    } else {
        const int64_t area = edge64(t.a.x, t.a.y, t.b.x, t.b.y, t.c.x, t.c.y);
        neg = area < 0, pos = area > 0;
    }
    t.swapped = neg;
    t.inside = t.inside && (two_sided ? neg || pos : KIND == 0 ? neg : pos);
    return t;
}

// Appends to the clip and large-triangle queues (wave-aggregated; called by
// the whole wave).
LH_DEV void queue_clip(const lh_view& v, uint32_t pass0, bool pred, uint32_t d, uint32_t t, uint32_t pi, bool alpha) {
    if (ballot(pred) == 0) return;
    const uint32_t slot = wave_append(&v.counters[LH_CNT_CLIP + pass0], pred);
    if (!pred) return;
    if (slot < v.clip_capacity)
        queues(v).clip[slot] = make_uint2((d << LH_KEY_TRI_BITS) | t, pi | (alpha ? kClipAlpha : 0u));
    else
        atomicOr(&v.counters[LH_CNT_OVERFLOW], LH_OVERFLOW_CLIP);
}
LH_DEV void store_big(BigTri* q, const WaveVerts& wv, const TriSetup& ts, uint32_t id, uint32_t pi, bool alpha) {
    const SV v0{ts.a.x, ts.a.y, wv.Z[ts.i0]}, v1{ts.b.x, ts.b.y, wv.Z[ts.i1]}, v2{ts.c.x, ts.c.y, wv.Z[ts.i2]};
    store_big(q, v0, ts.swapped ? v2 : v1, ts.swapped ? v1 : v2, id, ts.xlo, ts.xhi, ts.ylo, ts.yhi, pi, alpha);
}
// Returns whether the lane's triangle found the queue full.
LH_DEV bool queue_big(const lh_view& v, uint32_t pass0, bool pred, const WaveVerts& wv, const TriSetup& ts, uint32_t id,
                      uint32_t pi, bool alpha) {
    if (ballot(pred) == 0) return false;
    const uint32_t slot = wave_append(&v.counters[LH_CNT_BIG + pass0], pred);
    if (!pred) return false;
    if (slot >= v.big_capacity) return true;
    store_big(queues(v).big + slot, wv, ts, id, pi, alpha);
    return false;
}

// Triangles of up to kNarrow that are ready to be rasterized, collected over a
// wave's meshlets.  Most set-up triangles of a dense scene cover no pixel
// centre (4 of 64 do in the cascades of the 2,000-instance field), so the
// survivors of many rounds are put together here and rasterized 64 at a time
// instead of a few lanes per round.  An entry holds its box origin, the
// snapped vertices relative to the origin's pixel corner (16 bits each), the three depths and the key's id; triangles are
// oriented to positive area.  A round adds at most 64 entries to at most 63.
constexpr uint32_t kQueue = 128;
template <uint32_t N, class Own = int32_t>
struct TriQueueOf {
    uint4 box[N];     // xlo | ylo << 16, v0, v1, v2 (x & 0xFFFF | y << 16)
    uint4 att[N];     // z0, z1, z2, id
    Own own[64];      // owners of a pass's runs
    // a triangle of positive area; (xlo, ylo): first pixel of its clamped box
    LH_DEV void store(uint32_t k, int32_t xlo, int32_t ylo, const SV& v0, const SV& v1, const SV& v2, uint32_t id) {
        auto rel = [&](const SV& v) {
            return (uint32_t(v.X - xlo * 256) & 0xFFFFu) | uint32_t(v.Y - ylo * 256) << 16;
        };
        box[k] = make_uint4(uint32_t(xlo) | uint32_t(ylo) << 16, rel(v0), rel(v1), rel(v2));
        att[k] = make_uint4(__float_as_uint(v0.z), __float_as_uint(v1.z), __float_as_uint(v2.z), id);
    }
    LH_DEV void store(uint32_t k, const WaveVerts& wv, const TriSetup& ts, uint32_t id) {
        const SV v0{ts.a.x, ts.a.y, wv.Z[ts.i0]}, v1{ts.b.x, ts.b.y, wv.Z[ts.i1]}, v2{ts.c.x, ts.c.y, wv.Z[ts.i2]};
        store(k, ts.xlo, ts.ylo, v0, ts.swapped ? v2 : v1, ts.swapped ? v1 : v2, id);
    }
};
using TriQueue = TriQueueOf<kQueue>;

// shading::AlphaTri of up to 64 triangles, in LDS.
struct AlphaStore {
    float4 a[64], b[64], c[64], d[64], e[64];
    LH_DEV void store(uint32_t k, const shading::AlphaTri& t) {
        a[k] = make_float4(t.bary.invW.x, t.bary.invW.y, t.bary.invW.z, t.bary.n0.x);
        b[k] = make_float4(t.bary.n0.y, t.bary.ddx.x, t.bary.ddx.y, t.bary.ddx.z);
        c[k] = make_float4(t.bary.ddy.x, t.bary.ddy.y, t.bary.ddy.z, __uint_as_float(t.texture));
        d[k] = make_float4(t.uv[0].x, t.uv[0].y, t.uv[1].x, t.uv[1].y);
        e[k] = make_float4(t.uv[2].x, t.uv[2].y, t.offset.x, t.offset.y);
    }
    LH_DEV shading::AlphaTri load(uint32_t k) const {
        const float4 p = a[k], q = b[k], r = c[k], u = d[k], w = e[k];
        return {{{p.x, p.y, p.z}, {p.w, q.x}, {q.y, q.z, q.w}, {r.x, r.y, r.z}},
                {{u.x, u.y}, {u.z, u.w}, {w.x, w.y}},
                {w.z, w.w},
                __float_as_uint(r.w)};
    }
};
struct NoAlpha {};
LH_DEV int32_t lo16(uint32_t v) { return int32_t(int16_t(v & 0xFFFFu)); }
LH_DEV int32_t hi16(uint32_t v) { return int32_t(v) >> 16; }

// A queued triangle, coordinates relative to the corner of its box's first pixel.
struct QueuedTri {
    int32_t xlo, ylo, w, h;  // pixel box clamped to the target
    int32_t ax, ay, bx, by, cx, cy;
    float z0, d10, d20;
    uint32_t id;
    LH_DEV int32_t area() const { return __mul24(bx - ax, cy - ay) - __mul24(by - ay, cx - ax); }
};
template <class Q>
LH_DEV QueuedTri load_tri(const Q& q, uint32_t k, uint32_t W, uint32_t H) {
    const uint4 b = q.box[k], t = q.att[k];
    QueuedTri r;
    r.xlo = int32_t(b.x & 0xFFFFu), r.ylo = int32_t(b.x >> 16);
    r.ax = lo16(b.y), r.ay = hi16(b.y), r.bx = lo16(b.z), r.by = hi16(b.z), r.cx = lo16(b.w), r.cy = hi16(b.w);
    const int32_t maxX = max(r.ax, max(r.bx, r.cx)), maxY = max(r.ay, max(r.by, r.cy));
    r.w = min((maxX - 128) >> 8, int32_t(W) - 1 - r.xlo) + 1;
    r.h = min((maxY - 128) >> 8, int32_t(H) - 1 - r.ylo) + 1;
    r.z0 = __uint_as_float(t.x);
    r.d10 = __uint_as_float(t.y) - r.z0, r.d20 = __uint_as_float(t.z) - r.z0;
    r.id = t.w;
    return r;
}

// Edge functions of a queued triangle along one pixel row.  Every difference
// is within kNarrow, so the values are exact on the 24-bit multiplier and step
// exactly in integers: E_i(Px + 256) = E_i(Px) - 256 (Yb - Ya).  A pixel
// centre on an edge counts when the edge is a top or left one, so coverage
// (E > 0 || (E == 0 && top-left)) is E >= m with m = top-left ? 0 : 1.
struct RowEdges {
    int32_t e0, e1, e2, s0, s1, s2, m0, m1, m2;
    LH_DEV RowEdges(const QueuedTri& t, int32_t y) {
        const int32_t Py = y * 256 + 128, d0x = t.cx - t.bx, d0y = t.cy - t.by, d1x = t.ax - t.cx, d1y = t.ay - t.cy,
                      d2x = t.bx - t.ax, d2y = t.by - t.ay;
        e0 = __mul24(d0x, Py - t.by) - __mul24(d0y, 128 - t.bx);
        e1 = __mul24(d1x, Py - t.cy) - __mul24(d1y, 128 - t.cx);
        e2 = __mul24(d2x, Py - t.ay) - __mul24(d2y, 128 - t.ax);
        s0 = -d0y * 256, s1 = -d1y * 256, s2 = -d2y * 256;
        m0 = (d0y < 0 || (d0y == 0 && d0x > 0)) ? 0 : 1;
        m1 = (d1y < 0 || (d1y == 0 && d1x > 0)) ? 0 : 1;
        m2 = (d2y < 0 || (d2y == 0 && d2x > 0)) ? 0 : 1;
    }
};
// Narrows the covered columns [lo, hi] of a row by one edge, exactly: the
// quotient's estimate is within 1e-4 of (m - e) / s for the columns in
// question (0..120; others are clamped away), so the column it names or the
// next one inward is the edge's own, and one evaluation of the edge says which.
LH_DEV void clip_row(int32_t e, int32_t s, int32_t m, int32_t& lo, int32_t& hi) {
    const float q = float(m - e) * __builtin_amdgcn_rcpf(float(s));
    const float guess = s > 0 ? ceilf(q - 0.001f) : floorf(q + 0.001f);
    int32_t c = int32_t(fminf(fmaxf(guess, -1.0f), 121.0f));
    const int32_t miss = e + __mul24(c, s) < m ? 1 : 0;
    if (s > 0)
        lo = max(lo, c + miss);
    else if (s < 0)
        hi = min(hi, c - miss);
    else if (miss)  // the edge is horizontal: e itself, every column or none
        hi = -1;
}

// Depth test of the pixel at (x, y) of a queued triangle's box: in the pass's
// render target, or in another one that has its own test (a tile in LDS).
template <int KIND, bool ST, bool EARLY, class P, class F>
LH_DEV void raster_pixel(const P& p, const QueuedTri& t, float inv_area, int32_t e1, int32_t e2, int32_t x, int32_t y,
                         Tally<ST>& tally, F&& visible) {
    const int32_t px = t.xlo + x, py = t.ylo + y;
    const float l1 = float(e1) * inv_area, l2 = float(e2) * inv_area;
    const float z = (t.z0 + l1 * t.d10) + l2 * t.d20;
    if constexpr (std::is_same<P, Pass>::value)
        fragment<KIND, ST, EARLY>(p, px, py, z, t.id, tally, [&] { return visible(px, py); });
    else
        tally.hit(p.put(px, py, z, t.id));
}

// Numbers the `n` pieces of work of each lane in lane order and hands them out
// 64 at a time: f(owner lane, piece of that owner, active).  All lanes call f
// (the owners' registers are read across lanes).  A lane finds the owner of
// its piece as the last lane whose first piece is at or before it: first
// pieces are marked in LDS, and a running maximum spreads the marks.
template <class Own, class F>
LH_DEV void wave_spread(Own* own, uint32_t lane, uint32_t n, F&& f) {
    const uint32_t incl = wave_scan_add(n), excl = incl - n;
    const uint32_t total = readlane_u32(incl, 63);
    int32_t carry = 0;
    for (uint32_t base = 0; base < total; base += 64) {
        own[lane] = -1;
        lds_order();
        if (n && excl - base < 64u) own[excl - base] = Own(lane);  // excl >= base, unsigned
        lds_order();
        const int32_t o = max(wave_scan_max(int32_t(own[lane])), carry);
        lds_order();
        carry = __builtin_amdgcn_readlane(o, 63);
        const uint32_t k = base + lane;
        f(o, k - uint32_t(__shfl(int32_t(excl), o, 64)), k < total);
    }
}

// Part `part` of 2^lg equal parts of a triangle: rows (or runs of pixels) dealt
// out one by one.
struct Share {
    uint32_t part = 0, lg = 0;
    LH_DEV uint32_t count(uint32_t rows) const { return (rows + ((1u << lg) - 1u) - part) >> lg; }
    LH_DEV uint32_t nth(uint32_t k) const { return (k << lg) + part; }
    LH_DEV int32_t first(uint32_t k, uint32_t run) const { return int32_t(k + part * run); }
};
// log2 of the waves that share each of n triangles: all of `waves` are busy
// anyway and hold no more than `each` triangles then, or no more than `few`
// are busy (505x210, some 2,000 triangles of 8 px and more: 16.8 us shared by
// all 16,384 waves, 10.9 at 2,048, each of the others' cost being its fixed
// part; alpha-clipped samples are dearer: 1,500 cards of 60 and 150 px at
// 1920x1080 318 and 995 us a frame at 2,048, 278 and 652 at 4,096, 286 and 651
// at 8,192, where 4,000 of 20 px go from 289 to 308).
constexpr uint32_t kShareWaves = 2048, kShareWavesAlpha = 4096;
LH_DEV uint32_t share_out(uint32_t n, uint32_t waves, uint32_t each, uint32_t few, uint32_t most) {
    const uint32_t limit = n >= waves ? waves * each : few;
    uint32_t lg = 0;
    while (lg < most && (n << (lg + 1)) <= limit && waves >> (lg + 1)) lg++;
    return lg;
}

// Rasterizes entries [from, from + n) of the queue, n <= 64, one per lane.
// Boxes of up to P::kLanePx pixels (most of a dense scene's) are walked by their
// own lane.  The others are spread over the wave twice: first their rows, one
// per lane, each cut to the columns that the triangle covers (exactly, so no
// pixel is tested again); then the rows' covered pixels, one per lane.  So the
// cost follows the covered pixels, not the boxes: a sliver across a 120 px box
// costs its rows and the few pixels on each.  Against boxes walked in runs of
// four with the edges tested at each pixel: the main views of 12 cameras 2.77
// -> 1.96 ms, the alpha-clipped 720p view 1.12 -> 0.56 ms.
template <int KIND, bool ST, bool ALPHA, bool EARLY, class P, class Q, class A>
LH_DEV void raster_queue(const lh_scene& s, const LhMat4& M, const P& p, Q& q, A& alpha, uint32_t from, uint32_t n,
                         uint32_t lane, Tally<ST>& tally, Share share = {}) {
    lds_order();
    uint32_t rows = 0;
    float inv_area = 0.0f;
    if (lane < n) {
        const QueuedTri t = load_tri(q, from + lane, p.W, p.H);
        inv_area = rcp_exact(float(t.area()));
        if constexpr (ALPHA) alpha.store(lane, shading::alpha_setup(s, M, t.id));
        if (!ALPHA && share.lg == 0 && __mul24(t.w, t.h) <= P::kLanePx) {
            for (int32_t y = 0; y < t.h; y++) {
                RowEdges r(t, y);
                for (int32_t x = 0; x < t.w; x++) {
                    if (r.e0 >= r.m0 && r.e1 >= r.m1 && r.e2 >= r.m2)
                        raster_pixel<KIND, ST, EARLY>(p, t, inv_area, r.e1, r.e2, x, y, tally,
                                                      [](int32_t, int32_t) { return true; });
                    r.e0 += r.s0, r.e1 += r.s1, r.e2 += r.s2;
                }
            }
        } else {
            rows = share.count(uint32_t(t.h));
        }
    }
    wave_spread(q.own, lane, rows, [&](int32_t o, uint32_t k, bool active) {
        const uint32_t y = share.nth(k);
        uint32_t columns = 0, row = 0;  // row: first column | y << 8 | triangle << 16
        if (active) {
            const QueuedTri t = load_tri(q, from + uint32_t(o), p.W, p.H);
            const RowEdges r(t, int32_t(y));
            int32_t lo = 0, hi = t.w - 1;
            clip_row(r.e0, r.s0, r.m0, lo, hi);
            clip_row(r.e1, r.s1, r.m1, lo, hi);
            clip_row(r.e2, r.s2, r.m2, lo, hi);
            if (hi >= lo) {
                columns = uint32_t(hi - lo + 1);
                row = uint32_t(lo) | y << 8 | uint32_t(o) << 16;
            }
        }
        wave_spread(q.own, lane, columns, [&](int32_t ro, uint32_t k, bool on) {
            const uint32_t rw = uint32_t(__shfl(int32_t(row), ro, 64));
            const uint32_t to = rw >> 16;
            const float inv = __shfl(inv_area, int32_t(to), 64);
            if (on) {
                const QueuedTri t = load_tri(q, from + to, p.W, p.H);
                const int32_t ry = int32_t(rw >> 8 & 255u), x = int32_t((rw & 255u) + k);
                const RowEdges r(t, ry);
                raster_pixel<KIND, ST, EARLY>(p, t, inv, r.e1 + __mul24(x, r.s1), r.e2 + __mul24(x, r.s2), x, ry, tally,
                                              [&](int32_t px, int32_t py) {
                                                  if constexpr (ALPHA)
                                                      return shading::alpha_at(s, alpha.load(to), p.W, p.H, px, py);
                                                  else
                                                      return true;
                                              });
            }
        });
    });
}

// Segment lookup of a flattened draw index g.  One view: the segments are the
// passes of the set, offsets computed from the view's counters.  A batch: the
// segments are (view, pass) pairs, offsets planned on the device beforehand.
template <class VS>
struct Segments;

template <>
struct Segments<OneView> {
    // off[i]: first flattened index of pass i; only constant indices, so the
    // array lives in registers.
    uint32_t off[LH_NUM_CASCADES + 1];
    uint32_t first;  // draws before this index were rasterized by an earlier phase
    LH_DEV Segments(const OneView& vs, const PassSet& ps) {
        const lh_view& v = vs.v;
        first = ps.phase2 ? min(v.counters[LH_CNT_HIZ_PHASE1], v.draw_capacity) : 0u;
        off[0] = 0;
#pragma unroll
        for (uint32_t i = 0; i < LH_NUM_CASCADES; i++)
            off[i + 1] = off[i] + (i < ps.n ? min(v.counters[LH_CNT_DRAWS + ps.pass0 + i], v.draw_capacity) : 0u);
        if (ps.phase2) {  // one pass: [first, count) of the main view's draws
#pragma unroll
            for (uint32_t i = 1; i <= LH_NUM_CASCADES; i++) off[i] = off[i] > first ? off[i] - first : 0u;
        }
    }
    LH_DEV uint32_t total() const { return off[LH_NUM_CASCADES]; }
    // Flattened index of a block's k-th draw: a plain grid stride.
    LH_DEV uint32_t draw(uint32_t k) const { return blockIdx.x + k * gridDim.x; }
    LH_DEV void find(uint32_t g, uint32_t& view, uint32_t& pi, uint32_t& d) const {
        // the last pass whose range starts at or before g (empty passes are skipped)
        uint32_t base = 0;
        pi = 0;
#pragma unroll
        for (uint32_t i = 1; i < LH_NUM_CASCADES; i++)
            if (g >= off[i]) {
                pi = i;
                base = off[i];
            }
        view = 0;
        d = g - base + first;  // first is 0 unless this is the main view's second phase
    }
};

template <>
struct Segments<ViewTable> {
    const uint32_t* off;
    uint32_t nseg, np;
    LH_DEV Segments(const ViewTable& vs, const PassSet& ps) : off(vs.seg_offsets), nseg(vs.n * ps.n), np(ps.n) {}
    LH_DEV uint32_t total() const { return off[nseg]; }
    // A block takes runs of 8 consecutive draws, which mostly share their view
    // and pass (a change of either flushes the block's triangle queue).
    LH_DEV uint32_t draw(uint32_t k) const { return (blockIdx.x + (k >> 3) * gridDim.x) * 8 + (k & 7); }
    LH_DEV void find(uint32_t g, uint32_t& view, uint32_t& pi, uint32_t& d) const {
        uint32_t lo = 0, hi = nseg;  // last k with off[k] <= g
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (off[mid] <= g)
                lo = mid;
            else
                hi = mid;
        }
        view = lo / np;
        pi = lo % np;
        d = g - off[lo];
    }
};

}  // namespace lhr

namespace lhk {
// LDS-binned tiled raster of the main view (tile.hip): binning, fill and the
// tile kernel; the caller's launches then draw the direct list
// (PassSet::direct) and the queues.  bins_clear: the view's meshlet cull zeroed the tile counts.
template <bool ST>
hipError_t raster_tiles(const lh_scene& s, const lhd::OneView& vs, const lhr::PassSet& ps, const RasterTuning& t,
                        bool bins_clear, hipStream_t st);
}  // namespace lhk
