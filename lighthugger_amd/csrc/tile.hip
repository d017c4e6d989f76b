// Tiled visibility-buffer raster of the main view (LDS-binned 64x64 screen
// tiles).  Same coverage and depth rules as the per-meshlet raster
// (raster.h; the reference's visbuffer_opaque_vertex/pixel,
// src/shaders/rasterization.glsl:38-58, with the pipeline state of
// src/pipelines.cpp:10-77), so the keys are identical; what changes is where
// the depth test happens: in LDS, one 64x64 tile of 64-bit keys per work item,
// and each pixel of a tile reaches the visibility buffer once per item (a
// plain store when the item is the tile's only one), instead of one
// device-scope atomicMin per covered sample.
//
// Launches of one main-view raster (single view):
//   k_bin_meshlets  one wave per surviving meshlet (the first bin_capacity):
//                   vertices fetched, transformed and snapped once; the snapped
//                   vertices and the front-facing, unclipped triangles (oriented,
//                   compacted) go to the bin cache, the tile rectangle of their
//                   pixel bounding boxes to the bin header; clip-crossing
//                   triangles to the clip queue and triangles over the medium
//                   extent to the large-triangle queue, as in the per-meshlet
//                   raster.  The meshlet's tiles are counted; draws that
//                   cannot be binned (over bin_capacity, too many tiles) go to
//                   the direct list.
//   k_bin_fill      tile offsets, work items of at most `item_entries` entries
//                   per tile, and the (draw, part) entries.
//   k_tile_raster   persistent blocks of 8 waves over the items: LDS tile
//                   cleared, each wave rasterizes one binned meshlet at a time
//                   (two when their triangles fit one round) from the cache
//                   (ds_min_u64 per covered sample), then the tile's covered
//                   pixels are written out.
// The direct list is then drawn by the large-triangle launch (or, when the
// caller's bin_capacity is below its draw capacity, by the per-meshlet raster),
// followed by the alpha-clip launches (all device-scope atomicMin on top of
// what the tiles wrote).
#include "raster.h"

using namespace lhd;
using namespace lhr;
using lhs::BinCache;
using lhs::BinHeader;
using lhs::ScratchLayout;
using lhs::TileItem;

namespace {

constexpr uint32_t kTile = LH_TILE_SIDE;
constexpr uint32_t kTileWaves = 8;
constexpr uint32_t kTileThreads = 64 * kTileWaves;

struct Bins {
    BinHeader* hdr;
    BinCache* cache;
    uint32_t* tile_count;
    uint32_t* tile_cursor;
    TileItem* items;
    uint32_t* entries;
    uint32_t* direct;
    ScratchLayout L;
};
LH_DEV Bins bins(const lh_view& v) {
    const ScratchLayout L = lhs::scratch_layout(v);
    char* b = static_cast<char*>(v.scratch);
    return {reinterpret_cast<BinHeader*>(b + L.hdr),
            reinterpret_cast<BinCache*>(b + L.cache),
            reinterpret_cast<uint32_t*>(b + L.tile_count),
            reinterpret_cast<uint32_t*>(b + L.tile_cursor),
            reinterpret_cast<TileItem*>(b + L.items),
            reinterpret_cast<uint32_t*>(b + L.entries),
            reinterpret_cast<uint32_t*>(b + L.direct),
            L};
}

// Word of tile t in the count and cursor arrays.  Device atomics to one cache
// line serialize as those to one word do, and the busy tiles of a view are
// neighbours (the horizon's row): consecutive tiles lie in different 64-byte
// lines.  (Binning the 20,000-instance field at 4K: 1.71 ms with the tiles in
// order.)  The arrays end on a 256-byte boundary, so the last line is whole.
LH_DEV uint32_t tile_word(uint32_t t, uint32_t tiles) {
    const uint32_t lines = (tiles + 15) / 16;
    return (t % lines) * 16 + t / lines;
}

// Draws [0, n) of the launch binned by k_bin_meshlets.
LH_DEV uint32_t binned_draws(const Segments<OneView>& seg, const lh_view& v) { return min(seg.total(), v.bin_capacity); }

// ---------------------------------------------------------------- binning

// Zeroes the tile counts and cursors and the counters of a main-view raster
// that does not follow a meshlet cull which has done so (kClearBins).
__global__ void __launch_bounds__(256) k_bin_reset(OneView vs) {
    const Bins B = bins(vs.v);
    for (uint32_t t = blockIdx.x * 256 + threadIdx.x; t < lhs::tile_words(B.L.tiles); t += gridDim.x * 256)
        B.tile_count[t] = B.tile_cursor[t] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        vs.v.counters[LH_CNT_TILE_DIRECT] = 0;
        vs.v.counters[LH_CNT_TILE_ITEMS] = 0;
    }
}

// Occupancy (waves per SIMD), grid (two rounds of what is resident) and the
// fewest draws per wave of the binning.  Bound by VALU issue (about 400
// instructions a meshlet) and, with many large triangles, by the appends to
// their queue.  500 k meshlets of the 20,000-instance field at 4K: 446 us one
// draw at a time plus 15 for a launch that counted the tiles; 359, 311, 296 us
// on 7,168, 14,336, 28,672 blocks at 7 waves, 330 at 6, 363 at 8.  The 1080p
// field (59 k): 60 + 8 -> 53 us; 56 and 60 with at least 8 and 12 draws.
#define LH_BIN_WAVES 7
constexpr uint32_t kBinBlocks = 14336;
constexpr uint32_t kBinShare = 2;

// One wave per draw g < min(total, bin_capacity); later draws go to the direct
// list.  Alpha-clip meshlets are left to the alpha-clip raster (header with no
// triangles).  The heads of a wave's next 64 draws are loaded together, and a
// meshlet's vertices requested while the one before is in hand (as in the
// meshlet raster).  A wave's draws are consecutive, so that they share most of
// their tiles, and it adds their counts to the tiles' together: one atomic per
// distinct tile (one per meshlet and tile took the binning of the 1080p field
// from 55 to 82 us: same-address atomics serialize).
template <int KIND>
__global__ void __launch_bounds__(64) LH_WAVES_ATTR(LH_BIN_WAVES) k_bin_meshlets(lh_scene s, OneView vs, PassSet ps) {
    __shared__ WaveVerts wv;
    const uint32_t lane = threadIdx.x;
    const lh_view& v = vs.v;
    const Segments<OneView> seg(vs, ps);
    const uint32_t all = seg.total(), total = binned_draws(seg, v);
    const Bins B = bins(v);
    const Pass p = make_pass(v, ps.pass0);
    const LhMat4 M = load_mat4(reinterpret_cast<uint64_t>(&view_matrix<KIND>(v, p.pass)));
    for (uint32_t g0 = total + blockIdx.x * 64; g0 < all; g0 += gridDim.x * 64) {
        const uint32_t slot = wave_append(&v.counters[LH_CNT_TILE_DIRECT], g0 + lane < all);
        if (g0 + lane < all && slot < B.L.direct_capacity) B.direct[slot] = g0 + lane;
    }
    const uint32_t share = max((total + gridDim.x - 1) / gridDim.x, kBinShare), last = min((blockIdx.x + 1) * share, total);
    for (uint32_t k0 = blockIdx.x * share; k0 < last; k0 += 64) {
        const uint32_t my_g = k0 + lane;
        DrawHead head{};
        uint32_t my_d = 0, my_rect = 0, my_tiles = 0, my_parts = 0;
        if (my_g < last) {
            uint32_t view, pi;
            seg.find(my_g, view, pi, my_d);
            head = load_head(s, p.draws[my_d]);
            if (head.has(MESH_INFO_FLAGS_ALPHA_CLIP)) B.hdr[my_g] = BinHeader{0u, 0u, head.mid, 0u};
        }
        uint64_t todo = ballot(my_g < last && !head.has(MESH_INFO_FLAGS_ALPHA_CLIP));
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
            if (todo) {
                h = head_of_lane(head, first_lane(todo));
                next.request(h, lane);
            }
            const uint32_t g = k0 + l, d = readlane_u32(my_d, l);
            const LhMat4 T = load_mat4(reinterpret_cast<uint64_t>(&s.instances[cur.instance].transform));
            SV sv;
            lds_order();
            const bool clean = transform_vertices(cur, f, T, M, p.W, p.H, lane, wv, sv);
            lds_order();
            BinCache& c = B.cache[g];
            if (lane < cur.vertices()) {
                c.X[lane] = sv.X;
                c.Y[lane] = sv.Y;
                c.Z[lane] = sv.z;
            }
            if (todo) next.request_position(h, lane);
            const uint32_t ntri = cur.triangles();
            int32_t xlo_m = 0x7FFFFFFF, ylo_m = 0x7FFFFFFF, xhi_m = -1, yhi_m = -1;
            uint32_t nfront = 0, work = 0;  // work: pixels of the front triangles' boxes
            for (uint32_t round = 0; round * 64 < ntri; round++) {
                const uint32_t t = lane + 64 * round;
                const TriSetup ts = triangle_setup<KIND>(wv, f.corners(cur, lane, round), t < ntri, clean, false, p.W, p.H);
                if (!clean) queue_clip(v, ps.pass0, ts.clip, d, t, 0, false);
                // triangles over the medium extent: spread over many blocks by the large-triangle raster
                const bool big = ts.inside && ts.extent > ps.medium_extent, front = ts.inside && !big;
                queue_big(v, ps.pass0, big, wv, ts, (cur.mid << LH_KEY_TRI_BITS) | t, 0, false);
                const uint64_t fm = ballot(front);
                if (front) {
                    xlo_m = min(xlo_m, ts.xlo), ylo_m = min(ylo_m, ts.ylo);
                    xhi_m = max(xhi_m, ts.xhi), yhi_m = max(yhi_m, ts.yhi);
                    work += uint32_t(__mul24(ts.xhi - ts.xlo + 1, ts.yhi - ts.ylo + 1));
                    const uint32_t b = ts.swapped ? ts.i2 : ts.i1, e = ts.swapped ? ts.i1 : ts.i2;
                    c.tri[nfront + lanes_below(fm)] = ts.i0 | (b << 8) | (e << 16) | (t << 24);
                }
                nfront += uint32_t(__popcll(fm));
            }
            if (nfront == 0) {  // wave-uniform
                if (lane == 0) B.hdr[g] = BinHeader{0u, 0u, cur.mid, 0u};
                continue;
            }
            const uint32_t x0 = wave_min_u32(uint32_t(xlo_m)) >> lhs::kTileShift, y0 = wave_min_u32(uint32_t(ylo_m)) >> lhs::kTileShift;
            const uint32_t x1 = (wave_max_u32(uint32_t(xhi_m + 1)) - 1) >> lhs::kTileShift,
                           y1 = (wave_max_u32(uint32_t(yhi_m + 1)) - 1) >> lhs::kTileShift;
            const uint32_t total_work = wave_sum_u32(work);
            // a meshlet with much pixel work is split by triangle range into 2^lp parts, each its own
            // entry (so its work spreads over several waves), within LH_TILE_MAX_RECT entries in all
            const uint32_t nx = x1 - x0 + 1, tiles = nx * (y1 - y0 + 1);
            uint32_t lp = 0;
            while (lp < lhs::kMaxPartsLog2 && (total_work >> (lhs::kPartWorkLog2 + lp)) != 0 &&
                   (tiles << (lp + 1)) <= LH_TILE_MAX_RECT && (nfront >> (lp + 1)) >= 8)
                lp++;
            // too many tiles: left to the per-meshlet path
            const bool direct = tiles > LH_TILE_MAX_RECT;
            const uint32_t rect = x0 | (y0 << 8) | (x1 << 16) | (y1 << 24);
            if (lane == l) my_rect = rect, my_tiles = direct ? 0u : tiles, my_parts = 1u << lp;
            if (lane == 0) {
                B.hdr[g] = BinHeader{rect, nfront | (lp << lhs::kPartShift) | (direct ? lhs::kBinDirect : 0u), cur.mid, 0u};
                if (direct) {
                    const uint32_t slot = atomicAdd(&v.counters[LH_CNT_TILE_DIRECT], 1u);
                    if (slot < B.L.direct_capacity) B.direct[slot] = g | lhs::kBinDirect;
                }
            }
        }
        // the i-th tiles of all the wave's meshlets, merged
        uint32_t tx = my_rect & 255u, ty = (my_rect >> 8) & 255u;
        for (uint32_t i = 0, most = wave_max_u32(my_tiles); i < most; i++) {
            const uint32_t tile = ty * B.L.tiles_x + tx;
            for (uint64_t left = ballot(i < my_tiles); left;) {
                const uint32_t t = readlane_u32(tile, first_lane(left));
                const bool mine = i < my_tiles && tile == t;
                const uint32_t n = wave_sum_u32(mine ? my_parts : 0u);
                if (lane == 0) atomicAdd(&B.tile_count[tile_word(t, B.L.tiles)], n);
                left &= ~ballot(mine);
            }
            if (++tx > ((my_rect >> 16) & 255u)) tx = my_rect & 255u, ty++;
        }
    }
}

LH_DEV void for_each_tile(uint32_t rect, uint32_t tiles_x, auto&& f) {
    const uint32_t tx0 = rect & 255u, ty0 = (rect >> 8) & 255u, tx1 = (rect >> 16) & 255u, ty1 = rect >> 24;
    for (uint32_t ty = ty0; ty <= ty1; ty++)
        for (uint32_t tx = tx0; tx <= tx1; tx++) f(ty * tiles_x + tx);
}

// The entry lists and the work items.  Every block scans the tile counts into
// entry and item offsets by itself (a few loads per thread, from the L2)
// instead of waiting for a launch that would; the items, runs of at most
// `item_entries` entries per tile, are shared out over the blocks tile by
// tile.  Then one thread per binned draw puts its entries at the tiles'
// cursors: per run of kBinThreads draws a block counts its entries per tile in
// LDS, reserves each tile's range with one device atomic, and hands out the
// slots in LDS (same-address device atomics serialize).  In views of more than
// kHistTiles tiles the offsets fill the LDS: block 0 writes the items and every
// slot comes from the device cursor.
constexpr uint32_t kBinThreads = 256;
constexpr uint32_t kHistTiles = 8192;
constexpr uint32_t kMaxTiles = (LH_MAX_VIEW_SIDE / LH_TILE_SIDE) * (LH_MAX_VIEW_SIDE / LH_TILE_SIDE);
static_assert(kMaxTiles <= 2 * kHistTiles, "the offsets of the largest view fit the shared array");
__global__ void __launch_bounds__(kBinThreads) k_bin_fill(OneView vs, PassSet ps, uint32_t item_entries) {
    __shared__ uint32_t shared[2 * kHistTiles];
    __shared__ uint32_t wsum[2][kBinThreads / 64];
    const lh_view& v = vs.v;
    const Segments<OneView> seg(vs, ps);
    const uint32_t nb = binned_draws(seg, v);
    const Bins B = bins(v);
    const uint32_t tiles = B.L.tiles, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const bool wide = tiles > kHistTiles;
    uint32_t *off = shared, *item_off = shared + kHistTiles, *cnt = shared + kHistTiles;
    auto items_of = [&](uint32_t c) { return (c + item_entries - 1) / item_entries; };
    auto put_item = [&](uint32_t t, uint32_t at, uint32_t c, uint32_t item, uint32_t j) {
        if (item + j >= B.L.item_capacity) return;
        const uint32_t b = at + j * item_entries, e = min(b + item_entries, at + c);
        B.items[item + j] = TileItem{t, b, e | (c <= item_entries ? lhs::kItemOnly : 0u)};
    };
    {
        const uint32_t per = (tiles + kBinThreads - 1) / kBinThreads, t0 = threadIdx.x * per, t1 = min(t0 + per, tiles);
        uint32_t n = 0, ni = 0;
        for (uint32_t t = t0; t < t1; t++) {
            const uint32_t c = B.tile_count[tile_word(t, tiles)];
            n += c;
            ni += items_of(c);
        }
        const uint32_t in = wave_scan_add(n), ii = wave_scan_add(ni);
        if (lane == 63) {
            wsum[0][wave] = in;
            wsum[1][wave] = ii;
        }
        __syncthreads();
        uint32_t at = in - n, item = ii - ni;
        for (uint32_t w = 0; w < wave; w++) {
            at += wsum[0][w];
            item += wsum[1][w];
        }
        for (uint32_t t = t0; t < t1; t++) {
            const uint32_t c = B.tile_count[tile_word(t, tiles)];
            off[t] = at;
            if (!wide)
                item_off[t] = item;
            else if (blockIdx.x == 0)
                for (uint32_t j = 0; j < items_of(c); j++) put_item(t, at, c, item, j);
            at += c;
            item += items_of(c);
        }
        if (blockIdx.x == 0 && threadIdx.x == kBinThreads - 1) {
            v.counters[LH_CNT_TILE_ITEMS] = min(item, B.L.item_capacity);
            v.counters[LH_CNT_TILE_NEXT] = 0;  // the tile raster's work queue starts empty
        }
        __syncthreads();
        if (!wide)
            for (uint32_t t = blockIdx.x * (kBinThreads / 64) + wave; t < tiles; t += gridDim.x * (kBinThreads / 64)) {
                const uint32_t c = B.tile_count[tile_word(t, tiles)];
                for (uint32_t j = lane; j < items_of(c); j += 64) put_item(t, off[t], c, item_off[t], j);
            }
        __syncthreads();  // item_off becomes cnt
    }
    auto binned = [&](uint32_t g, uint32_t& rect, uint32_t& parts) {
        if (g >= nb) return false;
        const BinHeader h = B.hdr[g];
        rect = h.rect;
        parts = 1u << lhs::parts_log2(h.ntri);
        return h.ntri != 0 && (h.ntri & lhs::kBinDirect) == 0;
    };
    auto put = [&](uint32_t at, uint32_t g, uint32_t parts) {
        for (uint32_t q = 0; q < parts; q++)
            if (at + q < B.L.entry_capacity) B.entries[at + q] = g | (q << lhs::kEntryPartShift);
    };
    if (wide) {
        for (uint32_t g = blockIdx.x * kBinThreads + threadIdx.x; g < nb; g += gridDim.x * kBinThreads) {
            uint32_t rect, parts;
            if (binned(g, rect, parts))
                for_each_tile(rect, B.L.tiles_x,
                              [&](uint32_t t) { put(off[t] + atomicAdd(&B.tile_cursor[tile_word(t, tiles)], parts), g, parts); });
        }
        return;
    }
    for (uint32_t c0 = blockIdx.x * kBinThreads; c0 < nb; c0 += gridDim.x * kBinThreads) {
        for (uint32_t t = threadIdx.x; t < tiles; t += kBinThreads) cnt[t] = 0;
        __syncthreads();
        uint32_t rect = 0, parts = 0;
        const uint32_t g = c0 + threadIdx.x;
        const bool mine = binned(g, rect, parts);
        if (mine) for_each_tile(rect, B.L.tiles_x, [&](uint32_t t) { atomicAdd(&cnt[t], parts); });
        __syncthreads();
        for (uint32_t t = threadIdx.x; t < tiles; t += kBinThreads)
            if (cnt[t]) cnt[t] = off[t] + atomicAdd(&B.tile_cursor[tile_word(t, tiles)], cnt[t]);
        __syncthreads();
        if (mine) for_each_tile(rect, B.L.tiles_x, [&](uint32_t t) { put(atomicAdd(&cnt[t], parts), g, parts); });
        __syncthreads();
    }
}

// ---------------------------------------------------------------- tile raster

// LDS slot of pixel (lx, ly) of the tile.  A row of 64 keys spans the LDS
// banks twice, so every row starts on the same bank; the column is XORed
// with the row so that the rows of a box handed to one wave spread over them.
LH_DEV int32_t tile_slot(int32_t lx, int32_t ly) { return ly * int32_t(kTile) + (lx ^ ((ly & 7) << 3)); }

// Depth test of one covered sample in the LDS tile (lx, ly: pixel in the tile).
LH_DEV bool tile_fragment(uint64_t* tile, int32_t lx, int32_t ly, float z, uint32_t id) {
    z = fminf(fmaxf(z, 0.0f), 1.0f);
    if (!(z > 0.0f)) return false;  // depth GREATER against the 0.0 clear
    const unsigned long long key = ((unsigned long long)(~__float_as_uint(z)) << 32) | id;
    __hip_atomic_fetch_min(reinterpret_cast<unsigned long long*>(tile) + tile_slot(lx, ly), key, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
    return true;
}

// Materializes v in a register at this point.  The triangle's values come
// from LDS reads; left to itself the compiler recomputes them inside a pixel
// loop, and the LDS-counter wait those reads need then also waits for every
// depth atomic the loop has issued.
template <class T>
LH_DEV void pin(T& v) {
    asm volatile("" : "+v"(v));
}

// Coverage of one pixel centre by an oriented triangle (exact integer edges).
template <class E>
LH_DEV bool inside(E e0, E e1, E e2, bool tl0, bool tl1, bool tl2) {
    return (e0 > 0 || (e0 == 0 && tl0)) && (e1 > 0 || (e1 == 0 && tl1)) && (e2 > 0 || (e2 == 0 && tl2));
}

// In-lane raster of a triangle whose box inside the tile is small (at most
// small_extent pixels a side): the lane walks the box itself.
template <bool ST>
LH_DEV void tile_lane(uint64_t* tile, int32_t ox, int32_t oy, SV a, SV b, SV c, int32_t xlo, int32_t xhi, int32_t ylo,
                      int32_t yhi, float inv_area, uint32_t id, Tally<ST>& tally) {
    pin(a.X), pin(a.Y), pin(b.X), pin(b.Y), pin(c.X), pin(c.Y);
    float z0 = a.z, d10 = b.z - a.z, d20 = c.z - a.z;
    pin(z0), pin(d10), pin(d20), pin(inv_area);
    const bool tl0 = top_left(b.X, b.Y, c.X, c.Y), tl1 = top_left(c.X, c.Y, a.X, a.Y), tl2 = top_left(a.X, a.Y, b.X, b.Y);
    for (int32_t py = ylo; py <= yhi; py++) {
        const int32_t Py = py * 256 + 128;
        for (int32_t px = xlo; px <= xhi; px++) {
            const int32_t Px = px * 256 + 128;
            const int32_t e0 = (c.X - b.X) * (Py - b.Y) - (c.Y - b.Y) * (Px - b.X);
            const int32_t e1 = (a.X - c.X) * (Py - c.Y) - (a.Y - c.Y) * (Px - c.X);
            const int32_t e2 = (b.X - a.X) * (Py - a.Y) - (b.Y - a.Y) * (Px - a.X);
            if (inside(e0, e1, e2, tl0, tl1, tl2)) {
                const float l1 = float(e1) * inv_area, l2 = float(e2) * inv_area;
                tally.hit(tile_fragment(tile, px - ox, py - oy, (z0 + l1 * d10) + l2 * d20, id));
            }
        }
    }
}

// Load-balanced raster of one round of triangles (one per lane) over the
// wave.  A lane's clamped box is cut into runs of up to kRun pixels along its
// rows (`n` runs, 0 for none); the runs are numbered in lane order (exclusive
// scan) and handed out 64 at a time, so a wave spends ceil(sum n / 64) passes
// on a round instead of the largest box.  A lane finds the triangle of its
// run as the last one starting at or before it (start lanes mark their first
// run in `own`, an inclusive max-scan spreads the marks), fetches the
// triangle's corners, box and 1/area from that lane and its snapped vertices
// from the wave's LDS copy, and steps the edge functions along the run.
constexpr int32_t kRun = 4;
LH_DEV int32_t runs_per_row(int32_t w) { return (w + kRun - 1) / kRun; }

template <bool ST>
LH_DEV void tile_expand(uint64_t* tile, int32_t ox, int32_t oy, int32_t* own, const int32_t* sX, const int32_t* sY,
                        const float* sZ, uint32_t tri, uint32_t n, int32_t xlo, int32_t ylo, int32_t w, float inv_area,
                        uint32_t mid, uint32_t lane, Tally<ST>& tally) {
    const uint32_t incl = wave_scan_add(n), excl = incl - n;
    const uint32_t total = uint32_t(__builtin_amdgcn_readlane(int(incl), 63));
    const int32_t box = (xlo - ox) | ((ylo - oy) << 8) | (w << 16);  // tile-relative origin and width
    int32_t carry = 0;
    for (uint32_t base = 0; base < total; base += 64) {
        own[lane] = -1;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (n && excl >= base && excl < base + 64) own[excl - base] = int32_t(lane);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        int32_t o = max(wave_scan_max(own[lane]), carry);
        carry = __builtin_amdgcn_readlane(o, 63);
        // every lane takes part in the fetches (the owner lanes are active)
        const uint32_t otri = __shfl(tri, o, 64);
        const int32_t obox = __shfl(box, o, 64);
        const uint32_t oex = __shfl(excl, o, 64);
        const float oinv = __shfl(inv_area, o, 64);
        const uint32_t omid = uint32_t(__shfl(int(mid), o, 64));
        const uint32_t k = base + lane;
        if (k < total) {
            // run (local % wr, local / wr) of the owner's box; local < 4096, wr <= 16
            const int32_t ow = obox >> 16, wr = runs_per_row(ow);
            const int32_t local = int32_t(k - oex);
            int32_t q = int32_t(float(local) * __builtin_amdgcn_rcpf(float(wr)));
            int32_t r = local - q * wr;
            if (r < 0) q--, r += wr;
            if (r >= wr) q++, r -= wr;
            const int32_t lx0 = (obox & 255) + kRun * r, ly = ((obox >> 8) & 255) + q;
            const int32_t len = min(kRun, ow - kRun * r);
            const uint32_t i0 = otri & 255u, i1 = (otri >> 8) & 255u, i2 = (otri >> 16) & 255u;
            const SV a{sX[i0], sY[i0], sZ[i0]}, b{sX[i1], sY[i1], sZ[i1]}, c{sX[i2], sY[i2], sZ[i2]};
            const int32_t Px = (ox + lx0) * 256 + 128, Py = (oy + ly) * 256 + 128;
            int32_t e0 = (c.X - b.X) * (Py - b.Y) - (c.Y - b.Y) * (Px - b.X);
            int32_t e1 = (a.X - c.X) * (Py - c.Y) - (a.Y - c.Y) * (Px - c.X);
            int32_t e2 = (b.X - a.X) * (Py - a.Y) - (b.Y - a.Y) * (Px - a.X);
            int32_t s0 = -(c.Y - b.Y) * 256, s1 = -(a.Y - c.Y) * 256, s2 = -(b.Y - a.Y) * 256;
            bool tl0 = top_left(b.X, b.Y, c.X, c.Y), tl1 = top_left(c.X, c.Y, a.X, a.Y),
                 tl2 = top_left(a.X, a.Y, b.X, b.Y);
            float z0 = a.z, d10 = b.z - a.z, d20 = c.z - a.z, inv = oinv;
            pin(z0), pin(d10), pin(d20), pin(inv), pin(s0), pin(s1), pin(s2);
            const uint32_t id = (omid << LH_KEY_TRI_BITS) | (otri >> 24);
            for (int32_t j = 0; j < len; j++) {
                if (inside(e0, e1, e2, tl0, tl1, tl2)) {
                    const float l1 = float(e1) * inv, l2 = float(e2) * inv;
                    tally.hit(tile_fragment(tile, lx0 + j, ly, (z0 + l1 * d10) + l2 * d20, id));
                }
                e0 += s0;
                e1 += s1;
                e2 += s2;
            }
        }
    }
}

// Persistent blocks of kTileWaves waves over the work items.  Item: clear the
// LDS tile; each wave takes every kTileWaves-th entry (one binned meshlet),
// with the entry list of the item held one per lane and the next meshlet's
// cache lines requested while the current one is rasterized.  When an entry
// and the next hold at most 64 triangles together (an entry averages about
// 35), both go through one round: the second's vertices at LDS slots
// 64..127, its triangles on the lanes after the first's, each lane with its
// own meshlet id.  Then the covered pixels go out: a plain store when the
// item is the tile's only one (the visibility buffer holds the clear value
// there, as nothing else has drawn yet), an atomicMin otherwise and in the
// second occlusion phase.  Six waves per SIMD (80 VGPRs; the pairing's
// registers would otherwise take the kernel to five).
struct CacheLanes {
    int32_t X, Y;
    float Z;
    uint32_t t0, t1;
};
// The triangles [first, first + count) of an entry: the whole list, or one
// of the 2^lp parts it is split into.
LH_DEV void entry_range(uint32_t ntri_field, uint32_t part, uint32_t& first, uint32_t& count) {
    const uint32_t ntri = ntri_field & 255u, lp = lhs::parts_log2(ntri_field);
    first = (part * ntri) >> lp;
    count = (((part + 1) * ntri) >> lp) - first;
}
LH_DEV CacheLanes load_cache(const BinCache& c, uint32_t lane, uint32_t first) {
    // every lane reads its word whatever the meshlet's vertex and triangle
    // counts: the entry is allocated whole, and words past the counts are
    // never referenced
    return {c.X[lane], c.Y[lane], c.Z[lane], c.tri[min(first + lane, 127u)], c.tri[min(first + lane + 64, 127u)]};
}

template <bool ST>
__global__ void __launch_bounds__(kTileThreads) LH_WAVES_ATTR(6) k_tile_raster(OneView vs, PassSet ps) {
    __shared__ uint64_t tile[kTile * kTile];
    __shared__ int32_t sX[kTileWaves][128], sY[kTileWaves][128];
    __shared__ float sZ[kTileWaves][128];
    __shared__ int32_t own[kTileWaves][64];
    const lh_view& v = vs.v;
    const Bins B = bins(v);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t n_items = min(v.counters[LH_CNT_TILE_ITEMS], B.L.item_capacity);
    const int32_t W = int32_t(v.width), H = int32_t(v.height);
    Tally<ST> tally;
    // Block b starts on item b; each further item comes from a queue, so a
    // block that drew light items takes more of them instead of idling while
    // the heavy ones finish.
    __shared__ uint32_t next_item;
    for (uint32_t it = blockIdx.x; it < n_items;) {
        const TileItem item = B.items[it];
        const int32_t ox = int32_t(item.tile % B.L.tiles_x) * int32_t(kTile);
        const int32_t oy = int32_t(item.tile / B.L.tiles_x) * int32_t(kTile);
        const int32_t ex = min(ox + int32_t(kTile), W) - 1, ey = min(oy + int32_t(kTile), H) - 1;
        const uint32_t end = min(item.end & ~lhs::kItemOnly, B.L.entry_capacity);
        // this wave's entries: begin + wave + kTileWaves k, k < mine (<= 64: item_entries <= 512)
        const uint32_t first = item.begin + wave;
        const uint32_t mine = end > first ? min((end - first + kTileWaves - 1) / kTileWaves, 64u) : 0u;
        const uint32_t my_e = lane < mine ? B.entries[first + kTileWaves * lane] : 0u;
        const uint32_t my_g = my_e & lhs::kEntryDrawMask;
        uint32_t my_first = 0, my_count = 0, my_mid = 0;
        if (lane < mine) {
            const uint2 h = *reinterpret_cast<const uint2*>(&B.hdr[my_g].ntri);
            entry_range(h.x, my_e >> lhs::kEntryPartShift, my_first, my_count);
            my_mid = h.y;
        }
        for (uint32_t k = threadIdx.x; k < kTile * kTile; k += kTileThreads) tile[k] = LH_VISBUFFER_CLEAR;
        CacheLanes cur{};
        if (mine)
            cur = load_cache(B.cache[uint32_t(readlane(int32_t(my_g), 0))], lane,
                             uint32_t(readlane(int32_t(my_first), 0)));
        __syncthreads();
        for (uint32_t k = 0; k < mine;) {
            const uint32_t ntri = uint32_t(readlane(int32_t(my_count), k)), mid = uint32_t(readlane(int32_t(my_mid), k));
            const uint32_t ntri2 = k + 1 < mine ? uint32_t(readlane(int32_t(my_count), k + 1)) : 65u;
            const bool pair = ntri + ntri2 <= 64u;  // wave-uniform
            const uint32_t mid2 = pair ? uint32_t(readlane(int32_t(my_mid), k + 1)) : 0u;
            CacheLanes next{};
            if (k + 1 < mine)
                next = load_cache(B.cache[uint32_t(readlane(int32_t(my_g), k + 1))], lane,
                                  uint32_t(readlane(int32_t(my_first), k + 1)));
            sX[wave][lane] = cur.X;
            sY[wave][lane] = cur.Y;
            sZ[wave][lane] = cur.Z;
            uint32_t tri_pair = cur.t0, lane_mid = mid;
            if (pair) {
                sX[wave][64 + lane] = next.X;
                sY[wave][64 + lane] = next.Y;
                sZ[wave][64 + lane] = next.Z;
                const uint32_t from = uint32_t(__shfl(int(next.t0), int((lane - ntri) & 63u), 64));
                if (lane >= ntri) {
                    tri_pair = from + 0x404040u;  // corners of the second entry at slots 64..127
                    lane_mid = mid2;
                }
                // the second entry is consumed: its registers take the request
                // of the entry after the pair
                if (k + 2 < mine)
                    next = load_cache(B.cache[uint32_t(readlane(int32_t(my_g), k + 2))], lane,
                                      uint32_t(readlane(int32_t(my_first), k + 2)));
            }
            const uint32_t total = pair ? ntri + ntri2 : ntri;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            for (uint32_t round = 0; round < 2 && round * 64 < total; round++) {
                const uint32_t tri = pair ? tri_pair : (round ? cur.t1 : cur.t0);
                uint32_t n = 0;
                int32_t xlo = 0, ylo = 0, w = 1;
                float inv_area = 0.0f;
                if (lane + 64 * round < total) {
                    const uint32_t i0 = tri & 255u, i1 = (tri >> 8) & 255u, i2 = (tri >> 16) & 255u;
                    const SV a{sX[wave][i0], sY[wave][i0], sZ[wave][i0]};
                    const SV b{sX[wave][i1], sY[wave][i1], sZ[wave][i1]};
                    const SV c{sX[wave][i2], sY[wave][i2], sZ[wave][i2]};
                    const int32_t minX = min(a.X, min(b.X, c.X)), maxX = max(a.X, max(b.X, c.X));
                    const int32_t minY = min(a.Y, min(b.Y, c.Y)), maxY = max(a.Y, max(b.Y, c.Y));
                    xlo = max((minX + 127) >> 8, ox);
                    const int32_t xhi = min((maxX - 128) >> 8, ex);
                    ylo = max((minY + 127) >> 8, oy);
                    const int32_t yhi = min((maxY - 128) >> 8, ey);
                    if (xlo <= xhi && ylo <= yhi) {
                        w = xhi - xlo + 1;
                        const int32_t h = yhi - ylo + 1;
                        // positive area (oriented by the binning), every value within int32 (<= 64 px)
                        inv_area = rcp_exact(float((b.X - a.X) * (c.Y - a.Y) - (b.Y - a.Y) * (c.X - a.X)));
                        if (max(w, h) * 256 <= ps.small_extent)
                            tile_lane<ST>(tile, ox, oy, a, b, c, xlo, xhi, ylo, yhi, inv_area,
                                          (lane_mid << LH_KEY_TRI_BITS) | (tri >> 24), tally);
                        else
                            n = uint32_t(runs_per_row(w) * h);
                    }
                }
                tile_expand<ST>(tile, ox, oy, own[wave], sX[wave], sY[wave], sZ[wave], tri, n, xlo, ylo, w, inv_area,
                                lane_mid, lane, tally);
            }
            k += pair ? 2u : 1u;
            cur = next;
        }
        tally.flush(v, 0);
        __syncthreads();
        const bool only = (item.end & lhs::kItemOnly) && !ps.phase2;
        for (uint32_t k = threadIdx.x; k < kTile * kTile; k += kTileThreads) {
            const int32_t lx = int32_t(k & (kTile - 1)), ly = int32_t(k >> lhs::kTileShift);
            const int32_t px = ox + lx, py = oy + ly;
            const uint64_t key = tile[tile_slot(lx, ly)];
            if (px > ex || py > ey || key == LH_VISBUFFER_CLEAR) continue;
            unsigned long long* dst = reinterpret_cast<unsigned long long*>(v.visbuffer + size_t(py) * v.width + px);
            if (only)
                *dst = key;
            else
                atomicMin(dst, (unsigned long long)key);
        }
        if (threadIdx.x == 0) next_item = gridDim.x + atomicAdd(&v.counters[LH_CNT_TILE_NEXT], 1u);
        __syncthreads();  // the item's LDS tile is free; next_item is written
        it = next_item;   // rewritten only after the next item's barriers
    }
}

}  // namespace

namespace lhk {

template <bool ST>
hipError_t raster_tiles(const lh_scene& s, const OneView& vs, const PassSet& ps, const RasterTuning& t,
                        bool bins_clear, hipStream_t st) {
    const uint32_t item_entries = std::min(std::max(t.tile_item_entries, lhs::kMinItemEntries), 64u * kTileWaves);
    if (!bins_clear) {
        mark("bin_reset_view", st);
        hipLaunchKernelGGL(k_bin_reset, dim3(8), dim3(256), 0, st, vs);
    }
    mark("bin_meshlets_view", st);
    const uint32_t blocks = std::min<uint32_t>(kBinBlocks, std::max(s.total_meshlets, 1u));
    hipLaunchKernelGGL(k_bin_meshlets<0>, dim3(blocks), dim3(64), 0, st, s, vs, ps);
    // the draw count is on the device: the grid is sized for the most draws
    const uint32_t most = std::min(std::min(vs.v.draw_capacity, vs.v.bin_capacity), std::max(s.total_meshlets, 1u));
    const uint32_t chunks = std::max<uint32_t>(1, (std::min(most, 1u << 22) + kBinThreads - 1) / kBinThreads);
    mark("bin_fill_view", st);
    hipLaunchKernelGGL(k_bin_fill, dim3(std::min<uint32_t>(chunks, 256)), dim3(kBinThreads), 0, st, vs, ps, item_entries);
    mark("tile_raster_view", st);
    hipLaunchKernelGGL((k_tile_raster<ST>), dim3(t.tile_blocks), dim3(kTileThreads), 0, st, vs, ps);
    return hipGetLastError();
}

template hipError_t raster_tiles<false>(const lh_scene&, const OneView&, const PassSet&, const RasterTuning&, bool,
                                        hipStream_t);
template hipError_t raster_tiles<true>(const lh_scene&, const OneView&, const PassSet&, const RasterTuning&, bool,
                                       hipStream_t);

}  // namespace lhk
