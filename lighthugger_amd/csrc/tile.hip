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
//                   cleared, each wave collects the triangles of its binned
//                   meshlets that meet the tile, from the cache, and rasterizes
//                   up to 64 at a time (ds_min_u64 per covered sample), then the
//                   tile's covered pixels are written out.
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
                if (queue_big(v, ps.pass0, big, wv, ts, (cur.mid << LH_KEY_TRI_BITS) | t, 0, false))
                    atomicOr(&v.counters[LH_CNT_OVERFLOW], LH_OVERFLOW_BIG);
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
            // too many tiles: left to the direct list
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

// The LDS tile as a render target of raster_queue; coordinates are the tile's.
struct TileTarget {
    uint64_t* tile;
    uint32_t W, H;  // of the part inside the view
    // An LDS depth test costs a lane less than a device atomic: 0, 4, 8, 12, 16,
    // 24 px: stress tiles 503, 469, 457, 449, 443, 438 us, 1920x1080 84, 81,
    // 78, 74, 72, 72, 1280x720 50, 50, 52, 51, 51, 55.
    static constexpr int32_t kLanePx = 16;
    LH_DEV bool put(int32_t x, int32_t y, float z, uint32_t id) const { return tile_fragment(tile, x, y, z, id); }
};

// Persistent blocks of kTileWaves waves over the work items.  Item: clear the
// LDS tile; each wave takes every kTileWaves-th entry (one binned meshlet),
// with the entry list of the item held one per lane and the next meshlet's
// cache lines requested while the current one is set up.  The triangles whose
// box holds a pixel centre of the tile are collected in the wave's queue and
// rasterized when it is full (raster.h).  Then the covered pixels go out: a
// plain store when the item is the tile's only one (the visibility buffer holds
// the clear value there, as nothing else has drawn yet), an atomicMin otherwise
// and in the second occlusion phase.
//
// Bound by VALU issue.  With a round's triangles on one entry's lanes and boxes
// walked in runs of four, 27 of 64 lanes were active: 1920x1080 101 us, 720p
// 77, the 3840x2160 field 152, 20,000 instances 557; with the queue and the
// exact row spans 72, 51, 124, 443.
//
// LDS is what limits the blocks of a compute unit to three (six waves per
// SIMD): vertices are kept relative to the tile in 16 bits.  A triangle of at
// most 64 px that touches the tile lies within them; the clamp keeps any other
// vertex on its side of the tile.
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
    __shared__ uint2 verts8[kTileWaves][64];  // x & 0xFFFF | y << 16 (subpixels of the tile), z
    __shared__ TriQueueOf<64, int8_t> queues8[kTileWaves];
    const lh_view& v = vs.v;
    const Bins B = bins(v);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t n_items = min(v.counters[LH_CNT_TILE_ITEMS], B.L.item_capacity);
    const int32_t W = int32_t(v.width), H = int32_t(v.height);
    uint2* const verts = verts8[wave];
    auto& queue = queues8[wave];
    NoAlpha none;
    Tally<ST> tally;
    // Block b starts on item b; each further item comes from a queue, so a
    // block that drew light items takes more of them instead of idling while
    // the heavy ones finish.  (The word is a vertex's between the barriers.)
    uint32_t& next_item = verts8[0][0].x;
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
        const TileTarget target{tile, uint32_t(ex - ox + 1), uint32_t(ey - oy + 1)};
        uint32_t held = 0;  // triangles in the queue
        auto flush = [&] {
            if (held) raster_queue<0, ST, false, false>(lh_scene{}, LhMat4{}, target, queue, none, 0, held, lane, tally);
            held = 0;
            lds_order();
        };
        for (uint32_t k = 0; k < mine; k++) {
            const uint32_t ntri = uint32_t(readlane(int32_t(my_count), k)), mid = uint32_t(readlane(int32_t(my_mid), k));
            auto rel = [](int32_t X, int32_t o) { return min(max(X - o * 256, -32768), 32767); };
            lds_order();
            verts[lane] = make_uint2((uint32_t(rel(cur.X, ox)) & 0xFFFFu) | uint32_t(rel(cur.Y, oy)) << 16,
                                     __float_as_uint(cur.Z));
            lds_order();
            const uint32_t tris[2] = {cur.t0, cur.t1};
            if (k + 1 < mine)
                cur = load_cache(B.cache[uint32_t(readlane(int32_t(my_g), k + 1))], lane,
                                 uint32_t(readlane(int32_t(my_first), k + 1)));
#pragma unroll
            for (uint32_t round = 0; round < 2; round++) {
                if (round * 64 >= ntri) break;
                const uint32_t tri = tris[round];
                const uint2 a = verts[tri & 63u], b = verts[(tri >> 8) & 63u], c = verts[(tri >> 16) & 63u];
                const int32_t ax = lo16(a.x), ay = hi16(a.x), bx = lo16(b.x), by = hi16(b.x), cx = lo16(c.x), cy = hi16(c.x);
                const int32_t xlo = max((min(ax, min(bx, cx)) + 127) >> 8, 0);
                const int32_t ylo = max((min(ay, min(by, cy)) + 127) >> 8, 0);
                const int32_t xhi = min((max(ax, max(bx, cx)) - 128) >> 8, int32_t(target.W) - 1);
                const int32_t yhi = min((max(ay, max(by, cy)) - 128) >> 8, int32_t(target.H) - 1);
                const bool push = lane + 64 * round < ntri && xlo <= xhi && ylo <= yhi;
                const uint64_t pm = ballot(push);
                const uint32_t n = uint32_t(__popcll(pm));
                if (n == 0) continue;
                if (held + n > 64) flush();
                if (push)
                    queue.store(held + lanes_below(pm), xlo, ylo, SV{ax, ay, __uint_as_float(a.y)},
                                SV{bx, by, __uint_as_float(b.y)}, SV{cx, cy, __uint_as_float(c.y)},
                                (mid << LH_KEY_TRI_BITS) | (tri >> 24));
                held += n;
            }
        }
        flush();
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
