// Tiled raster path: bin-to-tile and LDS tile raster.
// The data flow is described in sloth_tiled.h.
#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "sloth_tiled.h"

namespace sloth {

constexpr int BIN_BLOCK = 256;
constexpr int RASTER_BLOCK = 256;

// k_tile_raster<true> walks a box with more than BIG_BOX pixels in a tile by
// the whole wavefront.  careful_cnt[BIG_CNT] is where the counting run of
// k_bin counts the triangles whose (unclipped) box has more.
constexpr uint32_t BIG_BOX = 128;
constexpr uint32_t BIG_CNT = 2 + MAX_GROUPS;
// careful_cnt[TALL_CNT]: triangles the counting run finds spanning more than
// TALL_ROWS rows (TiledPlan::bin_tree)
constexpr uint32_t TALL_CNT = BIG_CNT + 1;
// careful_cnt[WRAP_CNT]: the most tile columns odd_cols_of asks for in the
// counting run (TiledPlan::odd_wraps)
constexpr uint32_t WRAP_CNT = TALL_CNT + 1;
constexpr int TALL_ROWS = 16;

// ---------------------------------------------------------------------------
// k_tile_clear
// ---------------------------------------------------------------------------
__global__ void k_tile_clear(uint32_t* __restrict__ cursor, uint64_t n_tiles, int32_t* __restrict__ nl,
                             uint64_t n_rows, uint32_t* __restrict__ overflow, uint32_t n_frames,
                             uint32_t* __restrict__ careful_cnt)
{
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    uint64_t i0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (uint64_t i = i0; i < n_tiles; i += stride) cursor[i] = 0;
    for (uint64_t i = i0; i < n_rows; i += stride) nl[i] = -1;
    for (uint64_t i = i0; i < n_frames; i += stride) overflow[i] = 0;
    if (i0 == 0) careful_cnt[0] = careful_cnt[1] = careful_cnt[BIG_CNT] = careful_cnt[TALL_CNT] =
            careful_cnt[WRAP_CNT] = 0;   // list length, first group's start; the counting run's
}

// ---------------------------------------------------------------------------
// tile geometry shared by the binning kernels
// ---------------------------------------------------------------------------

// Pool entries: the frame triangle index of a CLS_TIGHT triangle, LOOSE_FLAG |
// the index of a CLS_BOX one (the raster recomputes either box from the
// triangle's x extent), or CAREFUL_FLAG | row of the careful-box table for
// triangles whose box k_careful computed.  Frames on this path hold fewer than
// TILED_MAX_TRIS triangles.
constexpr uint32_t CAREFUL_FLAG = 0x80000000u;
constexpr uint32_t LOOSE_FLAG = 0x40000000u;


// Tile rectangles (inclusive, in tile units) that a candidate box reaches:
// the direct part (2x < W, cell (2x, y)) and the wrapped part (2x >= W, cell
// (2x - W, y + 1)).  An empty rectangle has x0 > x1.
struct TileRects {
    int dx0, dx1, dy0, dy1;
    int wx0, wx1, wy0, wy1;
};

__device__ __forceinline__ void empty_rects(TileRects& r)
{
    r.dx0 = r.dy0 = r.wx0 = r.wy0 = 1;
    r.dx1 = r.dy1 = r.wx1 = r.wy1 = 0;
}

__device__ __forceinline__ void tile_rects(int bx0, int bx1, int by0, int by1, uint32_t W, int tws, int ths,
                                           TileRects& r)
{
    // direct pixels: 2x < W, i.e. x <= (W - 1) / 2; wrapped: x >= (W + 1) / 2
    empty_rects(r);
    int dxe = min(bx1, (int)((W - 1) >> 1));
    if (bx0 <= dxe && by0 <= by1) {
        r.dx0 = (2 * bx0) >> tws;
        r.dx1 = (2 * dxe) >> tws;
        r.dy0 = by0 >> ths;
        r.dy1 = by1 >> ths;
    }
    int wxs = max(bx0, (int)((W + 1) >> 1));
    if (wxs <= bx1 && by0 <= by1) {
        r.wx0 = (2 * wxs - (int)W) >> tws;
        r.wx1 = (2 * bx1 - (int)W) >> tws;
        r.wy0 = (by0 + 1) >> ths;
        r.wy1 = (by1 + 1) >> ths;
    }
}

// The tile columns of a frame of odd width that the raster's odd instance must
// take for a box that ends at column bx1: none while it ends before the last
// cell column (x = W / 2); the first for that column, whose slots' second cells
// are the next rows' first; and for wrapped columns those they reach and one
// more, whose first cells may be second cells of the last of them.
__device__ __forceinline__ int odd_cols_of(int bx1, uint32_t W, int tws)
{
    const int last = (int)(W >> 1);
    return bx1 < last ? 0 : bx1 == last ? 1 : ((2 * bx1 - (int)W) >> tws) + 2;
}

__device__ __forceinline__ bool in_direct(const TileRects& r, int tx, int ty)
{
    return tx >= r.dx0 && tx <= r.dx1 && ty >= r.dy0 && ty <= r.dy1;
}

// One entry appended to tile `gt` at `pos` (when the pool has room).
template <bool COUNT>
__device__ __forceinline__ void put_entry(uint64_t gt, uint32_t pos, uint32_t entry, const uint64_t* __restrict__ off,
                                          uint32_t* __restrict__ pool, uint32_t* __restrict__ overflow, uint32_t frame)
{
    if (COUNT) return;
    const uint64_t o = off[gt], cap = off[gt + 1] - o;
    if (pos < cap) pool[o + pos] = entry;
    else overflow[frame] = 1u;
}

// ---------------------------------------------------------------------------
// k_bin
// ---------------------------------------------------------------------------
constexpr int BIN_CELLS = 512;   // the block aggregates appends in a window of up to so many tiles

// Grid: x = blocks of TPT * BIN_BLOCK consecutive triangles of one draw,
// y = draw index - d_lo, so the draw, its frame and its matrix are uniform
// per block (scalar loads).  CLS_BOX / CLS_TIGHT triangles of few tiles are
// appended to them here; others and CLS_SPANS / CLS_FULL ones go to the
// careful list for k_careful.
//
// Each thread takes TPT triangles (k * BIN_BLOCK + thread), set up one after
// another with their loads in flight together, so that the block's barriers
// and its global atomic round trip serve TPT times as many triangles (the
// kernel is bound by latency, not by issue).  TPT is 1, 2 or 4
// (TiledPlan::bin_tpt; the autotuner picks it).  Per triangle a thread
// keeps two words between the phases (its tile rectangle and flags, and its
// rows) and two more of window counts between the last two.
//
// Appends: a block's consecutive triangles lie close together on screen.
// Triangles whose box touches at most 2 x 2 tiles, all in the direct region
// or all in the wrapped one (nearly all), count themselves into LDS counters
// of a window of tiles anchored at the block's smallest tile coordinates; one
// global atomicAdd per window tile then reserves that tile's run (the thread
// that reserves it also reads the tile's pool range), and each triangle
// writes its entry at run + its LDS count.  The window has 512 tiles in rows
// as long as the block's tiles need (a strip of a large mesh's face is wide
// and low, or slanted); those outside append with one global atomicAdd per
// tile, up to four in flight together.  Larger boxes and part-wrapping ones
// go to k_careful: appended here, one tile after another, they held up their
// block (972 triangles of about 20 tiles each on 2560x1440: 70 us, now 29 for
// the launch; 519,168 small ones, some across the wrap: 106 us, now 21).
// 30 unlike jobs: k_bin 110-255 us, now 53-59 (with bin_tree's rule).
//
// geo word: qx0 (bits 0-13), qy0 (14-27) of the tile rectangle, wide (28),
// tall (29), CLS_BOX (30); tile coordinates stay below 2^14 (frames of at
// most 65535 cells a side, tiles of at least 8 x 4 cells).
constexpr uint32_t GEO_WIDE = 1u << 28, GEO_TALL = 1u << 29, GEO_LOOSE = 1u << 30;

// Newline rows over a window of BIN_BLOCK rows: a max segment tree in LDS
// (node 1 spans the window, node i has children 2i and 2i + 1, row r's leaf
// is BIN_BLOCK + r).  A triangle raises the nodes that tile its rows [a, b)
// of the window, at most 2 log2(BIN_BLOCK) of them (a range of up to 4 rows
// takes its leaves); row r's value is the maximum on its leaf's path to the
// root.
__device__ __forceinline__ void nl_raise(int32_t* tree, int a, int b, int32_t v)
{
    if (b - a <= 4) {
        for (int y = a; y < b; ++y) atomicMax(&tree[BIN_BLOCK + y], v);
        return;
    }
    for (int l = a + BIN_BLOCK, r = b + BIN_BLOCK; l < r; l >>= 1, r >>= 1) {
        if (l & 1) atomicMax(&tree[l++], v);
        if (r & 1) atomicMax(&tree[--r], v);
    }
}
__device__ __forceinline__ int32_t nl_value(const int32_t* tree, int r)
{
    int32_t v = -1;
    for (int i = BIN_BLOCK + r; i >= 1; i >>= 1) v = max(v, tree[i]);
    return v;
}

template <bool COUNT, int TPT, bool TREE>
__global__ void __launch_bounds__(BIN_BLOCK) k_bin(const Draw* __restrict__ draws, uint32_t d_lo,
                                                   const Frame* __restrict__ frames, int tws, int ths,
                                                   uint32_t* __restrict__ cursor, const uint64_t* __restrict__ off,
                                                   uint32_t* __restrict__ pool, int32_t* __restrict__ nl,
                                                   uint32_t* __restrict__ overflow, uint32_t* __restrict__ careful_cnt,
                                                   uint4* __restrict__ careful_in, uint32_t careful_cap,
                                                   const uint2* __restrict__ flat_blocks, uint32_t odd_cols)
{
    __shared__ uint32_t w_cnt[BIN_CELLS];
    __shared__ uint64_t w_base[BIN_CELLS];   // pool index of the tile's reserved run
    __shared__ uint32_t w_room[BIN_CELLS];   // entries of it that the tile's pool range holds
    // newline rows: a window of rows, or (TREE) its segment tree (nl_raise)
    __shared__ int32_t s_nl[TREE ? 2 * BIN_BLOCK : BIN_BLOCK];
    constexpr int LEAF = TREE ? BIN_BLOCK : 0;   // row r of the window at s_nl[LEAF + r]
    __shared__ int s_tx0, s_ty0, s_tx1, s_ty1, s_lo, s_hi;

    // the block's draw and first triangle: from the grid, or (flat grids of
    // draws of different sizes) from its table entry
    uint32_t d, base;
    if (flat_blocks) {
        const uint2 e = flat_blocks[blockIdx.x];
        d = e.x;
        base = e.y;
    } else {
        d = d_lo + blockIdx.y;
        base = blockIdx.x * (BIN_BLOCK * TPT);
    }
    const Draw& dr = draws[d];
    if (base >= dr.n) return;
    const uint32_t frame = dr.frame;
    const Frame& fr = frames[frame];
    const uint32_t W = fr.W, H = fr.H;
    const uint64_t tile_begin = fr.tile_begin;
    const uint32_t tiles_x = fr.tiles_x;

    for (int c = threadIdx.x; c < BIN_CELLS; c += BIN_BLOCK) w_cnt[c] = 0;
    s_nl[threadIdx.x] = -1;
    if (TREE) s_nl[LEAF + threadIdx.x] = -1;
    if (threadIdx.x == 0) {
        s_tx0 = s_ty0 = s_lo = 1 << 30;
        s_tx1 = s_ty1 = s_hi = -1;
    }

    // Phase 1: set-up and classes.  Lanes past the draw's end set up its
    // last triangle and discard it, so that the set-up has no branch around
    // it (the lanes of a wavefront take different classes; selects cost less
    // than divergent paths).
    uint32_t geo[TPT], rows[TPT];
    uint32_t small = 0;   // bit k: triangle k has a small rectangle, appended here
    int acc_lo = 1 << 30, acc_hi = -1;
    uint32_t acc_t0 = 0x7FFF7FFFu, acc_t1 = 0;   // least and largest tile: x, y << 16
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
        const uint32_t local = base + (uint32_t)k * BIN_BLOCK + threadIdx.x;
        const bool valid = local < dr.n;
        Tri t;
        setup_draw_tri(dr, valid ? local : dr.n - 1, W, H, t);
        const uint32_t cls = valid ? setup_class(t) : CLS_EMPTY;
        const bool boxed = cls == CLS_BOX || cls == CLS_TIGHT;
        bool careful = cls == CLS_SPANS || cls == CLS_FULL;
        uint32_t g = cls == CLS_BOX ? GEO_LOOSE : 0u;
        // A wavefront whose triangles are all back faces or empty (half of
        // a closed mesh's, in runs) has no tiles to find: a uniform branch.
        if (__ballot(boxed)) {
            int bx0 = 1, bx1 = 0;
            if (boxed) box_x(t, cls == CLS_TIGHT, bx0, bx1);   // empty when not boxed
            if (COUNT) {
                const bool big = boxed && (int64_t)(bx1 - bx0 + 1) * (int64_t)(t.y1d - t.y0) > (int64_t)BIG_BOX;
                const uint64_t m = __ballot(big);
                if (__lane_id() == 0 && m) atomicAdd(&careful_cnt[BIG_CNT], (uint32_t)__popcll(m));
            }
            // A box in one region appends through that region's tile
            // rectangle [qx0, qx1] x [qy0, qy1]; k_careful takes a box that
            // wraps in part (it spans 2x = W).  (Meshes wider than the frame's
            // logical width put whole patches of triangles in the wrapped
            // region.)
            bool has_direct, has_wrap;
            int qx0, qx1, qy0, qy1;
            if (!__ballot(bx1 >= (int)(W >> 1))) {
                // no box of the wavefront reaches the wrapped region (x >=
                // (W + 1) / 2) or an odd frame's last column (x = W / 2):
                // tile_rects' direct rectangle with x <= bx1
                has_direct = bx0 <= bx1 && t.y0 < t.y1d;
                has_wrap = false;
                qx0 = (2 * bx0) >> tws;
                qx1 = (2 * bx1) >> tws;
                qy0 = t.y0 >> ths;
                qy1 = (t.y1d - 1) >> ths;
            } else {
                if (W & 1u) {
                    const uint32_t need = (uint32_t)wave_max(boxed ? odd_cols_of(bx1, W, tws) : 0);
                    if (__lane_id() == 0) {
                        if (COUNT) atomicMax(&careful_cnt[WRAP_CNT], need);
                        else if (need > odd_cols) overflow[frame] = 1u;
                    }
                }
                TileRects r;
                tile_rects(bx0, bx1, t.y0, t.y1d - 1, W, tws, ths, r);   // empty when bx0 > bx1
                has_direct = r.dx0 <= r.dx1 && r.dy0 <= r.dy1;
                has_wrap = r.wx0 <= r.wx1 && r.wy0 <= r.wy1;
                const bool wrap_only = has_wrap && !has_direct;
                qx0 = wrap_only ? r.wx0 : r.dx0;
                qx1 = wrap_only ? r.wx1 : r.dx1;
                qy0 = wrap_only ? r.wy0 : r.dy0;
                qy1 = wrap_only ? r.wy1 : r.dy1;
            }
            const bool sm = has_direct != has_wrap && qx1 - qx0 <= 1 && qy1 - qy0 <= 1;
            // larger and part-wrapping boxes: appended by k_careful
            careful = careful || ((has_direct || has_wrap) && !sm);
            if (sm) {
                small |= 1u << k;
                g |= (uint32_t)qx0 | ((uint32_t)qy0 << 14) | (qx1 > qx0 ? GEO_WIDE : 0u) | (qy1 > qy0 ? GEO_TALL : 0u);
                acc_t0 = min_u16x2(acc_t0, (uint32_t)qx0 | ((uint32_t)qy0 << 16));
                acc_t1 = max_u16x2(acc_t1, (uint32_t)qx1 | ((uint32_t)qy1 << 16));
            }
        }
        geo[k] = g;
        if (careful) {
            const uint32_t idx = atomicAdd(careful_cnt, 1u);
            if (idx < careful_cap) {
                // the screen vertices come along, so that k_careful starts
                // from them instead of the draw record and the mesh
                careful_in[2 * idx] = make_uint4(frame, dr.tri_begin + local, __float_as_uint(t.x1), __float_as_uint(t.y1));
                careful_in[2 * idx + 1] = make_uint4(__float_as_uint(t.x2), __float_as_uint(t.y2),
                                                     __float_as_uint(t.x3), __float_as_uint(t.y3));
            }
            else if (!COUNT) overflow[frame] = 1u;
        }
        const bool has_rows = fr.image && valid && t.y0 < t.y1d;
        rows[k] = has_rows ? (uint32_t)t.y0 | ((uint32_t)t.y1d << 16) : 0u;
        if (has_rows) {
            acc_lo = min(acc_lo, t.y0);
            acc_hi = max(acc_hi, t.y1d - 1);
        }
        if (COUNT) {
            const uint64_t m = __ballot(has_rows && t.y1d - t.y0 > TALL_ROWS);
            if (__lane_id() == 0 && m) atomicAdd(&careful_cnt[TALL_CNT], (uint32_t)__popcll(m));
        }
    }
    __syncthreads();   // LDS initialised

    {
        const int wlo = wave_min(acc_lo), whi = wave_max(acc_hi);
        if (__lane_id() == 0 && whi >= 0) {
            atomicMin(&s_lo, wlo);
            atomicMax(&s_hi, whi);
        }
        if (__ballot(small != 0)) {
            const uint32_t t0 = wave_reduce((int)acc_t0, [](int a, int b) { return (int)min_u16x2((uint32_t)a, (uint32_t)b); });
            const uint32_t t1 = wave_reduce((int)acc_t1, [](int a, int b) { return (int)max_u16x2((uint32_t)a, (uint32_t)b); });
            if (__lane_id() == 0) {
                atomicMin(&s_tx0, (int)(t0 & 0xFFFFu));
                atomicMin(&s_ty0, (int)(t0 >> 16));
                atomicMax(&s_tx1, (int)(t1 & 0xFFFFu));
                atomicMax(&s_ty1, (int)(t1 >> 16));
            }
        }
    }
    __syncthreads();

    // Phase 2: window counts and newline rows in LDS.
    // rasterizer.rs:89-91: a newline cell after every row of the domain; the
    // last triangle (in draw order) whose rows include r decides row r.
    // The block reduces its rows in LDS, one global atomicMax per row: here
    // when they span fewer than BIN_BLOCK rows, else in windows of BIN_BLOCK
    // rows at the end (tall triangles put every row of a tall frame under
    // the atomics of each triangle that covers it).
    const int ox = __builtin_amdgcn_readfirstlane(s_tx0), oy = __builtin_amdgcn_readfirstlane(s_ty0);
    const int lo = s_lo, hi = s_hi;
    // the window: the block's tiles, in rows of 2^ws, when there are that few
    // (one tile where no rectangle is small)
    const int tiles_w = max(__builtin_amdgcn_readfirstlane(s_tx1) - ox + 1, 1);
    const int tiles_h = max(__builtin_amdgcn_readfirstlane(s_ty1) - oy + 1, 1);
    const int ws_all = 31 - __builtin_clz(2 * tiles_w - 1);
    const int ws = ((int64_t)tiles_h << ws_all) <= BIN_CELLS ? ws_all : min(ws_all, 5);
    const bool nl_lds = hi >= lo && hi - lo < BIN_BLOCK;
    auto in_window = [&](uint32_t g, int& c) {
        const int qx0 = (int)(g & 0x3FFFu), qy0 = (int)((g >> 14) & 0x3FFFu);
        c = ((qy0 - oy) << ws) + (qx0 - ox);
        return qx0 + (int)((g >> 28) & 1u) - ox < 1 << ws && qy0 + (int)((g >> 29) & 1u) - oy < BIN_CELLS >> ws;
    };
    const uint32_t tri0 = dr.tri_begin + base + threadIdx.x;
    uint32_t lpa[TPT], lpb[TPT];   // LDS counts: tiles (0,0) | (1,0) << 16, (0,1) | (1,1) << 16
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
        lpa[k] = lpb[k] = 0;
        int c;
        if (((small >> k) & 1u) && in_window(geo[k], c)) {
            const bool wide = geo[k] & GEO_WIDE, tall = geo[k] & GEO_TALL;
            uint32_t l0 = atomicAdd(&w_cnt[c], 1u), l1 = 0, l2 = 0, l3 = 0;
            if (wide) l1 = atomicAdd(&w_cnt[c + 1], 1u);
            if (tall) l2 = atomicAdd(&w_cnt[c + (1 << ws)], 1u);
            if (wide && tall) l3 = atomicAdd(&w_cnt[c + (1 << ws) + 1], 1u);
            lpa[k] = l0 | (l1 << 16);
            lpb[k] = l2 | (l3 << 16);
        }
        if (nl_lds && rows[k]) {
            const int y0 = (int)(rows[k] & 0xFFFFu), y1d = (int)(rows[k] >> 16);
            if (TREE) nl_raise(s_nl, y0 - lo, y1d - lo, (int32_t)(tri0 + (uint32_t)k * BIN_BLOCK));
            else
                for (int y = y0; y < y1d; ++y) atomicMax(&s_nl[y - lo], (int32_t)(tri0 + (uint32_t)k * BIN_BLOCK));
        }
    }
    __syncthreads();

    int32_t* fnl = nl + fr.nl_off;
    const uint32_t cells = (uint32_t)min(tiles_h << ws, BIN_CELLS);
    for (uint32_t c = threadIdx.x; c < cells; c += BIN_BLOCK) {
        const uint32_t n = w_cnt[c];
        if (n) {
            const uint64_t gt = tile_begin + (uint64_t)(oy + (int)(c >> ws)) * tiles_x + (uint64_t)(ox + (int)(c & ((1u << ws) - 1)));
            const uint32_t pos = atomicAdd(&cursor[gt], n);
            if (!COUNT) {
                const uint64_t o = off[gt];
                const uint32_t cap = (uint32_t)(off[gt + 1] - o);
                w_base[c] = o + pos;
                w_room[c] = pos < cap ? cap - pos : 0u;
            }
        }
    }
    if (nl_lds && (int)threadIdx.x <= hi - lo) {
        const int32_t v = TREE ? nl_value(s_nl, (int)threadIdx.x) : s_nl[threadIdx.x];
        if (v >= 0) atomicMax(&fnl[lo + (int)threadIdx.x], v);
    }
    __syncthreads();

    // Phase 3: entries.
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
        if (!((small >> k) & 1u)) continue;
        const uint32_t local = base + (uint32_t)k * BIN_BLOCK + threadIdx.x;
        const uint32_t entry = (dr.tri_begin + local) | ((geo[k] & GEO_LOOSE) ? LOOSE_FLAG : 0u);
        const bool wide = geo[k] & GEO_WIDE, tall = geo[k] & GEO_TALL;
        int c;
        if (in_window(geo[k], c)) {
            if (!COUNT) {
                auto put = [&](int cc, uint32_t l) {
                    if (l < w_room[cc]) pool[w_base[cc] + l] = entry;
                    else overflow[frame] = 1u;
                };
                put(c, lpa[k] & 0xFFFFu);
                if (wide) put(c + 1, lpa[k] >> 16);
                if (tall) put(c + (1 << ws), lpb[k] & 0xFFFFu);
                if (wide && tall) put(c + (1 << ws) + 1, lpb[k] >> 16);
            }
        } else {
            // outside the window: one global atomic per tile, in flight together
            const uint64_t gt = tile_begin + (uint64_t)((geo[k] >> 14) & 0x3FFFu) * tiles_x + (uint64_t)(geo[k] & 0x3FFFu);
            uint32_t p1 = 0, p2 = 0, p3 = 0;
            const uint32_t p0 = atomicAdd(&cursor[gt], 1u);
            if (wide) p1 = atomicAdd(&cursor[gt + 1], 1u);
            if (tall) p2 = atomicAdd(&cursor[gt + tiles_x], 1u);
            if (wide && tall) p3 = atomicAdd(&cursor[gt + tiles_x + 1], 1u);
            put_entry<COUNT>(gt, p0, entry, off, pool, overflow, frame);
            if (wide) put_entry<COUNT>(gt + 1, p1, entry, off, pool, overflow, frame);
            if (tall) put_entry<COUNT>(gt + tiles_x, p2, entry, off, pool, overflow, frame);
            if (wide && tall) put_entry<COUNT>(gt + tiles_x + 1, p3, entry, off, pool, overflow, frame);
        }
    }
    if (hi >= lo && !nl_lds) {   // uniform per block
        for (int ws = lo; ws <= hi; ws += BIN_BLOCK) {
            __syncthreads();   // the previous window's reads are done
            s_nl[threadIdx.x] = -1;
            if (TREE) s_nl[LEAF + threadIdx.x] = -1;
            __syncthreads();
#pragma unroll
            for (int k = 0; k < TPT; ++k) {
                if (!rows[k]) continue;
                const int y0 = max((int)(rows[k] & 0xFFFFu), ws), y1d = min((int)(rows[k] >> 16), ws + BIN_BLOCK);
                if (TREE) {
                    if (y0 < y1d) nl_raise(s_nl, y0 - ws, y1d - ws, (int32_t)(tri0 + (uint32_t)k * BIN_BLOCK));
                } else {
                    for (int y = y0; y < y1d; ++y) atomicMax(&s_nl[y - ws], (int32_t)(tri0 + (uint32_t)k * BIN_BLOCK));
                }
            }
            __syncthreads();
            if (ws + (int)threadIdx.x <= hi) {
                const int32_t v = TREE ? nl_value(s_nl, (int)threadIdx.x) : s_nl[threadIdx.x];
                if (v >= 0) atomicMax(&fnl[ws + (int)threadIdx.x], v);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// k_careful: triangles of many tiles, and exact boxes of those the bound could not decide
// ---------------------------------------------------------------------------
// One wavefront per careful triangle.  CLS_SPANS: the lanes split the rows of
// the domain, each row's exact span comes from row_span(), and the box is the
// wave's min/max; CLS_FULL: the whole domain.  CLS_BOX / CLS_TIGHT triangles
// come here for their many tiles.  The lanes then append the triangle to every
// tile of the box, and lane 0 stores a box that the raster cannot derive.
template <bool COUNT>
__device__ __forceinline__ void careful_one(const Frame* __restrict__ frames, int tws,
                                            int ths, uint32_t* __restrict__ cursor, const uint64_t* __restrict__ off,
                                            uint32_t* __restrict__ pool, uint32_t* __restrict__ overflow,
                                            const uint4* __restrict__ careful_in, uint4* __restrict__ careful_box,
                                            uint32_t* __restrict__ careful_cnt, uint32_t odd_cols, uint32_t w, int lane)
{
    // (frame, frame triangle index, screen vertices as k_bin transformed them)
    const uint4 in = careful_in[2 * w], in2 = careful_in[2 * w + 1];
    const uint32_t frame = in.x;
    const Frame& fr = frames[frame];
    Tri t;
    t.x1 = __uint_as_float(in.z);
    t.y1 = __uint_as_float(in.w);
    t.x2 = __uint_as_float(in2.x);
    t.y2 = __uint_as_float(in2.y);
    t.x3 = __uint_as_float(in2.z);
    t.y3 = __uint_as_float(in2.w);
    tri_finish(fr.W, fr.H, t);
    const uint32_t T = in.y;
    const uint32_t cls = setup_class(t);
    int bx0 = t.x0, bx1 = t.x1d - 1, by0 = t.y0, by1 = t.y1d - 1;
    uint32_t entry = CAREFUL_FLAG | w;
    if (cls == CLS_SPANS) {
        int lo_x = 1 << 30, hi_x = -1, first = 1 << 30, last = -1;
        for (int y = t.y0 + lane; y < t.y1d; y += 64) {
            int l, h;
            if (row_span(t, y, l, h)) {
                lo_x = min(lo_x, l);
                hi_x = max(hi_x, h);
                first = min(first, y);
                last = max(last, y);
            }
        }
        bx0 = wave_min(lo_x);
        bx1 = wave_max(hi_x);
        by0 = wave_min(first);
        by1 = wave_max(last);
    } else if (cls == CLS_BOX || cls == CLS_TIGHT) {
        box_x(t, cls == CLS_TIGHT, bx0, bx1);
        entry = T | (cls == CLS_BOX ? LOOSE_FLAG : 0u);
    } else if (cls != CLS_FULL) {
        bx1 = -1;   // decided after all (cannot happen for entries k_bin sent here)
    }
    if (lane == 0 && !COUNT && entry == (CAREFUL_FLAG | w))
        careful_box[w] = make_uint4(T, (uint32_t)max(bx0, 0), (uint32_t)max(bx1, 0),
                                    (uint32_t)max(by0, 0) | ((uint32_t)max(by1, 0) << 16));
    if (bx0 > bx1 || by0 > by1) return;
    if ((fr.W & 1u) && lane == 0) {
        const uint32_t need = (uint32_t)odd_cols_of(bx1, fr.W, tws);
        if (COUNT) {
            if (need) atomicMax(&careful_cnt[WRAP_CNT], need);
        } else if (need > odd_cols) overflow[frame] = 1u;
    }
    TileRects r;
    tile_rects(bx0, bx1, by0, by1, fr.W, tws, ths, r);
    const int dw = r.dx1 - r.dx0 + 1, dh = r.dy1 - r.dy0 + 1;
    const int nd = (r.dx0 <= r.dx1 && r.dy0 <= r.dy1) ? dw * dh : 0;
    const int ww = r.wx1 - r.wx0 + 1, wh = r.wy1 - r.wy0 + 1;
    const int nw = (r.wx0 <= r.wx1 && r.wy0 <= r.wy1) ? ww * wh : 0;
    for (int k = lane; k < nd + nw; k += 64) {
        int tx, ty;
        if (k < nd) {
            tx = r.dx0 + k % dw;
            ty = r.dy0 + k / dw;
        } else {
            tx = r.wx0 + (k - nd) % ww;
            ty = r.wy0 + (k - nd) / ww;
            if (nd > 0 && in_direct(r, tx, ty)) continue;
        }
        const uint64_t gt = fr.tile_begin + (uint64_t)ty * fr.tiles_x + (uint64_t)tx;
        const uint32_t pos = atomicAdd(&cursor[gt], 1u);
        put_entry<COUNT>(gt, pos, entry, off, pool, overflow, frame);
    }
}

// careful_cnt[0] is the list length; careful_cnt[1 + g] the index where group
// g's triangles start (the bins of group g ran after those of group g - 1).
// Group g takes [careful_cnt[1 + g], length) and records the length as group
// g + 1's start.
template <bool COUNT>
__global__ void __launch_bounds__(256) k_careful(const Frame* __restrict__ frames, int tws, int ths, uint32_t* __restrict__ cursor,
                                                 const uint64_t* __restrict__ off, uint32_t* __restrict__ pool,
                                                 uint32_t* __restrict__ overflow, uint32_t* __restrict__ careful_cnt,
                                                 uint32_t group, const uint4* __restrict__ careful_in,
                                                 uint4* __restrict__ careful_box, uint32_t careful_cap,
                                                 uint32_t odd_cols)
{
    const int lane = (int)__lane_id();
    const uint32_t n = min(careful_cnt[0], careful_cap);
    const uint32_t first = careful_cnt[1 + group];
    const uint32_t n_waves = (gridDim.x * blockDim.x) >> 6;
    if (blockIdx.x == 0 && threadIdx.x == 0) careful_cnt[2 + group] = n;
    for (uint32_t w = first + ((blockIdx.x * blockDim.x + threadIdx.x) >> 6); w < n; w += n_waves)
        careful_one<COUNT>(frames, tws, ths, cursor, off, pool, overflow, careful_in, careful_box, careful_cnt, odd_cols,
                           w, lane);
}


// ---------------------------------------------------------------------------
// k_tile_raster
// ---------------------------------------------------------------------------
constexpr uint32_t CHUNK = RASTER_BLOCK;   // list entries whose triangles sit in LDS at once (one per thread)
// An entry's LDS row, an array per part (parts that are read together lie
// together, and rows drawn at random then spread over all banks): the shade
// factor or finished cell with the shader or ROW_CONST flag; the screen
// vertices' x and y; and, read by the big-box walk only, the depth terms.
struct Rows {
    uint2* end;
    float4* v12;
    float2* v3;
    float4* depth;
};
__host__ __device__ constexpr uint32_t row_bytes(bool big) { return big ? 48 : 32; }
// end.y of a row whose triangle has one glyph over its box (end.x is then the
// finished cell); ROW_NEGZ: its first vertex's depth is -0.  Other rows have the shader index (below 255) in the low byte.
constexpr uint32_t ROW_CONST = 0xFFu, ROW_NEGZ = 0x100u, ROW_MASK = 0x1FFu;
constexpr uint32_t LDS_RAMPS = 4;          // shaders staged in LDS per tile
static_assert(CHUNK <= 256, "tile keys hold a cache row index in one byte");

// A tile's z-test key: (depth code, frame triangle, sub) decide the order
// exactly as make_key's do; below them a `stored` flag and the cache row p
// of the entry that wrote the key (its lane in the chunk).  Two fragments
// with equal (depth code, triangle, sub) are the same fragment, so the low
// bits never change a comparison, and the resolve finds the winner's row from
// the key alone.  `stored` is set on keys whose winner's cell a multi-chunk
// tile has already put aside.
constexpr uint64_t TILE_KEY_STORED = 1u << 8;
// An empty slot: the code of f32::MAX, which no fragment reaches, so that its
// depth decodes like any other, and a low word of ones, which no fragment has
// (TILED_MAX_TRIS); its flag reads as stored.
constexpr uint64_t TILE_EMPTY = ((uint64_t)0xFF7FFFFFu << 32) | 0xFFFFFFFFu;
__device__ __forceinline__ bool tile_empty(uint64_t k) { return (uint32_t)k == 0xFFFFFFFFu; }
// (z is not -0: see walk_rect)
__device__ __forceinline__ uint64_t make_tile_key(float z, uint32_t tri, uint32_t sub, uint32_t p)
{
    return ((uint64_t)depth_bits_code(__float_as_uint(z)) << 32) | (uint64_t)((tri << 10) | (sub << 9) | p);
}
__device__ __forceinline__ uint32_t tile_key_tri(uint64_t k) { return (uint32_t)k >> 10; }
__device__ __forceinline__ uint32_t tile_key_sub(uint64_t k) { return ((uint32_t)k >> 9) & 1u; }
__device__ __forceinline__ uint32_t tile_key_row(uint64_t k) { return (uint32_t)k & 0xFFu; }

__device__ __forceinline__ const Draw& draw_of_t(const Draw* __restrict__ draws, const Frame& fr, uint32_t tri)
{
    uint32_t lo = fr.draw_begin, hi = fr.draw_end - 1;
    while (lo < hi) {
        uint32_t mid = (lo + hi + 1) >> 1;
        if (draws[mid].tri_begin <= tri) lo = mid; else hi = mid - 1;
    }
    return draws[lo];
}

// A tile's cells and z slots.  With W even a z slot id = y*W + 2x sits on an
// even column and owns its two cells: a tile row of TW cells holds TW/2
// slots (cs = 1).  With W odd, direct pixels land on even columns and
// wrapped ones (2x >= W, row y + 1) on odd columns, so every column holds a
// slot (cs = 0).  A pixel whose slot is cell column c of the tile's row r
// takes slot ((r - tr0) << sws) + ((c - tc0) >> cs).
struct TileGeom {
    int tc0, tc1, tr0, tr1;   // cell columns [tc0,tc1), rows [tr0,tr1)
    int sws;                  // log2(slots per tile row): log2(TW >> cs)
    int cs;                   // 1 for even W, 0 for odd W
    int W;
};

// Tests the pixels (x, y) in [xa, xb] x [ya, yb] of triangle t with the
// expressions of edges() and depth() and calls hit(slot, z, sub) for the
// covered ones: slot = row0 + ((y - ya) << sws) + (x - xa) * XS.
//
// WALK_COLS columns are taken at a time, all rows of them.  An edge function
// is fl(fl(A (py - ay)) - fl(B (px - ax))): its second product does not depend
// on the row, so the three of each column are made once and a pixel costs
// three subtractions of its own instead of nine operations; the slots of a
// row's columns differ by constants.  Columns past xb get an infinite product,
// which no pixel passes (the difference is -infinity or NaN).  Most boxes of a
// dense mesh are at most four wide: 1080p sweep, 4 columns 1.095 ms, 2 or 3
// 1.105, 5 1.09 and 6 1.12; a batch of unlike jobs 0.200, 0.221, 0.211, 0.202
// and 0.205 ms.  (Nine operations a pixel, one at a time: 1.195 and 0.241.)
//
// z is that of depth() but for -0, which reads +0: x + y is -0 only for two
// negative zeros, so adding +0 to the first vertex's depth is enough.  CHECK:
// z < f32::MAX (the z buffer's first value never loses, NaN never wins) is
// tested per pixel; without it the caller knows (depth_safe).
constexpr int WALK_COLS = 4;
template <int XS, bool CHECK, class Hit>
__device__ __forceinline__ void walk_rect(const Tri& t, int xa, int xb, int ya, int yb, int row0, int sws, uint32_t sub,
                                          Hit&& hit)
{
    const float z1 = t.z1 + 0.0f, dz2 = t.z2 - t.z1, dz3 = t.z3 - t.z1;
    for (int x = xa; x <= xb; x += WALK_COLS, row0 += WALK_COLS * XS) {
        float q0[WALK_COLS], q1[WALK_COLS], q2[WALK_COLS];
        float px = (float)x;   // below 2^16: stepping by 1.0f is exact
#pragma unroll
        for (int c = 0; c < WALK_COLS; ++c, px += 1.0f) {
            q0[c] = c == 0 || x + c <= xb ? t.B0 * (px - t.x2) : INFINITY;
            q1[c] = t.B1 * (px - t.x3);
            q2[c] = t.B2 * (px - t.x1);
        }
        int slot = row0;
        for (int y = ya; y <= yb; ++y, slot += 1 << sws) {
            const float py = (float)y;
            const float p0 = t.A0 * (py - t.y2), p1 = t.A1 * (py - t.y3), p2 = t.A2 * (py - t.y1);
#pragma unroll
            for (int c = 0; c < WALK_COLS; ++c) {
                const float w0 = p0 - q0[c], w1 = p1 - q1[c], w2 = p2 - q2[c];
                const float z = z1 + t.a * (w1 * dz2 + w2 * dz3);
                if (inside(w0, w1, w2) && (!CHECK || z < F32_MAX)) hit(slot + c * XS, z, sub);
            }
        }
    }
}

// Every pixel of a CLS_BOX / CLS_TIGHT triangle's box has a finite depth below
// f32::MAX: vertices within 2^22 and pixels below 2^16 give |w| < 2^47, so
// |z| < 2^60 + 2^15 2 2^47 2^61.
__device__ __forceinline__ bool depth_safe(const Tri& t)
{
    // (the IEEE 754-2019 maximum propagates NaN)
    const float m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(t.z1), fabsf(t.z2)), fabsf(t.z3));
    return m < 0x1p60f && fabsf(t.a) < 0x1p15f;
}

// walk_rect over the box's pixels that land in the tile's wrapped region
// (column 2x - W in [tc0,tc1), row y + 1).
template <int XS, class Hit>
__device__ __forceinline__ void walk_wrapped(const TileGeom& g, const Tri& t, int bx0, int bx1, int by0, int by1,
                                             Hit&& hit)
{
    const int xa = max(bx0, (g.tc0 + g.W + 1) >> 1), xb = min(bx1, (g.tc1 - 1 + g.W) >> 1);
    const int ya = max(by0, g.tr0 - 1), yb = min(by1, g.tr1 - 2);
    walk_rect<XS, true>(t, xa, xb, ya, yb, ((ya + 1 - g.tr0) << g.sws) + ((2 * xa - g.W - g.tc0) >> g.cs), g.sws, 0u, hit);
}

// Walks the candidate pixels of the box that land in the tile: the direct
// region (column 2x in [tc0,tc1), row y; safe: every lane is depth_safe), then
// the wrapped one.
template <int XS, class Hit>
__device__ __forceinline__ void walk_tile(const TileGeom& g, const Tri& t, int bx0, int bx1, int by0, int by1,
                                          bool safe, Hit&& hit)
{
    const int xa = max(bx0, (g.tc0 + 1) >> 1), xb = min(bx1, (g.tc1 - 1) >> 1);
    const int ya = max(by0, g.tr0), yb = min(by1, g.tr1 - 1);
    const int row0 = ((ya - g.tr0) << g.sws) + ((2 * xa - g.tc0) >> g.cs);
    if (safe) walk_rect<XS, false>(t, xa, xb, ya, yb, row0, g.sws, 1u, hit);
    else walk_rect<XS, true>(t, xa, xb, ya, yb, row0, g.sws, 1u, hit);
    walk_wrapped<XS>(g, t, bx0, bx1, by0, by1, hit);
}

// The direct part of the walk: the box clipped to the tile's logical pixels,
// as tile-relative [xa, xb] x [ya, yb] (empty when xa > xb or ya > yb).
__device__ __forceinline__ void direct_rect(const TileGeom& g, int bx0, int bx1, int by0, int by1, int& xa, int& xb,
                                            int& ya, int& yb)
{
    xa = max(bx0, g.tc0 >> 1) - (g.tc0 >> 1);
    xb = min(bx1, (g.tc1 - 1) >> 1) - (g.tc0 >> 1);
    ya = max(by0, g.tr0) - g.tr0;
    yb = min(by1, g.tr1 - 1) - g.tr0;
}

// The wrapped part, as the slots' columns and rows in the tile.
__device__ __forceinline__ void wrapped_rect(const TileGeom& g, int bx0, int bx1, int by0, int by1, int& xa, int& xb,
                                             int& ya, int& yb)
{
    const int ox = (g.tc0 + g.W + 1) >> 1;
    xa = max(bx0, ox) - ox;
    xb = min(bx1, (g.tc1 - 1 + g.W) >> 1) - ox;
    ya = max(by0, g.tr0 - 1) - (g.tr0 - 1);
    yb = min(by1, g.tr1 - 2) - (g.tr0 - 1);
}

// Order in which the pixels of a frame are written: by triangle, row, column
// (0: never).
__device__ __forceinline__ uint64_t pixel_time(uint32_t T, uint32_t py, uint32_t px)
{
    return (((uint64_t)T << 32) | ((uint64_t)py << 16) | px) + 1;
}

// Triangle index of a pool entry; the candidate box of a careful entry comes
// from its table row (given = true), the others' from box_x.
__device__ __forceinline__ uint32_t entry_tri(uint32_t e, const uint4* __restrict__ careful_box, int& bx0, int& bx1,
                                              int& by0, int& by1, bool& given, bool& tight)
{
    given = (e & CAREFUL_FLAG) != 0;
    tight = (e & LOOSE_FLAG) == 0;
    if (!given) return e & ~LOOSE_FLAG;
    const uint4 b = careful_box[e & ~CAREFUL_FLAG];
    bx0 = (int)b.y;
    bx1 = (int)b.z;
    by0 = (int)(b.w & 0xFFFFu);
    by1 = (int)(b.w >> 16);
    return b.x;
}

// One workgroup per tile; grid (tile x, tile y, frame - f_lo).  Blocks past a
// smaller frame's tile grid return at once.
//
// The tile's list is taken CHUNK entries at a time: each entry's row goes to
// the LDS row of its lane, and its fragments take a 64-bit LDS atomicMin of
// packed (depth, triangle, sub, row) keys (make_tile_key).  At the end every
// slot's cell comes from the row its key names and its depth from the key's
// code, and a thread stores two slots at a time.  With several chunks, after
// each but the last the slots whose key was written in that chunk put their
// cell aside in LDS and flag the key (a later winner comes from a later
// chunk), so that the frame is still written once, in 16-byte stores.
//
// What bounds it: VALU issue (a wave64 instruction takes four cycles of its
// SIMD).  A wavefront of entries costs about 240 instructions of set-up and 23
// per step of its largest box, and a slot pair about 35 at the end.
// 256 frames of 1920x1080, 327,680 triangles: 600M wavefront instructions, 0.98
// ms on 1024 SIMDs at 2.4 GHz, which is what it takes under the profiler (0.94 by
// events; the stores of its 4.26 GB alone take 0.75 ms).  Before,
// with rows of 48 bytes, nine operations more per pixel and chunk by chunk
// stores, 762M and 1.19 ms.
//
// BIG: an entry whose box covers more than BIG_BOX of the tile's pixels in
// its direct or its wrapped region is not walked there by its own lane; after its own walk, each
// wavefront takes its lanes' big boxes one at a time and all 64 lanes stride
// over the box.  The variant costs registers on every path, so it is launched
// only for lists with many big boxes (TiledPlan::big_walk).
//
// ONE: every frame of the launch has exactly one draw, so the draw is the
// same for the whole workgroup and its fields come through scalar loads that
// do not wait for the list entries.
//
// Frames of odd width: slots of direct pixels lie on even columns too, so most
// of their tiles take the same way as even frames' (rows then start at any
// 4-byte address, and a tile's last slot may have one cell).  Only wrapped
// pixels lie on odd columns, and the last column's pixels have their second
// cell in the next row: the first tile columns, as many as such boxes reach
// (odd_cols_of), take WRAP.  64 frames of 1919x1079 and 81,920 triangles, whose
// boxes reach one or two tile columns: 720 us a pass with all tiles WRAP, 420
// this way (0.06 ms of it the WRAP tiles', 0.007 k_tile_edges').
//
// WRAP: those tiles.  Every cell column holds a z slot (direct pixels
// on even columns, wrapped ones on odd columns) and a cell's final value is
// the later write of two slots' winners: its own slot's and the one to its
// left (rasterizer.rs:82-85 writes cells id and id + 1), and the row's
// newline for cell 1.  The tile first derives every slot's winner (depth
// and winner out, the cell into LDS), then resolves each cell whose two
// slots it holds; a first-column cell takes its own slot's winner here and
// is finished by k_tile_edges, from the winners this tile and its left
// neighbour leave in `edge_out` (first and last column, per row).
// Tile (tx, ty) of frame fr, global tile index gt, whose list is pool[o, o + n).
// KIND: EVEN for launches most of whose widths are multiples of 32 cells (a
// 128-byte line), RAGGED for the others of even widths, ANY for those with odd
// ones, WRAPPED for WRAP tiles.  FLAT is that of the calling kernel and changes nothing here: it gives each
// kernel its own copy of the lambdas below, which the compiler then inlines
// as it does for a single caller (shared by the two kernels, they cost the
// 3-D instances two VGPRs spilled to scratch).
enum RasterKind { EVEN, RAGGED, ANY, WRAPPED };
template <bool BIG, bool ONE, RasterKind KIND, bool FLAT>
__device__ __forceinline__ void raster_tile(const Draw* __restrict__ draws, const Ramp* __restrict__ ramps,
                                            const Ramp* s_ramp, uint32_t* s_negz, const Frame& fr, uint32_t tx,
                                            uint32_t ty, uint64_t gt, uint64_t o, uint32_t n, int tws, int ths,
                                            const uint32_t* __restrict__ pool, const int32_t* __restrict__ nl,
                                            const uint4* __restrict__ careful_box, uint32_t* __restrict__ cells,
                                            float* __restrict__ zbuf, int32_t* __restrict__ win, uint32_t win_raw,
                                            uint4* __restrict__ edge_out, uint64_t* smem, uint32_t keep)
{
    constexpr bool WRAP = KIND == WRAPPED, EVENS = KIND == EVEN || KIND == RAGGED;
    static_assert(!(BIG && WRAP), "the big-box walk maps slots of even columns only");
    const uint32_t W = fr.W, H = fr.H;
    const int sws = tws - (WRAP ? 0 : 1);
    const uint32_t S = 1u << (sws + ths);
    TileGeom g;
    g.tc0 = (int)(tx << tws);
    g.tc1 = min((int)W, g.tc0 + (1 << tws));
    g.tr0 = (int)(ty << ths);
    g.tr1 = min((int)H, g.tr0 + (1 << ths));
    g.sws = sws;
    g.cs = WRAP ? 0 : 1;
    g.W = (int)W;

    const uint32_t* list = pool + o;
    uint64_t* keys = smem;
    // (S, the tile's slots, is a power of two of at least 16)
    static_assert(CHUNK * sizeof(uint2) % 16 == 0 && CHUNK * sizeof(float4) % 16 == 0 && CHUNK * sizeof(float2) % 16 == 0,
                  "each array of the rows, and the cells after them, start on 16 bytes");
    Rows rows;
    rows.end = (uint2*)(keys + S);
    rows.v12 = (float4*)(rows.end + CHUNK);
    rows.v3 = (float2*)(rows.v12 + CHUNK);
    rows.depth = (float4*)(rows.v3 + CHUNK);   // BIG only
    // a cell per slot: WRAP, the winners' for the per-cell resolve; else, in
    // tiles of several chunks, those put aside
    uint32_t* wcell = (uint32_t*)(keys + S) + CHUNK * row_bytes(BIG) / 4;

    const int32_t* fnl = nl + fr.nl_off;
    uint32_t* fc = cells + fr.cell_off;
    float* fz = zbuf + fr.z_off;
    auto win_of = [&](uint64_t k) -> uint32_t {
        // win_raw gives triangle << 1 | sub for the shading pass
        return tile_empty(k) ? 0xFFFFFFFFu : win_raw ? (uint32_t)k >> 9 : tile_key_tri(k);
    };
    // WRAP: a thread owns the slots of one column of the tile, every
    // row_step-th row (the block is at least one tile row of slots wide):
    // fn(slot, row, id of the slot's first cell) over its slots in the frame.
    const uint32_t my_sc = threadIdx.x & ((1u << sws) - 1);
    const int my_col = g.tc0 + ((int)my_sc << g.cs);
    auto for_my_slots = [&](auto&& fn) {
        if (my_col >= g.tc1) return;
        const int row_step = (int)(blockDim.x >> sws);
        const uint64_t id_step = (uint64_t)row_step * W;
        int row = g.tr0 + (int)(threadIdx.x >> sws);
        uint64_t id = (uint64_t)row * W + (uint64_t)my_col;
        for (; row < g.tr1; row += row_step, id += id_step)
            fn(((uint32_t)(row - g.tr0) << sws) | my_sc, row, id);
    };
    // WRAP: stores slot s's depth and winner, its cell into wcell.
    auto store_slot = [&](uint32_t s, uint64_t id, uint64_t k, uint32_t cell, float z) {
        __builtin_nontemporal_store(z, fz + id);
        if (win) __builtin_nontemporal_store((int32_t)win_of(k), win + fr.z_off + id);
        if (!tile_empty(k)) wcell[s] = cell;
    };
    // Otherwise a thread takes the slot pairs (2q, 2q + 1) of a row, q = thread
    // mod (slots a row / 2), every (512 >> sws)-th row: fn(first slot, row, its
    // first cell's column, that cell's byte offset from the tile's first cell,
    // the cells of the four that lie in the frame).  Addresses are the tile's (uniform)
    // plus 32 bits a lane (a tile spans at most 64 rows of 65535 cells).
    auto for_my_pairs = [&](auto&& fn) {
        const uint32_t q = threadIdx.x & ((1u << (sws - 1)) - 1);
        const int col = g.tc0 + ((int)q << 2);
        if (col >= g.tc1) return;
        const int have = EVENS ? (col + 2 < g.tc1 ? 4 : 2) : min(g.tc1 - col, 4);
        const int step = (int)(blockDim.x >> (sws - 1));
        int r = (int)(threadIdx.x >> (sws - 1));
        uint32_t off = ((uint32_t)r * W + (q << 2)) * 4u;
        for (; r < g.tr1 - g.tr0; r += step, off += (uint32_t)step * W * 4u)
            fn(((uint32_t)r << sws) | (q << 1), g.tr0 + r, col, off, have);
    };
    const uint64_t tile0 = (uint64_t)g.tr0 * W + (uint64_t)g.tc0;
    uint8_t* tile_cells = (uint8_t*)(fc + tile0);
    uint8_t* tile_z = (uint8_t*)(fz + tile0);
    uint8_t* tile_win = win ? (uint8_t*)(win + fr.z_off + tile0) : nullptr;
    // Streaming stores: the frame is written once and not read back here.
    // Words need only their own alignment: a 16-byte store at any 4-byte
    // address is one instruction.
    typedef unsigned int v4u __attribute__((ext_vector_type(4), aligned(4)));
    typedef unsigned int v2u __attribute__((ext_vector_type(2), aligned(4)));
    // But where `keep` says so, the lines that a row shares with the tiles beside
    // it are written by ordinary stores, which stay in the L2 until the
    // neighbour's part has come (TiledPlan::keep_lines).
    const bool shared_lines = keep && (W & 31u);
    auto put4 = [&](uint8_t* p, uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
        const v4u v = {a, b, c, d};
        if (KIND != EVEN && shared_lines) {
            const uint32_t at = (uint32_t)(uintptr_t)p, row = at - ((threadIdx.x & ((1u << (tws - 2)) - 1)) << 4);
            if ((at & ~127u) < row || ((at + 15u) | 127u) >= row + (4u << tws)) {
                *(v4u*)p = v;
                asm volatile("");   // keeps the two stores two
                return;
            }
        }
        __builtin_nontemporal_store(v, (v4u*)p);
    };
    // the first `have` < 4 words (ANY: 1 and 3 at an odd width's last column)
    auto put_some = [](uint8_t* p, uint32_t a, uint32_t b, uint32_t c, int have) {
        if (EVENS || (have & 2)) {
            const v2u v = {a, b};
            __builtin_nontemporal_store(v, (v2u*)p);
        }
        if (KIND == ANY && (have & 1)) __builtin_nontemporal_store(have == 1 ? a : c, (uint32_t*)p + (have - 1));
    };
    const bool nl_here = fr.image && tx == 0;
    // Stores a pair from its keys' low words, cells and depths.
    auto store_pair = [&](int row, int col, uint32_t off, int have, uint32_t k0, uint32_t c0, float z0, uint32_t k1,
                          uint32_t c1, float z1) {
        uint32_t c0b = c0;
        if (nl_here && col == 0) {
            // cell row*W + 1: the newline of row `row` comes after every pixel
            // of its triangle's row and before its next row, so it overwrites
            // a wrapped pixel (drawn in row-1) of the same or an earlier
            // triangle
            const int32_t nlr = fnl[row];
            if (nlr >= 0 && (tile_empty(k0) || nlr >= (int32_t)tile_key_tri(k0))) c0b = CELL_NEWLINE;
        }
        if (have == 4) {
            put4(tile_cells + off, c0, c0b, c1, c1);
            put4(tile_z + off, __float_as_uint(z0), __float_as_uint(F32_MAX), __float_as_uint(z1), __float_as_uint(F32_MAX));
            if (win) put4(tile_win + off, win_of(k0), 0xFFFFFFFFu, win_of(k1), 0xFFFFFFFFu);
            return;
        }
        put_some(tile_cells + off, c0, c0b, c1, have);
        put_some(tile_z + off, __float_as_uint(z0), __float_as_uint(F32_MAX), __float_as_uint(z1), have);
        if (win) put_some(tile_win + off, win_of(k0), 0xFFFFFFFFu, win_of(k1), have);
        if (KIND == ANY && edge_out && (have & 1)) {
            // the last column of an odd width: its second cell is k_tile_edges'
            const uint32_t k = have == 1 ? k0 : k1;
            uint4 e = make_uint4(have == 1 ? c0 : c1, 0u, 0u, 0u);
            if (!tile_empty(k)) {
                const uint64_t t = pixel_time(tile_key_tri(k), (uint32_t)row, W >> 1);
                e.z = (uint32_t)t;
                e.w = (uint32_t)(t >> 32);
            }
            edge_out[(gt * (1u << ths) + (uint64_t)(row - g.tr0)) * 2 + 1] = e;
        }
    };

    if (n == 0) {
        // no triangle reaches the tile: blank cells, f32::MAX depths, and the
        // newline cells of column 1
        if constexpr (WRAP)
            for_my_slots([&](uint32_t s, int, uint64_t id) { store_slot(s, id, TILE_EMPTY, CELL_BLANK, F32_MAX); });
        else
            for_my_pairs([&](uint32_t, int row, int col, uint32_t off, int have) {
                store_pair(row, col, off, have, ~0u, CELL_BLANK, F32_MAX, ~0u, CELL_BLANK, F32_MAX);
            });
    } else {
        // glyph of shade sh under shader r: the first LDS_RAMPS shaders from
        // LDS, the others from global memory (two calls, so that each reads
        // its own address space rather than through generic pointers)
        auto glyph_of = [&](uint32_t r, float sh) -> uint32_t {
            if (r < LDS_RAMPS) return ramp_glyph(s_ramp[r], sh);
            return ramp_glyph(ramps[r], sh);
        };
        // The glyph a triangle gives every pixel of its box when that is
        // provably one glyph, else ~0u.  The pixel's shade is fl(na * S) with
        // S = fl(fl(w0 + w1) + w2) (rasterizer.rs:76).  Each FP32 edge
        // function errs from the exact one by at most
        // 4.0003u (|A| |py - ay| + |B| |px - ax|) (u = 2^-24), the exact ones
        // sum to the exact orient, the two additions add at most 2.0001u of
        // their inputs' magnitudes, and the FP32 orient o errs from the exact
        // one by at most 4.0002u (|A2| |y3 - y1| + |B2| |x3 - x1|).  So every
        // S lies within E = 10u (Sb + Q) of o, with Sb the edge terms' sum
        // over the box and Q o's terms; 10u also covers the rounding of E
        // and of o -+ E (Sb >= |o|).  `terms` is Sb + Q or more.  fl(na * .)
        // and the step index are monotone, so equal indices at the two ends
        // mean one glyph for the whole box.  Shaders that are not
        // non-decreasing, and non-finite values, take the per-pixel
        // evaluation.
        //
        // na comes here from the hardware reciprocal square root: na_h =
        // fl(fl(nz rsq(n2)) a), rsq within 1 ulp, so for n2 in [2^-100,
        // 2^100] na_h lies within 2^-21 |na| of the reference's fl(fl(nz /
        // sqrt(n2)) a) (two roundings each side).  Every fl(na S) then lies
        // between fl(na_h (o - E')) and fl(na_h (o + E')) with E' = E +
        // 2^-19 (|o| + E).  The lower end's step index i is counted, and the
        // upper end compared with threshold i: both ends have index i when
        // it is at most thr[i] (thresholds are non-decreasing).
        auto box_glyph = [&](const Ramp& rp, const Tri& t, float na, float terms) -> uint32_t {
            if (!rp.sorted) return ~0u;
            const float ey = t.y3 - t.y1, ex = t.x3 - t.x1;
            const float o = t.A2 * ey - t.B2 * ex;
            const float E = 5.9604645e-07f * terms;
            const float E2 = E + 0x1p-19f * (fabsf(o) + E);
            const float s1 = na * (o - E2), s2 = na * (o + E2);
            // NaN or infinity anywhere fails the finite test (v_maximum3 propagates NaN)
            const float mag = __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(na), fabsf(s1)), fabsf(s2));
            if (!(mag < INFINITY)) return ~0u;
            const float lo = fminf(s1, s2), hi = fmaxf(s1, s2);
            const uint32_t i = ramp_index_sorted(rp, lo);
            if (i < rp.n && !(hi <= rp.thr[i])) return ~0u;
            return i < rp.n ? rp.glyph[i] : rp.fallback;
        };
        const bool one_draw = fr.draw_end - fr.draw_begin == 1;
        const bool multi = n > CHUNK;
        auto draw_of_tri = [&](uint32_t T) -> const Draw& {
            return ONE ? draws[fr.draw_begin] : one_draw ? draws[fr.draw_begin] : draw_of_t(draws, fr, T);
        };
        // the pixel that key k denotes at the slot of cell (row, col)
        auto pixel_of = [&](int col, int row, uint64_t k, float& px, float& py) {
            const uint32_t sub = tile_key_sub(k);
            px = (float)(sub ? (col >> 1) : ((col + g.W) >> 1));
            py = (float)(sub ? row : row - 1);
        };
        // The depth of slot (row, col)'s winner from its mesh: zero depths,
        // whose sign the code does not keep.
        auto mesh_depth = [&](int col, int row, uint64_t k) -> float {
            const uint32_t T = tile_key_tri(k);
            const Draw& dr = draw_of_tri(T);
            Tri t;
            setup_draw_tri(dr, T - dr.tri_begin, W, H, t);
            float px, py, w0, w1, w2;
            pixel_of(col, row, k, px, py);
            edges(t, px, py, w0, w1, w2);
            return depth(t, w1, w2);
        };
        // Cell and depth of a winner whose row is not plainly ROW_CONST: the
        // expressions of edges() and shade_value() on the row's vertices.
        // A zero depth is -0 only when its first vertex's is (x + y = -0 only
        // for two negative zeros), so a ROW_CONST row without ROW_NEGZ never
        // comes here for its sign.
        auto winner_slow = [&](int col, int row, uint64_t k, uint32_t& cell, float& z) {
            const uint32_t r = tile_key_row(k);
            const uint2 end = rows.end[r];
            const uint32_t cw = end.y;
            const uint32_t code = (uint32_t)(k >> 32);
            cell = end.x;
            z = depth_of_code(code);
            if (code == DEPTH_CODE_ZERO) z = mesh_depth(col, row, k);
            if ((cw & 0xFFu) == ROW_CONST) return;
            float px, py;
            pixel_of(col, row, k, px, py);
            const float4 v12 = rows.v12[r];
            const float2 v3 = rows.v3[r];
            const float x1 = v12.x, y1 = v12.y, x2 = v12.z, y2 = v12.w, x3 = v3.x, y3 = v3.y;
            const float w0 = (x3 - x2) * (py - y2) - (y3 - y2) * (px - x2);
            const float w1 = (x1 - x3) * (py - y3) - (y1 - y3) * (px - x3);
            const float w2 = (x2 - x1) * (py - y1) - (y2 - y1) * (px - x1);
            const float sh = __uint_as_float(end.x) * (w0 + w1 + w2);
            cell = glyph_of(cw & 0xFFu, sh) | (cw & 0xFFFFFF00u);
        };
        auto row_end = [&](uint64_t k) -> uint2 { return rows.end[tile_key_row(k)]; };
        auto plain = [](uint2 w) { return (w.y & ROW_MASK) == ROW_CONST; };

        for (uint32_t s = threadIdx.x; s < S; s += blockDim.x) keys[s] = TILE_EMPTY;
        if (!WRAP && threadIdx.x == 0) *s_negz = 0;
        // the next chunk's entry, read while this one's slots are looked over (a
        // 4K frame of 1,310,720 triangles: 65.7 -> 64.7 us)
        uint32_t next = threadIdx.x < n ? list[threadIdx.x] : 0u;
        for (uint32_t base = 0; base < n; base += CHUNK) {
            __syncthreads();   // keys cleared / the previous chunk's cells no longer read its rows
            const uint32_t p = threadIdx.x;
            // BIG: the direct / wrapped part of this lane's box is walked by its
            // wavefront (the wrapped part by its lane alone: a few triangles of
            // 200 pixels a side on a 2560x1440 frame took 97 us, now 27)
            bool big = false, big_w = false;
            uint32_t big_T = 0, big_rect = 0, big_rect_w = 0;
            // the entry of this thread.  BIG: a list of a few entries is dealt
            // out over the wavefronts, which walk their big boxes one by one
            // (30 unlike jobs in turn: 171 -> 158 us; dealing out up to 40
            // entries costs batches of small triangles their set-up in four
            // wavefronts: 523 -> 590 us for 64 frames of 1919x1079 at 64 x 16)
            const uint32_t at = BIG && n <= 16 ? ((p & 63u) << 2) | (p >> 6) : base + p;
            if (at < n) {
                int bx0, bx1, by0, by1;
                bool given, tight;
                const uint32_t T = entry_tri(BIG && n <= 16 ? list[at] : next, careful_box, bx0, bx1, by0, by1, given, tight);
                const Draw& dr = draw_of_tri(T);
                const uint32_t li = T - dr.tri_begin;
                Tri t;
                setup_draw_tri(dr, li, W, H, t);
                float nz, n2;
                normal_parts(t, nz, n2);
                const auto* c = global_ptr(dr.rgb + (size_t)li * 3);
                const uint32_t rgb = ((uint32_t)c[0] << 8) | ((uint32_t)c[1] << 16) | ((uint32_t)c[2] << 24);
                // Sb + Q of the glyph proof.  Boxes of box_x lie within a
                // pixel of the vertices' extent in x and inside it in y, the
                // |A_k| sum to 2 wx and the |B_k| to 2 wy (the extents), and
                // Q <= 2 wx wy: at most 2 wx wy + 2 wy (wx + 1) + 2 wx wy.
                const float wx = t.maxx - t.minx, wy = t.maxy - t.miny;
                float terms = wy * (6.0f * wx + 2.0f);
                if (!given) {
                    box_x(t, tight, bx0, bx1);
                    by0 = t.y0;
                    by1 = t.y1d - 1;
                } else {
                    // careful boxes: the edge terms' exact maximum over the
                    // box, edge by edge (an empty box has no pixels, so its
                    // glyph is never used)
                    const float X0 = (float)bx0, X1 = (float)bx1, Y0 = (float)by0, Y1 = (float)by1;
                    terms = fabsf(t.A0) * fmaxf(fabsf(Y0 - t.y2), fabsf(Y1 - t.y2)) + fabsf(t.B0) * fmaxf(fabsf(X0 - t.x2), fabsf(X1 - t.x2)) +
                            fabsf(t.A1) * fmaxf(fabsf(Y0 - t.y3), fabsf(Y1 - t.y3)) + fabsf(t.B1) * fmaxf(fabsf(X0 - t.x3), fabsf(X1 - t.x3)) +
                            fabsf(t.A2) * fmaxf(fabsf(Y0 - t.y1), fabsf(Y1 - t.y1)) + fabsf(t.B2) * fmaxf(fabsf(X0 - t.x1), fabsf(X1 - t.x1)) +
                            fabsf(t.A2) * fabsf(t.y3 - t.y1) + fabsf(t.B2) * fabsf(t.x3 - t.x1);
                }
                // a triangle with one glyph over its box keeps its finished
                // cell where the shade factor would be
                uint32_t bg = ~0u;
                if (n2 >= 0x1p-100f && n2 <= 0x1p100f) {
                    const float na_h = nz * __builtin_amdgcn_rsqf(n2) * t.a;
                    const uint32_t r = dr.ramp;
                    bg = r < LDS_RAMPS ? box_glyph(s_ramp[r], t, na_h, terms) : box_glyph(ramps[r], t, na_h, terms);
                }
                uint32_t w2 = bg | rgb;
                uint32_t w3 = ROW_CONST | (__float_as_uint(t.z1) == 0x80000000u ? ROW_NEGZ : 0u);
                // the others keep the shade factor (rasterizer.rs:76
                // multiplies the unit normal's z by a first)
                if (bg == ~0u) {
                    w2 = __float_as_uint(nz / sqrtf(n2) * t.a);
                    w3 = rgb | dr.ramp;
                }
                rows.end[p] = make_uint2(w2, w3);
                rows.v12[p] = make_float4(t.x1, t.y1, t.x2, t.y2);
                rows.v3[p] = make_float2(t.x3, t.y3);
                if constexpr (BIG) rows.depth[p] = make_float4(t.z1 + 0.0f, t.z2 - t.z1, t.z3 - t.z1, t.a);   // no -0, as walk_rect
                const bool safe = __ballot(given || !depth_safe(t)) == 0;
                if (bx0 <= bx1 && by0 <= by1) {
                    auto hit = [&](int slot, float z, uint32_t sub) {
                        atomicMin((unsigned long long*)&keys[slot], (unsigned long long)make_tile_key(z, T, sub, p));
                    };
                    constexpr int XS = WRAP ? 2 : 1;
                    if constexpr (BIG) {
                        int xa, xb, ya, yb;
                        direct_rect(g, bx0, bx1, by0, by1, xa, xb, ya, yb);
                        if (xa <= xb && ya <= yb && (xb - xa + 1) * (yb - ya + 1) > (int)BIG_BOX) {
                            big = true;
                            big_rect =
                                (uint32_t)xa | ((uint32_t)xb << 8) | ((uint32_t)ya << 16) | ((uint32_t)yb << 24);
                        } else {
                            if (safe)
                                walk_rect<XS, false>(t, xa + (g.tc0 >> 1), xb + (g.tc0 >> 1), ya + g.tr0, yb + g.tr0,
                                                     (ya << sws) + xa, sws, 1u, hit);
                            else
                                walk_rect<XS, true>(t, xa + (g.tc0 >> 1), xb + (g.tc0 >> 1), ya + g.tr0, yb + g.tr0,
                                                    (ya << sws) + xa, sws, 1u, hit);
                        }
                        wrapped_rect(g, bx0, bx1, by0, by1, xa, xb, ya, yb);
                        if (xa <= xb && ya <= yb) {
                            big_w = (xb - xa + 1) * (yb - ya + 1) > (int)BIG_BOX;
                            big_rect_w =
                                (uint32_t)xa | ((uint32_t)xb << 8) | ((uint32_t)ya << 16) | ((uint32_t)yb << 24);
                            if (!big_w) walk_wrapped<XS>(g, t, bx0, bx1, by0, by1, hit);
                        }
                        big_T = T;
                    } else {
                        walk_tile<XS>(g, t, bx0, bx1, by0, by1, safe, hit);
                    }
                }
            }
            if constexpr (BIG) {
                // The wavefront's big boxes, one at a time: lane l of the box
                // takes pixels i = l, l + 64, ... (row i / nx, column i % nx),
                // with the expressions of edges() and depth() on the box's
                // row (row p of the lane that holds it, written by this
                // wavefront above).
                uint64_t m = __ballot(big), m_w = __ballot(big_w);
                while (m | m_w) {
                    const bool direct = m != 0;
                    const int l = __builtin_ctzll(direct ? m : m_w);
                    if (direct) m &= m - 1;
                    else m_w &= m_w - 1;
                    const uint32_t T = __builtin_amdgcn_readlane(big_T, l);
                    const uint32_t rc = direct ? __builtin_amdgcn_readlane(big_rect, l) : __builtin_amdgcn_readlane(big_rect_w, l);
                    // the pixel of the tile's first slot
                    const int ox = direct ? g.tc0 >> 1 : (g.tc0 + g.W + 1) >> 1, oy = direct ? g.tr0 : g.tr0 - 1;
                    const uint32_t prow = (threadIdx.x & ~63u) + (uint32_t)l;   // the owner lane's row
                    const float4 v12 = rows.v12[prow], q2 = rows.depth[prow];
                    const float2 v3 = rows.v3[prow];
                    const float x1 = v12.x, y1 = v12.y, x2 = v12.z, y2 = v12.w, x3 = v3.x, y3 = v3.y;
                    const float A0 = x3 - x2, B0 = y3 - y2, A1 = x1 - x3, B1 = y1 - y3, A2 = x2 - x1, B2 = y2 - y1;
                    const float z1 = q2.x, dz2 = q2.y, dz3 = q2.z, a = q2.w;
                    const int xa = (int)(rc & 0xFFu), nx = (int)((rc >> 8) & 0xFFu) - xa + 1;
                    const int ya = (int)((rc >> 16) & 0xFFu), ny = (int)(rc >> 24) - ya + 1;
                    const int dy = 64 / nx, dx = 64 - dy * nx;
                    int i = (int)__lane_id(), yy = i / nx, xx = i - yy * nx;
                    for (; i < nx * ny; i += 64) {
                        const int x = xa + xx, y = ya + yy;
                        const float px = (float)(x + ox), py = (float)(y + oy);
                        const float w0 = A0 * (py - y2) - B0 * (px - x2);
                        const float w1 = A1 * (py - y3) - B1 * (px - x3);
                        const float w2 = A2 * (py - y1) - B2 * (px - x1);
                        const float z = z1 + a * (w1 * dz2 + w2 * dz3);
                        if (inside(w0, w1, w2) && z < F32_MAX)
                            atomicMin((unsigned long long*)&keys[(y << sws) + x],
                                      (unsigned long long)make_tile_key(z, T, direct ? 1u : 0u, prow));
                        xx += dx;
                        yy += dy;
                        if (xx >= nx) {
                            xx -= nx;
                            ++yy;
                        }
                    }
                }
            }
            if (base + CHUNK + p < n) next = list[base + CHUNK + p];
            __syncthreads();
            if constexpr (WRAP) {
                if (multi)
                    // slots whose key was written in this chunk (no stored
                    // flag) store that winner and flag the key; a later chunk
                    // that changes the key stores again.  The same thread
                    // owns slot s throughout, so its last store lands last.
                    for_my_slots([&](uint32_t s, int row, uint64_t id) {
                        const uint64_t k = keys[s];
                        if (k & TILE_KEY_STORED) return;   // or empty
                        const uint2 w = row_end(k);
                        uint32_t cell = w.x;
                        float z = depth_of_code((uint32_t)(k >> 32));
                        if (!plain(w)) winner_slow(my_col, row, k, cell, z);
                        store_slot(s, id, k, cell, z);
                        keys[s] = k | TILE_KEY_STORED;
                    });
            } else {
                if (multi && base + CHUNK < n)
                    // slots whose key was written in this chunk put their
                    // cell aside (the rows go to the next chunk); a slot whose
                    // depth is -0 is remembered for the tile
                    for (uint32_t s = threadIdx.x; s < S; s += blockDim.x) {
                        const uint64_t k = keys[s];
                        if (k & TILE_KEY_STORED) continue;   // or empty
                        const uint2 w = row_end(k);
                        uint32_t cell = w.x;
                        if (!plain(w)) {
                            float z;
                            winner_slow(g.tc0 + (int)((s & ((1u << sws) - 1)) << 1), g.tr0 + (int)(s >> sws), k, cell, z);
                            if (__float_as_uint(z) == 0x80000000u) *s_negz = 1;
                        }
                        wcell[s] = cell;
                        *(uint32_t*)(keys + s) = (uint32_t)k | (uint32_t)TILE_KEY_STORED;
                    }
            }
        }
        if constexpr (WRAP) {
            for_my_slots([&](uint32_t s, int row, uint64_t id) {
                const uint64_t k = keys[s];
                if (multi && !tile_empty(k)) return;   // stored after its chunk
                uint32_t cell = CELL_BLANK;
                float z = F32_MAX;
                if (!tile_empty(k)) {
                    const uint2 w = row_end(k);
                    cell = w.x;
                    z = depth_of_code((uint32_t)(k >> 32));
                    if (!plain(w)) winner_slow(my_col, row, k, cell, z);
                }
                store_slot(s, id, k, cell, z);
            });
        } else {
            const bool negz = multi && *s_negz != 0;
            for_my_pairs([&](uint32_t s, int row, int col, uint32_t off, int have) {
                const uint4 kk = *(const uint4*)(keys + s);   // low and high words of the two keys
                const uint2 w0 = rows.end[kk.x & 0xFFu], w1 = rows.end[kk.z & 0xFFu];
                uint32_t c0 = w0.x, c1 = w1.x;
                float z0 = depth_of_code(kk.y), z1 = depth_of_code(kk.w);
                const bool own0 = !(kk.x & (uint32_t)TILE_KEY_STORED), own1 = !(kk.z & (uint32_t)TILE_KEY_STORED);
                if (multi) {
                    const uint2 st = *(const uint2*)(wcell + s);
                    c0 = own0 ? c0 : st.x;
                    c1 = own1 ? c1 : st.y;
                }
                // the few whose row does not say it all (empty and stored
                // slots read some row too: never here), one after another
                uint32_t rest = (own0 && !plain(w0) ? 1u : 0u) | (own1 && !plain(w1) ? 2u : 0u);
                while (rest) {
                    const bool second = rest == 2u;
                    uint32_t cell;
                    float zz;
                    winner_slow(second ? col + 2 : col, row,
                                second ? ((uint64_t)kk.w << 32) | kk.z : ((uint64_t)kk.y << 32) | kk.x, cell, zz);
                    c0 = second ? c0 : cell;
                    z0 = second ? z0 : zz;
                    c1 = second ? cell : c1;
                    z1 = second ? zz : z1;
                    rest &= rest - 1;
                }
                if (negz) {
                    // a stored winner's zero depth: its sign from its mesh
                    for (int i = 0; i < 2; ++i) {
                        const uint32_t lo = i ? kk.z : kk.x, hi = i ? kk.w : kk.y;
                        if ((lo & (uint32_t)TILE_KEY_STORED) && hi == DEPTH_CODE_ZERO) {
                            const float zi = mesh_depth(col + 2 * i, row, lo);
                            z0 = i ? z0 : zi;
                            z1 = i ? zi : z1;
                        }
                    }
                }
                store_pair(row, col, off, have, kk.x, tile_empty(kk.x) ? CELL_BLANK : c0, z0, kk.z,
                           tile_empty(kk.z) ? CELL_BLANK : c1, z1);
            });
        }
    }
    if constexpr (WRAP) {
        // Each cell: the later write of its own slot's winner and the left
        // slot's (write time = triangle, then the pixel's row and column,
        // as the sequential loop orders them), and for cell 1 the row's
        // newline, which follows its triangle's pixels of that row.
        const bool any = n > 0;
        if (any) __syncthreads();   // every slot's winner cell is in wcell
        auto slot_time = [&](uint64_t k, int row, int col) -> uint64_t {
            const uint32_t sub = tile_key_sub(k);
            const uint32_t py = sub ? (uint32_t)row : (uint32_t)row - 1u;
            const uint32_t px = sub ? (uint32_t)col >> 1 : (uint32_t)(col + (int)W) >> 1;
            return pixel_time(tile_key_tri(k), py, px);
        };
        for_my_slots([&](uint32_t s, int row, uint64_t id) {
            uint64_t t_own = 0, t_best = 0;
            uint32_t c_own = CELL_BLANK, best = CELL_BLANK;
            if (any) {
                const uint64_t k = keys[s];
                if (!tile_empty(k)) {
                    t_own = slot_time(k, row, my_col);
                    c_own = wcell[s];
                }
                t_best = t_own;
                best = c_own;
                if (my_col > g.tc0) {
                    const uint64_t kl = keys[s - 1];
                    if (!tile_empty(kl)) {
                        const uint64_t tl = slot_time(kl, row, my_col - 1);
                        if (tl > t_best) {
                            t_best = tl;
                            best = wcell[s - 1];
                        }
                    }
                }
            }
            if (fr.image && my_col == 1) {
                const int32_t nlr = fnl[row];
                if (nlr >= 0) {
                    const uint64_t tn = (((uint64_t)(uint32_t)nlr << 32) | ((uint64_t)row << 16) | 0xFFFFu) + 1;
                    if (tn > t_best) best = CELL_NEWLINE;
                }
            }
            __builtin_nontemporal_store(best, fc + id);
            uint4* e = edge_out + (gt * (1u << ths) + (uint64_t)(row - g.tr0)) * 2;
            if (my_col == g.tc0) e[0] = make_uint4(c_own, 0u, (uint32_t)t_own, (uint32_t)(t_own >> 32));
            if (my_col == g.tc1 - 1) e[1] = make_uint4(c_own, 0u, (uint32_t)t_own, (uint32_t)(t_own >> 32));
        });
    }
    // image mode: the H cells after the W*H grid are never written (context.rs:38-40)
    if (fr.image && tx == 0 && ty == 0)
        for (uint32_t i = threadIdx.x; i < H; i += blockDim.x) __builtin_nontemporal_store(CELL_BLANK, fc + (uint64_t)W * H + i);
}

// The tile of a frame's workgroup r, RAGGED and ANY (3-D grids; flat ones keep
// their table's order): workgroups go to the eight
// XCDs in turn, so taking eight tile rows at a time gives each XCD, and its L2,
// whole rows.  The rows of such widths start within a line, and the lines that
// two tiles of a row share are then put together before they leave for memory:
// 64 frames of 1919x1079 at 128 x 16 cells 474 -> 416 us, at 32 x 32 1020 -> 727;
// of 1918x1079 at 128 x 16 465 -> 410, at 64 x 32 620 -> 524.  Where tiles share
// no line, 256 frames of 1920x1080 lose (1.79 -> 1.825 ms) and keep the plain order.
__device__ __forceinline__ void tile_of(uint32_t r, uint32_t nx, uint32_t ny, uint32_t& tx, uint32_t& ty)
{
    const uint32_t full = (ny & ~7u) * nx;
    if (r < full) {
        const uint32_t j = r >> 3, g = j / nx;
        tx = j - g * nx;
        ty = 8u * g + (r & 7u);
    } else {
        const uint32_t j = r - full, g = j / nx;
        tx = j - g * nx;
        ty = (ny & ~7u) + g;
    }
}

// One workgroup per tile; grid (tile x, tile y, frame - f_lo).  Blocks past a
// smaller frame's tile grid return at once.
// Occupancy: LDS allows 7 workgroups of 4 wavefronts per CU at 64 x 32 cells,
// and the instances fit the 72 VGPRs of 7 wavefronts per SIMD (1.10 ms for the
// sweep at 7 wavefronts, 1.18 at 6, and 1.13 at 8, which spill).
template <bool BIG, bool ONE, RasterKind KIND, bool FLAT>
__global__ void __launch_bounds__(RASTER_BLOCK) __attribute__((amdgpu_waves_per_eu(7, 8))) k_tile_raster(
    const Draw* __restrict__ draws, const Ramp* __restrict__ ramps, const Frame* __restrict__ frames, uint32_t f_lo,
    int tws, int ths, uint32_t* __restrict__ cursor, const uint64_t* __restrict__ off,
    const uint32_t* __restrict__ pool, int32_t* __restrict__ nl, const uint4* __restrict__ careful_box,
    uint32_t* __restrict__ cells, float* __restrict__ zbuf, int32_t* __restrict__ win, uint32_t win_raw,
    uint32_t n_ramps, uint4* __restrict__ edge_out, uint32_t* __restrict__ careful_reset,
    const uint2* __restrict__ tile_frame, uint32_t t_lo, uint32_t odd_cols, uint32_t keep)
{
    // keys, rows and cells are read and written in 16-byte words (declared for 8
    // it began at 360: 256 frames of 1920x1080 1495 us, now 1471)
    extern __shared__ __align__(16) uint64_t smem[];
    // the job's first LDS_RAMPS shaders, so that a glyph lookup reads LDS
    // (read only after the tile's first barrier)
    __shared__ Ramp s_ramp[LDS_RAMPS];
    __shared__ uint32_t s_negz;

    // the careful list was read by k_careful, which ran before this launch
    if (careful_reset && (blockIdx.x | blockIdx.y | blockIdx.z | threadIdx.x) == 0) careful_reset[0] = 0;
    // the block's tile: (x, y, frame) from a 3-D grid, or (FLAT: frames of
    // different tile grids) the (tile, frame) of entry t_lo + x of a flat one
    uint32_t f, tx, ty;
    if constexpr (FLAT) {
        const uint2 e = tile_frame[t_lo + blockIdx.x];
        f = e.y;
        const uint32_t local = e.x - (uint32_t)frames[f].tile_begin;
        ty = local / frames[f].tiles_x;
        tx = local - ty * frames[f].tiles_x;
    } else {
        f = f_lo + blockIdx.z;
        tx = blockIdx.x;
        ty = blockIdx.y;
        if constexpr (KIND == RAGGED || KIND == ANY) tile_of(ty * gridDim.x + tx, gridDim.x, gridDim.y, tx, ty);
    }
    const Frame& fr = frames[f];
    constexpr bool WRAP = KIND == WRAPPED;
    if (tx >= fr.tiles_x || ty >= fr.tiles_y) return;
    if ((KIND == ANY || WRAP) && ((fr.W & 1u) && tx < odd_cols) != WRAP) return;
    const uint64_t gt = fr.tile_begin + (uint64_t)ty * fr.tiles_x + tx;
    const uint64_t o = off[gt];
    const uint32_t c = cursor[gt];
    const uint32_t n = min(c, (uint32_t)(off[gt + 1] - o));
    if (n > 0)
        for (uint32_t i = threadIdx.x; i < min(n_ramps, LDS_RAMPS) * (uint32_t)sizeof(Ramp) / 4; i += blockDim.x)
            ((uint32_t*)s_ramp)[i] = ((const uint32_t*)ramps)[i];
    raster_tile<BIG, ONE, KIND, FLAT>(draws, ramps, s_ramp, &s_negz, fr, tx, ty, gt, o, n, tws, ths, pool, nl, careful_box,
                                      cells, zbuf, win, win_raw, edge_out, smem, keep);
    // The tile leaves its binning state as k_tile_clear would for the next
    // render: its cursor at 0 and, but for frames one column wide (k_tile_edges
    // reads their rows after this), the newline rows of its tile row back at -1
    // (the first tile of the row is the one that read them).  Every wave
    // has read the cursor and the rows once the block has met here.
    const bool reset_nl = fr.image && tx == 0 && !(WRAP && fr.W == 1);
    if (c != 0 || reset_nl) {
        __syncthreads();
        if (c != 0 && threadIdx.x == 0) cursor[gt] = 0;
        if (reset_nl) {
            const uint32_t r0 = ty << ths, r1 = min(fr.H, r0 + (1u << ths));
            for (uint32_t r = r0 + threadIdx.x; r < r1; r += blockDim.x) nl[fr.nl_off + r] = -1;
        }
    }
}

// Frames of odd width: the first-column cells of the odd instance's tiles.  Cell (r, c)
// with c the first column of a tile is the later write of slot (r, c)'s
// winner and slot (r, c - 1)'s, which the tile to the left holds; cell
// (r, 0) takes the last slot of row r - 1 instead (id + 1 of the row's last
// direct pixel wraps to the next row).  The tiles left each first and last
// column slot's winning cell and write time in `edges` (time 0: none).  A
// frame one column wide has no pixels (the domain's x range is empty), and
// its cell (r, 0) is row r - 1's newline cell (r - 1) * W + 1.
// Grid (rows / 256, odd_cols, frame - f_lo).
__global__ void __launch_bounds__(256) k_tile_edges(const Frame* __restrict__ frames, uint32_t f_lo, int tws,
                                                    int ths, const uint4* __restrict__ edges,
                                                    const int32_t* __restrict__ nl, uint32_t* __restrict__ cells)
{
    const Frame& fr = frames[f_lo + blockIdx.z];
    const uint32_t b = blockIdx.y;
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (!(fr.W & 1u) || b >= fr.tiles_x || r >= fr.H || (b == 0 && r == 0)) return;
    const uint32_t TH = 1u << ths;
    const uint64_t own = fr.tile_begin + (uint64_t)(r >> ths) * fr.tiles_x + b;
    const uint4 e_own = edges[(own * TH + (r & (TH - 1))) * 2];
    uint4 e_left;
    if (b > 0) {
        e_left = edges[((own - 1) * TH + (r & (TH - 1))) * 2 + 1];
    } else {
        const uint32_t rl = r - 1;
        const uint64_t left = fr.tile_begin + (uint64_t)(rl >> ths) * fr.tiles_x + (fr.tiles_x - 1);
        e_left = edges[(left * TH + (rl & (TH - 1))) * 2 + 1];
    }
    const uint64_t t_own = ((uint64_t)e_own.w << 32) | e_own.z, t_left = ((uint64_t)e_left.w << 32) | e_left.z;
    uint32_t cell = CELL_BLANK;
    if (t_own | t_left) cell = t_own > t_left ? e_own.x : e_left.x;
    if (fr.W == 1 && fr.image && nl[fr.nl_off + r - 1] >= 0) cell = CELL_NEWLINE;
    cells[fr.cell_off + (uint64_t)r * fr.W + ((uint64_t)b << tws)] = cell;
}

// ---------------------------------------------------------------------------
// TiledPlan
// ---------------------------------------------------------------------------
static unsigned blocks(uint64_t n, unsigned per) { return (unsigned)((n + per - 1) / per); }

static int log2u(uint32_t v)
{
    int s = 0;
    while ((1u << s) < v) ++s;
    return s;
}

int TiledPlan::set_tile(uint32_t tw, uint32_t th)
{
    if (tw < 8 || tw > 512 || th < 4 || th > 64 || (tw & (tw - 1)) || (th & (th - 1)))
        return fail(SLOTH_EINVAL, "tile size %ux%u: width must be a power of two in 8..512, height in 4..64", tw, th);
    if (tw != TW || th != TH) sized = false;
    TW = tw;
    TH = th;
    user_tile = true;
    return SLOTH_OK;
}

size_t TiledPlan::raster_lds(bool odd) const
{
    // keys (8 B per slot), rows, and a cell per slot where a list may be
    // longer than a chunk; odd widths: a slot and its cell per cell
    const size_t S = (size_t)(odd ? TW : TW / 2) * TH;
    return S * 8 + (size_t)CHUNK * row_bytes(!odd && walk()) + (odd || multi ? S * 4 : 0);
}

bool TiledPlan::tile_fits() const
{
    // the raster's threads own whole columns of slots: a tile row holds at
    // most one workgroup's worth (odd widths: a slot per cell).  Sizes are
    // taken or refused for any list: 12 KiB of rows, 8 bytes a slot (12 for
    // odd widths).
    auto fits = [&](bool odd) {
        const size_t S = (size_t)(odd ? TW : TW / 2) * TH;
        return S * (odd ? 12 : 8) + 12288 <= 65536 && (odd ? TW : TW / 2) <= (uint32_t)RASTER_BLOCK;
    };
    return (!has_even || fits(false)) && (!has_odd || fits(true));
}

TiledPlan::Range TiledPlan::range(const std::vector<Frame>& frames, const std::vector<Draw>& draws, uint32_t f_lo,
                                  uint32_t f_hi) const
{
    if (f_lo == 0 && f_hi == n_frames) return whole;
    Range r;
    uint64_t slots = 0, ragged = 0;
    for (uint32_t f = f_lo; f < f_hi; ++f) {
        const Frame& fr = frames[f];
        r.tiles_x = std::max(r.tiles_x, fr.tiles_x);
        r.tiles_y = std::max(r.tiles_y, fr.tiles_y);
        r.H = std::max(r.H, fr.H);
        r.one = r.one && fr.draw_end - fr.draw_begin == 1;
        ((fr.W & 1u) ? r.odd : r.even) = true;
        slots += (uint64_t)fr.W * fr.H;
        if (fr.W & 31u) ragged += (uint64_t)fr.W * fr.H;
        for (uint32_t d = fr.draw_begin; d < fr.draw_end; ++d) r.max_draw = std::max(r.max_draw, draws[d].n);
    }
    r.ragged = ragged * 2 > slots;
    return r;
}

int TiledPlan::plan(std::vector<Frame>& frames, const std::vector<Draw>& draws, uint64_t rows)
{
    bool ev = false, od = false;
    odd_narrow = false;
    for (const Frame& f : frames) {
        ((f.W & 1u) ? od : ev) = true;
        odd_narrow = odd_narrow || f.W == 1;
    }
    if (ev != has_even || od != has_odd) sized = false;
    has_even = ev;
    has_odd = od;
    // Jobs that were not tuned.  Tiles of 64 x 32 cells when there are as many
    // as the chip takes at once (7 workgroups per CU); else lower ones, and for
    // the smallest jobs 16 x 16, since a launch lasts as long as one tile then.
    // Odd widths hold twice the slots in some tiles: half the height of the
    // smaller two (120 frames of 641x480 at 64 x 32 / 64 x 16 158 / 199 us).  A render
    // at 64 x 32 / 64 x 16 / 16 x 16 cells: 80x24 (2 tiles of 64 x 32) 17.3 /
    // 16.5 / 14.4 us, 240x70 (12) 23.3 / 19.0 / 15.9, four meshes on 640x480
    // (150) 30.0 / 27.1 / 27.9, 100 frames of 100x100 (800) 29.0 / 23.6 / 29.1,
    // six meshes on 1920x1080 (1020) 60.1 / 43.7 / 43.7, four frames of 1280x720
    // (1840) 38.2 / 45.1 / 80.7; 641x481 at half the heights 52.1 / 46.6 / 47.6.
    if (!user_tile) {
        auto count = [&](uint32_t tw, uint32_t th) {
            uint64_t n = 0;
            for (const Frame& f : frames) n += (uint64_t)((f.W + tw - 1) / tw) * ((f.H + th - 1) / th);
            return n;
        };
        const uint32_t odd = has_odd ? 2 : 1;
        const uint32_t tw = TW, th = TH;
        TW = 64;
        TH = 32;
        if (count(TW, TH) < 1792) {
            TH = 16;
            if (count(TW, TH) < 256) TW = 16;
            TH /= odd;
        }
        if (tw != TW || th != TH) sized = false;
    }
    // k_bin's triangles per thread: several serve jobs whose blocks wait in
    // line, one the others (the same jobs: 10.6 us with 4 / 6.7 with 1, 11.3 /
    // 6.9, 13.0 / 7.4, 12.5 / 8.3, 16.4 / 12.9, 14.4 / 7.9; 1,310,720 triangles
    // 17.9 / 14.8, and 15.5 with 2; 5 million in 30 draws 57 / 113)
    if (!user_tpt) {
        uint64_t n = 0;
        for (const Draw& d : draws) n += d.n;
        bin_tpt = n <= 1u << 20 ? 1 : n <= 1u << 21 ? 2 : 4;
    }
    uint64_t tiles = 0;
    for (Frame& f : frames) {
        f.tiles_x = (f.W + TW - 1) / TW;
        f.tiles_y = (f.H + TH - 1) / TH;
        f.tile_begin = tiles;
        tiles += (uint64_t)f.tiles_x * f.tiles_y;
    }
    // a context's draws may have changed since the tables were made: the
    // padded grid takes any
    flat_bin = flat_bin && flat_draws.size() == draws.size();
    for (size_t d = 0; flat_bin && d < draws.size(); ++d) flat_bin = draws[d].n == flat_draws[d];
    n_frames = UINT32_MAX;   // not the whole, while that is made
    whole = range(frames, draws, 0, (uint32_t)frames.size());
    n_frames = (uint32_t)frames.size();
    if (tiles != n_tiles) sized = false;
    n_tiles = tiles;
    n_rows = rows;
    int rc;
    if ((rc = d_cursor.reserve(sizeof(uint32_t) * std::max<uint64_t>(1, n_tiles)))) return rc;
    if ((rc = d_off.reserve(sizeof(uint64_t) * (n_tiles + 1)))) return rc;
    if ((rc = d_nl.reserve(sizeof(int32_t) * std::max<uint64_t>(1, n_rows)))) return rc;
    if ((rc = d_careful_cnt.reserve(sizeof(uint32_t) * (WRAP_CNT + 1)))) return rc;
    return reserve_edges();
}

int TiledPlan::reserve_edges()
{
    return odd_cols() ? d_edges.reserve(sizeof(uint4) * 2 * std::max<uint64_t>(1, n_tiles) * TH) : SLOTH_OK;
}

uint32_t* TiledPlan::pool_of(const std::vector<Frame>& frames, uint32_t part_begin) const
{
    // off counts through all parts; each part's lists start at the pool's start
    return (uint32_t*)((uintptr_t)d_pool.p - sizeof(uint32_t) * off[frames[part_begin].tile_begin]);
}

int TiledPlan::launch_clear(const std::vector<Frame>& frames, uint32_t f_lo, uint32_t f_hi, hipStream_t s)
{
    const Frame& a = frames[f_lo];
    const Frame& b = frames[f_hi - 1];
    uint64_t t_lo = a.tile_begin, t_hi = b.tile_begin + (uint64_t)b.tiles_x * b.tiles_y;
    uint64_t r_lo = a.nl_off, r_hi = b.nl_off + b.H;
    uint64_t n = std::max(t_hi - t_lo, r_hi - r_lo);
    unsigned g = std::max(1u, std::min(blocks(n, 256), 4096u));
    hipLaunchKernelGGL(k_tile_clear, dim3(g), dim3(256), 0, s, d_cursor.as<uint32_t>() + t_lo, t_hi - t_lo,
                       d_nl.as<int32_t>() + r_lo, r_hi - r_lo, overflow + f_lo, f_hi - f_lo,
                       d_careful_cnt.as<uint32_t>());
    HIP_TRY(hipGetLastError());
    return SLOTH_OK;
}

int TiledPlan::launch_bin(const std::vector<Frame>& frames, const std::vector<Draw>& draws, const Frame* d_frames,
                          const Draw* d_draws, uint32_t f_lo, uint32_t f_hi, uint32_t* pool, bool count_only, hipStream_t s)
{
    const uint32_t d_lo = frames[f_lo].draw_begin, d_hi = frames[f_hi - 1].draw_end;
    const int tws = log2u(TW), ths = log2u(TH);
    auto go = [&](dim3 grid, uint32_t d0, const uint2* flat) {
        auto run = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(BIN_BLOCK), 0, s, d_draws, d0, d_frames, tws, ths,
                               d_cursor.as<uint32_t>(), d_off.as<uint64_t>(), pool,
                               d_nl.as<int32_t>(), overflow, d_careful_cnt.as<uint32_t>(),
                               d_careful_in.as<uint4>(), careful_cap, flat, odd_cols());
        };
        // the counting run takes the tree variant (it counts the tall triangles)
        if (bin_tpt == 1)
            count_only ? run(k_bin<true, 1, true>) : bin_tree ? run(k_bin<false, 1, true>) : run(k_bin<false, 1, false>);
        else if (bin_tpt == 2)
            count_only ? run(k_bin<true, 2, true>) : bin_tree ? run(k_bin<false, 2, true>) : run(k_bin<false, 2, false>);
        else
            count_only ? run(k_bin<true, 4, true>) : bin_tree ? run(k_bin<false, 4, true>) : run(k_bin<false, 4, false>);
        HIP_TRY(hipGetLastError());
        return SLOTH_OK;
    };
    if (flat_bin) {
        // one block per (draw, BIN_BLOCK * TPT triangles) of the range
        const int ti = bin_tpt == 1 ? 0 : bin_tpt == 2 ? 1 : 2;
        const uint64_t b0 = bin_block_begin[ti][d_lo], b1 = bin_block_begin[ti][d_hi];
        if (b1 - b0 > 0x7FFFFFFFull) return fail(SLOTH_EINVAL, "too many binning blocks in one launch");
        if (b1 > b0) return go(dim3((unsigned)(b1 - b0)), d_lo, d_bin_blocks[ti].as<uint2>() + b0);
        return SLOTH_OK;
    }
    int rc;
    const uint32_t max_n = range(frames, draws, f_lo, f_hi).max_draw;
    for (uint32_t d0 = d_lo; d0 < d_hi; d0 += 65535u) {
        const uint32_t d1 = std::min(d_hi, d0 + 65535u);
        if (max_n == 0) continue;
        if ((rc = go(dim3(blocks(max_n, BIN_BLOCK * (uint32_t)bin_tpt), d1 - d0), d0, nullptr))) return rc;
    }
    return SLOTH_OK;
}

int TiledPlan::launch_careful(const Frame* d_frames, const Draw* d_draws, uint32_t* pool, bool count_only,
                              uint32_t group, hipStream_t s)
{
    if (careful_cap == 0) return SLOTH_OK;
    const int tws = log2u(TW), ths = log2u(TH);
    // a grid of up to 16,384 wavefronts (the chip holds about 8,192 of
    // these at once) strides over the careful list, one triangle per
    // wavefront at a time (the sweep's pass 0.015 -> 0.012 ms against 4,096)
    dim3 grid(std::min(blocks(careful_cap, 4), 4096u));
    if (count_only)
        hipLaunchKernelGGL(k_careful<true>, grid, dim3(256), 0, s, d_frames, tws, ths,
                           d_cursor.as<uint32_t>(), d_off.as<uint64_t>(), pool,
                           overflow, d_careful_cnt.as<uint32_t>(), group, d_careful_in.as<uint4>(),
                           d_careful_box.as<uint4>(), careful_cap, odd_cols());
    else
        hipLaunchKernelGGL(k_careful<false>, grid, dim3(256), 0, s, d_frames, tws, ths,
                           d_cursor.as<uint32_t>(), d_off.as<uint64_t>(), pool,
                           overflow, d_careful_cnt.as<uint32_t>(), group, d_careful_in.as<uint4>(),
                           d_careful_box.as<uint4>(), careful_cap, odd_cols());
    HIP_TRY(hipGetLastError());
    return SLOTH_OK;
}

int TiledPlan::size(const std::vector<Frame>& frames, const std::vector<Draw>& draws, const Frame* d_frames,
                    const Draw* d_draws, hipStream_t s)
{
    if (frames.empty()) return SLOTH_OK;
    const uint32_t F = (uint32_t)frames.size();
    int rc;
    // 0. flat k_bin grids (draws of different sizes): each block's (draw,
    // first triangle) for TPT 1, 2, 4
    flat_bin = false;
    for (const Draw& d : draws) flat_bin = flat_bin || d.n != draws[0].n;
    if (flat_bin) {
        flat_draws.resize(draws.size());
        for (size_t d = 0; d < draws.size(); ++d) flat_draws[d] = draws[d].n;
        for (int ti = 0; ti < 3; ++ti) {
            const uint32_t per = (uint32_t)BIN_BLOCK << ti;
            std::vector<uint2> tbl;
            std::vector<uint64_t>& beg = bin_block_begin[ti];
            beg.assign(draws.size() + 1, 0);
            for (size_t d = 0; d < draws.size(); ++d) {
                beg[d] = tbl.size();
                for (uint32_t b = 0; b < draws[d].n; b += per) tbl.push_back(make_uint2((uint32_t)d, b));
            }
            beg[draws.size()] = tbl.size();
            if ((rc = d_bin_blocks[ti].reserve(sizeof(uint2) * std::max<size_t>(1, tbl.size())))) return rc;
            if (!tbl.empty())
                HIP_TRY(hipMemcpyAsync(d_bin_blocks[ti].p, tbl.data(), sizeof(uint2) * tbl.size(),
                                       hipMemcpyHostToDevice, s));
            HIP_TRY(hipStreamSynchronize(s));   // before tbl goes
        }
    }
    // 1. count tile entries of CLS_BOX triangles and the careful triangles
    const uint32_t cap_before = careful_cap;
    auto careful_room = [&] { return (uint32_t)(std::min(d_careful_in.bytes / 2, d_careful_box.bytes) / sizeof(uint4)); };
    careful_cap = careful_room();
    if ((rc = launch_clear(frames, 0, F, s))) return rc;
    if ((rc = launch_bin(frames, draws, d_frames, d_draws, 0, F, nullptr, true, s))) return rc;
    uint32_t cnt[WRAP_CNT + 1];
    HIP_TRY(hipMemcpyAsync(cnt, d_careful_cnt.p, sizeof(cnt), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    const uint32_t n_careful = cnt[0];
    // the wavefront walk of big boxes pays once about one wavefront in ten
    // holds one (a big box costs its lane's wavefront 10x the common walk)
    uint64_t n_tri = 0;
    for (const Draw& d : draws) n_tri += d.n;
    big_walk = (uint64_t)cnt[BIG_CNT] * 512 >= n_tri && cnt[BIG_CNT] > 0;
    if (const char* e = getenv("SLOTH_BIG_WALK")) big_walk = e[0] == '1';
    // the binning kernel's segment-tree newline rows pay once one triangle
    // in 256 spans more than TALL_ROWS rows (a wavefront's row loop lasts as
    // long as its tallest triangle's); among draws of different sizes a block
    // of them is enough, since the launch waits for the few blocks of a small
    // draw of tall triangles (30 unlike jobs: 104-131 -> 53-59 us)
    bin_tree = cnt[TALL_CNT] > 0 && ((uint64_t)cnt[TALL_CNT] * 256 >= n_tri || (flat_bin && cnt[TALL_CNT] >= (uint32_t)BIN_BLOCK));
    if (const char* e = getenv("SLOTH_BIN_TREE")) bin_tree = e[0] == '1';
    // (those of other tiles than the present ones do not count: their boxes
    // take other paths)
    const uint32_t want = std::max(n_careful ? n_careful + n_careful / 2 + 1024 : 0u, outgrown ? cap_before : 0u);
    if (n_careful > careful_cap) {
        // 2. room for the careful list, then count again so that it is filled
        careful_cap = want;
        if ((rc = d_careful_in.reserve(2 * sizeof(uint4) * careful_cap))) return rc;
        if ((rc = d_careful_box.reserve(sizeof(uint4) * careful_cap))) return rc;
        if ((rc = launch_clear(frames, 0, F, s))) return rc;
        if ((rc = launch_bin(frames, draws, d_frames, d_draws, 0, F, nullptr, true, s))) return rc;
    }
    // 3. the careful triangles' tile entries
    if ((rc = launch_careful(d_frames, d_draws, nullptr, true, 0, s))) return rc;
    std::vector<uint32_t> counts(n_tiles);
    if (n_tiles)
        HIP_TRY(hipMemcpyAsync(counts.data(), d_cursor.p, sizeof(uint32_t) * n_tiles, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipMemcpyAsync(cnt, d_careful_cnt.p, sizeof(cnt), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    careful_cap = std::min(want, careful_room());
    // a reach that outgrew its columns may go on growing: room for a third more.
    // (Columns kept, or one more at least, cost a view that moves to and fro more
    // than its re-sizes: 641x480 turned by 3.6 degrees a frame 99 -> 115 us.)
    const uint32_t need = cnt[WRAP_CNT];
    odd_wraps = need + (outgrown && need > odd_wraps ? need / 3 : 0u);
    if ((rc = reserve_edges())) return rc;
    off.assign(n_tiles + 1, 0);
    multi = false;
    for (uint64_t t = 0; t < n_tiles; ++t) {
        uint64_t c = counts[t];
        uint64_t cap = c ? c + c / 8 + 16 : 0;
        multi = multi || cap > CHUNK;
        off[t + 1] = off[t] + cap;
    }
    // the parts: frames in order, of near equal lists
    const uint64_t n_parts = off[n_tiles] * sizeof(uint32_t) / PART_BYTES + 1;
    parts.assign(1, 0);
    uint64_t most = 0;
    auto lists_from = [&](uint32_t f) { return f < F ? off[frames[f].tile_begin] : off[n_tiles]; };
    for (uint32_t f = 1; f <= F; ++f)
        if (f == F || (parts.size() < n_parts && lists_from(f) * n_parts >= off[n_tiles] * parts.size())) {
            most = std::max(most, lists_from(f) - lists_from(parts.back()));
            parts.push_back(f);
        }
    if ((rc = d_pool.reserve(sizeof(uint32_t) * std::max<uint64_t>(1, most)))) return rc;
    HIP_TRY(hipMemcpyAsync(d_off.p, off.data(), sizeof(uint64_t) * (n_tiles + 1), hipMemcpyHostToDevice, s));
    // 4. flat raster grids (frames of different tile grids): each tile's
    // (tile, frame) in tile order, and the same with the tiles of more than
    // four chunks of entries moved to the front, longest first (the rest
    // keep tile order, whose neighbouring tiles share cached vertices and
    // lists: sorting every tile by length made the uneven batch slower)
    flat_raster = false;
    for (const Frame& f : frames)
        flat_raster = flat_raster || f.tiles_x != frames[0].tiles_x || f.tiles_y != frames[0].tiles_y;
    std::vector<uint2> tf, heavy;
    if (flat_raster) {
        tf.resize(n_tiles);
        for (uint32_t f = 0; f < F; ++f)
            for (uint64_t t = 0; t < (uint64_t)frames[f].tiles_x * frames[f].tiles_y; ++t)
                tf[frames[f].tile_begin + t] = make_uint2((uint32_t)(frames[f].tile_begin + t), f);
        heavy = tf;
        for (size_t p = 0; p + 1 < parts.size(); ++p) {
            const auto end = heavy.begin() + (parts[p + 1] < F ? frames[parts[p + 1]].tile_begin : n_tiles);
            const auto begin = heavy.begin() + frames[parts[p]].tile_begin;
            const auto split = std::stable_partition(begin, end, [&](const uint2& a) { return counts[a.x] > 4 * CHUNK; });
            std::stable_sort(begin, split, [&](const uint2& a, const uint2& b) { return counts[a.x] > counts[b.x]; });
        }
        if ((rc = d_tile_frame.reserve(sizeof(uint2) * std::max<uint64_t>(1, n_tiles))) ||
            (rc = d_tile_heavy.reserve(sizeof(uint2) * std::max<uint64_t>(1, n_tiles))))
            return rc;
        if (n_tiles) {
            HIP_TRY(hipMemcpyAsync(d_tile_frame.p, tf.data(), sizeof(uint2) * n_tiles, hipMemcpyHostToDevice, s));
            HIP_TRY(hipMemcpyAsync(d_tile_heavy.p, heavy.data(), sizeof(uint2) * n_tiles, hipMemcpyHostToDevice, s));
        }
    }
    // renders start from cleared cursors, rows and careful list (each leaves them so)
    if ((rc = launch_clear(frames, 0, F, s))) return rc;
    HIP_TRY(hipStreamSynchronize(s));
    sized = true;
    outgrown = false;
    return SLOTH_OK;
}

// The common raster instance: odd widths, ragged ones or neither, big-box walk or not, one
// draw per frame or not, flat grid (frames of different tile grids) or 3-D.  Each instance is compiled
// on its own, so the 3-D instances carry no flat-grid mapping and its
// registers.
template <bool FLAT, RasterKind KIND>
static auto raster_kernel(bool walk, bool one)
{
    return walk ? (one ? k_tile_raster<true, true, KIND, FLAT> : k_tile_raster<true, false, KIND, FLAT>)
                : (one ? k_tile_raster<false, true, KIND, FLAT> : k_tile_raster<false, false, KIND, FLAT>);
}

template <bool FLAT>
static auto raster_kernel(bool walk, bool one, bool odd, bool ragged)
{
    return odd ? raster_kernel<FLAT, ANY>(walk, one)
               : ragged ? raster_kernel<FLAT, RAGGED>(walk, one) : raster_kernel<FLAT, EVEN>(walk, one);
}

int TiledPlan::launch_raster(const std::vector<Frame>& frames, const std::vector<Draw>& draws, const Frame* d_frames,
                             const Draw* d_draws, const Ramp* d_ramps, uint32_t f_lo, uint32_t f_hi, uint32_t* pool, uint32_t* cells, float* z,
                             int32_t* win, bool win_raw, uint32_t n_ramps, bool reset_careful, hipStream_t s)
{
    // the first raster launch resets the careful list's length (k_careful
    // has read it) when asked
    uint32_t* careful_reset = reset_careful ? d_careful_cnt.as<uint32_t>() : nullptr;
    // grid (tile x, tile y, frame) over the largest tile grid of the range,
    // at most 65535 frames per launch
    for (uint32_t f0 = f_lo; f0 < f_hi; f0 += 65535u) {
        const uint32_t f1 = std::min(f_hi, f0 + 65535u);
        const Range rg = range(frames, draws, f0, f1);
        const uint32_t mx = rg.tiles_x, my = rg.tiles_y;
        if (mx == 0 || my == 0) continue;
        // one launch for the common instance's tiles and one for the odd
        // one's; each skips the other's.  The grid: (tile x, tile y, frame)
        // over the largest tile grid, or one workgroup per tile when the
        // frames' tile grids differ
        const bool one = rg.one, od = rg.odd && odd_cols(), ev = rg.even || !od || mx > odd_cols();
        const uint64_t t_lo = frames[f0].tile_begin;
        const uint64_t t_hi = frames[f1 - 1].tile_begin + (uint64_t)frames[f1 - 1].tiles_x * frames[f1 - 1].tiles_y;
        if (flat_raster && t_hi > 0x7FFFFFFFull) return fail(SLOTH_EINVAL, "too many tiles for a flat raster grid");
        const dim3 grid = flat_raster ? dim3((unsigned)(t_hi - t_lo)) : dim3(mx, my, f1 - f0);
        const uint2* tf = !flat_raster ? nullptr
                          : is_part(f0, f1) ? d_tile_heavy.as<uint2>()
                                            : d_tile_frame.as<uint2>();
        uint4* edges = od ? d_edges.as<uint4>() : nullptr;
        auto go = [&](auto kern, dim3 grid, size_t lds) {
            hipLaunchKernelGGL(kern, grid, dim3(RASTER_BLOCK), lds, s, d_draws, d_ramps, d_frames, f0, log2u(TW),
                               log2u(TH), d_cursor.as<uint32_t>(), d_off.as<uint64_t>(), pool,
                               d_nl.as<int32_t>(), d_careful_box.as<uint4>(), cells, z, win, win_raw ? 1u : 0u,
                               n_ramps, edges, careful_reset, tf, (uint32_t)t_lo, odd_cols(), keep_lines() ? 1u : 0u);
            careful_reset = nullptr;
        };
        if (ev) {
            go(flat_raster ? raster_kernel<true>(walk(), one, rg.odd, rg.ragged) : raster_kernel<false>(walk(), one, rg.odd, rg.ragged),
               grid, raster_lds(false));
            HIP_TRY(hipGetLastError());
        }
        if (od) {
            const unsigned nx = std::min(odd_cols(), mx);
            go(one ? k_tile_raster<false, true, WRAPPED, false> : k_tile_raster<false, false, WRAPPED, false>,
               dim3(nx, my, f1 - f0), raster_lds(true));
            HIP_TRY(hipGetLastError());
            hipLaunchKernelGGL(k_tile_edges, dim3(blocks(rg.H, 256), nx, f1 - f0), dim3(256), 0, s, d_frames, f0,
                               log2u(TW), log2u(TH), (const uint4*)d_edges.as<uint4>(),
                               (const int32_t*)d_nl.as<int32_t>(), cells);
            HIP_TRY(hipGetLastError());
        }
    }
    // no raster block ran (frames without tiles): reset the length here
    if (careful_reset) return launch_clear(frames, f_lo, f_hi, s);
    return SLOTH_OK;
}

int TiledPlan::launch(const std::vector<Frame>& frames, const std::vector<Draw>& draws, const Frame* d_frames,
                      const Draw* d_draws, const Ramp* d_ramps, uint32_t f_lo, uint32_t f_hi, uint32_t* cells,
                      float* z, int32_t* win, bool win_raw, uint32_t n_ramps, hipStream_t s,
                      std::vector<hipEvent_t>* ev, hipStream_t s2, const std::vector<hipEvent_t>* join)
{
    if (!sized) return fail(SLOTH_ESTATE, "tile lists not sized");
    if (!tile_fits())
        return fail(SLOTH_EINVAL,
                    "tile %ux%u does not fit a workgroup: %zu bytes of LDS (at most 65536), %u slots a row "
                    "(at most %d)", TW, TH, raster_lds(has_odd), has_odd ? TW : TW / 2, RASTER_BLOCK);
    int rc;
    const uint32_t nf = f_hi - f_lo;
    uint32_t groups = 1;
    if (s2 && join && !ev && parts.size() == 2)
        groups = std::min<uint32_t>({MAX_GROUPS, nf / PIPE_MIN_FRAMES, (uint32_t)join->size() - 1});
    if (groups < 2) {
        // Every render leaves the tile cursors, the even frames' newline
        // rows and the careful list's length as k_tile_clear sets them
        // (k_tile_raster resets what it has read; size() ends with a
        // clear), but for frames one column wide, whose newline rows
        // k_tile_edges reads after the raster.
        size_t n_ev = 0;
        auto mark = [&]() -> int {
            if (!ev) return SLOTH_OK;
            if (n_ev == ev->size()) {
                ev->push_back(nullptr);
                HIP_TRY(hipEventCreate(&ev->back()));
            }
            HIP_TRY(hipEventRecord((*ev)[n_ev++], s));
            return SLOTH_OK;
        };
        for (size_t p = 0; p + 1 < parts.size(); ++p) {
            const uint32_t a = std::max(f_lo, parts[p]), b = std::min(f_hi, parts[p + 1]);
            if (a >= b) continue;
            uint32_t* pool = pool_of(frames, parts[p]);
            if ((rc = mark())) return rc;
            if (odd_narrow && (rc = launch_clear(frames, a, b, s))) return rc;
            if ((rc = mark())) return rc;
            if ((rc = launch_bin(frames, draws, d_frames, d_draws, a, b, pool, false, s))) return rc;
            if ((rc = mark())) return rc;
            if ((rc = launch_careful(d_frames, d_draws, pool, false, 0, s))) return rc;
            if ((rc = mark())) return rc;
            if ((rc = launch_raster(frames, draws, d_frames, d_draws, d_ramps, a, b, pool, cells, z, win, win_raw,
                                    n_ramps, true, s)))
                return rc;
            if ((rc = mark())) return rc;
        }
        return SLOTH_OK;
    }
    // Pipeline over frame groups: s bins group g + 1 while s2 rasters group
    // g.  Group g's raster waits for its bins and careful boxes (event g); s
    // joins s2 at the end.
    uint32_t* pool = d_pool.as<uint32_t>();
    if ((rc = launch_clear(frames, f_lo, f_hi, s))) return rc;
    for (uint32_t g = 0; g < groups; ++g) {
        const uint32_t a = f_lo + (uint32_t)((uint64_t)nf * g / groups);
        const uint32_t b = f_lo + (uint32_t)((uint64_t)nf * (g + 1) / groups);
        if ((rc = launch_bin(frames, draws, d_frames, d_draws, a, b, pool, false, s))) return rc;
        if ((rc = launch_careful(d_frames, d_draws, pool, false, g, s))) return rc;
        HIP_TRY(hipEventRecord((*join)[g], s));
        HIP_TRY(hipStreamWaitEvent(s2, (*join)[g], 0));
        // the last group's raster runs after every group's careful pass
        if ((rc = launch_raster(frames, draws, d_frames, d_draws, d_ramps, a, b, pool, cells, z, win, win_raw, n_ramps,
                                g + 1 == groups, s2)))
            return rc;
    }
    HIP_TRY(hipEventRecord((*join)[groups], s2));
    HIP_TRY(hipStreamWaitEvent(s, (*join)[groups], 0));
    return SLOTH_OK;
}

int TiledPlan::overflowed(uint32_t nf, hipStream_t s, bool& ovf)
{
    ovf = false;
    HIP_TRY(hipStreamSynchronize(s));
    for (uint32_t f = 0; f < nf; ++f) ovf |= (((volatile uint32_t*)overflow)[f] != 0);
    return SLOTH_OK;
}

}  // namespace sloth
