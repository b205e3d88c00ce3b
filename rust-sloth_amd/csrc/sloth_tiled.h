// Tiled raster path (internal).
//
// The W x H cell grid of every frame is cut into TW x TH cell tiles (TW even,
// tiles start on even columns).  With W even, z slot ids = y*W + 2x are even,
// so a tile's slots and the two cells each slot writes (id, id+1) never cross
// a tile edge, and a tile can resolve its cells alone.  So can a tile of a frame
// of odd width that wrapped pixels do not reach; the others take the raster's
// odd instance (described there).
//
//   k_tile_clear   tile cursors <- 0, newline rows <- -1, overflow <- 0,
//                  careful-list length <- 0; after sizing and before
//                  renders of frames one column wide: k_tile_raster leaves
//                  what it read in this state for the next render
//   k_bin          1, 2 or 4 triangles per thread: setup, classification,
//                  candidate box, newline rows (LDS max per block, one
//                  atomicMax per row), and the triangle index appended to
//                  every tile its box reaches: boxes within 2 x 2 tiles of one
//                  region count into an LDS window of tiles, with one global
//                  atomicAdd per window tile per block; others go to the
//                  careful list
//   k_careful      one wavefront per careful triangle (many tiles, or an
//                  exact box from row spans): its tile entries
//   k_tile_raster  one 256-thread workgroup per tile, grid (tile x, tile y,
//                  frame): each list entry is set up by a lane and its row
//                  kept in LDS, its fragments do a 64-bit LDS atomicMin of
//                  packed keys that also name that row, then a thread takes
//                  two slots at a time: cells from the rows their keys name
//                  (evaluated per pixel only where the glyph is not constant
//                  over the box), depths from the keys, 16-byte streaming
//                  stores.  Lists longer than the 256 LDS rows run in chunks,
//                  whose winners' cells are put aside in LDS.  The image-mode
//                  tail cells are written by the frame's first tile.  When
//                  many boxes are big, a variant has each wavefront walk its
//                  lanes' big boxes with all 64 lanes.
//
// Tile lists live in one pool at fixed per-tile offsets (large jobs: per part
// of their frames, see PART_BYTES), sized from an exact
// counting run of k_bin plus headroom.  If a later run would exceed a tile's
// capacity (the transforms changed), k_bin raises the overflow flag and the
// host re-plans and renders again.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "sloth_device.h"
#include "sloth_host.h"

namespace sloth {

constexpr uint32_t MAX_GROUPS = 8;        // frame groups of a pipelined launch
// Frames on the tiled path hold fewer triangles than this: the raster's
// 64-bit LDS keys carry the triangle index, the pixel's `sub` bit, a stored
// flag and the entry's 8-bit cache row in their low 32 bits.
constexpr uint32_t TILED_MAX_TRIS = (1u << 22) - 1;
constexpr uint32_t PIPE_MIN_FRAMES = 16;  // frames per group at least
// A job whose tile lists take more is rendered in parts of whole frames that
// share one pool.  k_bin writes a list and the raster reads it a launch later:
// from the 256 MB last-level cache when the pool's lines are still there,
// else from HBM between the frames' stores, which costs more than the bytes
// do (the list's lines read ahead by other blocks cost the same).  A part
// costs a launch's tail, about 15 us.  256 frames of 1920x1080 with 0.2 GB
// of lists, three such batches in turn / one after another, each waited for:
// one part 1.80 / 1.65 ms, two 1.79 / 1.57, three 1.60 / 1.52, four 1.49 /
// 1.48, five 1.48 / 1.51, six 1.49 / 1.57.  A batch rendered over and over
// with nothing in between, which finds its lists cached either way: 1.42 in
// one part, 1.46 in four.
constexpr uint64_t PART_BYTES = 64ull << 20;

struct TiledPlan {
    uint32_t TW = 64, TH = 32;       // tile size in cells (TW even)
    bool user_tile = false;          // set_tile was called (keeps the size on a re-plan)
    // Frames of even / odd width in the job.  A frame of odd width has its
    // first odd_cols() tile columns rendered by the raster's odd instance
    // (each launch skips the other's tiles), which holds a z slot on every
    // cell column, resolves cells from two slots and finishes first-column
    // cells in k_tile_edges.
    bool has_even = true, has_odd = false;
    // odd_wraps: the tile columns that the counting run's boxes ask for
    // (odd_cols_of), a third more after a run that found more and so raised the
    // overflow flag.
    // odd_narrow: frames one column wide (only newline cells).
    uint32_t odd_wraps = 0;
    bool odd_narrow = false;
    uint32_t odd_cols() const { return !has_odd ? 0u : odd_narrow && !odd_wraps ? 1u : odd_wraps; }
    bool multi = false;              // set by size(): some tile's list may grow past one chunk of the raster
    DevBuf d_edges;                  // odd_cols() > 0: per tile and row, the first and last column slots' winners
    uint64_t n_tiles = 0;
    uint64_t n_rows = 0;
    bool sized = false;              // pool offsets match the current layout
    // a render outgrew its lists: the next sizing keeps what room they had
    bool outgrown = false;
    void outgrow()
    {
        sized = false;
        outgrown = true;
    }
    std::vector<uint64_t> off;       // host copy of the per-tile pool offsets (n_tiles + 1)
    // set by size(): the first frame of each part and, last, the number of
    // frames.  The parts are binned and rendered one after another and share
    // the pool.
    std::vector<uint32_t> parts;
    bool is_part(uint32_t f_lo, uint32_t f_hi) const
    {
        const auto it = std::lower_bound(parts.begin(), parts.end(), f_lo);
        return it != parts.end() && *it == f_lo && it + 1 != parts.end() && it[1] == f_hi;
    }
    DevBuf d_cursor, d_off, d_pool, d_nl;
    uint32_t* overflow = nullptr;    // per frame, the job's pinned memory: kernels write it (rarely), the host reads it after a wait
    // triangles whose candidate box k_careful computes: (frame, triangle,
    // screen vertices) in, 32 bytes each, (triangle, box) out.  careful_cap is
    // the counting run's number plus headroom, 0 for none (k_careful is then
    // not launched); the memory only grows.
    DevBuf d_careful_cnt, d_careful_in, d_careful_box;
    uint32_t careful_cap = 0;
    // Batches whose draws differ in size, or whose frames differ in tile
    // grid, launch flat grids instead of grids padded to the largest draw
    // (k_bin) or tile grid (the raster), whose extra blocks would only exit:
    // k_bin takes one block per (draw, BIN_BLOCK * TPT triangles) from a
    // table per TPT, the raster one workgroup per tile of the range.
    bool flat_bin = false, flat_raster = false;
    std::vector<uint32_t> flat_draws;            // the draws' sizes that the flat_bin tables are of
    DevBuf d_bin_blocks[3];                      // per TPT 1, 2, 4: (draw, first triangle) of each block
    std::vector<uint64_t> bin_block_begin[3];    // per TPT: each draw's first block (draws + 1)
    // flat raster grids: workgroup i of a launch over tiles [t_lo, t_hi) takes
    // entry t_lo + i, a (tile, frame) pair: in tile order, or (launches of the
    // whole batch) with the tiles of more than four chunks of entries first,
    // so that a tile of thousands of entries (a dense mesh in a small frame)
    // does not start last
    DevBuf d_tile_frame, d_tile_heavy;
    // set by size(): the lists hold enough big boxes (more than 128 pixels,
    // one triangle in 512 or more) for the raster variant whose wavefronts
    // walk those boxes together; SLOTH_BIG_WALK=0/1 overrides
    bool big_walk = false;
    // set by size(): k_bin reduces newline rows through a segment tree
    // (one triangle in 256 or more spans more than 16 rows, or a block's worth
    // among draws of different sizes); SLOTH_BIN_TREE
    // =0/1 overrides
    bool bin_tree = false;
    // -1: the raster variant big_walk picks; 0 / 1: without / with the
    // wavefront walk of big boxes (set by the autotuner)
    int walk_force = -1;

    // What a launch over frames [f_lo, f_hi) needs to know of them; that of
    // the whole job is made by plan(), so that launching it does not look at
    // every frame and draw again.
    struct Range {
        uint32_t max_draw = 0;                     // triangles of the largest draw
        uint32_t tiles_x = 0, tiles_y = 0, H = 0;  // of the largest frame, each
        bool one = true;                           // every frame has exactly one draw
        bool even = false, odd = false;            // width parities
        bool ragged = false;                       // most cells lie in frames whose width is no multiple of 32
    };
    Range whole;
    uint32_t n_frames = 0;
    Range range(const std::vector<Frame>& frames, const std::vector<Draw>& draws, uint32_t f_lo, uint32_t f_hi) const;

    // Sets the tile grid of every frame and allocates per-tile and per-row
    // state.  Pool offsets become invalid until size() runs.
    int plan(std::vector<Frame>& frames, const std::vector<Draw>& draws, uint64_t rows);

    // Tile size in cells: TW a power of two in 8..512, TH in 4..64.
    int set_tile(uint32_t tw, uint32_t th);
    // The raster variant the next launches use (-1 = the sizing run's choice).
    void set_walk(int mode) { walk_force = mode; }
    // the common instance's variant (the odd one has no big-box walk)
    bool walk() const { return walk_force >= 0 ? walk_force == 1 : big_walk; }
    // Triangles per thread of k_bin: 1, 2 or 4 (plan()'s choice until set).
    int bin_tpt = 4;
    bool user_tpt = false;
    void set_bin_tpt(int t)
    {
        bin_tpt = t;
        user_tpt = true;
    }
    // The default plan's tiles of 64 x 32 cells keep the memory lines that they
    // share with the tiles beside them (widths that are no multiples of 32
    // cells) in the L2 until those have written their part; memory reads a line
    // that it is given a part of.  Three batches in turn: 64 frames of 1918x1079
    // 513 -> 406 us, of 1919x1079 527 -> 427, 120 of 641x480 162 -> 130.  Narrower
    // and lower tiles lose (32 x 16: 838 -> 930, 64 x 16: 506 -> 597), and the wider
    // ones that tuning finds are as fast without (128 x 16: 402 and 411, 512 x 8:
    // 371 and 404), which repeated renders of one batch do not tell it.
    bool keep_lines() const { return !user_tile && TW == 64 && TH == 32; }
    // LDS of the even- or odd-width raster instance at the current tile size
    size_t raster_lds(bool odd) const;
    // Both parities' instances the job needs can take the current tile size
    // (LDS, slots per row).
    bool tile_fits() const;

    // Counting run over all frames (synchronous): per-tile list lengths ->
    // pool offsets with headroom.
    int size(const std::vector<Frame>& frames, const std::vector<Draw>& draws, const Frame* d_frames,
             const Draw* d_draws, hipStream_t s);

    // clear + bin + careful + raster over frames [f_lo, f_hi), part by part.
    // ev (optional) gets 5 events recorded around the 4 stages of each part,
    // more of them made when it holds too few.  With a second stream s2
    // and join events (and no ev), ranges of at least 2 * PIPE_MIN_FRAMES
    // frames run as a pipeline of frame groups: the bins of one group overlap
    // the raster of the previous one (join needs groups + 1 events).
    int launch(const std::vector<Frame>& frames, const std::vector<Draw>& draws, const Frame* d_frames,
               const Draw* d_draws, const Ramp* d_ramps, uint32_t f_lo, uint32_t f_hi, uint32_t* cells, float* z,
               int32_t* win, bool win_raw, uint32_t n_ramps, hipStream_t s, std::vector<hipEvent_t>* ev,
               hipStream_t s2 = nullptr, const std::vector<hipEvent_t>* join = nullptr);

    // Reads the overflow flags of frames [0, nf) (synchronises the stream).
    int overflowed(uint32_t nf, hipStream_t s, bool& ovf);

    static std::vector<const char*> stage_names() { return {"k_tile_clear", "k_bin", "k_careful", "k_tile_raster"}; }

  private:
    int launch_clear(const std::vector<Frame>& frames, uint32_t f_lo, uint32_t f_hi, hipStream_t s);
    int launch_bin(const std::vector<Frame>& frames, const std::vector<Draw>& draws, const Frame* d_frames,
                   const Draw* d_draws, uint32_t f_lo, uint32_t f_hi, uint32_t* pool, bool count_only, hipStream_t s);
    int reserve_edges();
    uint32_t* pool_of(const std::vector<Frame>& frames, uint32_t part_begin) const;
    int launch_careful(const Frame* d_frames, const Draw* d_draws, uint32_t* pool, bool count_only, uint32_t group, hipStream_t s);
    int launch_raster(const std::vector<Frame>& frames, const std::vector<Draw>& draws, const Frame* d_frames, const Draw* d_draws,
                      const Ramp* d_ramps, uint32_t f_lo, uint32_t f_hi, uint32_t* pool, uint32_t* cells, float* z, int32_t* win,
                      bool win_raw, uint32_t n_ramps, bool reset_careful, hipStream_t s);
};

}  // namespace sloth
