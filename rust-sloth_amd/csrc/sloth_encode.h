// Output encoders (internal); see sloth_encode.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sloth_device.h"
#include "sloth_host.h"

namespace sloth {

// A stream: frames [first, first + count) of a job, with the `-j` export's
// framing around each (framing) or as they are.  It is encoded in runs of
// frames [lo, hi) of the stream.
struct EncodeJob {
    const uint32_t* cells;
    const Frame* frames;
    uint32_t first, count;
    uint32_t lo, hi;
    uint32_t max_blocks;     // blocks of the largest frame of the run
    int mode, framing;
    uint32_t* block_len;     // [hi - lo][max_blocks]
    uint64_t* block_off;     // [hi - lo][max_blocks]
    uint64_t* frame_off;     // [count + 1], host memory
};

// A run's grids and tables hold the largest frame's blocks for each of its
// frames: it takes frames while at least half of those are in use, or they are
// fewer than this in all (12 bytes each).
constexpr uint64_t ENC_RUN_BLOCKS = 65536;

// A stream of one frame of up to this many cells takes launch_encode_one: a
// block reads at most 64 KiB of cells before its own, and the stream (672 KB
// at most) fits a small pinned buffer that the kernel writes itself.  80x24:
// one launch and one wait instead of three and three (a terminal frame 146 ->
// 102 us).
constexpr uint64_t ENC_ONE_CELLS = 16384;

uint32_t encode_blocks(uint64_t n_cells);
// most bytes a frame of n_cells can take, framing included
uint64_t encode_bound(uint64_t n_cells, int mode);
// block lengths of the run, their offsets, frame_off[lo .. hi] (after the run before)
int launch_encode_len(const EncodeJob& j, hipStream_t s);
// frames [f_lo, f_hi) of the run to out, which holds the stream from byte `base` on
int launch_encode_write(const EncodeJob& j, uint32_t f_lo, uint32_t f_hi, uint64_t base, uint8_t* out, hipStream_t s);
// one frame: frame_off and (out not null) its bytes
int launch_encode_one(const EncodeJob& j, uint8_t* out, hipStream_t s);

}  // namespace sloth
