// Output encoders of Context::flush (context.rs:50-92) on the device.
//
//   plain  (context.rs:58-61): every cell's char, then println!'s '\n'
//   ansi   (context.rs:62-78): per cell crossterm 0.18.0's PrintStyledContent
//          of the char with RGB foreground on RGB (25,25,25): CSI
//          "48;2;25;25;25m", CSI "38;2;R;G;Bm", the char, CSI "0m"
//   html   (context.rs:79-87): per cell `<span style="color:rgb(R,G,B)">` and
//          the char (the `-j` export format)
//
// A cell's glyph byte is a Unicode code point below 256 (`char` in the
// reference), written as UTF-8: one byte below 0x80, two bytes otherwise.
//
// A stream is the frames [first, first + count) of a job one after another,
// each as prefix + cells + suffix (frame_prefix / frame_suffix), in blocks of
// ENC_CELLS cells.  One launch sequence covers a run of frames, which is all of
// them unless their sizes are far apart (ENC_RUN_BLOCKS):
//   k_enc_len    bytes of every block
//   k_enc_scan   exclusive scan of those (one workgroup), frame starts
//   k_enc_write  each block lays its bytes out in LDS and stores them in
//                aligned 16-byte words
// and a single frame of up to ENC_ONE_CELLS cells takes k_enc_one alone: its
// blocks read the cells before them instead of a scan's result.
//
// What bounds it: the stream leaves over PCIe at 57 GB/s, so 141 MB (four
// 1280x720 HTML frames) cost 2.5 ms there; the kernels take 0.07 ms for them
// (write 0.056 ms = 2.5 TB/s, lengths 0.007, scan 0.005).  Cells that wrote
// their ~38 bytes to memory one by one took 0.17 ms, and a launch pair with a
// wait per frame cost 0.1 ms a frame (100 frames of 100x100: 26.2 -> 16.0 ms
// a call, and 1.55 with the bytes copied out through pinned memory).
#include "sloth_encode.h"

namespace sloth {

constexpr int ENC_BLOCK = 256;
constexpr uint32_t ENC_ITEMS = 4;                       // cells per thread: one 16-byte load
constexpr uint32_t ENC_CELLS = ENC_BLOCK * ENC_ITEMS;   // cells per block
constexpr int SCAN_BLOCK = 1024;
constexpr uint32_t SCAN_ITEMS = 4;

__device__ __forceinline__ uint32_t utf8_len(uint32_t g) { return g < 0x80u ? 1u : 2u; }

__device__ __forceinline__ uint32_t dec_len(uint32_t v) { return 1u + (v >= 10u ? 1u : 0u) + (v >= 100u ? 1u : 0u); }

// `<span style="color:rgb(` = 23 bytes, `)">` = 3 bytes, plus 2 commas
constexpr uint32_t HTML_FIXED = 23 + 3 + 2;
// ESC "[48;2;25;25;25m" = 16 bytes, ESC "[38;2;" = 7, two ';' and 'm' = 3,
// ESC "[0m" = 4
constexpr uint32_t ANSI_FIXED = 16 + 7 + 3 + 4;

// Most bytes of a cell: three 3-digit channels and a two-byte char.
constexpr uint32_t max_cell_len(int mode) { return mode == 0 ? 2 : (mode == 1 ? ANSI_FIXED : HTML_FIXED) + 9 + 2; }

__device__ __forceinline__ uint32_t cell_len(uint32_t c, int mode)
{
    const uint32_t g = c & 0xFFu;
    if (mode == 0) return utf8_len(g);
    const uint32_t digits = dec_len((c >> 8) & 0xFFu) + dec_len((c >> 16) & 0xFFu) + dec_len(c >> 24);
    return (mode == 1 ? ANSI_FIXED : HTML_FIXED) + digits + utf8_len(g);
}

// What precedes a frame's cells: with export framing (main.rs:55-58, 85-106)
// the script's header before the first frame and a backtick line before each;
// in terminal mode crossterm's MoveTo(0, 0) (context.rs:53-55).
template <uint32_t N>
__device__ __forceinline__ uint32_t put_text(uint8_t* p, const char (&s)[N])
{
#pragma unroll
    for (uint32_t k = 0; k + 1 < N; ++k) p[k] = (uint8_t)s[k];
    return N - 1;
}
__device__ __forceinline__ void frame_prefix(uint8_t* p, const EncodeJob& j, uint32_t f, bool image)
{
    if (j.framing) {
        if (f == 0) p += put_text(p, "let frames = [\n");
        p += put_text(p, "`\n");
    }
    if (!image) put_text(p, "\x1b[1;1H");
}
// What follows them: println!'s newline after plain text (context.rs:61), and
// with export framing "`," or after the last frame "`];".
__device__ __forceinline__ void frame_suffix(uint8_t* p, const EncodeJob& j, uint32_t f)
{
    if (j.mode == 0) p += put_text(p, "\n");
    if (j.framing) {
        if (f + 1 < j.count) put_text(p, "`,\n");
        else put_text(p, "`];\n");
    }
}
__device__ __forceinline__ uint32_t prefix_len(const EncodeJob& j, uint32_t f, bool image)
{
    return (j.framing ? (f == 0 ? 17u : 2u) : 0u) + (image ? 0u : 6u);
}
__device__ __forceinline__ uint32_t suffix_len(const EncodeJob& j, uint32_t f)
{
    return (j.mode == 0 ? 1u : 0u) + (j.framing ? (f + 1 < j.count ? 3u : 4u) : 0u);
}
constexpr uint32_t PREFIX_MAX = 17 + 6, SUFFIX_MAX = 1 + 4;

// This thread's ENC_ITEMS cells [i0, i0 + ENC_ITEMS) of a frame of n cells,
// and their number inside it.  Frames start on 256-byte boundaries, so a
// whole group is one aligned 16-byte load.
__device__ __forceinline__ uint32_t load_cells(const uint32_t* __restrict__ cells, uint64_t n, uint64_t i0, uint32_t* c)
{
    static_assert(ENC_ITEMS == 4, "one uint4");
    if (i0 + ENC_ITEMS <= n) {
        const uint4 v = *(const uint4*)(cells + i0);
        c[0] = v.x;
        c[1] = v.y;
        c[2] = v.z;
        c[3] = v.w;
        return ENC_ITEMS;
    }
    const uint32_t m = i0 < n ? (uint32_t)(n - i0) : 0u;
    for (uint32_t k = 0; k < ENC_ITEMS; ++k) c[k] = k < m ? cells[i0 + k] : 0u;
    return m;
}

__device__ __forceinline__ uint32_t cells_len(const uint32_t* c, uint32_t m, int mode)
{
    uint32_t t = 0;
#pragma unroll
    for (uint32_t k = 0; k < ENC_ITEMS; ++k) t += k < m ? cell_len(c[k], mode) : 0u;
    return t;
}

template <class T>
__device__ __forceinline__ T wave_inclusive(T v)
{
    for (int d = 1; d < 64; d <<= 1) {
        const T u = __shfl_up(v, d);
        if ((int)__lane_id() >= d) v += u;
    }
    return v;
}

// Exclusive scan of v over a block of WAVES wavefronts; *total gets the sum.
template <int WAVES, class T>
__device__ __forceinline__ T block_exclusive(T v, T* s_wave, T* total)
{
    const T inc = wave_inclusive(v);
    const int w = (int)(threadIdx.x >> 6);
    if (__lane_id() == 63) s_wave[w] = inc;
    __syncthreads();
    T before = 0, sum = 0;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) {
        before += k < w ? s_wave[k] : (T)0;
        sum += s_wave[k];
    }
    *total = sum;
    return before + inc - v;
}

// Bytes of block (x, frame f_lo + y), its frame's prefix and suffix
// included; 0 past the frame's last block.
__global__ void __launch_bounds__(ENC_BLOCK) k_enc_len(EncodeJob j, uint32_t f_lo)
{
    __shared__ uint32_t s_wave[ENC_BLOCK / 64];
    const uint32_t f = f_lo + blockIdx.y, b = blockIdx.x;
    const Frame& fr = j.frames[j.first + f];
    const uint64_t n = frame_cells(fr);
    const uint32_t nb = (uint32_t)((n + ENC_CELLS - 1) / ENC_CELLS);
    uint32_t* out = j.block_len + (uint64_t)(f - j.lo) * j.max_blocks + b;
    if (b >= nb) {
        if (threadIdx.x == 0) *out = 0;
        return;
    }
    uint32_t c[ENC_ITEMS];
    const uint32_t m = load_cells(j.cells + fr.cell_off, n, (uint64_t)b * ENC_CELLS + threadIdx.x * ENC_ITEMS, c);
    uint32_t total;
    block_exclusive<ENC_BLOCK / 64>(cells_len(c, m, j.mode), s_wave, &total);
    if (threadIdx.x == 0)
        *out = total + (b == 0 ? prefix_len(j, f, fr.image != 0) : 0u) + (b == nb - 1 ? suffix_len(j, f) : 0u);
}

// Exclusive scan of the run's block lengths (one workgroup, SCAN_ITEMS a thread
// and round), from where the run before ended.  frame_off[f] = where frame f
// starts, frame_off[hi] = the length so far (host memory: the caller reads it
// after the stream).
__global__ void __launch_bounds__(SCAN_BLOCK) k_enc_scan(EncodeJob j)
{
    __shared__ uint64_t s_wave[SCAN_BLOCK / 64];
    const uint64_t n = (uint64_t)(j.hi - j.lo) * j.max_blocks;
    uint64_t carry = j.lo ? j.frame_off[j.lo] : 0;
    for (uint64_t base = 0; base < n; base += SCAN_BLOCK * SCAN_ITEMS) {
        const uint64_t i0 = base + threadIdx.x * SCAN_ITEMS;
        uint32_t l[SCAN_ITEMS];
        uint64_t t = 0;
#pragma unroll
        for (uint32_t k = 0; k < SCAN_ITEMS; ++k) {
            l[k] = i0 + k < n ? j.block_len[i0 + k] : 0u;
            t += l[k];
        }
        uint64_t total;
        uint64_t run = carry + block_exclusive<SCAN_BLOCK / 64>(t, s_wave, &total);
#pragma unroll
        for (uint32_t k = 0; k < SCAN_ITEMS; ++k) {
            if (i0 + k < n) {
                j.block_off[i0 + k] = run;
                if ((i0 + k) % j.max_blocks == 0) j.frame_off[j.lo + (i0 + k) / j.max_blocks] = run;
            }
            run += l[k];
        }
        carry += total;
        __syncthreads();   // s_wave is free for the next round
    }
    if (threadIdx.x == 0) j.frame_off[j.hi] = carry;
}

__device__ __forceinline__ uint32_t put_dec(uint8_t* p, uint32_t v)
{
    if (v >= 100u) {
        p[0] = (uint8_t)('0' + v / 100u);
        p[1] = (uint8_t)('0' + (v / 10u) % 10u);
        p[2] = (uint8_t)('0' + v % 10u);
        return 3;
    }
    if (v >= 10u) {
        p[0] = (uint8_t)('0' + v / 10u);
        p[1] = (uint8_t)('0' + v % 10u);
        return 2;
    }
    p[0] = (uint8_t)('0' + v);
    return 1;
}

__device__ __forceinline__ uint32_t put_utf8(uint8_t* p, uint32_t g)
{
    if (g < 0x80u) {
        p[0] = (uint8_t)g;
        return 1;
    }
    p[0] = (uint8_t)(0xC0u | (g >> 6));
    p[1] = (uint8_t)(0x80u | (g & 0x3Fu));
    return 2;
}

template <int MODE>
__device__ __forceinline__ uint32_t put_cell(uint8_t* p, uint32_t c)
{
    if (MODE == 0) return put_utf8(p, c & 0xFFu);
    const char* head = MODE == 1 ? "\x1b[48;2;25;25;25m\x1b[38;2;" : "<span style=\"color:rgb(";
    const uint8_t sep = MODE == 1 ? ';' : ',';
    uint32_t k = 0;
#pragma unroll
    for (; k < 23; ++k) p[k] = (uint8_t)head[k];
    k += put_dec(p + k, (c >> 8) & 0xFFu);
    p[k++] = sep;
    k += put_dec(p + k, (c >> 16) & 0xFFu);
    p[k++] = sep;
    k += put_dec(p + k, c >> 24);
    if (MODE == 1) {
        p[k++] = 'm';
        k += put_utf8(p + k, c & 0xFFu);
        p[k++] = 0x1b;
        p[k++] = '[';
        p[k++] = '0';
        p[k++] = 'm';
    } else {
        p[k++] = ')';
        p[k++] = '"';
        p[k++] = '>';
        k += put_utf8(p + k, c & 0xFFu);
    }
    return k;
}

// LDS of a block's bytes: the stage starts up to 15 bytes in, at the
// destination's offset in its 16-byte word, and is read in whole words.
template <int MODE>
constexpr uint32_t stage_bytes()
{
    return (15u + PREFIX_MAX + ENC_CELLS * max_cell_len(MODE) + SUFFIX_MAX + 15u) & ~15u;
}

// Writes block b of frame f (nb blocks, n cells) to dst.
template <int MODE>
__device__ __forceinline__ void enc_block(const EncodeJob& j, uint32_t f, const Frame& fr, uint64_t n, uint32_t b,
                                          uint32_t nb, uint8_t* __restrict__ dst, uint8_t* stage, uint32_t* s_wave)
{
    uint32_t c[ENC_ITEMS];
    const uint32_t m = load_cells(j.cells + fr.cell_off, n, (uint64_t)b * ENC_CELLS + threadIdx.x * ENC_ITEMS, c);
    uint32_t len;
    const uint32_t at = block_exclusive<ENC_BLOCK / 64>(cells_len(c, m, MODE), s_wave, &len);
    const uint32_t shift = (uint32_t)((uintptr_t)dst & 15u);
    const uint32_t pre = b == 0 ? prefix_len(j, f, fr.image != 0) : 0u;
    const uint32_t suf = b == nb - 1 ? suffix_len(j, f) : 0u;
    if (threadIdx.x == 0) {
        if (pre) frame_prefix(stage + shift, j, f, fr.image != 0);
        if (suf) frame_suffix(stage + shift + pre + len, j, f);
    }
    uint32_t p = shift + pre + at;
#pragma unroll
    for (uint32_t k = 0; k < ENC_ITEMS; ++k)
        if (k < m) p += put_cell<MODE>(stage + p, c[k]);
    __syncthreads();
    // words of the stage that the block fills whole go out as such; the
    // first and last, which it may share with its neighbours, by bytes
    const uint32_t end = shift + pre + len + suf;
    uint8_t* word0 = dst - shift;
    for (uint32_t w = threadIdx.x; w * 16u < end; w += ENC_BLOCK) {
        const uint32_t lo = w * 16u;
        if (lo >= shift && lo + 16u <= end) {
            *(uint4*)(word0 + lo) = *(const uint4*)(stage + lo);
        } else {
            for (uint32_t i = max(lo, shift); i < min(lo + 16u, end); ++i) word0[i] = stage[i];
        }
    }
}

// Block (x, frame f_lo + y) of the stream, at block_off - base of out.
template <int MODE>
__global__ void __launch_bounds__(ENC_BLOCK) k_enc_write(EncodeJob j, uint32_t f_lo, uint64_t base,
                                                         uint8_t* __restrict__ out)
{
    __shared__ __align__(16) uint8_t stage[stage_bytes<MODE>()];
    __shared__ uint32_t s_wave[ENC_BLOCK / 64];
    const uint32_t f = f_lo + blockIdx.y, b = blockIdx.x;
    const Frame& fr = j.frames[j.first + f];
    const uint64_t n = frame_cells(fr);
    const uint32_t nb = (uint32_t)((n + ENC_CELLS - 1) / ENC_CELLS);
    if (b >= nb) return;
    enc_block<MODE>(j, f, fr, n, b, nb, out + (j.block_off[(uint64_t)(f - j.lo) * j.max_blocks + b] - base), stage, s_wave);
}

// A stream of one frame of few cells, in one launch: block b finds its place
// by adding up the lengths of the cells before it (at most ENC_ONE_CELLS,
// from L2), and the last block gives the length.  out = null: the length only.
template <int MODE>
__global__ void __launch_bounds__(ENC_BLOCK) k_enc_one(EncodeJob j, uint8_t* __restrict__ out)
{
    __shared__ __align__(16) uint8_t stage[stage_bytes<MODE>()];
    __shared__ uint32_t s_wave[2][ENC_BLOCK / 64];
    const Frame& fr = j.frames[j.first];
    const uint64_t n = frame_cells(fr);
    const uint32_t nb = gridDim.x, b = blockIdx.x;
    const uint32_t* cells = j.cells + fr.cell_off;
    // cells before this block; the last one counts its own too
    const uint64_t upto = b == nb - 1 ? n : (uint64_t)b * ENC_CELLS;
    if (!out && b != nb - 1) return;
    uint32_t t = 0, own = 0;
    for (uint64_t i0 = threadIdx.x * ENC_ITEMS; i0 < upto; i0 += ENC_CELLS) {
        uint32_t c[ENC_ITEMS];
        const uint32_t m = load_cells(cells, n, i0, c);
        own = cells_len(c, m, MODE);
        t += own;
    }
    uint32_t total;
    block_exclusive<ENC_BLOCK / 64>(t, s_wave[0], &total);
    const uint32_t pre = prefix_len(j, 0, fr.image != 0);
    if (b == nb - 1 && threadIdx.x == 0) {
        j.frame_off[0] = 0;
        j.frame_off[1] = (uint64_t)pre + total + suffix_len(j, 0);
    }
    if (!out) return;
    uint32_t before = total;
    if (b == nb - 1) {
        // take the block's own cells off again
        const uint64_t i0 = (uint64_t)b * ENC_CELLS + threadIdx.x * ENC_ITEMS;
        uint32_t mine = i0 < n ? own : 0u, sum;
        __syncthreads();
        block_exclusive<ENC_BLOCK / 64>(mine, s_wave[0], &sum);
        before -= sum;
    }
    enc_block<MODE>(j, 0, fr, n, b, nb, out + (b ? pre + before : 0u), stage, s_wave[1]);
}

uint32_t encode_blocks(uint64_t n_cells) { return (uint32_t)((n_cells + ENC_CELLS - 1) / ENC_CELLS); }

uint64_t encode_bound(uint64_t n_cells, int mode)
{
    return n_cells * max_cell_len(mode) + PREFIX_MAX + SUFFIX_MAX;
}

int launch_encode_len(const EncodeJob& j, hipStream_t s)
{
    for (uint32_t f = j.lo; f < j.hi; f += 65535u) {
        hipLaunchKernelGGL(k_enc_len, dim3(j.max_blocks, std::min(65535u, j.hi - f)), dim3(ENC_BLOCK), 0, s, j, f);
        HIP_TRY(hipGetLastError());
    }
    hipLaunchKernelGGL(k_enc_scan, dim3(1), dim3(SCAN_BLOCK), 0, s, j);
    HIP_TRY(hipGetLastError());
    return SLOTH_OK;
}

int launch_encode_write(const EncodeJob& j, uint32_t f_lo, uint32_t f_hi, uint64_t base, uint8_t* out, hipStream_t s)
{
    const auto kernel = j.mode == 0 ? k_enc_write<0> : j.mode == 1 ? k_enc_write<1> : k_enc_write<2>;
    for (uint32_t f = f_lo; f < f_hi; f += 65535u) {
        hipLaunchKernelGGL(kernel, dim3(j.max_blocks, std::min(65535u, f_hi - f)), dim3(ENC_BLOCK), 0, s, j, f, base, out);
        HIP_TRY(hipGetLastError());
    }
    return SLOTH_OK;
}

int launch_encode_one(const EncodeJob& j, uint8_t* out, hipStream_t s)
{
    const auto kernel = j.mode == 0 ? k_enc_one<0> : j.mode == 1 ? k_enc_one<1> : k_enc_one<2>;
    hipLaunchKernelGGL(kernel, dim3(j.max_blocks), dim3(ENC_BLOCK), 0, s, j, out);
    HIP_TRY(hipGetLastError());
    return SLOTH_OK;
}

}  // namespace sloth
