// Differentiable shading of the visible fragments (added form; the reference
// shades with a flat glyph only, rasterizer.rs:76).
//
// Visibility is fixed: for every z slot, the raster's winner (triangle and
// pixel) is kept as (triangle << 1 | sub).  For that pixel, with the
// triangle's screen vertices and edge functions exactly as draw_triangle
// computes them (rasterizer.rs:56-74),
//   lambda_k = a * w_k                      (a = 1/orient, rasterizer.rs:67)
//   I        = L . sum_k lambda_k G n[v_k]  (G = cof(M3) / |det M3|^(2/3): the
//                                            model-to-screen normal map, scale-free)
//   C        = sum_k lambda_k c[v_k]
//   out      = I * C                         (RGB, float)
//   loss     = sum (out - target)^2          (accumulated in double)
// With n[v_k] = the face's unit normal and L = (0,0,1), I equals the flat
// shade nz_unit * a * (w0 + w1 + w2) up to rounding order.
//
// Backward: per fragment, with g = 2 (out - target) and dI = g . C,
//   d c[v_k] += lambda_k I g,  d n[v_k] += dI lambda_k G^T L,  d L += dI n.
// The pass goes by triangles: the visibility is kept as lists of each
// triangle's visible pixels (k_frag_plan), a lane sums its triangle's terms in
// binary64, and the vertices' sums are formed per workgroup in LDS, added to
// binary64 accumulators with hardware atomics and converted to binary32.
#include "sloth_shade.h"

namespace sloth {

constexpr int SHADE_BLOCK = 256;

__device__ __forceinline__ const Draw& shade_draw(const Draw* __restrict__ draws, const Frame& fr, uint32_t tri)
{
    uint32_t lo = fr.draw_begin, hi = fr.draw_end - 1;
    while (lo < hi) {
        uint32_t mid = (lo + hi + 1) >> 1;
        if (draws[mid].tri_begin <= tri) lo = mid; else hi = mid - 1;
    }
    return draws[lo];
}

// What every fragment of triangle `li` of a draw (normal map G) uses: its screen vertices,
// edge deltas and 1/orient as draw_triangle computes them (rasterizer.rs:56-67),
// its vertex ids, the normal map G applied to each vertex normal, the vertex
// colours, and G^T L (the light in model space for this view).
struct ShadeTri {
    float x1, y1, x2, y2, x3, y3, A0, B0, A1, B1, A2, B2, a;
    float gn[3][3];    // G n[v_k]
    float col[3][3];   // c[v_k]
    float gl[3];       // G^T L
    uint32_t vid[3];
};

__device__ __forceinline__ void shade_tri(const ShadeArgs& p, const Draw& dr, const float* G, uint32_t li, uint32_t W,
                                          uint32_t H, ShadeTri& s)
{
    Tri t;
    setup_draw_tri(dr, li, W, H, t);
    s.x1 = t.x1;
    s.y1 = t.y1;
    s.x2 = t.x2;
    s.y2 = t.y2;
    s.x3 = t.x3;
    s.y3 = t.y3;
    s.A0 = t.A0;
    s.B0 = t.B0;
    s.A1 = t.A1;
    s.B1 = t.B1;
    s.A2 = t.A2;
    s.B2 = t.B2;
    s.a = t.a;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const uint32_t vid = p.faces[(size_t)li * 3 + k];
        s.vid[k] = vid;
        const float* nk = p.vnormal + (size_t)vid * 3;
        const float* ck = p.vcolor + (size_t)vid * 3;
        const float a0 = nk[0], a1 = nk[1], a2 = nk[2];
        s.gn[k][0] = G[0] * a0 + G[1] * a1 + G[2] * a2;
        s.gn[k][1] = G[3] * a0 + G[4] * a1 + G[5] * a2;
        s.gn[k][2] = G[6] * a0 + G[7] * a1 + G[8] * a2;
        s.col[k][0] = ck[0];
        s.col[k][1] = ck[1];
        s.col[k][2] = ck[2];
    }
    const float L0 = p.light[0], L1 = p.light[1], L2 = p.light[2];
    s.gl[0] = G[0] * L0 + G[3] * L1 + G[6] * L2;
    s.gl[1] = G[1] * L0 + G[4] * L1 + G[7] * L2;
    s.gl[2] = G[2] * L0 + G[5] * L1 + G[8] * L2;
}

// One visible fragment of triangle s at pixel (px, py): the barycentric
// weights, the interpolated normal (mapped by G) and colour, and the shade I.
struct Fragment {
    float lam[3];
    float n0, n1, n2, c0, c1, c2, I;
};

__device__ __forceinline__ Fragment shade_at(const ShadeArgs& p, const ShadeTri& s, float px, float py)
{
    Fragment f;
    // the expressions of edges() (rasterizer.rs:71-74)
    const float w0 = s.A0 * (py - s.y2) - s.B0 * (px - s.x2);
    const float w1 = s.A1 * (py - s.y3) - s.B1 * (px - s.x3);
    const float w2 = s.A2 * (py - s.y1) - s.B2 * (px - s.x1);
    f.lam[0] = s.a * w0;
    f.lam[1] = s.a * w1;
    f.lam[2] = s.a * w2;
    f.n0 = f.n1 = f.n2 = f.c0 = f.c1 = f.c2 = 0.f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        f.n0 += f.lam[k] * s.gn[k][0];
        f.n1 += f.lam[k] * s.gn[k][1];
        f.n2 += f.lam[k] * s.gn[k][2];
        f.c0 += f.lam[k] * s.col[k][0];
        f.c1 += f.lam[k] * s.col[k][1];
        f.c2 += f.lam[k] * s.col[k][2];
    }
    f.I = p.light[0] * f.n0 + p.light[1] * f.n1 + p.light[2] * f.n2;
    return f;
}

// The pixel of z entry (row, col) of a frame of width W whose winner has
// `sub` (key_pixel without the division).
__device__ __forceinline__ void entry_pixel(uint32_t row, uint32_t col, uint32_t sub, uint32_t W, float& px, float& py)
{
    px = (float)(sub ? col >> 1 : (col + W) >> 1);
    py = (float)(sub ? row : row - 1);
}

// Block sums of up to four doubles in a fixed order, written to partial[block * 4 + k].
__device__ __forceinline__ void block_partials(double v0, double v1, double v2, double v3, double* partial,
                                               uint32_t block)
{
    __shared__ double s_red[4][SHADE_BLOCK / 64];
    for (int sh = 32; sh >= 1; sh >>= 1) {
        v0 += __shfl_xor(v0, sh);
        v1 += __shfl_xor(v1, sh);
        v2 += __shfl_xor(v2, sh);
        v3 += __shfl_xor(v3, sh);
    }
    const int wv = threadIdx.x >> 6;
    if (__lane_id() == 0) {
        s_red[0][wv] = v0;
        s_red[1][wv] = v1;
        s_red[2][wv] = v2;
        s_red[3][wv] = v3;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double s = 0.0;
        for (int w = 0; w < SHADE_BLOCK / 64; ++w) s += s_red[threadIdx.x][w];
        partial[(size_t)block * 4 + threadIdx.x] = s;
    }
}

// Forward: one thread per z slot; output colours and per-block loss sums.
__global__ void __launch_bounds__(SHADE_BLOCK) k_shade_fwd(ShadeArgs p)
{
    const uint64_t g = (uint64_t)blockIdx.x * SHADE_BLOCK + threadIdx.x;
    double loss = 0.0;
    if (g < p.n_slots) {
        uint32_t lo = 0, hi = p.n_frames - 1;
        while (lo < hi) {
            uint32_t mid = (lo + hi + 1) >> 1;
            if (p.frames[mid].z_off <= g) lo = mid; else hi = mid - 1;
        }
        const int32_t v = p.vis[g];
        if (v >= 0) {
            const Frame& fr = p.frames[lo];
            const uint32_t id = (uint32_t)(g - fr.z_off), row = id / fr.W;
            ShadeTri st;
            const Draw& dr = shade_draw(p.draws, fr, (uint32_t)v >> 1);
            shade_tri(p, dr, p.G + (size_t)(&dr - p.draws) * 9, ((uint32_t)v >> 1) - dr.tri_begin, fr.W, fr.H, st);
            float px, py;
            entry_pixel(row, id - row * fr.W, (uint32_t)v & 1u, fr.W, px, py);
            const Fragment f = shade_at(p, st, px, py);
            const float o0 = f.I * f.c0, o1 = f.I * f.c1, o2 = f.I * f.c2;
            if (p.out) {
                p.out[g * 3 + 0] = o0;
                p.out[g * 3 + 1] = o1;
                p.out[g * 3 + 2] = o2;
            }
            if (p.target) {
                const float r0 = o0 - p.target[g * 3 + 0];
                const float r1 = o1 - p.target[g * 3 + 1];
                const float r2 = o2 - p.target[g * 3 + 2];
                loss = (double)r0 * r0 + (double)r1 * r1 + (double)r2 * r2;
            }
        }
    }
    block_partials(loss, 0.0, 0.0, 0.0, p.partial, blockIdx.x);
}

// ---------------------------------------------------------------------------
// fragment lists
// ---------------------------------------------------------------------------
// An entry is a triangle of a draw and an 8 x 8 block of logical pixels at
// (x0, y0), with a bit for each pixel whose z slot the triangle won:
//   x = triangle in the draw, y = x0 | y0 << 16, z, w = the 64 bits (row-major).
// Entries of one segment (FRAG_BLOCK consecutive triangles of one draw) lie
// together, segments in (triangle block, draw) order, and a chunk is up to 64
// entries of one segment:
//   x, y = first entry (64 bits), z = entries, w = draw.
// So a chunk is one wavefront's work with a uniform draw, and neighbouring
// chunks, also those of other views, are of the same triangles.  Making the
// lists takes 0.18 ms for 32 views of 99,904 triangles (0.074 counted, 0.034
// scanned, 0.073 filled), at the first backward pass after a visibility.
constexpr uint32_t FRAG_BLOCK = SHADE_BLOCK;
constexpr int FRAG_SIDE = 8;
constexpr int FRAG_OWN = 4;   // pixel blocks of a box that its lane scans by itself

// Visible pixels of triangle word `want` (triangle << 1) in the pixel block at
// (x0, y0) of the box that ends at (bx1, by1).
__device__ __forceinline__ uint64_t frag_mask(const int32_t* __restrict__ fvis, uint32_t W, int32_t want, int x0, int y0,
                                              int bx1, int by1)
{
    uint64_t m = 0;
    const int xe = min(bx1, x0 + FRAG_SIDE - 1), ye = min(by1, y0 + FRAG_SIDE - 1);
    for (int y = y0; y <= ye; ++y) {
        const int32_t* row = fvis + (uint64_t)y * W;
        for (int x = x0; x <= xe; x += 4) {
            int32_t v[4];   // four loads in flight, past the end the last pixel again
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = row[2 * min(x + i, xe)];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int32_t key = want | (2u * (uint32_t)(x + i) < W ? 1 : 0);   // the raster's triangle << 1 | sub
                m |= (uint64_t)(v[i] == key && x + i <= xe) << ((y - y0) * FRAG_SIDE + (x + i - x0));
            }
        }
    }
    return m;
}

// Grid (triangle blocks, draws).  COUNT: the entries of each segment's four
// wavefronts; otherwise the entries and the chunks at the offsets that
// k_frag_scan made (so the lists' order is always the same).  A winner lies in
// the box that the raster's proof gives its triangle (tri_box), so no visible
// pixel is missed.  A lane scans its own box unless that holds more than
// FRAG_OWN pixel blocks; those boxes are scanned by the wavefront, one pixel
// block a lane.
template <bool COUNT>
__global__ void __launch_bounds__(FRAG_BLOCK) k_frag_plan(FragPlan p, uint32_t d_lo)
{
    static_assert(FRAG_BLOCK == 256, "a segment is four wavefronts (uint4 counts)");
    const uint32_t d = d_lo + blockIdx.y;
    const Draw& dr = p.draws[d];
    const Frame& fr = p.frames[dr.frame];
    const uint32_t W = fr.W;
    const uint64_t seg = (uint64_t)blockIdx.x * p.n_draws + d;
    const int32_t* fvis = p.vis + fr.z_off;
    const uint32_t base = blockIdx.x * FRAG_BLOCK;
    const bool valid = base + threadIdx.x < dr.n;
    const uint32_t local = valid ? base + threadIdx.x : dr.n - 1;   // dr.n > 0: the grid is empty otherwise
    const uint32_t wave = threadIdx.x >> 6;
    uint64_t first = 0;
    uint32_t n = 0;   // entries of this wavefront so far
    uint4 counts = make_uint4(0, 0, 0, 0);
    if (!COUNT) {
        counts = p.seg_count[seg];
        first = p.seg_first[seg] + (wave > 0 ? counts.x : 0u) + (wave > 1 ? counts.y : 0u) + (wave > 2 ? counts.z : 0u);
    }
    // (all lanes of the wavefront, each with its own entry or mask 0)
    auto emit = [&](uint32_t li, int x, int y, uint64_t m) {
        const uint64_t who = __ballot(m != 0);
        if (!COUNT && m) {
            const uint32_t at = n + (uint32_t)__popcll(who & ((1ull << __lane_id()) - 1));
            p.entries[first + at] = make_uint4(li, (uint32_t)x | (uint32_t)y << 16, (uint32_t)m, (uint32_t)(m >> 32));
        }
        n += (uint32_t)__popcll(who);
    };
    Tri t;
    setup_draw_tri(dr, local, W, fr.H, t);
    const uint32_t cls = valid ? setup_class(t) : CLS_EMPTY;
    int bx0 = 0, bx1 = -1, by0 = 0, by1 = -1;
    const bool any = tri_box(t, cls, bx0, bx1, by0, by1);
    const int cx = any ? (bx1 - bx0) / FRAG_SIDE + 1 : 0, cy = any ? (by1 - by0) / FRAG_SIDE + 1 : 0;
    const bool big = cx * cy > FRAG_OWN;   // at most 2^13 blocks a side
    const int own = big ? 0 : cx * cy;
    for (int k = 0; __ballot(k < own); ++k) {
        const int x = bx0 + FRAG_SIDE * (k < cx ? k : k < 2 * cx ? k - cx : k < 3 * cx ? k - 2 * cx : k - 3 * cx);
        const int y = by0 + FRAG_SIDE * (k < cx ? 0 : k < 2 * cx ? 1 : k < 3 * cx ? 2 : 3);
        emit(local, x, y,
             k < own ? frag_mask(fvis, W, (int32_t)((dr.tri_begin + local) << 1), x, y, bx1, by1) : 0ull);
    }
    for (uint64_t m = __ballot(big); m; m &= m - 1) {
        const int l = __builtin_ctzll(m);
        const int ux0 = __builtin_amdgcn_readlane(bx0, l), ux1 = __builtin_amdgcn_readlane(bx1, l);
        const int uy0 = __builtin_amdgcn_readlane(by0, l), uy1 = __builtin_amdgcn_readlane(by1, l);
        const int ucx = __builtin_amdgcn_readlane(cx, l), ucy = __builtin_amdgcn_readlane(cy, l);
        const uint32_t li = (uint32_t)__builtin_amdgcn_readlane((int)local, l);
        for (int k0 = 0; k0 < ucx * ucy; k0 += 64) {
            const int k = k0 + (int)__lane_id();
            const int x = ux0 + FRAG_SIDE * (k % ucx), y = uy0 + FRAG_SIDE * (k / ucx);
            emit(li, x, y,
                 k < ucx * ucy ? frag_mask(fvis, W, (int32_t)((dr.tri_begin + li) << 1), x, y, ux1, uy1) : 0ull);
        }
    }
    if (COUNT) {
        if (__lane_id() == 0) ((uint32_t*)(p.seg_count + seg))[wave] = n;
        return;
    }
    const uint32_t total = counts.x + counts.y + counts.z + counts.w;
    const uint64_t c0 = p.seg_chunk[seg];
    for (uint32_t c = threadIdx.x; c * 64u < total; c += FRAG_BLOCK) {
        const uint64_t e = p.seg_first[seg] + c * 64u;
        p.chunks[c0 + c] = make_uint4((uint32_t)e, (uint32_t)(e >> 32), min(64u, total - c * 64u), d);
    }
}

// Exclusive scans of the segments' entries and chunks (one workgroup); the
// totals go to host memory.
constexpr int FRAG_SCAN = 1024;
__global__ void __launch_bounds__(FRAG_SCAN) k_frag_scan(FragPlan p)
{
    __shared__ uint64_t s_e[FRAG_SCAN / 64], s_c[FRAG_SCAN / 64];
    uint64_t ce = 0, cc = 0;
    for (uint64_t b = 0; b < p.n_segs; b += FRAG_SCAN) {
        const uint64_t i = b + threadIdx.x;
        const uint4 q = i < p.n_segs ? p.seg_count[i] : make_uint4(0, 0, 0, 0);
        const uint64_t n = (uint64_t)q.x + q.y + q.z + q.w, c = (n + 63) / 64;
        uint64_t e = n, k = c;
        for (int d = 1; d < 64; d <<= 1) {
            const uint64_t ue = __shfl_up(e, d), uk = __shfl_up(k, d);
            if ((int)__lane_id() >= d) {
                e += ue;
                k += uk;
            }
        }
        const int w = (int)(threadIdx.x >> 6);
        if (__lane_id() == 63) {
            s_e[w] = e;
            s_c[w] = k;
        }
        __syncthreads();
        uint64_t be = ce, bc = cc;
#pragma unroll
        for (int j = 0; j < FRAG_SCAN / 64; ++j) {
            be += j < w ? s_e[j] : 0;
            bc += j < w ? s_c[j] : 0;
            ce += s_e[j];
            cc += s_c[j];
        }
        if (i < p.n_segs) {
            p.seg_first[i] = be + e - n;
            p.seg_chunk[i] = bc + k - c;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        p.totals[0] = ce;
        p.totals[1] = cc;
    }
}

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------
constexpr uint32_t BWD_TABLE = 512;     // LDS rows for the workgroup's distinct vertices
constexpr uint32_t BWD_PROBES = 32;     // a vertex that finds no row adds to HBM directly
constexpr uint64_t BWD_EMPTY = ~0ull;
constexpr uint32_t BWD_ROW = 7;         // 64-bit LDS words per vertex row (6 terms, padded)
constexpr uint32_t BWD_WAVES = SHADE_BLOCK / 64;
constexpr uint32_t BWD_MAX_CHUNKS = 32;   // chunks a workgroup at most takes

// Vertex rows hold their 6 sums in fixed point: term t is added as the
// integer round(t 2^(FIX_BITS - e)), with e fixed per row when the row is
// claimed (the claiming sums' largest binary exponent + FIX_HEADROOM), so
// that |integer| < 2^FIX_BITS for every |t| < 2^e and 2^(63 - FIX_BITS)
// adds cannot overflow (a row takes at most three adds per entry of the
// workgroup's chunks).  A term outside the row's range (or not finite) goes to
// the binary64 accumulator directly.  The rounding error of an add is at most
// 2^(e - FIX_BITS - 1), i.e. 2^-39 of the claiming sums' magnitude.  LDS has
// integer atomics at full rate, while a float atomic add takes several
// cycles per lane.
constexpr int FIX_BITS = 50;
constexpr int FIX_HEADROOM = 12;
static_assert(BWD_MAX_CHUNKS * 64 * 3 <= (1u << (63 - FIX_BITS)), "a row's adds stay within int64");

__device__ __forceinline__ int fix_exponent(const double* t)
{
    int e = -100;
#pragma unroll
    for (int m = 0; m < 6; ++m)
        if (t[m] != 0.0) e = max(e, __builtin_amdgcn_frexp_exp(t[m]));
    return min(e, 100) + FIX_HEADROOM;
}

// round(v) for |v| < 2^51, to nearest even: adding 1.5 2^52 leaves the integer
// in the low mantissa bits.
__device__ __forceinline__ int64_t round_small(double v)
{
    const double magic = 6755399441055744.0;
    return __double_as_longlong(v + magic) - __double_as_longlong(magic);
}

// Backward: a workgroup takes p.chunks_per_block consecutive chunks, wavefront
// w chunks w, w + BWD_WAVES, ...; a lane takes one entry.  It sets its triangle
// up once, walks the entry's visible pixels (the next one's target is loaded
// while this one is worked on) and sums the 3 x 3 colour terms and the three
// normal weights in binary64; the six terms of each vertex then go into an LDS
// table keyed by vertex, in fixed point (above).  At the end each table row
// adds its sums to the vertex's binary64 accumulators, six lanes a row: the
// six words of a row lie together, and the memory system takes such a
// run as one request.  A vertex that finds no free row adds its terms to the
// accumulators directly.  The loss and the light gradient are summed per
// block.
//
// What bounds it: arithmetic, about 125 instructions a fragment with half of
// the lanes busy (a wavefront walks as long as its fullest entry).  32 views of
// 1024 x 1024 and 99,904 triangles, 6.6M fragments: 0.096 ms.  (By z entries,
// with the triangle set up and its 18 sums converted and added for every two
// fragments, and each table row's six global atomics issued by one lane,
// 0.489 ms; with those by six lanes 0.353 ms.)
__global__ void __launch_bounds__(SHADE_BLOCK) k_shade_bwd(ShadeArgs p)
{
    // key: exponent << 32 | vertex id (set together by the claiming CAS)
    __shared__ uint64_t s_key[BWD_TABLE];
    __shared__ uint64_t s_acc[BWD_TABLE * BWD_ROW];
    for (uint32_t i = threadIdx.x; i < BWD_TABLE; i += SHADE_BLOCK) s_key[i] = BWD_EMPTY;
    for (uint32_t i = threadIdx.x; i < BWD_TABLE * BWD_ROW; i += SHADE_BLOCK) s_acc[i] = 0;
    __syncthreads();
    double loss = 0.0, dl0 = 0.0, dl1 = 0.0, dl2 = 0.0;
    const uint64_t c0 = (uint64_t)blockIdx.x * p.chunks_per_block;
    const uint64_t c1 = min(p.n_chunks, c0 + p.chunks_per_block);
    const uint32_t lane = __lane_id();
    for (uint64_t c = c0 + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); c < c1; c += BWD_WAVES) {
        const uint4 ck = p.chunks[c];
        const uint32_t d = (uint32_t)__builtin_amdgcn_readfirstlane((int)ck.w);
        const Draw& dr = p.draws[d];
        const Frame& fr = p.frames[dr.frame];
        const uint32_t W = fr.W;
        if (lane >= ck.z) continue;
        const uint4 e = p.entries[(((uint64_t)ck.y << 32) | ck.x) + lane];
        uint64_t mask = ((uint64_t)e.w << 32) | e.z;   // never 0
        const uint32_t x0 = e.y & 0xFFFFu, y0 = e.y >> 16;
        const float* ftarget = p.target + fr.z_off * 3;
        // the target of the mask's first pixel
        auto load_target = [&](uint64_t m, float* tg) {
            const uint32_t bit = (uint32_t)__builtin_ctzll(m);
            const float* q = ftarget + ((uint64_t)(y0 + bit / FRAG_SIDE) * W + 2u * (x0 + bit % FRAG_SIDE)) * 3;
            tg[0] = q[0];
            tg[1] = q[1];
            tg[2] = q[2];
        };
        float tg[3];
        load_target(mask, tg);
        ShadeTri st;
        shade_tri(p, dr, p.G + (size_t)d * 9, e.x, W, fr.H, st);
        double gc[3][3], gn[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) gn[k] = gc[k][0] = gc[k][1] = gc[k][2] = 0.0;
        for (;;) {
            const uint32_t bit = (uint32_t)__builtin_ctzll(mask);
            mask &= mask - 1;
            float next[3] = {0.0f, 0.0f, 0.0f};
            if (mask) load_target(mask, next);
            const Fragment f = shade_at(p, st, (float)(x0 + bit % FRAG_SIDE), (float)(y0 + bit / FRAG_SIDE));
            const float r0 = f.I * f.c0 - tg[0];
            const float r1 = f.I * f.c1 - tg[1];
            const float r2 = f.I * f.c2 - tg[2];
            loss += (double)r0 * r0 + (double)r1 * r1 + (double)r2 * r2;   // as the forward pass sums it
            const float g0 = 2.f * r0, g1 = 2.f * r1, g2 = 2.f * r2;
            const float dI = g0 * f.c0 + g1 * f.c1 + g2 * f.c2;
            const float i0 = f.I * g0, i1 = f.I * g1, i2 = f.I * g2;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                gc[k][0] += (double)(f.lam[k] * i0);
                gc[k][1] += (double)(f.lam[k] * i1);
                gc[k][2] += (double)(f.lam[k] * i2);
                gn[k] += (double)(dI * f.lam[k]);
            }
            dl0 += (double)(dI * f.n0);
            dl1 += (double)(dI * f.n1);
            dl2 += (double)(dI * f.n2);
            if (!mask) break;
            tg[0] = next[0];
            tg[1] = next[1];
            tg[2] = next[2];
        }
        // the triangle's sums to the table: the three vertices' first probes
        // are issued together
        double acc[3][6];
        uint64_t mine[3], old[3];
        uint32_t h[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                acc[k][m] = gc[k][m];
                acc[k][3 + m] = gn[k] * (double)st.gl[m];
            }
            mine[k] = ((uint64_t)(uint32_t)fix_exponent(acc[k]) << 32) | st.vid[k];
            h[k] = (st.vid[k] * 0x9E3779B1u) >> 23;   // BWD_TABLE = 512 rows
            old[k] = atomicCAS((unsigned long long*)&s_key[h[k]], (unsigned long long)BWD_EMPTY,
                               (unsigned long long)mine[k]);
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint32_t vid = st.vid[k];
            bool found = old[k] == BWD_EMPTY || (uint32_t)old[k] == vid;
            for (uint32_t probe = 1; !found && probe < BWD_PROBES; ++probe) {
                h[k] = (h[k] + 1) & (BWD_TABLE - 1);
                old[k] = atomicCAS((unsigned long long*)&s_key[h[k]], (unsigned long long)BWD_EMPTY,
                                   (unsigned long long)mine[k]);
                found = old[k] == BWD_EMPTY || (uint32_t)old[k] == vid;
            }
            // the row's exponent: the claimer's (this lane's when it claimed the row)
            const int ex = (int)(uint32_t)((old[k] == BWD_EMPTY ? mine[k] : old[k]) >> 32);
            double* dst = p.vert_acc + (size_t)vid * 6;
            const double lim = __builtin_ldexp(1.0, ex), sc = __builtin_ldexp(1.0, FIX_BITS - ex);
#pragma unroll
            for (int m = 0; m < 6; ++m) {
                const double t = acc[k][m];
                if (found && fabs(t) < lim)
                    atomicAdd((unsigned long long*)&s_acc[h[k] * BWD_ROW + m], (unsigned long long)round_small(t * sc));
                else
                    unsafeAtomicAdd(dst + m, t);
            }
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < BWD_TABLE * 6; i += SHADE_BLOCK) {
        const uint32_t r = i / 6, m = i - r * 6;
        const uint64_t key = s_key[r];
        if (key != BWD_EMPTY) {
            const double sc = __builtin_ldexp(1.0, (int)(uint32_t)(key >> 32) - FIX_BITS);
            unsafeAtomicAdd(p.vert_acc + (size_t)(uint32_t)key * 6 + m, (double)(int64_t)s_acc[r * BWD_ROW + m] * sc);
        }
    }
    block_partials(loss, dl0, dl1, dl2, p.partial, blockIdx.x);
}

// The vertices' binary64 sums as the binary32 gradients; the sums are left at
// zero for the next pass.  Six lanes a vertex, so that loads and stores are
// contiguous.
__global__ void __launch_bounds__(SHADE_BLOCK) k_shade_finish(double* __restrict__ vert_acc, uint32_t n_verts,
                                                              float* __restrict__ d_color, float* __restrict__ d_normal)
{
    const uint64_t i = (uint64_t)blockIdx.x * SHADE_BLOCK + threadIdx.x;
    if (i >= (uint64_t)n_verts * 6) return;
    const uint64_t v = i / 6;
    const uint32_t m = (uint32_t)(i - v * 6);
    const float g = (float)vert_acc[i];
    vert_acc[i] = 0.0;
    if (m < 3) d_color[v * 3 + m] = g;
    else d_normal[v * 3 + (m - 3)] = g;
}

// Sums of the blocks' partials (n blocks, four each), in an order fixed by n.
constexpr int SUM_BLOCK = 1024;
__global__ void __launch_bounds__(SUM_BLOCK) k_shade_sum(const double* __restrict__ partial, uint32_t n,
                                                         double* __restrict__ sum)
{
    __shared__ double s[4][SUM_BLOCK / 64];
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (uint32_t i = threadIdx.x; i < n; i += SUM_BLOCK)
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] += partial[(size_t)i * 4 + k];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        for (int sh = 32; sh >= 1; sh >>= 1) v[k] += __shfl_xor(v[k], sh);
        if (__lane_id() == 0) s[k][threadIdx.x >> 6] = v[k];
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double t = 0.0;
        for (int w = 0; w < SUM_BLOCK / 64; ++w) t += s[threadIdx.x][w];
        sum[threadIdx.x] = t;
    }
}

__global__ void __launch_bounds__(SHADE_BLOCK) k_fill_f64(double* __restrict__ a, uint64_t n)
{
    const uint64_t stride = (uint64_t)gridDim.x * SHADE_BLOCK;
    for (uint64_t i = (uint64_t)blockIdx.x * SHADE_BLOCK + threadIdx.x; i < n; i += stride) a[i] = 0.0;
}

uint32_t shade_blocks(uint64_t n_slots) { return (uint32_t)((n_slots + SHADE_BLOCK - 1) / SHADE_BLOCK); }

uint64_t frag_segments(uint32_t n_tris, uint32_t n_draws)
{
    return (uint64_t)((n_tris + FRAG_BLOCK - 1) / FRAG_BLOCK) * n_draws;
}

// A workgroup takes as many chunks as leave about BWD_GRID workgroups (two
// rounds of what the chip holds): more chunks merge more of a vertex's sums
// before the global adds (0.096 ms at 1024 and 2048, 0.101 at 4096, 0.125 from
// 8192 on).
constexpr uint64_t BWD_GRID = 2048;
uint32_t bwd_chunks_per_block(uint64_t n_chunks)
{
    const uint64_t per = (n_chunks / BWD_GRID + BWD_WAVES - 1) / BWD_WAVES * BWD_WAVES;
    return (uint32_t)std::min<uint64_t>(BWD_MAX_CHUNKS, std::max<uint64_t>(BWD_WAVES, per));
}
uint32_t bwd_blocks(uint64_t n_chunks)
{
    const uint64_t per = bwd_chunks_per_block(n_chunks);
    return (uint32_t)((n_chunks + per - 1) / per);
}

static int launch_frag(const FragPlan& p, bool count, uint32_t n_tris, hipStream_t s)
{
    const uint32_t nb = (n_tris + FRAG_BLOCK - 1) / FRAG_BLOCK;
    if (nb == 0) return SLOTH_OK;
    for (uint32_t d = 0; d < p.n_draws; d += 65535u) {
        const dim3 grid(nb, std::min(65535u, p.n_draws - d));
        if (count) hipLaunchKernelGGL(k_frag_plan<true>, grid, dim3(FRAG_BLOCK), 0, s, p, d);
        else hipLaunchKernelGGL(k_frag_plan<false>, grid, dim3(FRAG_BLOCK), 0, s, p, d);
        HIP_TRY(hipGetLastError());
    }
    return SLOTH_OK;
}

int launch_frag_count(const FragPlan& p, uint32_t n_tris, hipStream_t s)
{
    int rc = launch_frag(p, true, n_tris, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_frag_scan, dim3(1), dim3(FRAG_SCAN), 0, s, p);
    HIP_TRY(hipGetLastError());
    return SLOTH_OK;
}

int launch_frag_fill(const FragPlan& p, uint32_t n_tris, hipStream_t s) { return launch_frag(p, false, n_tris, s); }

int launch_shade_fwd(const ShadeArgs& a, double* sum, hipStream_t s)
{
    const uint32_t nb = shade_blocks(a.n_slots);
    if (nb) {
        hipLaunchKernelGGL(k_shade_fwd, dim3(nb), dim3(SHADE_BLOCK), 0, s, a);
        HIP_TRY(hipGetLastError());
    }
    hipLaunchKernelGGL(k_shade_sum, dim3(1), dim3(SUM_BLOCK), 0, s, (const double*)a.partial, nb, sum);
    HIP_TRY(hipGetLastError());
    return SLOTH_OK;
}

int launch_shade_zero(const ShadeArgs& a, hipStream_t s)
{
    const uint64_t n = (uint64_t)a.n_verts * 6;
    if (n == 0) return SLOTH_OK;
    hipLaunchKernelGGL(k_fill_f64, dim3((unsigned)std::min<uint64_t>(4096, (n + SHADE_BLOCK - 1) / SHADE_BLOCK)),
                       dim3(SHADE_BLOCK), 0, s, a.vert_acc, n);
    HIP_TRY(hipGetLastError());
    return SLOTH_OK;
}

int launch_shade_bwd(const ShadeArgs& a, float* d_color, float* d_normal, double* sum, hipStream_t s)
{
    const uint32_t nb = bwd_blocks(a.n_chunks);
    if (nb) {
        hipLaunchKernelGGL(k_shade_bwd, dim3(nb), dim3(SHADE_BLOCK), 0, s, a);
        HIP_TRY(hipGetLastError());
    }
    hipLaunchKernelGGL(k_shade_sum, dim3(1), dim3(SUM_BLOCK), 0, s, (const double*)a.partial, nb, sum);
    HIP_TRY(hipGetLastError());
    if (a.n_verts) {
        hipLaunchKernelGGL(k_shade_finish, dim3((unsigned)(((uint64_t)a.n_verts * 6 + SHADE_BLOCK - 1) / SHADE_BLOCK)),
                           dim3(SHADE_BLOCK), 0, s, a.vert_acc, a.n_verts, d_color, d_normal);
        HIP_TRY(hipGetLastError());
    }
    return SLOTH_OK;
}

}  // namespace sloth
