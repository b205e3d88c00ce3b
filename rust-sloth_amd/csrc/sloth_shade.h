// Differentiable shading kernels (internal); see sloth_shade.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sloth_device.h"
#include "sloth_host.h"

namespace sloth {

struct ShadeArgs {
    const Frame* frames;
    uint32_t n_frames;
    const Draw* draws;
    const int32_t* vis;       // per z slot: (triangle << 1 | sub), -1 = none
    const uint32_t* faces;    // [n_tris][3] vertex ids (mesh-local triangle index)
    const float* vcolor;      // [n_verts][3]
    const float* vnormal;     // [n_verts][3]
    const float* light;       // [3]
    const float* G;           // per draw, 3x3 row-major normal map
    const float* target;      // per z slot [3], or null (no loss)
    float* out;               // per z slot [3], or null
    double* partial;          // per block: loss, dL.x, dL.y, dL.z
    double* vert_acc;         // [n_verts][6]: d color, d normal (binary64 sums)
    uint64_t n_slots;
    uint32_t n_tris, n_verts;
    const uint4* entries;     // fragment lists (k_frag_plan)
    const uint4* chunks;
    uint64_t n_chunks;
    uint32_t chunks_per_block;
};

// The fragment lists: which pixels of each triangle are visible.
struct FragPlan {
    const Frame* frames;
    const Draw* draws;
    uint32_t n_draws;
    const int32_t* vis;
    uint64_t n_segs;
    uint4* seg_count;         // per segment: entries of its wavefronts
    uint64_t* seg_first;      // its first entry
    uint64_t* seg_chunk;      // its first chunk
    uint64_t* totals;         // entries, chunks (host memory)
    uint4* entries;
    uint4* chunks;
};

uint32_t shade_blocks(uint64_t n_slots);
uint64_t frag_segments(uint32_t n_tris, uint32_t n_draws);
// chunks per workgroup of the backward pass, and its workgroups (per-block
// partial sums)
uint32_t bwd_chunks_per_block(uint64_t n_chunks);
uint32_t bwd_blocks(uint64_t n_chunks);
// Entries of every segment, their offsets and totals; then the lists.  Every
// draw has n_tris triangles.
int launch_frag_count(const FragPlan& p, uint32_t n_tris, hipStream_t s);
int launch_frag_fill(const FragPlan& p, uint32_t n_tris, hipStream_t s);
// sum: loss, and from the backward pass the light gradient
int launch_shade_fwd(const ShadeArgs& a, double* sum, hipStream_t s);
// vert_acc to zero
int launch_shade_zero(const ShadeArgs& a, hipStream_t s);
// vert_acc is zero before and after
int launch_shade_bwd(const ShadeArgs& a, float* d_color, float* d_normal, double* sum, hipStream_t s);

}  // namespace sloth
