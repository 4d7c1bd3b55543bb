// Internal structures shared by the HIP kernels and the C-ABI host code.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/bmf.h"

namespace bmf {

constexpr int kRowThreads = 256;      // word kernels: 4 waves, an item of label words each
constexpr int kItemWords = 16;        // label words per item: enough active cells for a wave's lanes near a surface
constexpr int kItemSamples = 64 * kItemWords;
constexpr int kWaveBlocks = 16;       // 4 x 4 x 4 sample blocks per wave of k_blocks
constexpr int kSmoothThreads = 256;   // one vertex per thread
constexpr int kMaxRowWords = 4;       // ceil(BMF_MAX_DIM / 64)
constexpr int kXcds = 8;              // MI355X: 8 XCDs, each with its own L2

enum ChunkState : int32_t {
    kStateAir = 0,      // culled: every sample is air (d < 0 everywhere)
    kStateSolid = 1,    // culled: every sample is solid
    kStateSampled = 2,  // densities and labels computed
    kStateSkipped = 3   // did not fit an arena
};

// Device view of the sampler (Sampler + NoiseSamplerProperties).
struct SamplerDev {
    int32_t kind;
    float world_size;
    float amp, y0;
    int32_t octaves;
    float inv_norm;
    uint32_t seed;
    int32_t n_spheres, n_boxes;
    float fo[BMF_MAX_OCTAVES];  // per-octave frequency f0 * L^o (FP32 product chain)
    float ao[BMF_MAX_OCTAVES];  // per-octave amplitude g^o
    // reach[k] >= the most the FP32 partial sum after k octaves can still
    // move: sum of |a_o| for o >= k plus the rounding slack of those steps
    float reach[BMF_MAX_OCTAVES + 1];
    int32_t expand_ok;          // terrain: the noise sum can be expanded about block centres (k_blocks)
    const float* spheres;       // device, n_spheres x 4
    const float* boxes;         // device, n_boxes x 6
    float csg_slack;            // CSG: bounds the FP32 error of a primitive's value and of its cull (csg_reach)
    const float* ext;           // EXTERNAL: caller's densities, chunks packed in descriptor order
    // NOISE: basis, fractal, density map and perturbation (bmf_sampler_desc)
    int32_t noise_dims, noise_basis, noise_fractal;
    float g_scale, y_scale, height;
    int32_t perturb, perturb_octaves;
    float perturb_amp;
    float pf[BMF_MAX_PERTURB_OCTAVES];  // perturbation frequency f * 2^k (FP32 chain)
    float pa[BMF_MAX_PERTURB_OCTAVES];  // GRADIENT: amp * gain^k; OFFSET_XZ: gain^k
    float pinv;                         // OFFSET_XZ: 1 / sum of pa
    // k_plan's chunk culling: n lies in [nlo, nhi] for every sample (cull = 0: no bound)
    float nlo, nhi;
    int32_t cull;
    // 3D NOISE (k_field): the fractal's sum after k octaves moves at most
    // field_dn[k] down and field_up[k] up (1, then every step's rounding
    // included); early_ok = 0: the terms are too large for such bounds
    float field_dn[BMF_MAX_OCTAVES + 1], field_up[BMF_MAX_OCTAVES + 1];
    int32_t early_ok;
};

// How k_blocks expands a terrain chunk's noise: octaves per block and per
// sub-block (0: the level is left out), and the error quad * r^2 + base of
// the sum at a sample r sample steps from the centre.
struct BlockPlan {
    int32_t k4, k2;
    float quad4, base4, quad2, base2;
};

// Per-chunk state in device memory.
struct ChunkMeta {
    float opos[3];
    float delta;
    int32_t dim;
    int32_t iters;
    int32_t bp;
    int32_t state;
    int64_t dens_off;   // float index into the density arena
    int64_t lab_off;    // u64 index into the label bitmap arena
    int64_t lab_words;  // u64 words of this chunk's bitmap
    uint32_t any_air;   // set by the sampling kernel
    uint32_t any_solid;
    int32_t contains_mesh;
    int32_t status;
    int32_t V;          // vertices
    int32_t T;          // primitives (triangles, or quads in the quad mode)
    int32_t ipp;        // indices per primitive: 3 or 4
    int32_t csg_ns;     // CSG: spheres and boxes that can reach above the floor in this chunk,
    int32_t csg_nb;     //      listed in Arenas::csg_list (sphere ids, then box ids, in order)
    int64_t v_off;      // output offsets
    int64_t i_off;
    BlockPlan blocks;   // adaptive terrain
    int64_t item_slot;  // the chunk's first item of the word kernels (sampled chunks)
};

// Global counters, reset by the plan kernel.
struct Counters {
    unsigned long long v_bump;
    unsigned long long i_bump;
    unsigned long long need_v;
    unsigned long long need_i;
    int64_t total_samples;
    int32_t xcd_vtiles[kXcds]; // smoothing tiles of each XCD's maps
    int32_t xcd_ttiles[kXcds];
    int32_t n_smooth;
    int32_t overflow;
    int32_t error;
    int64_t total_items;       // items of the word kernels
    int32_t n_work;            // of these, the ones with edges or cells
};

// A tile of a chunk's vertices or primitives in the smoothing: what its
// kernels need of the chunk, so that a tile is one load and not a tour of the
// chunk table.
struct alignas(16) SmoothTile {
    int32_t chunk, tile;
    int32_t V, T;
    int64_t v_off, i_off, t_off;  // first vertex, index and primitive (t_off = i_off / ipp)
    int32_t iters;
    uint8_t bp, ipp;
    uint16_t dim;
};

// One label word's sign-changing edges per axis (in the quad mode only those
// whose four cells lie in the chunk) and active cells, as bits of its samples.
struct EdgeWord {
    uint64_t ex, ey, ez, ac;
};

// Device pointers of one context.
struct Arenas {
    ChunkMeta* meta;           // [max_chunks]
    bmf_chunk_desc* descs;     // [max_chunks]
    bmf_chunk_result* results; // [max_chunks]
    int64_t* block_prefix;     // [max_chunks + 1] items of the sampler's pre-pass: kWaveBlocks sample blocks
                               // (k_blocks) or 64 columns (k_columns)
    uint8_t* signs;            // [max_samples + 16] adaptive terrain: k_blocks' decisions, from the chunk's first
                               // sample on a byte per four samples of a row (x, y), ceil(dim / 4) bytes a row:
                               // undecided samples in the low bits, air samples in the high ones
    int64_t* plan_part;        // [8 nb + 1] multi-block plan passes (nb = max_chunks / 1024 rounded up): block
                               // totals and bases, overflow flag
    unsigned long long* stat_blocks;  // [3][stat_cap] terrain octaves evaluated per workgroup of the
                                      // sampling, refinement and block kernels (plain stores, no atomics)
    int32_t stat_cap;
    int2* item_map;            // [max_items] (chunk, item within the chunk) of the word kernels' items
                               // (written by the sampling)
    int2* work;                // [max_items] (chunk, item within the chunk) of the items with edges or cells, a
                               // chunk's in order (k_scan): what the emission takes
    SmoothTile* smooth_vmap;   // [kXcds][cap_vtiles] the smoothing's vertex tiles of each XCD (k_scan)
    SmoothTile* smooth_tmap;   // [kXcds][cap_ttiles] the same for the triangle tiles
    int64_t cap_vtiles, cap_ttiles;
    EdgeWord* edges;           // same layout as labels: edge and active-cell bits of each word
    uint32_t* word_pre;        // same layout: edges of the item before the word
    uint32_t* item_e;          // [max_items] edges of each item, then their exclusive prefix in the chunk
    uint32_t* item_c;          // [max_items] the same for triangles (polygons in the quad mode)
    float* dens;               // [max_samples]
    uint64_t* labels;          // [max_samples / 64 + max_chunks]
    uint64_t* exact;           // same layout as labels: density of the sample is final
    uint32_t* cell_tb;         // [max_samples] first triangle of each surface cell
    uint8_t* cell_mask;        // [max_samples] corner mask of each surface cell
    float* pos;                // [max_vertices * 3]
    float4* pos4;              // [max_vertices] positions during the smoothing
    float4* cen4;              // [max_indices / 3] triangle centroids
    uint8_t* boundary;         // [max_vertices]
    uint32_t* vedge;           // [max_vertices] lattice edge of each vertex: x | y<<8 | z<<16 | axis<<24
    uint4* vring;              // [max_vertices] ring cells of each vertex, packed by the first smoothing step
    uint32_t* idx;             // [max_indices]
    Counters* ctr;
    // The host's copies, in pinned memory that the kernels write: the results
    // and counters by the emit kernel, the error flag where it is raised.  Two copies after the pipeline took 4 us of
    // the device and 10 of the calling thread.
    bmf_chunk_result* host_results;  // [max_chunks]
    Counters* host_ctr;
    SamplerDev* sampler;
    const float* ext;          // the caller's densities of this call, before the EXTERNAL sampler's own
    int64_t cap_samples, cap_vertices, cap_indices;
    int32_t cap_chunks;
    int64_t ext_base;          // EXTERNAL: offset of this launch's first chunk in the caller's densities
    int32_t smoothing_follows; // the launch runs the smoothing kernels after the emit kernel (which then
                               // leaves the output positions of the vertices they move to them)
    uint16_t* csg_list;        // CSG: [chunk][csg_stride] primitives per chunk (k_plan), or null
    int32_t csg_stride;        // n_spheres + n_boxes
    // mesh options (BMF_MESH_*, BMF_PLACE_*): the quad mode's extra arenas
    int32_t mesh_mode;
    int32_t placement;
    float qef_tol;
    int32_t quad_tris;         // quads written as two triangles each
    uint32_t* ring;            // [kRingSlots][cap_vertices] primitives around each vertex (quad mode)
    uint32_t* ring_n;          // [cap_vertices] ring sizes
    float* qef_err;            // [cap_vertices] QEF residual of each vertex (QEF placement)
    // vertex normals of the triangle path (bmf_mesh_options::normals)
    int32_t normals;
    float4* nrm4;              // [cap_vertices] normal state during the smoothing
    float4* fn4;               // [cap_indices / 3] per-triangle normal of the current step
    float* nrm;                // [cap_vertices * 3] unit normals (output)
};

// Quad mode: a vertex (one polygon of a cell) has at most 7 edges, so at most
// 7 quads, or 14 triangles when quads are written as triangles.
constexpr int kRingSlots = 16;

// Workgroups that sample one chunk of ns samples: a wave per 256 of them, the
// finest of the sampling kernels' items.
inline int sample_blocks_of(int64_t ns) { return (int)((ns + 1023) / 1024); }
// Workgroups that give every item of one chunk's word kernels its wave.
inline int word_blocks(int dim) {
    const int64_t items = ((int64_t)dim * dim * dim + kItemSamples - 1) / kItemSamples;
    return (int)((items + kRowThreads / 64 - 1) / (kRowThreads / 64));
}

// What k_count evaluates again: nothing, or the endpoints of sign-changing
// edges that the adaptive terrain or 3D field sampling labelled early.
constexpr int kRefineNone = 0, kRefineTerrain = 1, kRefineField = 2;
inline int refinement(const SamplerDev& S) {
    return S.kind == BMF_SAMPLER_TERRAIN                        ? kRefineTerrain
           : S.kind == BMF_SAMPLER_NOISE && S.noise_dims == 3 ? kRefineField
                                                              : kRefineNone;
}

// Launch wrappers (bmf_kernels.hip).
// one: the single descriptor by value (n = 1), instead of A.descs
hipError_t launch_plan(const Arenas& A, int n, int allow_cull, int reset_bumps, hipStream_t s,
                       const bmf_chunk_desc* one = nullptr);
// adaptive: signs everywhere and densities where the surface reads them (terrain, CSG); 0: every density
// kind: the sampler the device struct holds for this launch (BMF_SAMPLER_*)
// slab: the sampler is a 2D noise field (its columns are evaluated in a pass of their own)
hipError_t launch_sample(const Arenas& A, int n, int blocks, int adaptive, int kind, int slab, hipStream_t s);
// refine: give early-labelled edge endpoints their full density (after an adaptive terrain launch_sample)
hipError_t launch_count(const Arenas& A, int blocks, int refine, hipStream_t s);
hipError_t launch_scan(const Arenas& A, int n, int blocks, hipStream_t s);
hipError_t launch_emit(const Arenas& A, int n, int blocks, hipStream_t s);
hipError_t launch_smooth(const Arenas& A, int m, int blocks, hipStream_t s);
// Quad mode (bmf_dmc.hip): emission after launch_count / launch_scan,
// smoothing over the per-vertex rings.
hipError_t launch_dmc_emit(const Arenas& A, int n, int blocks, hipStream_t s);
hipError_t launch_dmc_smooth(const Arenas& A, int m, int blocks, hipStream_t s);
hipError_t launch_ref_labels(const Arenas& A, uint32_t* words, hipStream_t s);
hipError_t launch_ref_masks(const Arenas& A, uint64_t* masks, hipStream_t s);

}  // namespace bmf
