// Seams between the chunks of a world octree (C ABI bmf_stitch in
// include/bmf.h): the marching-cubes triangles of the dual cells that
// straddle chunk boundaries, the output of WorldStitcher::stitch_all
// (WorldStitcher.cpp:26-49) over the chunks' shell octrees
// (DMCChunk::generate_octree, DMCChunk.cpp:700-778).
//
// The reference walks the world octree recursively (stitch_cell, the face
// and edge recursions, stitch_indexes: WorldStitcher.cpp:184-572); here the
// same dual cells are enumerated point by point, the candidate points in a
// fixed order (the chunks of the leaf list in order, the lattice
// points of each chunk's closed cube [0, dim]^3 on the cube's boundary in
// x-major order):
//   - integer geometry in units of the finest unit node: a node at level l
//     with morton code 1 d1 .. dl spans [sum_k d_k 2^(L-k) dim, + 2^(L-l) dim)
//     per axis (L the deepest level);
//   - a point is stitched when its 8 octant neighbourhoods lie in the world
//     but not all in one chunk, by the finest of those chunks (the lowest
//     node index among equals);
//   - corner c (4*dx + 2*dy + dz) is the unit node of octant c's chunk that
//     contains the point's octant c, placed where the shell octree places it
//     (pos + MCD * size/2 + MCD * size/4 + ..., FP32 in that order), valued
//     by the sampler there;
//   - marching cubes as stitch_indexes: crossing (v1 - v0) * mu + v0,
//     mu = (0 - s0) / (s1 - s0), triangles from the tri_table.
// Four launches: the world's root and deepest level, count (triangles per
// candidate, and per 256-candidate tile: a thread per candidate finds its
// chunks, 8 lanes its corners' signs, of the terrain by no more octaves than
// they take to be certain), a one-workgroup scan of the tile totals, emit (the
// cells of the candidates with triangles again, 8 lanes each and every octave,
// written at their offsets).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "../../include/bmf.h"
#include "bmf_context.h"
#include "bmf_device_tables.h"
#include "bmf_internal.h"
#include "bmf_rows.h"
#include "samplers.h"

namespace bmf {
namespace {

constexpr int kStitchThreads = 256;  // candidates per tile
constexpr int kScanThreads = 1024;

#define BMF_HIP(call)                          \
    do {                                       \
        hipError_t e_ = (call);                \
        if (e_ != hipSuccess) return BMF_EHIP; \
    } while (0)

// the child of a node in direction (dx, dy, dz), index dx | dy << 1 | dz << 2
// (children are numbered by the corner tables MCDX/Y/Z, Tables.hpp:7-9)
__constant__ int c_child_of[8] = {0, 1, 4, 5, 3, 2, 7, 6};
// corners of the 12 local edges in the tables' numbering
__constant__ int c_edge[12][2] = {{0, 4}, {1, 5}, {2, 6}, {3, 7}, {0, 2}, {1, 3},
                                  {4, 6}, {5, 7}, {0, 1}, {2, 3}, {4, 5}, {6, 7}};

struct World {
    const bmf_world_node* nodes;
    int n_nodes;
    int dim;             // unit nodes per chunk edge (a power of two)
    int log_dim;
    const int* root_level;  // device: the root's index (-1: none) and the deepest level L
    const float* max_size;  // device: the largest size of a leaf (0: none)
};

// Integer coordinates (twice the lattice's, so that octant points are whole)
// reach 2^(L + 1) dim: 32-bit arithmetic up to this many bits, 64-bit beyond.
constexpr int kNarrowBits = 28;
// Deepest level whose coordinates fit 64 bits for the largest dim.
constexpr int kMaxLevel = 62 - 9;

template <typename I>
struct Box {
    I o[3], e;  // origin and edge, in finest unit nodes
    int id;
};

// The box of node i from its level and morton code.
template <typename I>
__device__ __forceinline__ Box<I> node_box(const World& W, int L, int i) {
    const int l = W.nodes[i].level;
    const uint64_t m = W.nodes[i].morton;
    Box<I> b{{0, 0, 0}, (I)1 << (L - l + W.log_dim), i};
    for (int k = 1; k <= l; k++) {
        const int d = (int)((m >> (3 * (l - k))) & 7u);
        const I w = (I)1 << (L - k + W.log_dim);
        b.o[0] += (d & 1) ? w : 0;
        b.o[1] += ((d >> 1) & 1) ? w : 0;
        b.o[2] += ((d >> 2) & 1) ? w : 0;
    }
    return b;
}

// Whether the point p2 / 2 lies in the half-open box.
template <typename I>
__device__ __forceinline__ bool inside(const Box<I>& b, const I (&p2)[3]) {
    bool in = true;
#pragma unroll
    for (int a = 0; a < 3; a++) in = in && p2[a] >= 2 * b.o[a] && p2[a] < 2 * (b.o[a] + b.e);
    return in;
}

// The world leaf containing the point p2 / 2 (id -1: none), its box halved
// on the way down: one dependent load per level.
template <typename I>
__device__ __forceinline__ Box<I> locate(const World& W, int L, const Box<I>& root, const I (&p2)[3]) {
    Box<I> b = root;
    if (!inside(b, p2)) b.id = -1;
    for (int guard = 0; guard <= L + 1; guard++) {
        if (b.id < 0 || b.id >= W.n_nodes) break;
        const int h[3] = {p2[0] >= 2 * b.o[0] + b.e, p2[1] >= 2 * b.o[1] + b.e, p2[2] >= 2 * b.o[2] + b.e};
        const bmf_world_node& q = W.nodes[b.id];
        const int leaf = q.world_leaf, next = q.children[c_child_of[h[0] | (h[1] << 1) | (h[2] << 2)]];
        if (leaf) return b;
        b.e >>= 1;
#pragma unroll
        for (int a = 0; a < 3; a++) b.o[a] += h[a] ? b.e : 0;
        b.id = next;
    }
    b.id = -1;
    return b;
}

// Lattice index (i, j, k) of candidate t among the boundary points of the
// cube [0, d]^3 in x-major order.
__device__ __forceinline__ void boundary_point(uint32_t t, int d, int& i, int& j, int& k) {
    const uint32_t face = (uint32_t)(d + 1) * (uint32_t)(d + 1), ring = 4u * (uint32_t)d;
    if (t < face) {
        i = 0;
        j = (int)(t / (d + 1));
        k = (int)(t % (d + 1));
        return;
    }
    t -= face;
    if (t >= (uint32_t)(d - 1) * ring) {
        t -= (uint32_t)(d - 1) * ring;
        i = d;
        j = (int)(t / (d + 1));
        k = (int)(t % (d + 1));
        return;
    }
    i = 1 + (int)(t / ring);
    int s = (int)(t % ring);
    if (s < d + 1) {
        j = 0;
        k = s;
    } else if (s < d + 1 + 2 * (d - 1)) {
        const int u = s - (d + 1);
        j = 1 + u / 2;
        k = (u & 1) * d;
    } else {
        j = d;
        k = s - (d + 1) - 2 * (d - 1);
    }
}

// The chunk of a leaf list entry: its box, and whether the points of its box
// are found in it by descent (`own`; false when the entry is no leaf of the
// tree), which spares the octants on its side theirs.
template <typename I>
struct LeafBox {
    Box<I> b;
    int own;
};
template <typename I>
__device__ __forceinline__ LeafBox<I> leaf_box(const World& W, int L, const Box<I>& root, int leaf) {
    LeafBox<I> r{{{0, 0, 0}, 0, -1}, 0};
    if (leaf < 0 || leaf >= W.n_nodes) return r;
    r.b = node_box<I>(W, L, leaf);
    const I mid[3] = {2 * r.b.o[0] + 1, 2 * r.b.o[1] + 1, 2 * r.b.o[2] + 1};
    const Box<I> f = locate<I>(W, L, root, mid);
    r.own = f.id == leaf && f.e == r.b.e;
    return r;
}

// Twice the lattice point of candidate t of the leaf.
template <typename I>
__device__ __forceinline__ void candidate_point(const World& W, const Box<I>& leaf, uint32_t t, I (&P2)[3]) {
    int i, j, k;
    boundary_point(t, W.dim, i, j, k);
    const int ul = W.log_dim;  // the unit node's edge is the chunk's / dim
    P2[0] = 2 * (leaf.o[0] + (leaf.e >> ul) * (I)i);
    P2[1] = 2 * (leaf.o[1] + (leaf.e >> ul) * (I)j);
    P2[2] = 2 * (leaf.o[2] + (leaf.e >> ul) * (I)k);
}

// A point of octant c (4 dx + 2 dy + dz) around P.
template <typename I>
__device__ __forceinline__ void octant_point(const I (&P2)[3], int c, I (&p2)[3]) {
    p2[0] = P2[0] + ((c & 4) ? 1 : -1);
    p2[1] = P2[1] + ((c & 2) ? 1 : -1);
    p2[2] = P2[2] + ((c & 1) ? 1 : -1);
}

// Where corner c of the dual cell lies: the unit node of octant c's chunk
// (box b) that holds the octant, placed as the shell octree places it.
template <typename I>
__device__ __forceinline__ void corner_position(const World& W, int L, const Box<I>& b, const I (&P2)[3], int c,
                                                float (&p)[3]) {
    const bmf_world_node& q = W.nodes[b.id];
    int n[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const I rel = (P2[a] >> 1) - b.o[a], u = b.e >> W.log_dim;  // u a power of two
        const int sh = 63 - __clzll((long long)u);
        n[a] = ((c >> (2 - a)) & 1) ? (int)(rel >> sh) : (int)((rel + u - 1) >> sh) - 1;
        p[a] = q.pos[a];
    }
    float size = q.size;
    for (int half = W.log_dim - 1; half >= 0; half--) {
        const float cs = size * 0.5f;
#pragma unroll
        for (int a = 0; a < 3; a++) p[a] = p[a] + (float)((n[a] >> half) & 1) * cs;
        size = cs;
    }
}

// Whether the density at p is negative: the terrain's octaves only until the
// sign is certain (decide_label), every other sampler in full.
__device__ __forceinline__ bool corner_air(const SamplerDev& S, const float (&p)[3]) {
    if (S.kind != BMF_SAMPLER_TERRAIN) return sample_density(S, p[0], p[1], p[2]) < 0.0f;
    const TerrainTerms T{S.amp, S.y0, S.inv_norm};
    const float t2 = p[1] - T.y0;
    float sum = 0.0f;
    for (int k = 0; k < S.octaves; k++) {
        const int d = decide_label(T, S.reach[k], sum, t2);
        if (d) return d == 1;
        const float f = S.fo[k];
        sum = __builtin_fmaf(S.ao[k], snoise3(p[0] * f, p[1] * f, p[2] * f, S.seed + (uint32_t)k), sum);
    }
    return density_from_sum(T, sum, t2) < 0.0f;
}

__device__ __forceinline__ int tri_count(int mask) {
    return (mask == 0 || mask == 255) ? 0 : (int)(c_tri_table[mask] >> 60) / 3;
}

// Leaf list entries that one tile of candidates can touch: a chunk has at
// least 26 boundary points (dim 2).
constexpr int kTileLeaves = (kStitchThreads - 1) / 26 + 2;

// Triangles of the tile's candidates.  A thread per candidate finds the
// chunks of its 8 octants (most lie in the candidate's own chunk or in the one
// last found, so that a face point descends once); the candidates this chunk
// stitches, about half, are compacted, and 8 lanes each take their corners'
// signs.  Bound by the samplers' instructions within the terrain band and by
// the descents' load latency next to it; candidates off the band descend not
// at all.  288 chunks of 32^3 unit nodes, 1.77 M candidates, 5-octave terrain:
// 96 us (8 descents and 8 full samplers in each candidate's lane: about 620).
template <typename I>
__device__ __forceinline__ void count_tile(const World& W, int L, int root, const SamplerDev& S,
                                           const int32_t* __restrict__ leaves, uint32_t per_leaf, int64_t cand0,
                                           int ncand, LeafBox<I>* s_leaf, int (*s_oc)[8], uint16_t* s_list, int* s_n,
                                           uint8_t* s_cnt) {
    const int tid = threadIdx.x, lane = lane_id();
    const int64_t l0 = cand0 / per_leaf;
    const uint32_t t0 = (uint32_t)(cand0 - l0 * per_leaf);
    const Box<I> rb = node_box<I>(W, L, root);
    if (tid < kTileLeaves && (int64_t)tid * per_leaf < (int64_t)t0 + ncand)
        s_leaf[tid] = leaf_box<I>(W, L, rb, leaves[l0 + tid]);
    if (tid == 0) *s_n = 0;
    s_cnt[tid] = 0;
    __syncthreads();
    bool take = tid < ncand;
    int oc[8];
    I P2[3];
    if (take) {
        const uint32_t g = t0 + (uint32_t)tid, q = g / per_leaf;
        const LeafBox<I> lf = s_leaf[q];
        take = lf.b.id >= 0;
        if (take) {
            candidate_point<I>(W, lf.b, g - q * per_leaf, P2);
            // a corner lies within one unit node (of the coarsest chunk) of
            // its point, here with as much again for rounding: off the
            // sampler's band all corners have one sign
            const bmf_world_node& lq = W.nodes[lf.b.id];
            const float part = (float)((P2[1] >> 1) - lf.b.o[1]) / (float)lf.b.e;
            const float y = lq.pos[1] + part * lq.size;
            const float reach = 2.0f * *W.max_size / (float)W.dim + 1e-5f * (fabsf(lq.pos[1]) + lq.size);
            take = band_sign(S, y - reach, y + reach) == 0;
        }
        if (take) {
            Box<I> last = lf.b;
            if (!lf.own) last.id = -1;
            bool same = true;
            int owner = -1;
            I owner_e = 0;
#pragma unroll
            for (int c = 0; c < 8; c++) {
                I p2[3];
                octant_point<I>(P2, c, p2);
                Box<I> b = last;
                if (lf.own && inside(lf.b, p2)) b = lf.b;
                else if (last.id < 0 || !inside(last, p2)) b = last = locate<I>(W, L, rb, p2);
                oc[c] = b.id;
                if (b.id < 0) {
                    take = false;
                    break;
                }
                same = same && b.id == oc[0];
                if (owner < 0 || b.e < owner_e || (b.e == owner_e && b.id < owner)) {
                    owner = b.id;
                    owner_e = b.e;
                }
            }
            take = take && !same && owner == lf.b.id;
        }
    }
    const uint64_t bal = __ballot(take);
    int base = 0;
    if (lane == 0 && bal) base = atomicAdd(s_n, __popcll(bal));
    base = __shfl(base, 0);
    if (take) {
        const int r = base + (int)__popcll(bal & lanemask_lt());
        s_list[r] = (uint16_t)tid;
#pragma unroll
        for (int c = 0; c < 8; c++) s_oc[r][c] = oc[c];
    }
    __syncthreads();
    const int ns = *s_n;
    for (int r0 = 0; r0 < ns; r0 += kStitchThreads / 8) {
        const int r = r0 + tid / 8, c = tid & 7;
        bool air = false;
        int src = 0;
        if (r < ns) {
            src = s_list[r];
            const uint32_t g = t0 + (uint32_t)src, q = g / per_leaf;
            I Q2[3];
            candidate_point<I>(W, s_leaf[q].b, g - q * per_leaf, Q2);
            float p[3];
            corner_position<I>(W, L, node_box<I>(W, L, s_oc[r][c]), Q2, c, p);
            air = corner_air(S, p);
        }
        const int mask = (int)((__ballot(air) >> (lane & 56)) & 255u);
        if (r < ns && c == 0) s_cnt[src] = (uint8_t)tri_count(mask);
    }
    __syncthreads();
}

__global__ void __launch_bounds__(kStitchThreads) k_stitch_count(World W, const SamplerDev* __restrict__ S,
                                                                 const int32_t* __restrict__ leaves, uint32_t per_leaf,
                                                                 int64_t n_cand, uint8_t* __restrict__ counts,
                                                                 int64_t* __restrict__ tile_tot) {
    __shared__ int s_oc[kStitchThreads][8];
    __shared__ LeafBox<int64_t> s_leaf[kTileLeaves];
    __shared__ uint16_t s_list[kStitchThreads];
    __shared__ uint8_t s_cnt[kStitchThreads];
    __shared__ int s_n;
    __shared__ int s_w[kStitchThreads / 64];
    load_gradients();
    const int root = uniform_int(W.root_level[0]), L = uniform_int(W.root_level[1]);
    const int64_t cand0 = (int64_t)blockIdx.x * kStitchThreads;
    const int ncand = (int)(n_cand - cand0 < kStitchThreads ? n_cand - cand0 : kStitchThreads);
    int n = 0;
    if (root >= 0 && L <= kMaxLevel) {
        if (L + W.log_dim <= kNarrowBits)
            count_tile<int32_t>(W, L, root, *S, leaves, per_leaf, cand0, ncand,
                                reinterpret_cast<LeafBox<int32_t>*>(s_leaf), s_oc, s_list, &s_n, s_cnt);
        else
            count_tile<int64_t>(W, L, root, *S, leaves, per_leaf, cand0, ncand, s_leaf, s_oc, s_list, &s_n, s_cnt);
        n = s_cnt[threadIdx.x];
    }
    if ((int)threadIdx.x < ncand) counts[cand0 + threadIdx.x] = (uint8_t)n;
    int x = n;
    for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off);
    if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t t = 0;
        for (int w = 0; w < kStitchThreads / 64; w++) t += s_w[w];
        tile_tot[blockIdx.x] = t;
    }
}

// Exclusive scan of the tile totals in place; out_total[0] = the sum.
__global__ void __launch_bounds__(kScanThreads) k_stitch_scan(int64_t* __restrict__ tile, int64_t n_tiles,
                                                              int64_t* __restrict__ out_total,
                                                              int64_t* __restrict__ host_total) {
    __shared__ int64_t s_w[1][kScanThreads / 64 + 1];
    const int t = threadIdx.x;
    const int64_t seg = (n_tiles + kScanThreads - 1) / kScanThreads;
    const int64_t a0 = std::min<int64_t>(n_tiles, t * seg), a1 = std::min<int64_t>(n_tiles, a0 + seg);
    int64_t sum[1] = {0}, excl[1], tot[1];
#pragma unroll 8
    for (int64_t i = a0; i < a1; i++) sum[0] += tile[i];
    block_scan<1, kScanThreads>(sum, excl, tot, s_w);
    int64_t run = excl[0];
    for (int64_t i = a0; i < a1; i++) {
        const int64_t v = tile[i];
        tile[i] = run;
        run += v;
    }
    if (t == 0) out_total[0] = host_total[0] = tot[0];
}

// Triangles: a block takes kEmitTiles tiles, compacts their candidates with
// triangles (a few in a hundred) and gives each 8 lanes: a corner's chunk,
// position and density per lane, then the crossings, then the vertices.
// Bound by the chain of a round (descent, octaves, two exchanges), so a block
// has few rounds: 30 us with 2 tiles for the world above, 45 with 8.
constexpr int kEmitTiles = 2;
constexpr int kEmitCands = kEmitTiles * kStitchThreads;
constexpr int kEmitRound = kStitchThreads / 8;  // candidates per round

template <typename I>
__device__ __forceinline__ void emit_corner(const World& W, int L, int root, const SamplerDev& S,
                                            const int32_t* __restrict__ leaves, uint32_t per_leaf, int64_t cand, int c,
                                            float4& out) {
    const int64_t li = cand / per_leaf;
    I P2[3], p2[3];
    candidate_point<I>(W, node_box<I>(W, L, leaves[li]), (uint32_t)(cand - li * per_leaf), P2);
    octant_point<I>(P2, c, p2);
    const Box<I> b = locate<I>(W, L, node_box<I>(W, L, root), p2);
    if (b.id < 0) return;  // not for a counted candidate
    float p[3];
    corner_position<I>(W, L, b, P2, c, p);
    out = make_float4(p[0], p[1], p[2], sample_density(S, p[0], p[1], p[2]));
}

__global__ void __launch_bounds__(kStitchThreads) k_stitch_emit(World W, const SamplerDev* __restrict__ S,
                                                                const int32_t* __restrict__ leaves, uint32_t per_leaf,
                                                                int64_t n_cand, const uint8_t* __restrict__ counts,
                                                                const int64_t* __restrict__ tile_off,
                                                                const int64_t* __restrict__ total,
                                                                float* __restrict__ out, int64_t cap) {
    __shared__ uint32_t s_list[kEmitCands];  // candidate within the block | its first triangle's offset << 11
    __shared__ uint32_t s_wt[kStitchThreads / 64], s_wn[kStitchThreads / 64];
    __shared__ float4 s_corner[kEmitRound][8];
    __shared__ float s_cross[kEmitRound][12][3];
    static_assert(kEmitCands <= 1 << 11, "list entry layout");
    constexpr int kPer = kEmitCands / kStitchThreads;  // consecutive candidates per thread
    load_gradients();
    if (total[0] > cap) return;  // reported by the host: nothing is written
    const int root = uniform_int(W.root_level[0]), L = uniform_int(W.root_level[1]);
    const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
    const int64_t cand0 = (int64_t)blockIdx.x * kEmitCands;
    // the counts are padded to whole blocks
    uint8_t cn[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) cn[k] = counts[cand0 + kPer * tid + k];
    uint32_t nt = 0, nn = 0;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const uint32_t v = cand0 + kPer * tid + k < n_cand ? cn[k] : 0u;
        nt += v;
        nn += v != 0u;
    }
    uint32_t it = nt, in = nn;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t a = __shfl_up(it, off), b = __shfl_up(in, off);
        if (lane >= off) {
            it += a;
            in += b;
        }
    }
    if (lane == 63) {
        s_wt[wave] = it;
        s_wn[wave] = in;
    }
    __syncthreads();
    uint32_t ot = it - nt, on = in - nn, ns = 0;
    for (int w = 0; w < kStitchThreads / 64; w++) {
        if (w < wave) {
            ot += s_wt[w];
            on += s_wn[w];
        }
        ns += s_wn[w];
    }
    if (ns == 0) return;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const uint32_t v = cand0 + kPer * tid + k < n_cand ? cn[k] : 0u;
        if (v) {
            s_list[on++] = (uint32_t)(kPer * tid + k) | (ot << 11);
            ot += v;
        }
    }
    float* __restrict__ O = out + 9 * tile_off[(int64_t)blockIdx.x * kEmitTiles];
    const bool narrow = L + W.log_dim <= kNarrowBits;
    for (uint32_t r0 = 0; r0 < ns; r0 += kEmitRound) {
        __syncthreads();  // the list is written; the previous round is done with the corners
        const int q = tid / 8, c = tid & 7;
        const uint32_t r = r0 + (uint32_t)q;
        const uint32_t item = r < ns ? s_list[r] : 0u;
        if (r < ns) {
            float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const int64_t cand = cand0 + (item & 2047u);
            if (narrow) emit_corner<int32_t>(W, L, root, *S, leaves, per_leaf, cand, c, v);
            else emit_corner<int64_t>(W, L, root, *S, leaves, per_leaf, cand, c, v);
            s_corner[q][c] = v;
        }
        __syncthreads();
        int mask = 0;
        if (r < ns) {
#pragma unroll
            for (int k = 0; k < 8; k++) mask |= (s_corner[q][k].w < 0.0f) << k;
            for (int e = c; e < 12; e += 8) {
                const int a = c_edge[e][0], b = c_edge[e][1];
                if (((mask >> a) & 1) == ((mask >> b) & 1)) continue;
                const float4 A = s_corner[q][a], B = s_corner[q][b];
                const float mu = (0.0f - A.w) / (B.w - A.w);
                const float dx = (B.x - A.x) * mu, dy = (B.y - A.y) * mu, dz = (B.z - A.z) * mu;
                s_cross[q][e][0] = dx + A.x;
                s_cross[q][e][1] = dy + A.y;
                s_cross[q][e][2] = dz + A.z;
            }
        }
        __syncthreads();
        if (r < ns) {
            const uint64_t row = c_tri_table[mask];
            const int nv = 3 * tri_count(mask);
            float* __restrict__ T = O + 9 * (int64_t)(item >> 11);
            for (int v = c; v < nv; v += 8) {
                const int e = (int)((row >> (4 * v)) & 15);
                T[3 * v] = s_cross[q][e][0];
                T[3 * v + 1] = s_cross[q][e][1];
                T[3 * v + 2] = s_cross[q][e][2];
            }
        }
    }
}

__global__ void k_stitch_world(const bmf_world_node* __restrict__ nodes, int n_nodes, int* __restrict__ out,
                               float* __restrict__ max_size, int* __restrict__ host) {
    // out[0]: the first node without a parent, out[1]: the deepest level; both for the host too
    __shared__ int s_root, s_level, s_size;
    if (threadIdx.x == 0) {
        s_root = 0x7FFFFFFF;
        s_level = 0;
        s_size = 0;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n_nodes; i += blockDim.x) {
        if (nodes[i].parent < 0) atomicMin(&s_root, i);
        atomicMax(&s_level, nodes[i].level);
        // sizes are positive: their bits order as they do
        if (nodes[i].world_leaf && nodes[i].size > 0.0f) atomicMax(&s_size, __float_as_int(nodes[i].size));
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        out[0] = s_root == 0x7FFFFFFF ? -1 : s_root;
        out[1] = s_level;
        host[0] = out[0];
        host[1] = out[1];
        *max_size = __int_as_float(s_size);
    }
}

}  // namespace
}  // namespace bmf

using namespace bmf;

extern "C" {

int bmf_stitch(bmf_ctx* c, const bmf_world_node* nodes, int32_t n_nodes, const int32_t* leaves, int32_t n_leaves,
               const bmf_stitch_params* params, float* triangles, int64_t cap_triangles, int64_t* n_triangles) {
    if (!c || !params || n_nodes < 0 || n_leaves < 0 || cap_triangles < 0) return BMF_EINVAL;
    if ((n_nodes > 0 && !nodes) || (n_leaves > 0 && !leaves) || (cap_triangles > 0 && !triangles)) return BMF_EINVAL;
    const int dim = params->chunk_resolution;
    if (dim < 2 || dim > BMF_MAX_DIM || (dim & (dim - 1))) return BMF_EINVAL;
    if (!c->sampler_set) return BMF_ESTATE;
    if (c->h_sampler.kind == BMF_SAMPLER_EXTERNAL) return BMF_EINVAL;
    BMF_HIP(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    const int64_t per_leaf = 2ll * (dim + 1) * (dim + 1) + 4ll * dim * (dim - 1);
    const int64_t n_cand = per_leaf * n_leaves;
    const int64_t n_tiles = (n_cand + kStitchThreads - 1) / kStitchThreads;
    if (n_tiles > 0x7FFFFFFF) return BMF_EINVAL;
    // whole blocks of the emit kernel
    const int64_t n_room = (n_cand + kEmitCands - 1) / kEmitCands * kEmitCands;
    if (n_cand > c->stitch_cap_cand) {
        if (c->d_stitch_counts) (void)hipFree(c->d_stitch_counts);
        if (c->d_stitch_tiles) (void)hipFree(c->d_stitch_tiles);
        c->d_stitch_counts = nullptr;
        c->d_stitch_tiles = nullptr;
        c->stitch_cap_cand = 0;
        BMF_HIP(hipMalloc((void**)&c->d_stitch_counts, (size_t)std::max<int64_t>(n_room, 1)));
        BMF_HIP(hipMalloc((void**)&c->d_stitch_tiles, sizeof(int64_t) * (size_t)std::max<int64_t>(n_tiles, 1)));
        c->stitch_cap_cand = n_cand;
    }
    if (!c->d_stitch_misc) BMF_HIP(hipMalloc((void**)&c->d_stitch_misc, sizeof(int64_t) * 3));
    if (!c->h_stitch_total) BMF_HIP(host_alloc(&c->h_stitch_total, 2, &c->m_stitch_total));
    // the world's root and deepest level, and the triangle total: the kernels
    // read the first two on the device, the host all three at the end
    int* dw = reinterpret_cast<int*>(c->d_stitch_misc);
    int64_t* total = c->d_stitch_misc + 1;
    float* max_size = reinterpret_cast<float*>(c->d_stitch_misc + 2);
    hipLaunchKernelGGL(k_stitch_world, dim3(1), dim3(1024), 0, s, nodes, n_nodes, dw, max_size,
                       reinterpret_cast<int*>(c->m_stitch_total));
    if (n_cand > 0) {
        int log_dim = 0;
        while ((1 << log_dim) < dim) log_dim++;
        const World W{nodes, n_nodes, dim, log_dim, dw, max_size};
        hipLaunchKernelGGL(k_stitch_count, dim3((unsigned)n_tiles), dim3(kStitchThreads), 0, s, W, c->A.sampler, leaves,
                           (uint32_t)per_leaf, n_cand, c->d_stitch_counts, c->d_stitch_tiles);
        hipLaunchKernelGGL(k_stitch_scan, dim3(1), dim3(kScanThreads), 0, s, c->d_stitch_tiles, n_tiles, total,
                           c->m_stitch_total + 1);
        hipLaunchKernelGGL(k_stitch_emit, dim3((unsigned)(n_room / kEmitCands)), dim3(kStitchThreads), 0, s, W,
                           c->A.sampler, leaves, (uint32_t)per_leaf, n_cand, c->d_stitch_counts, c->d_stitch_tiles,
                           total, triangles, cap_triangles);
    }
    BMF_HIP(hipGetLastError());
    BMF_HIP(hipStreamSynchronize(s));
    int hw[2];
    std::memcpy(hw, c->h_stitch_total, sizeof(hw));
    const int64_t nt = n_cand > 0 && hw[0] >= 0 ? c->h_stitch_total[1] : 0;
    if (n_cand > 0 && hw[0] >= 0 && hw[1] > kMaxLevel) return BMF_EINVAL;  // integer coordinates must fit
    if (n_triangles) *n_triangles = nt;
    return nt > cap_triangles ? BMF_ECAPACITY : BMF_OK;
}

}  // extern "C"
