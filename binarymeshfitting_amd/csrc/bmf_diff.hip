// Differentiable extraction of one chunk (C ABI in include/bmf.h):
//   forward   the extraction kernels with every octave evaluated, then the
//             smoothing on the tape's own copy of the mesh, keeping the
//             positions every `checkpoint_every` iterations;
//   loss      mean squared distance to the nearest of a set of targets
//             (exact nearest neighbour: an implicit binary box hierarchy
//             over Morton-sorted targets, traversed nearest child first);
//   backward  the transpose of the K smoothing steps (linear in the
//             positions for the frozen topology) and of vertex placement
//             mu = (0 - s0) / (s1 - s0) (DMCChunk.cpp:657-674), gathered per
//             density sample in a fixed order (deterministic, no atomics).
//
// Tape layout in HBM (one chunk, V vertices, T triangles):
//   dens  FP32 [dim^3]      the densities of the forward
//   vid0  u32 [dim^3]       first vertex id owned by each sample (valid
//                           where the sample owns a sign-changing edge)
//   vedge u32 [V], boundary u8 [V], idx u32 [3T]   copies of the mesh
//   ring  u32x2 [kMaxRing][V] ring of each vertex: its triangles in
//                           ascending id (the adjacency of
//                           MeshProcessor::set_adj, MeshProcessor.cpp:98-128),
//                           each as its two other corners and the vertex's
//                           place among the three; slot-major so that a
//                           wave's loads of one slot are contiguous
//   deg u8 [V], mv u8 [V]   ring size; whether the primal step moves the
//                           vertex (MeshProcessor.cpp:247)
//   bscale f32 [V]          1 / (3 |ring|) for moved vertices, else 1 (the
//                           scale of the backward's gradient records)
//   p4, q4 float4 [V]       working positions (ping-pong); ckpt float4 [slots][V]
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <new>

#include "../../include/bmf.h"
#include "bmf_context.h"
#include "bmf_device_tables.h"
#include "bmf_internal.h"
#include "bmf_rows.h"

using namespace bmf;

namespace {

constexpr int kThreads = 256;
constexpr int kStepThreads = 64;  // smoothing steps: one wave per workgroup spreads a small mesh over more CUs
// A vertex's lattice edge borders 4 cells and one cell's triangulation uses
// one edge in at most 5 table slots (MCTable.h:27-283), so a ring holds at
// most 20 triangles.
constexpr int kMaxRing = 20;
// Vertex ids share a word with a corner place (2 bits) in the ring records.
constexpr uint32_t kVidMask = 0x3FFFFFFFu;
constexpr int64_t kMaxTapeVertices = int64_t(1) << 30;
constexpr int kLeaf = 64;      // targets per leaf box of the nearest-target hierarchy
constexpr int kNNFan = 6;      // a wave tests 2^kNNFan = 64 boxes of one subtree level at once
constexpr int kNNFrames = 4;   // inner frames of the walk: ceil(25 / kNNFan) levels less the leaves, n < 2^31

#define BMF_HIP(call)                          \
    do {                                       \
        hipError_t e_ = (call);                \
        if (e_ != hipSuccess) return BMF_EHIP; \
    } while (0)

template <class T>
hipError_t dalloc(T** p, int64_t count) {
    return hipMalloc((void**)p, (size_t)std::max<int64_t>(count, 1) * sizeof(T));
}

template <class T>
void dfree(T*& p) {
    if (p) (void)hipFree(p);
    p = nullptr;
}

unsigned blocks_for(int64_t n) { return (unsigned)std::max<int64_t>(1, (n + kThreads - 1) / kThreads); }
unsigned step_blocks(int64_t n) { return (unsigned)std::max<int64_t>(1, (n + kStepThreads - 1) / kStepThreads); }

// ------------------------------------------------------------------------
// forward
// ------------------------------------------------------------------------
// Vertices are ordered by lattice cells of 4^3 samples (8^3 in chunks of more
// than 132), so that consecutive ones are near each other in every direction:
// vertex ids follow the rows of the chunk, and a row meets a surface in few
// and far places.  A counting order: rank within the cell (k_tape_take), the
// cells' places in any sequence (k_order_cells), the order (k_order).
constexpr int kOrderCells = 33 * 33 * 33;
constexpr int kPacket = 4;  // vertices that k_nn_query takes together
__device__ __forceinline__ uint32_t order_cell(uint32_t code, int dim) {
    const uint32_t s = dim <= 132 ? 2u : 3u, nb = ((uint32_t)dim + (1u << s) - 1u) >> s;
    const uint32_t x = (code & 255u) >> s, y = ((code >> 8) & 255u) >> s, z = ((code >> 16) & 255u) >> s;
    return min((x * nb + y) * nb + z, (uint32_t)kOrderCells - 1u);
}

// The first place of each cell that holds vertices (one atomic per wave), its
// count cleared for the next forward.  A cell takes whole packets, its spare
// places -1: packets across two cells would hold vertices that are far apart
// (a quarter more leaves searched per packet).
__global__ void __launch_bounds__(kThreads) k_order_cells(uint32_t* __restrict__ cell_n, uint32_t* __restrict__ base,
                                                          int* __restrict__ places, int32_t* __restrict__ order) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t n = i < kOrderCells ? cell_n[i] : 0u, room = (n + kPacket - 1) / kPacket * kPacket;
    const uint32_t inc = wave_scan(room);
    uint32_t at = 0;
    if (lane_id() == 63 && inc) at = (uint32_t)atomicAdd(places, (int)inc);
    at = (uint32_t)__builtin_amdgcn_readlane((int)at, 63) + inc - room;
    if (!n) return;
    base[i] = at;
    cell_n[i] = 0u;
    for (uint32_t k = n; k < room; k++) order[at + k] = -1;
}
__global__ void __launch_bounds__(kThreads) k_order(const uint32_t* __restrict__ vedge, int V, int dim,
                                                    const uint32_t* __restrict__ base,
                                                    const uint32_t* __restrict__ rank, const int* __restrict__ taken,
                                                    int* __restrict__ host_places, int32_t* __restrict__ order) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v == 0) *host_places = *taken;
    if (v < V) order[base[order_cell(vedge[v], dim)] + rank[v]] = v;
}

// Takes the chunk's extraction into the tape in one launch: densities, edge
// codes, boundary flags and triangles copied out of the context's arenas,
// the positions as float4 (working copy and checkpoint 0, and as float3
// when no smoothing follows), each sample's first vertex id (vertices
// are numbered in sample order, x-, y-, z-edge within a sample), and each
// vertex's rank among those of its order cell (k_nn_query's packets).
__global__ void k_tape_take(const float* __restrict__ dens_in, const uint32_t* __restrict__ vedge_in,
                            const uint8_t* __restrict__ bnd_in, const uint32_t* __restrict__ idx_in,
                            const float* __restrict__ pos_in, int64_t n3, int V, int64_t n_idx, int dim,
                            float* __restrict__ dens, uint32_t* __restrict__ vedge, uint8_t* __restrict__ bnd,
                            uint32_t* __restrict__ idx, float4* __restrict__ p4, float4* __restrict__ ck0,
                            float* __restrict__ pos3, uint32_t* __restrict__ vid0, uint32_t* __restrict__ cell_n,
                            uint32_t* __restrict__ rank, int* __restrict__ taken, int* __restrict__ err) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *taken = *err = 0;
    const int64_t total = std::max<int64_t>(n3, std::max<int64_t>(n_idx, V));
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        if (i < n3) dens[i] = dens_in[i];
        if (i < n_idx) idx[i] = idx_in[i];
        if (i < V) {
            const uint32_t code = vedge_in[i];
            vedge[i] = code;
            bnd[i] = bnd_in[i];
            rank[i] = atomicAdd(&cell_n[order_cell(code, dim)], 1u);
            const float x = pos_in[3 * i], y = pos_in[3 * i + 1], z = pos_in[3 * i + 2];
            p4[i] = make_float4(x, y, z, 0.0f);
            ck0[i] = make_float4(x, y, z, 0.0f);
            if (pos3) {
                pos3[3 * i] = x;
                pos3[3 * i + 1] = y;
                pos3[3 * i + 2] = z;
            }
            const uint32_t smp = code & 0xFFFFFFu;
            if (i == 0 || (vedge_in[i - 1] & 0xFFFFFFu) != smp) {
                const int sx = (int)(smp & 255u), sy = (int)((smp >> 8) & 255u), sz = (int)(smp >> 16);
                vid0[((int64_t)sx * dim + sy) * dim + sz] = (uint32_t)i;
            }
        }
    }
}

// Ring of each vertex from the per-cell triangle bases and masks written by
// the emit kernel: the 4 cells around its edge in lexicographic order and,
// in each, the triangles that use the edge in slot order.  Each triangle
// is stored as its other two corners in corner order, the first with the
// vertex's own place (0, 1, 2) in bits 30-31.  Also the vertex's backward
// scale: 1 / (3 |ring|) if the primal step moves it, else 1.  Bound by its
// chain of gathers (edge code, cells, triangles): the four cells load
// together, then the corners of kAdjRound triangles (44,392 vertices: 8 us;
// a cell and a triangle at a time 21).
constexpr int kAdjRound = 4;
__global__ void __launch_bounds__(kStepThreads) k_tape_adj(
    const uint32_t* __restrict__ vedge, const uint8_t* __restrict__ boundary, const uint32_t* __restrict__ cell_tb,
    const uint8_t* __restrict__ cell_mask, const uint32_t* __restrict__ idx, int dim, int V, int T, int bp,
    int stride, uint2* __restrict__ ring, uint8_t* __restrict__ deg, uint8_t* __restrict__ mv,
    float* __restrict__ bscale, int* __restrict__ err) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const uint32_t code = vedge[v];
    const uint8_t bnd = boundary[v];
    const int ex = (int)(code & 255u), ey = (int)((code >> 8) & 255u), ez = (int)((code >> 16) & 255u);
    const int ax = (int)(code >> 24);
    uint32_t tb[4], tm[4];
    bool in[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {  // the rows of c_ring
        const int u = (c >> 1) - 1, w = (c & 1) - 1;
        const int cx = ex + (ax == 0 ? 0 : u), cy = ey + (ax == 0 ? u : (ax == 1 ? 0 : w)), cz = ez + (ax == 2 ? 0 : w);
        in[c] = cx >= 0 && cy >= 0 && cz >= 0 && cx <= dim - 2 && cy <= dim - 2 && cz <= dim - 2;
        const int64_t ci = in[c] ? ((int64_t)cx * dim + cy) * dim + cz : 0;
        tb[c] = cell_tb[ci];
        tm[c] = cell_mask[ci];
    }
    // the ring's triangles as bits 5 c + triangle of the cell
    uint32_t bits = 0;
#pragma unroll
    for (int c = 0; c < 4; c++) bits |= (in[c] ? (uint32_t)c_edge_tris.m[tm[c]][4 * ax + 3 - c] : 0u) << (5 * c);
    const int count = __popc(bits);
    int n = 0;
    while (bits) {
        uint32_t t[kAdjRound], a[kAdjRound], b[kAdjRound], d[kAdjRound];
        bool ok[kAdjRound];
#pragma unroll
        for (int k = 0; k < kAdjRound; k++) {
            ok[k] = bits != 0u;
            const uint32_t q = ok[k] ? (uint32_t)(__ffs(bits) - 1) : 0u;
            const uint32_t f = q < 5u ? tb[0] : (q < 10u ? tb[1] - 5u : (q < 15u ? tb[2] - 10u : tb[3] - 15u));
            t[k] = f + q;
            bits &= bits - 1u;
            if (ok[k] && t[k] >= (uint32_t)T) {  // counts and ids disagree
                *err = 1;
                ok[k] = false;
            }
            if (!ok[k]) t[k] = 0u;
        }
#pragma unroll
        for (int k = 0; k < kAdjRound; k++) {
            a[k] = idx[3 * t[k]];
            b[k] = idx[3 * t[k] + 1];
            d[k] = idx[3 * t[k] + 2];
        }
#pragma unroll
        for (int k = 0; k < kAdjRound; k++) {
            if (!ok[k]) continue;
            const uint32_t place = a[k] == (uint32_t)v ? 0u : (b[k] == (uint32_t)v ? 1u : 2u);
            if (place == 2u && d[k] != (uint32_t)v) *err = 1;
            const uint32_t o1 = place == 0u ? b[k] : a[k], o2 = place == 2u ? b[k] : d[k];
            ring[(int64_t)n * stride + v] = make_uint2(o1 | (place << 30), o2);
            n++;
        }
    }
    if (n != count) *err = 1;
    const bool moved = (bp || !bnd) && n > 0;
    deg[v] = (uint8_t)n;
    mv[v] = (uint8_t)moved;
    bscale[v] = moved ? 1.0f / (3.0f * (float)n) : 1.0f;
}

// x / 3 rounded to nearest in three FP32 operations: q0 = x RN(1/3), the
// exact remainder r = x - 3 q0 (one fma), then q0 + r RN(1/3) (one fma) --
// the correction step of Markstein's division (IA-64 and Elementary
// Functions, 2000, ch. 8); zeros and infinities take q0.  Equal to the IEEE
// quotient for every float (tests/test_exact_division.py runs the same
// operations on the host over all 2^32 of them).
__device__ __forceinline__ float div3(float x) {
    const float third = 1.0f / 3.0f;
    const float q0 = x * third;
    const float q = __builtin_fmaf(__builtin_fmaf(-q0, 3.0f, x), third, q0);
    // v_cmp_class mask: -inf (bit 2), -0 (5), +0 (6), +inf (9)
    return __builtin_amdgcn_classf(x, (1 << 2) | (1 << 5) | (1 << 6) | (1 << 9)) ? q0 : q;
}

// The new position of one moved vertex: its ring's centroids summed from +0
// in ascending triangle order, divided by the ring size.
__device__ __forceinline__ float4 smooth_vertex(const uint2* __restrict__ ring, int stride, int n,
                                               const float4* __restrict__ in, float4 pv, int v) {
    float sx = 0.0f, sy = 0.0f, sz = 0.0f;
#pragma unroll 4
    for (int k = 0; k < n; k++) {
        const uint2 e = ring[(int64_t)k * stride + v];
        const uint32_t place = e.x >> 30;
        const float4 a = in[e.x & kVidMask], b = in[e.y];
        const float4 c0 = place == 0u ? pv : a;
        const float4 c1 = place == 0u ? a : (place == 1u ? pv : b);
        const float4 c2 = place == 2u ? pv : b;
        float cx = 0.0f, cy = 0.0f, cz = 0.0f;
        cx = cx + c0.x;
        cy = cy + c0.y;
        cz = cz + c0.z;
        cx = cx + c1.x;
        cy = cy + c1.y;
        cz = cz + c1.z;
        cx = cx + c2.x;
        cy = cy + c2.y;
        cz = cz + c2.z;
        sx = sx + div3(cx);
        sy = sy + div3(cy);
        sz = sz + div3(cz);
    }
    const float fc = (float)n;
    return make_float4(sx / fc, sy / fc, sz / fc, 0.0f);
}

// One smoothing iteration (MeshProcessor.cpp:130-306) in one launch: the new
// position of a moved vertex is its ring's centroids summed from +0 in
// ascending triangle order and divided by the ring size, each centroid
// ((0 + p0) + p1) + p2, / 3 recomputed from the corners by every vertex of
// the triangle (the same FP32 value each time, so no separate dual pass);
// other vertices keep theirs.  Reads `in`, writes `out` (ping-pong buffers)
// and, when given, a checkpoint copy `ck` and float3 positions `pos3`.
__global__ void __launch_bounds__(kStepThreads) k_tape_step(const uint2* __restrict__ ring, int stride,
                                                            const uint8_t* __restrict__ deg,
                                                            const uint8_t* __restrict__ mv,
                                                            const float4* __restrict__ in, int V,
                                                            float4* __restrict__ out, float4* __restrict__ ck,
                                                            float* __restrict__ pos3) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const float4 pv = in[v];
    float4 r = pv;
    if (mv[v]) r = smooth_vertex(ring, stride, deg[v], in, pv, v);
    out[v] = r;
    if (ck) ck[v] = r;
    if (pos3) {
        pos3[3 * v] = r.x;
        pos3[3 * v + 1] = r.y;
        pos3[3 * v + 2] = r.z;
    }
}

__global__ void k_tape_out(const float4* __restrict__ p4, int V, float* __restrict__ pos) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const float4 q = p4[v];
    pos[3 * v] = q.x;
    pos[3 * v + 1] = q.y;
    pos[3 * v + 2] = q.z;
}

// ------------------------------------------------------------------------
// backward
// ------------------------------------------------------------------------
// The backward's working record of vertex v: .w = [v moved] and .xyz =
// dL/dp_v scaled by bscale_v = 1 / (3 |ring(v)|) for moved vertices, so that
// a row of the transposed step needs nothing of its neighbours but their
// records.  With no smoothing (`scaled` = 0) the record is dL/dp_v itself.
__global__ void k_bwd_init(const float* __restrict__ g3, int V, const uint8_t* __restrict__ mv,
                           const float* __restrict__ bscale, int scaled, float4* __restrict__ g) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const float sc = scaled ? bscale[v] : 1.0f;
    g[v] = make_float4(g3[3 * v] * sc, g3[3 * v + 1] * sc, g3[3 * v + 2] * sc, scaled ? (float)mv[v] : 0.0f);
}

// A round of ring records and the other corners' data.  A transposed step is
// bound by latency (a mesh of 44,392 vertices is 0.7 waves per SIMD), so a
// round's records load beside the vertex's own data, before its ring size is
// known (slots past it hold anything and are not used), and their corners
// together: two round trips, where a loop over the ring takes two for every four
// records and the remainder one by one (4.6 us, this 4.0; the smoothing step,
// whose arithmetic is four times that, gains nothing by it).
constexpr int kStepRound = 8;
struct RingRound {
    uint2 e[kStepRound];
    __device__ __forceinline__ void load(const uint2* __restrict__ ring, int stride, int k0, int v) {
#pragma unroll
        for (int k = 0; k < kStepRound; k++) e[k] = ring[(int64_t)(k0 + k < kMaxRing ? k0 + k : k0) * stride + v];
    }
    // the two other corners of each of the records before the n-th, v's own
    // value for the others
    __device__ __forceinline__ void corners(const float4* __restrict__ in, int left, int v, float4 (&a)[kStepRound],
                                            float4 (&b)[kStepRound]) const {
#pragma unroll
        for (int k = 0; k < kStepRound; k++) {
            a[k] = in[k < left ? e[k].x & kVidMask : (uint32_t)v];
            b[k] = in[k < left ? e[k].y : (uint32_t)v];
        }
        // all of them at once: left alone, loads move behind the selects that use them
#pragma unroll
        for (int k = 0; k < kStepRound; k++) {
            asm volatile("" : "+v"(a[k].x), "+v"(a[k].y), "+v"(a[k].z), "+v"(a[k].w));
            asm volatile("" : "+v"(b[k].x), "+v"(b[k].y), "+v"(b[k].z), "+v"(b[k].w));
        }
    }
};

// One transposed smoothing iteration.  The forward step is
// p'_u = [u not moved] p_u + [u moved] / (3 |ring(u)|) * (sum over the
// triangles of ring(u) of their corners), so
//   dL/dp_v = [v not moved] dL/dp'_v
//             + sum over the triangles t of ring(v), over the corners u of t,
//               of [u moved] dL/dp'_u / (3 |ring(u)|);
// with the records x_u = [u moved] dL/dp'_u / (3 |ring(u)|) (w = [u moved])
// that is m_self x_v plus, per ring triangle, its two other corners' records
// times their w (m_self = |ring(v)| for a moved v, whose own record is
// scaled; 1 otherwise).  Writes v's record for the step before, or dL/dp_v
// itself after the first iteration (`last`).
__global__ void __launch_bounds__(kStepThreads) k_bwd_step(const uint2* __restrict__ ring, int stride,
                                                           const uint8_t* __restrict__ deg,
                                                           const uint8_t* __restrict__ mv,
                                                           const float* __restrict__ bscale,
                                                           const float4* __restrict__ in, int V, int last,
                                                           float4* __restrict__ out) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    RingRound R;
    R.load(ring, stride, 0, v);
    const int n = deg[v];
    const bool moved = mv[v] != 0;
    const float4 own = in[v];
    const float scale = bscale[v];
    const float ms = moved ? (float)n : 1.0f;
    float sx = ms * own.x, sy = ms * own.y, sz = ms * own.z;
    for (int k0 = 0; k0 < n; k0 += kStepRound) {
        if (k0) R.load(ring, stride, k0, v);
        float4 a[kStepRound], b[kStepRound];
        R.corners(in, n - k0, v, a, b);
#pragma unroll
        for (int k = 0; k < kStepRound; k++) {
            const bool ok = k0 + k < n;
            const float tx = __builtin_fmaf(a[k].w, a[k].x, sx), ty = __builtin_fmaf(a[k].w, a[k].y, sy),
                        tz = __builtin_fmaf(a[k].w, a[k].z, sz);
            sx = ok ? __builtin_fmaf(b[k].w, b[k].x, tx) : sx;
            sy = ok ? __builtin_fmaf(b[k].w, b[k].y, ty) : sy;
            sz = ok ? __builtin_fmaf(b[k].w, b[k].z, tz) : sz;
        }
    }
    const float sc = last ? 1.0f : scale;
    out[v] = make_float4(sx * sc, sy * sc, sz * sc, moved ? 1.0f : 0.0f);
}

// dL/d(density) per sample: the sample is s0 of its own sign-changing edges
// (+x, +y, +z, vertex ids vid0[i] + 0, 1, ...) and s1 of the sign-changing
// edges of its -x, -y, -z neighbours.  mu = -s0 / (s1 - s0), so
// dmu/ds0 = -s1 / (s1 - s0)^2 and dmu/ds1 = s0 / (s1 - s0)^2; the vertex
// moves along its edge axis by mu (grid units).
// Nearly every sample has no such edge: its six neighbours are compared
// first.  Bound by VALU issue (129^3 samples: 13 us; with 32-bit divisions
// and both edge loops at every sample 17).
__global__ void __launch_bounds__(kThreads) k_bwd_place(const float* __restrict__ dens,
                                                        const uint32_t* __restrict__ vid0,
                                                        const float4* __restrict__ g, int dim,
                                                        float* __restrict__ out) {
    const uint32_t d1 = (uint32_t)dim, d2 = d1 * d1, n3 = d2 * d1;  // dim <= 256
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n3) return;
    const uint32_t x = udiv24(i, d2, 1.0f / (float)d2), r = i - x * d2;
    const uint32_t y = udiv24(r, d1, 1.0f / (float)d1), z = r - y * d1;
    const uint32_t st[3] = {d2, d1, 1u}, co[3] = {x, y, z};
    const float di = dens[i];
    const bool li = di < 0.0f;
    float up[3], dn[3];  // neighbours along each axis, the sample itself at a face
#pragma unroll
    for (int a = 0; a < 3; a++) {
        up[a] = dens[co[a] + 1 < d1 ? i + st[a] : i];
        dn[a] = dens[co[a] > 0 ? i - st[a] : i];
    }
    bool any = false;
#pragma unroll
    for (int a = 0; a < 3; a++) any = any || (up[a] < 0.0f) != li || (dn[a] < 0.0f) != li;
    float acc = 0.0f;
    if (any) {
        uint32_t k = 0;
#pragma unroll
        for (int a = 0; a < 3; a++) {  // own edges: this sample is s0
            const float dj = up[a];
            if ((dj < 0.0f) == li) continue;
            const float4 q = g[vid0[i] + k];
            k++;
            const float ds = dj - di;
            const float ga = a == 0 ? q.x : (a == 1 ? q.y : q.z);
            acc = acc + ga * (-dj / (ds * ds));
        }
#pragma unroll
        for (int a = 0; a < 3; a++) {  // edges of the -a neighbour: this sample is s1
            const float dj = dn[a];
            const bool lj = dj < 0.0f;
            if (lj == li) continue;
            const uint32_t j = i - st[a];
            // rank of j's axis-a edge among j's sign-changing edges
            uint32_t rank = 0;
#pragma unroll
            for (int b = 0; b < a; b++)
                if (co[b] + 1 < d1 && ((dens[j + st[b]] < 0.0f) != lj)) rank++;
            const float4 q = g[vid0[j] + rank];
            const float ds = di - dj;
            const float ga = a == 0 ? q.x : (a == 1 ? q.y : q.z);
            acc = acc + ga * (dj / (ds * ds));
        }
    }
    out[i] = acc;
}

// ------------------------------------------------------------------------
// nearest-target loss
// ------------------------------------------------------------------------
__device__ __forceinline__ int float_order(float f) {
    const int b = __float_as_int(f);
    return b >= 0 ? b : b ^ 0x7FFFFFFF;
}
__device__ __forceinline__ float order_float(int b) { return __int_as_float(b >= 0 ? b : b ^ 0x7FFFFFFF); }

__global__ void k_nn_bbox_init(int* bb) {
    if (threadIdx.x < 3) bb[threadIdx.x] = 0x7FFFFFFF;
    else if (threadIdx.x < 6) bb[threadIdx.x] = (int)0x80000000;
}

// Bounding box of the targets: per-thread, per-wave, per-block reductions,
// then one atomic per block and coordinate (min/max are order-independent).
__global__ void __launch_bounds__(kThreads) k_nn_bbox(const float* __restrict__ t, int64_t n, int* bb) {
    __shared__ float s_r[6][kThreads / 64];
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        for (int a = 0; a < 3; a++) {
            lo[a] = fminf(lo[a], t[3 * i + a]);
            hi[a] = fmaxf(hi[a], t[3 * i + a]);
        }
    const int wave = threadIdx.x >> 6;
    for (int a = 0; a < 3; a++) {
        for (int off = 32; off > 0; off >>= 1) {
            lo[a] = fminf(lo[a], __shfl_xor(lo[a], off));
            hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], off));
        }
        if ((threadIdx.x & 63) == 0) {
            s_r[a][wave] = lo[a];
            s_r[3 + a][wave] = hi[a];
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        float v = s_r[a][0];
        for (int w = 1; w < kThreads / 64; w++) v = a < 3 ? fminf(v, s_r[a][w]) : fmaxf(v, s_r[a][w]);
        if (a < 3) atomicMin(&bb[a], float_order(v));
        else atomicMax(&bb[a], float_order(v));
    }
}

__device__ __forceinline__ uint32_t spread10(uint32_t v) {
    v &= 1023u;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

__device__ __forceinline__ uint32_t morton_key(const int* bb, float x, float y, float z) {
    const float p[3] = {x, y, z};
    uint32_t q[3];
    for (int a = 0; a < 3; a++) {
        const float lo = order_float(bb[a]), hi = order_float(bb[3 + a]);
        const float ext = hi - lo;
        float u = ext > 0.0f ? (p[a] - lo) * (1024.0f / ext) : 0.0f;
        u = fminf(fmaxf(u, 0.0f), 1023.0f);
        q[a] = (uint32_t)u;
    }
    return (spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2]);
}

__global__ void k_nn_keys(const float* __restrict__ t, int64_t n, const int* __restrict__ bb,
                          uint32_t* __restrict__ keys, int32_t* __restrict__ vals) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    keys[i] = morton_key(bb, t[3 * i], t[3 * i + 1], t[3 * i + 2]);
    vals[i] = (int32_t)i;
}

// fmin with the value DPP control CTRL brings from another lane (+inf where
// the source lane is outside the row or the row is not in ROW_MASK).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_fmin(float v) {
    const int o = __builtin_amdgcn_update_dpp(__float_as_int(INFINITY), __float_as_int(v), CTRL, ROW_MASK, 0xf, false);
    return fminf(v, __int_as_float(o));
}

// Minimum over the 64 lanes of a wave (all lanes active): prefix minima
// within each row of 16 lanes (row_shr 1, 2, 4, 8), then row 0's last lane
// into row 1 and row 2's into row 3 (row_bcast:15), then lane 31 into rows 2
// and 3 (row_bcast:31); lane 63 then holds the minimum.
__device__ __forceinline__ float wave_min(float x) {
    x = dpp_fmin<0x111, 0xf>(x);
    x = dpp_fmin<0x112, 0xf>(x);
    x = dpp_fmin<0x114, 0xf>(x);
    x = dpp_fmin<0x118, 0xf>(x);
    x = dpp_fmin<0x142, 0xa>(x);
    x = dpp_fmin<0x143, 0xc>(x);
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

// Sum over the 64 lanes of a wave (all lanes active), the same way.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_fadd(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xf, false));
}
__device__ __forceinline__ float wave_sum(float x) {
    x = dpp_fadd<0x111, 0xf>(x);
    x = dpp_fadd<0x112, 0xf>(x);
    x = dpp_fadd<0x114, 0xf>(x);
    x = dpp_fadd<0x118, 0xf>(x);
    x = dpp_fadd<0x142, 0xa>(x);
    x = dpp_fadd<0x143, 0xc>(x);
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

// Leaves of the implicit hierarchy: heap-numbered nodes 1 .. 2P-1 over P (a
// power of two) leaves; leaf l is node P + l and holds sorted targets
// [kLeaf l, kLeaf (l+1)), the last one filled up with points at infinity; leaves
// past the targets are empty boxes.  A wave per leaf, a lane per target, which it
// also brings into sorted order as (x, y, z, id) (a lane per leaf walked its 64
// targets four times: 47 us for 313 leaves with the gather, this takes 12).
//
// Box, and oriented bound: the centre c of the targets, the principal
// axes of their covariance (cyclic Jacobi, then re-orthonormalised) and the
// largest |(q - c) . axis| per axis; four float4 per leaf (c, then each axis
// with its extent in w).  A patch of a curved target set is thin along its
// normal, where the axis-aligned box of a tilted patch is not.  Empty leaves
// get a zero record (their axis-aligned box already excludes them).
__global__ void __launch_bounds__(kThreads) k_nn_leaves(const float* __restrict__ t, const int32_t* __restrict__ perm,
                                                        int64_t n, int64_t P, float4* __restrict__ st,
                                                        float4* __restrict__ lo, float4* __restrict__ hi,
                                                        float4* __restrict__ ob) {
    const int64_t l = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (l >= P) return;  // uniform across the wave
    const int lane = lane_id();
    const int64_t b = l * kLeaf;
    const bool has = b + lane < n;
    float4* o = ob + 4 * l;
    if (b >= n) {
        if (lane < 4) o[lane] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (lane == 0) {
            lo[P + l] = make_float4(INFINITY, INFINITY, INFINITY, 0.0f);
            hi[P + l] = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
        }
        return;
    }
    float4 q = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (has) {
        const int32_t id = perm[b + lane];
        q = make_float4(t[3 * (int64_t)id], t[3 * (int64_t)id + 1], t[3 * (int64_t)id + 2], __int_as_float(id));
    }
    st[b + lane] = has ? q : make_float4(INFINITY, INFINITY, INFINITY, __int_as_float(0x7FFFFFFF));
    const float qa[3] = {q.x, q.y, q.z};
    float bl[3], bh[3], c[3];
    const float inv = 1.0f / (float)std::min<int64_t>(kLeaf, n - b);
#pragma unroll
    for (int k = 0; k < 3; k++) {
        bl[k] = wave_min(has ? qa[k] : INFINITY);
        bh[k] = -wave_min(has ? -qa[k] : INFINITY);
        c[k] = wave_sum(has ? qa[k] : 0.0f) * inv;
    }
    if (lane == 0) {
        lo[P + l] = make_float4(bl[0], bl[1], bl[2], 0.0f);
        hi[P + l] = make_float4(bh[0], bh[1], bh[2], 0.0f);
    }
    const float dq[3] = {has ? q.x - c[0] : 0.0f, has ? q.y - c[1] : 0.0f, has ? q.z - c[2] : 0.0f};
    float a[3][3];
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int k = r; k < 3; k++) a[r][k] = a[k][r] = wave_sum(dq[r] * dq[k]);
    float v[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
    for (int sw = 0; sw < 8; sw++)
#pragma unroll
        for (int pq = 0; pq < 3; pq++) {
            const int p0 = pq == 2 ? 1 : 0, q0 = pq == 0 ? 1 : 2;
            const float apq = a[p0][q0];
            if (!(fabsf(apq) > 1e-30f)) continue;
            const float th = (a[q0][q0] - a[p0][p0]) / (2.0f * apq);
            const float t = (th >= 0.0f ? 1.0f : -1.0f) / (fabsf(th) + sqrtf(th * th + 1.0f));
            const float cs = 1.0f / sqrtf(t * t + 1.0f), sn = t * cs;
#pragma unroll
            for (int k = 0; k < 3; k++) {  // columns p0, q0 of A J
                const float akp = a[k][p0], akq = a[k][q0];
                a[k][p0] = cs * akp - sn * akq;
                a[k][q0] = sn * akp + cs * akq;
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {  // rows p0, q0 of J^T (A J)
                const float apk = a[p0][k], aqk = a[q0][k];
                a[p0][k] = cs * apk - sn * aqk;
                a[q0][k] = sn * apk + cs * aqk;
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const float vkp = v[k][p0], vkq = v[k][q0];
                v[k][p0] = cs * vkp - sn * vkq;
                v[k][q0] = sn * vkp + cs * vkq;
            }
        }
    // axes: the first two eigenvector columns, Gram-Schmidt, and their cross product
    float u[3] = {v[0][0], v[1][0], v[2][0]}, w[3] = {v[0][1], v[1][1], v[2][1]};
    float lu = sqrtf(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
    for (int k = 0; k < 3; k++) u[k] /= lu;
    const float dw = w[0] * u[0] + w[1] * u[1] + w[2] * u[2];
    for (int k = 0; k < 3; k++) w[k] -= dw * u[k];
    const float lw = sqrtf(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
    for (int k = 0; k < 3; k++) w[k] /= lw;
    const float nn[3] = {u[1] * w[2] - u[2] * w[1], u[2] * w[0] - u[0] * w[2], u[0] * w[1] - u[1] * w[0]};
    const float ax[3][3] = {{u[0], u[1], u[2]}, {w[0], w[1], w[2]}, {nn[0], nn[1], nn[2]}};
    if (lane == 0) o[0] = make_float4(c[0], c[1], c[2], 0.0f);
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float e = -wave_min(-fabsf(dq[0] * ax[k][0] + dq[1] * ax[k][1] + dq[2] * ax[k][2]));
        if (lane == 0) o[1 + k] = make_float4(ax[k][0], ax[k][1], ax[k][2], e);
    }
}

// Inner boxes of one wide level [level, 2 level).
__global__ void k_nn_level(int64_t level, float4* __restrict__ lo, float4* __restrict__ hi) {
    const int64_t i = level + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * level) return;
    const float4 a = lo[2 * i], b = lo[2 * i + 1], c = hi[2 * i], d = hi[2 * i + 1];
    lo[i] = make_float4(fminf(a.x, b.x), fminf(a.y, b.y), fminf(a.z, b.z), 0.0f);
    hi[i] = make_float4(fmaxf(c.x, d.x), fmaxf(c.y, d.y), fmaxf(c.z, d.z), 0.0f);
}

// Inner boxes of the levels from `top` up to the root (one workgroup).
__global__ void __launch_bounds__(1024) k_nn_inner(int64_t top, float4* __restrict__ lo, float4* __restrict__ hi) {
    for (int64_t level = top; level >= 1; level >>= 1) {
        for (int64_t i = level + threadIdx.x; i < 2 * level; i += blockDim.x) {
            const float4 a = lo[2 * i], b = lo[2 * i + 1], c = hi[2 * i], d = hi[2 * i + 1];
            lo[i] = make_float4(fminf(a.x, b.x), fminf(a.y, b.y), fminf(a.z, b.z), 0.0f);
            hi[i] = make_float4(fmaxf(c.x, d.x), fmaxf(c.y, d.y), fmaxf(c.z, d.z), 0.0f);
        }
        __syncthreads();
    }
}

__device__ __forceinline__ float dist2(float px, float py, float pz, float4 q) {
    const float dx = px - q.x, dy = py - q.y, dz = pz - q.z;
    return (dx * dx + dy * dy) + dz * dz;
}

// Squared distance from p to the box [l, h] (0 inside, +inf for an empty box);
// never above the distance of p to any point in it in FP32 (every step rounds
// monotonically).
__device__ __forceinline__ float box_lb2(float px, float py, float pz, float4 l, float4 h) {
    const float dx = fmaxf(fmaxf(l.x - px, px - h.x), 0.0f);
    const float dy = fmaxf(fmaxf(l.y - py, py - h.y), 0.0f);
    const float dz = fmaxf(fmaxf(l.z - pz, pz - h.z), 0.0f);
    return (dx * dx + dy * dy) + dz * dz;
}

// Squared-distance lower bound from p to the targets of a leaf from its
// oriented record: per axis max(0, |(p - c) . axis| - extent - slack), summed
// and scaled down.  The slack (1e-5 of |p - c|_1 and of the extent per axis,
// then 1 - 1e-5 on the sum) is far above the FP32 errors of the projections, of
// the axes' orthonormality and of the targets' own FP32 distances (each of order
// 1e-7 relative), so the bound stays below the FP32 distance of p to every
// target of the leaf.  e: the extents with their share of the slack added.
__device__ __forceinline__ float obb_lb2(float px, float py, float pz, float4 c, float4 u, float4 w, float4 nrm,
                                         const float (&e)[3]) {
    const float dx = px - c.x, dy = py - c.y, dz = pz - c.z;
    const float s = 1e-5f * ((fabsf(dx) + fabsf(dy)) + fabsf(dz));
    const float tu = fabsf((dx * u.x + dy * u.y) + dz * u.z), tw = fabsf((dx * w.x + dy * w.y) + dz * w.z),
                tn = fabsf((dx * nrm.x + dy * nrm.y) + dz * nrm.z);
    const float su = fmaxf((tu - e[0]) - s, 0.0f), sw = fmaxf((tw - e[1]) - s, 0.0f),
                sn = fmaxf((tn - e[2]) - s, 0.0f);
    return ((su * su + sw * sw) + sn * sn) * (1.0f - 1e-5f);
}

// A wave-uniform 64-bit value held in every lane, moved to scalar registers.
__device__ __forceinline__ uint64_t uniform_u64(uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// Lowest lane of the (non-empty) set m whose value x is smallest.
__device__ __forceinline__ int wave_argmin(float x, uint64_t m, int lane) {
    const float y = (m >> lane) & 1 ? x : INFINITY;
    const float mn = wave_min(y);
    return __ffsll((unsigned long long)(__ballot(y == mn) & m)) - 1;
}

// Value x from the lane XOR 1, 2 or (within 8 or 16 lanes, lane i <-> 7 - i, 15 - i) mirrored.
template <int CTRL>
__device__ __forceinline__ int dpp_lane(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kMirror8 = 0x141, kMirror16 = 0x140;

// Nearest target of each vertex, one wave per packet of kPacket vertices that
// are consecutive in the tape's order, so near each other.  The hierarchy
// (heap nodes 1 .. 2P-1, leaves at depth D = log2 P) is walked once for the
// packet, in frames of the 2^f descendants, f <= kNNFan levels down, of the
// node popped from the frame above (the first, of the root, takes D mod kNNFan
// levels or kNNFan so that the leaf frames are full).  Lane j holds descendant
// j and bounds its distance from each vertex in turn (leaves also by their
// oriented bound); it is live while some vertex's bound is no farther than that
// vertex's best target distance U so far.  Frames pop their nearest live box
// first.  Leaves are evaluated in pairs (one load latency and one set of
// minima), by kPart lanes per vertex, kEach of a leaf's targets each, and the
// frame re-pruned.  Pruning drops a box only when it is strictly farther than U
// from every vertex, and each U is an actual target distance, so every target
// at a vertex's minimum distance is evaluated and the result is the lowest
// (distance, original index), as a brute-force scan gives.
//
// Bound by VALU issue, and with few packets by the longest walk.  A wave per
// vertex (7 frames and 17 leaves each, a wave-wide minimum after every leaf) took
// 168 us for 44,392 vertices and 200,000 targets, 33 us for 7,819 and 20,000;
// packets share boxes, leaves and minima: 80 and 47 us with four
// vertices, 92 and 86 with eight (the walks are longer and fewer).  The small
// case pays less than its hierarchy's leaves gain.  One bound for the whole
// packet instead of one per vertex is cheaper a box and loses all of it:
// far from the targets, boxes differ by less than the packet's width (2,455 us).
constexpr int kPart = 64 / kPacket;    // lanes per vertex
constexpr int kEach = kLeaf / kPart;   // targets of a leaf per lane
static_assert(kPart == 8 || kPart == 16, "the minima over a vertex's lanes");
static_assert(kNNFan == 6, "a frame is a wave's lanes");
__global__ void __launch_bounds__(64) k_nn_query(const float* __restrict__ pos, const int32_t* __restrict__ order,
                                                 int V, const float4* __restrict__ st, int64_t n, int64_t P,
                                                 const float4* __restrict__ lo, const float4* __restrict__ hi,
                                                 const float4* __restrict__ ob, int32_t* __restrict__ nearest,
                                                 float* __restrict__ dldp, double* __restrict__ d2) {
    const int64_t first = (int64_t)blockIdx.x * kPacket;
    const int lane = (int)threadIdx.x, slot = lane / kPart, part = lane % kPart;
    const int mine = order[first + slot];  // -1: a packet's spare slot, which repeats its first vertex
    const bool own = mine >= 0;
    const int v = own ? mine : __builtin_amdgcn_readlane(mine, 0);
    const float px = pos[3 * (int64_t)v], py = pos[3 * (int64_t)v + 1], pz = pos[3 * (int64_t)v + 2];
    // no box is near enough for a spare slot, nor for a vertex that is not a
    // number (it has no distance)
    const bool counts = own && px == px && py == py && pz == pz;
    auto slot_value = [](float x, int s) {
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), kPart * s));
    };
    float vx[kPacket], vy[kPacket], vz[kPacket], U[kPacket];  // scalar registers
#pragma unroll
    for (int s = 0; s < kPacket; s++) {
        vx[s] = slot_value(px, s);
        vy[s] = slot_value(py, s);
        vz[s] = slot_value(pz, s);
        U[s] = slot_value(counts ? INFINITY : -INFINITY, s);
    }
    int D = 0;
    while ((int64_t)1 << D < P) D++;
    const int f0 = D == 0 ? 0 : D - kNNFan * ((D - 1) / kNNFan);
    float bd = INFINITY;  // this lane's best (distance, original index, sorted position) for its vertex
    int bi = 0x7FFFFFFF;
    int bs = -1;  // sorted position (n < 2^31, heap indices < 2^30)
    // inner frames: per lane and vertex box distances, the live set, heap index of descendant 0
    __shared__ float s_lb[kNNFrames][kPacket][64];
    __shared__ unsigned long long s_mk[kNNFrames];
    __shared__ int s_base[kNNFrames];
    const int Pi = (int)P, leaves = (int)((n + kLeaf - 1) / kLeaf);
    float lb[kPacket];
    auto live = [&]() {
        unsigned long long m = 0;
#pragma unroll
        for (int s = 0; s < kPacket; s++) m |= __ballot(lb[s] <= U[s]);
        return m;
    };
    auto nearest_of = [&](unsigned long long m) {
        float x = lb[0];
#pragma unroll
        for (int s = 1; s < kPacket; s++) x = fminf(x, lb[s]);
        return wave_argmin(x, m, lane);
    };
    auto lower = [](float& a, int& ai, int& as, float b, int bj, int bt) {
        const bool t = (b < a) | ((b == a) & (bj < ai));
        a = t ? b : a;
        ai = t ? bj : ai;
        as = t ? bt : as;
    };
    // The targets of two leaves (heap indices; twice the same where one is
    // left), then every vertex's U: this lane's targets, the nearest by a tree
    // of selects, the minimum over the vertex's lanes.
    auto eval = [&](int leaf, int also) {
        const uint32_t i0 = (uint32_t)(leaf - Pi) * kLeaf + (uint32_t)part;
        const uint32_t i1 = (uint32_t)(also - Pi) * kLeaf + (uint32_t)part;
        float4 q[2 * kEach];
        float e[2 * kEach];
        int ei[2 * kEach], es[2 * kEach];
#pragma unroll
        for (int u = 0; u < 2 * kEach; u++) {
            es[u] = (int)((u & 1 ? i1 : i0) + kPart * (u >> 1));
            q[u] = st[es[u]];
        }
#pragma unroll
        for (int u = 0; u < 2 * kEach; u++) {
            const float x = dist2(px, py, pz, q[u]);
            e[u] = x == x ? x : INFINITY;  // at a point that is not a number: as one past the targets
            ei[u] = x == x ? __float_as_int(q[u].w) : 0x7FFFFFFF;
        }
#pragma unroll
        for (int w = kEach; w; w >>= 1)
#pragma unroll
            for (int u = 0; u < w; u++) lower(e[u], ei[u], es[u], e[u + w], ei[u + w], es[u + w]);
        lower(bd, bi, bs, e[0], ei[0], es[0]);
        float m = bd;
        m = fminf(m, __int_as_float(dpp_lane<kXor1>(__float_as_int(m))));
        m = fminf(m, __int_as_float(dpp_lane<kXor2>(__float_as_int(m))));
        m = fminf(m, __int_as_float(dpp_lane<kMirror8>(__float_as_int(m))));
        if (kPart == 16) m = fminf(m, __int_as_float(dpp_lane<kMirror16>(__float_as_int(m))));
        m = counts ? m : -INFINITY;
#pragma unroll
        for (int s = 0; s < kPacket; s++) U[s] = slot_value(m, s);
    };
    int k = 0, f = f0, base = 1 << f0;
    while (k >= 0) {
        const int level = f0 + kNNFan * k;
        // a frame of leaves ends with the last that holds targets
        const int width = level == D ? min(1 << f, Pi + leaves - base) : 1 << f;
        const unsigned long long all = width < 64 ? (1ull << max(width, 0)) - 1ull : ~0ull;
        const int node = lane < (1 << f) ? base + lane : base;
        const float4 l = lo[node], h = hi[node];
#pragma unroll
        for (int s = 0; s < kPacket; s++) lb[s] = box_lb2(vx[s], vy[s], vz[s], l, h);
        if (level == D) {
            const float4* o = ob + 4 * (int64_t)(node - Pi);
            const float4 c = o[0], u = o[1], w = o[2], nrm = o[3];
            const float e[3] = {u.w * (1.0f + 2e-5f), w.w * (1.0f + 2e-5f), nrm.w * (1.0f + 2e-5f)};
#pragma unroll
            for (int s = 0; s < kPacket; s++)
                if (__ballot(lb[s] <= U[s]))
                    lb[s] = fmaxf(lb[s], obb_lb2(vx[s], vy[s], vz[s], c, u, w, nrm, e));
            unsigned long long m = all & live();
            while (m) {
                // the nearest, with its sibling or else any other live one
                const int j = nearest_of(m);
                m &= ~(1ull << j);
                const int h = m >> (j ^ 1) & 1 || !m ? j ^ 1 : __ffsll(m) - 1, i = m ? h : j;
                eval(base + j, base + i);
                m = m & ~(1ull << i) & live();
            }
            k--;
        } else {
#pragma unroll
            for (int s = 0; s < kPacket; s++) s_lb[k][s][lane] = lb[s];
            s_mk[k] = all;
            s_base[k] = base;
        }
        // the next node: the nearest live one of the lowest frame that has any
        for (; k >= 0; k--) {
#pragma unroll
            for (int s = 0; s < kPacket; s++) lb[s] = s_lb[k][s][lane];
            const unsigned long long m = uniform_u64(s_mk[k]) & live();
            if (!m) continue;
            const int j = nearest_of(m);
            s_mk[k] = m & ~(1ull << j);
            base = (__builtin_amdgcn_readfirstlane(s_base[k]) + j) << kNNFan;
            f = kNNFan;
            k++;
            break;
        }
    }
    // each vertex's lowest (distance, index) over its kPart lanes
    auto take = [&](float od, int oi, int os) {
        if (od < bd || (od == bd && oi < bi)) {
            bd = od;
            bi = oi;
            bs = os;
        }
    };
    take(__int_as_float(dpp_lane<kXor1>(__float_as_int(bd))), dpp_lane<kXor1>(bi), dpp_lane<kXor1>(bs));
    take(__int_as_float(dpp_lane<kXor2>(__float_as_int(bd))), dpp_lane<kXor2>(bi), dpp_lane<kXor2>(bs));
    take(__int_as_float(dpp_lane<kMirror8>(__float_as_int(bd))), dpp_lane<kMirror8>(bi), dpp_lane<kMirror8>(bs));
    if (kPart == 16)
        take(__int_as_float(dpp_lane<kMirror16>(__float_as_int(bd))), dpp_lane<kMirror16>(bi), dpp_lane<kMirror16>(bs));
    if (part != 0 || !own) return;
    const float4 q = bs >= 0 ? st[bs] : make_float4(px, py, pz, 0.0f);
    nearest[v] = bs >= 0 ? bi : -1;
    const float sc = 2.0f / (float)V;
    dldp[3 * (int64_t)v] = (px - q.x) * sc;
    dldp[3 * (int64_t)v + 1] = (py - q.y) * sc;
    dldp[3 * (int64_t)v + 2] = (pz - q.z) * sc;
    d2[v] = bs >= 0 ? (double)bd : 0.0;
}

// Deterministic sum: thread t adds x[t], x[t + 1024], ... in order, then a
// fixed tree.
__global__ void __launch_bounds__(1024) k_sum(const double* __restrict__ x, int n, double* __restrict__ out) {
    __shared__ double s[1024];
    const int tid = threadIdx.x;
    double a = 0.0;
    int i = tid;
    // the same order as one add per stride step; the loads of 8 steps are
    // issued together
    for (; i + 7 * 1024 < n; i += 8 * 1024) {
        double v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = x[i + j * 1024];
#pragma unroll
        for (int j = 0; j < 8; j++) a += v[j];
    }
    for (; i < n; i += 1024) a += x[i];
    s[tid] = a;
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
        if (tid < w) s[tid] += s[tid + w];
        __syncthreads();
    }
    if (tid == 0) out[0] = s[0] / (double)n;
}

}  // namespace

struct bmf_tape {
    bmf_ctx* ctx = nullptr;
    int32_t max_dim = 0;
    int64_t cap_v = 0, cap_i = 0;
    int32_t ckpt_every = 1;
    bool valid = false;
    int32_t dim = 0, K = 0, bp = 0, V = 0, T = 0, contains_mesh = 0;
    float* dens = nullptr;
    uint32_t* vid0 = nullptr;
    // vertices by lattice cell, for the packets of the nearest-target query
    int32_t* order = nullptr;
    uint32_t* rank = nullptr;     // of each vertex within its cell
    uint32_t* cell_n = nullptr;   // [kOrderCells] vertices of each cell (0 between forwards)
    uint32_t* cell_base = nullptr;  // [kOrderCells] first place of each cell
    int places = 0;                 // of `order` in use, a multiple of kPacket
    uint32_t* vedge = nullptr;
    uint8_t* boundary = nullptr;
    uint32_t* idx = nullptr;
    uint2* ring = nullptr;
    float* bscale = nullptr;
    uint8_t* deg = nullptr;
    uint8_t* mv = nullptr;
    float4* p4 = nullptr;
    float4* q4 = nullptr;
    float* pos = nullptr;
    float4* g = nullptr;
    float4* g2 = nullptr;   // ping-pong partner of g in the backward
    float4* r4 = nullptr;   // ping-pong partner of q4 in bmf_tape_positions
    int* taken = nullptr;         // places of `order` taken
    struct Host {                 // what the host reads, written by the kernels
        double loss;
        int err;                  // the adjacency's check
        int places;
    };
    Host* host = nullptr;         // pinned
    Host* mhost = nullptr;        // its device address
    SamplerDev* ext_sampler = nullptr;  // device: EXTERNAL, the densities named by each call (Arenas::ext)
    hipEvent_t ev[6] = {};  // start / end of the last forward, loss and backward
    bool timed[3] = {false, false, false};
    float4* ckpt = nullptr;
    int64_t ckpt_slots = 0;
    // nearest-target search: hierarchy buffers for up to nn_cap targets and
    // the target set last built into them (nn_n targets, 0 = none)
    int64_t nn_cap = 0;
    int64_t nn_n = 0;
    uint32_t* keys[2] = {nullptr, nullptr};
    int32_t* vals[2] = {nullptr, nullptr};
    float4* st = nullptr;
    float4* blo = nullptr;  // hierarchy boxes, heap-numbered [2P]
    float4* bhi = nullptr;
    float4* obb = nullptr;  // oriented bound of each leaf [4P]
    int* bb = nullptr;
    void* cub_tmp = nullptr;
    size_t cub_bytes = 0;
    double* d2 = nullptr;
    double* loss = nullptr;
    int32_t* nearest_tmp = nullptr;
};

namespace {

// Leaves of the target hierarchy, rounded up to a power of two.
int64_t leaf_pow2(int64_t n) {
    const int64_t leaves = (n + kLeaf - 1) / kLeaf;
    int64_t P = 1;
    while (P < leaves) P <<= 1;
    return P;
}

void free_nn(bmf_tape* t) {
    for (int i = 0; i < 2; i++) {
        dfree(t->keys[i]);
        dfree(t->vals[i]);
    }
    dfree(t->st);
    dfree(t->blo);
    dfree(t->bhi);
    dfree(t->obb);
    if (t->cub_tmp) (void)hipFree(t->cub_tmp);
    t->cub_tmp = nullptr;
    t->cub_bytes = 0;
    t->nn_cap = 0;
    t->nn_n = 0;
}

int reserve_nn(bmf_tape* t, int64_t n) {
    if (n <= t->nn_cap) return BMF_OK;
    free_nn(t);
    const int64_t P = leaf_pow2(n);
    bool ok = true;
    for (int i = 0; i < 2; i++)
        ok = ok && dalloc(&t->keys[i], n) == hipSuccess && dalloc(&t->vals[i], n) == hipSuccess;
    ok = ok && dalloc(&t->st, (n + kLeaf - 1) / kLeaf * kLeaf) == hipSuccess && dalloc(&t->blo, 2 * P) == hipSuccess &&
         dalloc(&t->bhi, 2 * P) == hipSuccess && dalloc(&t->obb, 4 * P) == hipSuccess;
    if (ok) {
        hipcub::DoubleBuffer<uint32_t> kb(t->keys[0], t->keys[1]);
        hipcub::DoubleBuffer<int32_t> vb(t->vals[0], t->vals[1]);
        size_t bytes = 0;
        ok = hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, kb, vb, (int)n, 0, 30) == hipSuccess;
        ok = ok && hipMalloc(&t->cub_tmp, std::max<size_t>(bytes, 1)) == hipSuccess;
        t->cub_bytes = bytes;
    }
    if (!ok) {
        free_nn(t);
        return BMF_EHIP;
    }
    t->nn_cap = n;
    return BMF_OK;
}

// Buffers of the nearest-target hierarchy of n targets: Morton keys and
// target ids (double-buffered for the radix sort), the targets in Morton
// order (x, y, z, id), the boxes of the heap-numbered nodes 1 .. 2P-1 and
// the oriented bound of each leaf.
struct NNBuffers {
    uint32_t* keys[2];
    int32_t* vals[2];
    float4* st;
    float4* blo;
    float4* bhi;
    float4* ob;
    void* cub_tmp;
    size_t cub_bytes;
};

NNBuffers tape_nn(bmf_tape* t) {
    return NNBuffers{{t->keys[0], t->keys[1]}, {t->vals[0], t->vals[1]}, t->st, t->blo, t->bhi, t->obb, t->cub_tmp,
                     t->cub_bytes};
}

// Enqueues the hierarchy build of the n targets [n][3] into b: bounding box,
// Morton keys, radix sort of (key, id), sorted targets, leaf and inner boxes.
int nn_build(const float* targets, int64_t n, int* bb, const NNBuffers& b, hipStream_t s) {
    const int64_t P = leaf_pow2(n);
    hipLaunchKernelGGL(k_nn_bbox_init, dim3(1), dim3(64), 0, s, bb);
    hipLaunchKernelGGL(k_nn_bbox, dim3((unsigned)std::min<int64_t>(256, blocks_for(n))), dim3(kThreads), 0, s, targets,
                       n, bb);
    hipLaunchKernelGGL(k_nn_keys, dim3(blocks_for(n)), dim3(kThreads), 0, s, targets, n, bb, b.keys[0], b.vals[0]);
    BMF_HIP(hipGetLastError());
    hipcub::DoubleBuffer<uint32_t> kb(b.keys[0], b.keys[1]);
    hipcub::DoubleBuffer<int32_t> vb(b.vals[0], b.vals[1]);
    size_t bytes = b.cub_bytes;
    BMF_HIP(hipcub::DeviceRadixSort::SortPairs(b.cub_tmp, bytes, kb, vb, (int)n, 0, 30, s));
    hipLaunchKernelGGL(k_nn_leaves, dim3(blocks_for(64 * P)), dim3(kThreads), 0, s, targets, vb.Current(), n, P, b.st,
                       b.blo, b.bhi, b.ob);
    int64_t level = P >> 1;
    for (; level >= 2048; level >>= 1)
        hipLaunchKernelGGL(k_nn_level, dim3(blocks_for(level)), dim3(kThreads), 0, s, level, b.blo, b.bhi);
    if (level >= 1) hipLaunchKernelGGL(k_nn_inner, dim3(1), dim3(1024), 0, s, level, b.blo, b.bhi);
    BMF_HIP(hipGetLastError());
    return BMF_OK;
}

// Enqueues the nearest-target query of the tape's V final positions against
// a hierarchy of n targets, dL/dp, and the loss (FP64, fixed order) into
// loss_out (device).
int nn_query(bmf_tape* t, const NNBuffers& b, int64_t n, float* dldp, int32_t* nearest, double* loss_out,
             hipStream_t s) {
    const int64_t P = leaf_pow2(n);
    hipLaunchKernelGGL(k_nn_query, dim3((unsigned)(t->places / kPacket)), dim3(64), 0, s, t->pos, t->order, t->V, b.st, n, P, b.blo, b.bhi, b.ob,
                       nearest ? nearest : t->nearest_tmp, dldp, t->d2);
    hipLaunchKernelGGL(k_sum, dim3(1), dim3(1024), 0, s, t->d2, t->V, loss_out);
    BMF_HIP(hipGetLastError());
    return BMF_OK;
}

// Runs k smoothing iterations starting from `a` (float4 [V]), ping-ponging
// between a and b, one launch per iteration; the state after iteration m is
// kept in checkpoint slot (from + m + 1) / every when that divides (from >= 0),
// and the final state is written as float3 to pos3.
int smooth_steps(bmf_tape* t, float4* a, float4* b, int k, hipStream_t s, float* pos3, int ckpt_from = -1) {
    float4* cur = a;
    float4* nxt = b;
    if (k == 0) {
        hipLaunchKernelGGL(k_tape_out, dim3(blocks_for(t->V)), dim3(kThreads), 0, s, a, t->V, pos3);
        BMF_HIP(hipGetLastError());
        return BMF_OK;
    }
    for (int m = 0; m < k; m++) {
        float4* ck = nullptr;
        if (ckpt_from >= 0 && (ckpt_from + m + 1) % t->ckpt_every == 0)
            ck = t->ckpt + (int64_t)((ckpt_from + m + 1) / t->ckpt_every) * t->cap_v;
        hipLaunchKernelGGL(k_tape_step, dim3(step_blocks(t->V)), dim3(kStepThreads), 0, s, t->ring, (int)t->cap_v,
                           t->deg, t->mv, cur, t->V, nxt, ck, m == k - 1 ? pos3 : nullptr);
        BMF_HIP(hipGetLastError());
        std::swap(cur, nxt);
    }
    return BMF_OK;
}

// ---- scratch of bmf_loss_nearest_noalloc ---------------------------------
// The hierarchy of up to BMF_NOALLOC_MAX_TARGETS targets lives in one
// file-scope device array, so that entry point allocates nothing: Morton
// keys and target ids (2 x 2 x 1 MiB), the sorted targets (4 MiB), the boxes
// of 2 x 4096 heap nodes of 64-target leaves (2 x 128 KiB), the oriented
// bounds of the 4096 leaves (256 KiB) and the radix sort's temporary storage
// (2 MiB), 10.5 MiB per GPU for the life of the process.  Host code
// never passes the array's name to a kernel (on the host it is a stand-in,
// not a device address): each device's address comes from
// hipGetSymbolAddress, taken once per device with that device current.
constexpr int64_t kNAMax = BMF_NOALLOC_MAX_TARGETS;
constexpr int64_t kNALeaves = kNAMax / kLeaf;
static_assert(kNAMax % kLeaf == 0 && (kNALeaves & (kNALeaves - 1)) == 0, "leaves of the maximum set: a power of two");
constexpr size_t kNAKeyBytes = sizeof(uint32_t) * kNAMax;
constexpr size_t kNATgtBytes = sizeof(float4) * kNAMax;
constexpr size_t kNABoxBytes = sizeof(float4) * 2 * kNALeaves;
constexpr size_t kNAObbBytes = sizeof(float4) * 4 * kNALeaves;
constexpr size_t kNACubBytes = 2u << 20;
constexpr size_t kScratchBytes = 4 * kNAKeyBytes + kNATgtBytes + 2 * kNABoxBytes + kNAObbBytes + kNACubBytes;
static_assert(kScratchBytes == (42u << 18), "10.5 MiB of scratch with 64-target leaves");
static_assert(kNAKeyBytes % 256 == 0 && kNATgtBytes % 256 == 0 && kNABoxBytes % 256 == 0 && kNAObbBytes % 256 == 0,
              "256-byte aligned parts");

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_dev[kMaxDevices] = {};

// Device address of `scratch` on `device` (which must be current), looked up
// on the first call for that device.
int scratch_acquire(int device) {
    if (device < 0 || device >= kMaxDevices) return BMF_EINVAL;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_dev[device]) return BMF_OK;
    void* ptr = nullptr;
    BMF_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) return BMF_EHIP;
    g_scratch_dev[device] = ptr;
    return BMF_OK;
}

void* scratch_on(int device) {
    if (device < 0 || device >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    return g_scratch_dev[device];
}

NNBuffers scratch_nn(void* base) {
    unsigned char* p = static_cast<unsigned char*>(base);
    NNBuffers b;
    b.keys[0] = reinterpret_cast<uint32_t*>(p);
    b.keys[1] = reinterpret_cast<uint32_t*>(p + kNAKeyBytes);
    b.vals[0] = reinterpret_cast<int32_t*>(p + 2 * kNAKeyBytes);
    b.vals[1] = reinterpret_cast<int32_t*>(p + 3 * kNAKeyBytes);
    p += 4 * kNAKeyBytes;
    b.st = reinterpret_cast<float4*>(p);
    p += kNATgtBytes;
    b.blo = reinterpret_cast<float4*>(p);
    b.bhi = reinterpret_cast<float4*>(p + kNABoxBytes);
    p += 2 * kNABoxBytes;
    b.ob = reinterpret_cast<float4*>(p);
    p += kNAObbBytes;
    b.cub_tmp = p;
    b.cub_bytes = kNACubBytes;
    return b;
}

__global__ void k_store_f64(double* __restrict__ out, double v) { out[0] = v; }

}  // namespace

extern "C" {

int bmf_tape_create(bmf_tape** out, bmf_ctx* ctx, int32_t max_dim, int64_t max_vertices, int64_t max_indices,
                    int32_t checkpoint_every) {
    if (!out || !ctx) return BMF_EINVAL;
    *out = nullptr;
    if (max_dim < 2 || max_dim > BMF_MAX_DIM || max_vertices < 1 || max_vertices > kMaxTapeVertices ||
        max_indices < 3 || checkpoint_every < 1)
        return BMF_EINVAL;
    BMF_HIP(hipSetDevice(ctx->device));
    bmf_tape* t = new (std::nothrow) bmf_tape();
    if (!t) return BMF_EHIP;
    t->ctx = ctx;
    t->max_dim = max_dim;
    t->cap_v = max_vertices;
    t->cap_i = max_indices;
    t->ckpt_every = checkpoint_every;
    const int64_t n3 = (int64_t)max_dim * max_dim * max_dim;
    const bool ok = dalloc(&t->dens, n3) == hipSuccess && dalloc(&t->vid0, n3) == hipSuccess &&
                    dalloc(&t->order, max_vertices + (kPacket - 1) * std::min<int64_t>(max_vertices, kOrderCells)) ==
                        hipSuccess && dalloc(&t->rank, max_vertices) == hipSuccess &&
                    dalloc(&t->cell_n, kOrderCells) == hipSuccess &&
                    dalloc(&t->cell_base, kOrderCells) == hipSuccess &&
                    hipMemsetAsync(t->cell_n, 0, sizeof(uint32_t) * kOrderCells, ctx->stream) == hipSuccess &&
                    dalloc(&t->vedge, max_vertices) == hipSuccess && dalloc(&t->boundary, max_vertices) == hipSuccess &&
                    dalloc(&t->idx, max_indices) == hipSuccess &&
                    dalloc(&t->ring, (int64_t)kMaxRing * max_vertices) == hipSuccess &&
                    dalloc(&t->bscale, max_vertices) == hipSuccess &&
                    dalloc(&t->deg, max_vertices) == hipSuccess && dalloc(&t->mv, max_vertices) == hipSuccess &&
                    dalloc(&t->p4, max_vertices) == hipSuccess && dalloc(&t->q4, max_vertices) == hipSuccess &&
                    dalloc(&t->pos, 3 * max_vertices) == hipSuccess &&
                    dalloc(&t->g, max_vertices) == hipSuccess && dalloc(&t->g2, max_vertices) == hipSuccess &&
                    dalloc(&t->r4, max_vertices) == hipSuccess && dalloc(&t->taken, 1) == hipSuccess &&
                    host_alloc(&t->host, 1, &t->mhost) == hipSuccess && dalloc(&t->ext_sampler, 1) == hipSuccess &&
                    dalloc(&t->bb, 8) == hipSuccess && dalloc(&t->d2, max_vertices) == hipSuccess &&
                    dalloc(&t->loss, 1) == hipSuccess && dalloc(&t->nearest_tmp, max_vertices) == hipSuccess;
    bool evs = ok;
    for (int i = 0; i < 6 && evs; i++) evs = hipEventCreate(&t->ev[i]) == hipSuccess;
    SamplerDev ext{};
    ext.kind = BMF_SAMPLER_EXTERNAL;
    if (!evs || hipMemcpy(t->ext_sampler, &ext, sizeof ext, hipMemcpyHostToDevice) != hipSuccess) {
        bmf_tape_destroy(t);
        return BMF_EHIP;
    }
    // set-up of bmf_loss_nearest_noalloc: the scratch address on this device
    // (the device is current); a failure here only disables that entry point
    (void)scratch_acquire(ctx->device);
    *out = t;
    return BMF_OK;
}

void bmf_tape_destroy(bmf_tape* t) {
    if (!t) return;
    (void)hipSetDevice(t->ctx->device);
    (void)hipStreamSynchronize(t->ctx->stream);
    dfree(t->dens);
    dfree(t->vid0);
    dfree(t->order);
    dfree(t->rank);
    dfree(t->cell_n);
    dfree(t->cell_base);
    dfree(t->vedge);
    dfree(t->boundary);
    dfree(t->idx);
    dfree(t->ring);
    dfree(t->bscale);
    dfree(t->deg);
    dfree(t->mv);
    dfree(t->p4);
    dfree(t->q4);
    dfree(t->pos);
    dfree(t->g);
    dfree(t->g2);
    dfree(t->r4);
    for (int i = 0; i < 6; i++)
        if (t->ev[i]) (void)hipEventDestroy(t->ev[i]);
    dfree(t->taken);
    dfree(t->ext_sampler);
    if (t->host) (void)hipHostFree(t->host);
    dfree(t->ckpt);
    dfree(t->bb);
    dfree(t->d2);
    dfree(t->loss);
    dfree(t->nearest_tmp);
    free_nn(t);
    delete t;
}

int bmf_forward_diff(bmf_ctx* c, const bmf_chunk_desc* d, const float* densities, bmf_tape* t) {
    if (!c || !d || !t || t->ctx != c) return BMF_EINVAL;
    int rc = check_desc(*d);
    if (rc) return rc;
    if (d->dim > t->max_dim) return BMF_ECAPACITY;
    if (!densities && !c->sampler_set) return BMF_ESTATE;
    const int dim = d->dim;
    const int64_t n3 = (int64_t)dim * dim * dim;
    if (n3 > c->A.cap_samples) return BMF_ECAPACITY;
    BMF_HIP(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    BMF_HIP(hipStreamSynchronize(s));
    t->valid = false;
    t->timed[0] = false;
    BMF_HIP(hipEventRecord(t->ev[0], s));
    c->have_extract = false;
    c->results_valid = false;
    c->queued_n = -1;  // as after an extraction
    Arenas A = c->A;
    A.ext_base = 0;
    if (densities) {  // this call's sampler, the context's own is not touched
        A.sampler = t->ext_sampler;
        A.ext = densities;
        A.csg_list = nullptr;
    }
    A.mesh_mode = BMF_MESH_TRIANGLES;  // the adjoint is defined on the triangle path
    A.quad_tris = 0;
    A.smoothing_follows = 0;  // the tape smooths its own copy: every output position is written by emit
    A.normals = 0;
    // extraction with every octave evaluated (densities exact everywhere),
    // no smoothing: the tape smooths its own copy
    hipError_t e = launch_plan(A, 1, 0, 1, s, d);
    if (e == hipSuccess)
        e = launch_sample(A, 1, sample_blocks_of(n3),
                          0, densities ? (int)BMF_SAMPLER_EXTERNAL : (int)c->h_sampler.kind,
                          !densities && c->h_sampler.noise_dims == 2, s);
    if (e == hipSuccess) e = launch_count(A, word_blocks(dim), 0, s);
    if (e == hipSuccess) e = launch_scan(A, 1, 1, s);
    if (e == hipSuccess) e = launch_emit(A, 1, word_blocks(dim), s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return BMF_EHIP;
    const bmf_chunk_result r = c->h_results[0];
    if (c->h_ctr->error) return BMF_EHIP;
    if (r.status != BMF_OK) return r.status;
    if (r.vertex_count > t->cap_v || r.index_count > t->cap_i) return BMF_ECAPACITY;
    t->dim = dim;
    t->K = d->iters;
    t->bp = d->boundary_processing;
    t->V = r.vertex_count;
    t->T = r.index_count / 3;
    t->contains_mesh = r.contains_mesh;
    const int64_t slots = t->K / t->ckpt_every + 1;
    if (slots > t->ckpt_slots) {
        dfree(t->ckpt);
        t->ckpt_slots = 0;  // a failed reallocation leaves no slots, so the next forward retries it
        BMF_HIP(dalloc(&t->ckpt, slots * t->cap_v));
        t->ckpt_slots = slots;
    }
    const int V = t->V, T = t->T;
    const bool smooth = t->K > 0 && T > 0;  // per-cell triangle bases and masks exist for chunks with K > 0
    {
        const int64_t most = std::max<int64_t>(n3, std::max<int64_t>(3 * (int64_t)T, V));
        const unsigned blocks = (unsigned)std::min<int64_t>((most + kThreads - 1) / kThreads, 4096);
        hipLaunchKernelGGL(k_tape_take, dim3(blocks), dim3(kThreads), 0, s, A.dens, A.vedge + r.vertex_offset,
                           A.boundary + r.vertex_offset, A.idx + r.index_offset, A.pos + 3 * r.vertex_offset, n3, V,
                           3 * (int64_t)T, dim, t->dens, t->vedge, t->boundary, t->idx, t->p4, t->ckpt,
                           smooth ? nullptr : t->pos, t->vid0, t->cell_n, t->rank, t->taken,
                           &t->mhost->err);
        BMF_HIP(hipGetLastError());
    }
    if (V > 0) {
        hipLaunchKernelGGL(k_order_cells, dim3(blocks_for(kOrderCells)), dim3(kThreads), 0, s, t->cell_n, t->cell_base,
                           t->taken, t->order);
        hipLaunchKernelGGL(k_order, dim3(blocks_for(V)), dim3(kThreads), 0, s, t->vedge, V, dim, t->cell_base, t->rank,
                           t->taken, &t->mhost->places, t->order);
        BMF_HIP(hipGetLastError());
        if (smooth) {
            hipLaunchKernelGGL(k_tape_adj, dim3(step_blocks(V)), dim3(kStepThreads), 0, s, t->vedge, t->boundary,
                               A.cell_tb, A.cell_mask, t->idx, dim, V, T, t->bp, (int)t->cap_v, t->ring, t->deg, t->mv,
                               t->bscale, &t->mhost->err);
            BMF_HIP(hipGetLastError());
            rc = smooth_steps(t, t->p4, t->q4, t->K, s, t->pos, 0);
            if (rc) return rc;
        } else {
            BMF_HIP(hipMemsetAsync(t->deg, 0, V, s));
            BMF_HIP(hipMemsetAsync(t->mv, 0, V, s));
            for (int64_t q = 1; q < slots; q++)
                BMF_HIP(hipMemcpyAsync(t->ckpt + q * t->cap_v, t->p4, sizeof(float4) * V, hipMemcpyDeviceToDevice, s));
        }
    }
    BMF_HIP(hipEventRecord(t->ev[1], s));
    BMF_HIP(hipStreamSynchronize(s));
    if (V > 0 && t->host->err) return BMF_EHIP;
    t->places = t->host->places;
    t->valid = true;
    t->timed[0] = true;
    return BMF_OK;
}

int bmf_tape_get(bmf_tape* t, bmf_tape_info* info) {
    if (!t || !info) return BMF_EINVAL;
    if (!t->valid) return BMF_ESTATE;
    info->dim = t->dim;
    info->iters = t->K;
    info->checkpoint_every = t->ckpt_every;
    info->vertex_count = t->V;
    info->index_count = 3 * t->T;
    info->contains_mesh = t->contains_mesh;
    info->positions = t->pos;
    info->indices = t->idx;
    info->boundary = t->boundary;
    info->densities = t->dens;
    return BMF_OK;
}

int bmf_tape_positions(bmf_tape* t, int32_t iteration, float* out) {
    if (!t || !out) return BMF_EINVAL;
    if (!t->valid) return BMF_ESTATE;
    if (iteration < 0 || iteration > t->K) return BMF_EINVAL;
    if (t->V == 0) return BMF_OK;
    hipStream_t s = t->ctx->stream;
    BMF_HIP(hipSetDevice(t->ctx->device));
    const int64_t slot = iteration / t->ckpt_every;
    BMF_HIP(hipMemcpyAsync(t->q4, t->ckpt + slot * t->cap_v, sizeof(float4) * t->V, hipMemcpyDeviceToDevice, s));
    const int rest = t->T > 0 ? iteration - (int)(slot * t->ckpt_every) : 0;
    int rc = smooth_steps(t, t->q4, t->r4, rest, s, out);
    if (rc) return rc;
    BMF_HIP(hipStreamSynchronize(s));
    return BMF_OK;
}

int bmf_loss_nearest(bmf_tape* t, const float* targets, int64_t n, float* dldp, int32_t* nearest, float* loss) {
    if (!t || !targets || n < 1 || n > (int64_t)0x7FFFFFFF || !dldp) return BMF_EINVAL;
    if (!t->valid) return BMF_ESTATE;
    BMF_HIP(hipSetDevice(t->ctx->device));
    hipStream_t s = t->ctx->stream;
    int rc = reserve_nn(t, n);
    if (rc) return rc;
    t->nn_n = 0;
    t->timed[1] = false;
    BMF_HIP(hipEventRecord(t->ev[2], s));
    rc = nn_build(targets, n, t->bb, tape_nn(t), s);
    if (rc) return rc;
    t->nn_n = n;
    if (t->V == 0) {
        BMF_HIP(hipStreamSynchronize(s));
        if (loss) *loss = 0.0f;
        return BMF_OK;
    }
    rc = nn_query(t, tape_nn(t), n, dldp, nearest, &t->mhost->loss, s);
    if (rc) return rc;
    BMF_HIP(hipEventRecord(t->ev[3], s));
    BMF_HIP(hipStreamSynchronize(s));
    if (loss) *loss = (float)t->host->loss;
    t->timed[1] = true;
    return BMF_OK;
}

int bmf_tape_set_targets(bmf_tape* t, const float* targets, int64_t n) {
    if (!t || !targets || n < 1 || n > (int64_t)0x7FFFFFFF) return BMF_EINVAL;
    BMF_HIP(hipSetDevice(t->ctx->device));
    hipStream_t s = t->ctx->stream;
    int rc = reserve_nn(t, n);
    if (rc) return rc;
    t->nn_n = 0;
    rc = nn_build(targets, n, t->bb, tape_nn(t), s);
    if (rc) return rc;
    BMF_HIP(hipStreamSynchronize(s));
    t->nn_n = n;
    return BMF_OK;
}

int bmf_tape_loss_nearest(bmf_tape* t, float* dldp, int32_t* nearest, float* loss) {
    if (!t || !dldp) return BMF_EINVAL;
    if (!t->valid || t->nn_n < 1) return BMF_ESTATE;
    BMF_HIP(hipSetDevice(t->ctx->device));
    hipStream_t s = t->ctx->stream;
    if (t->V == 0) {
        if (loss) *loss = 0.0f;
        return BMF_OK;
    }
    t->timed[1] = false;
    BMF_HIP(hipEventRecord(t->ev[2], s));
    int rc = nn_query(t, tape_nn(t), t->nn_n, dldp, nearest, &t->mhost->loss, s);
    if (rc) return rc;
    BMF_HIP(hipEventRecord(t->ev[3], s));
    BMF_HIP(hipStreamSynchronize(s));
    if (loss) *loss = (float)t->host->loss;
    t->timed[1] = true;
    return BMF_OK;
}

int bmf_loss_nearest_noalloc(bmf_tape* t, const float* targets, int64_t n, float* dldp, int32_t* nearest,
                             double* loss) {
    if (!t || !targets || n < 1 || !dldp) return BMF_EINVAL;
    if (n > BMF_NOALLOC_MAX_TARGETS) return BMF_ECAPACITY;
    if (!t->valid) return BMF_ESTATE;
    void* base = scratch_on(t->ctx->device);
    if (!base) return BMF_EHIP;  // the address lookup at bmf_tape_create failed
    BMF_HIP(hipSetDevice(t->ctx->device));
    hipStream_t s = t->ctx->stream;
    const NNBuffers b = scratch_nn(base);
    // the radix sort's temporary storage for n pairs must fit its share (a
    // size query: nothing is launched or allocated)
    size_t need = 0;
    {
        hipcub::DoubleBuffer<uint32_t> kb(b.keys[0], b.keys[1]);
        hipcub::DoubleBuffer<int32_t> vb(b.vals[0], b.vals[1]);
        BMF_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, need, kb, vb, (int)n, 0, 30, s));
    }
    if (need > b.cub_bytes) return BMF_ECAPACITY;
    int rc = nn_build(targets, n, t->bb, b, s);
    if (rc) return rc;
    if (t->V == 0) {
        if (loss) hipLaunchKernelGGL(k_store_f64, dim3(1), dim3(1), 0, s, loss, 0.0);
        BMF_HIP(hipGetLastError());
        return BMF_OK;
    }
    return nn_query(t, b, n, dldp, nearest, loss ? loss : t->loss, s);
}

int bmf_backward_diff(bmf_tape* t, const float* dldp, float* dldd) {
    if (!t || !dldd || (!dldp && t->V > 0)) return BMF_EINVAL;
    if (!t->valid) return BMF_ESTATE;
    BMF_HIP(hipSetDevice(t->ctx->device));
    hipStream_t s = t->ctx->stream;
    const int64_t n3 = (int64_t)t->dim * t->dim * t->dim;
    if (t->V == 0) {
        BMF_HIP(hipMemsetAsync(dldd, 0, sizeof(float) * n3, s));
        BMF_HIP(hipStreamSynchronize(s));
        return BMF_OK;
    }
    t->timed[2] = false;
    BMF_HIP(hipEventRecord(t->ev[4], s));
    const bool smooth = t->K > 0 && t->T > 0;
    hipLaunchKernelGGL(k_bwd_init, dim3(blocks_for(t->V)), dim3(kThreads), 0, s, dldp, t->V, t->mv, t->bscale,
                       (int)smooth, t->g);
    float4* cur = t->g;
    float4* nxt = t->g2;
    if (smooth)
        for (int m = t->K - 1; m >= 0; m--) {
            hipLaunchKernelGGL(k_bwd_step, dim3(step_blocks(t->V)), dim3(kStepThreads), 0, s, t->ring, (int)t->cap_v,
                               t->deg, t->mv, t->bscale, cur, t->V, (int)(m == 0), nxt);
            std::swap(cur, nxt);
        }
    hipLaunchKernelGGL(k_bwd_place, dim3(blocks_for(n3)), dim3(kThreads), 0, s, t->dens, t->vid0, cur, t->dim, dldd);
    BMF_HIP(hipGetLastError());
    BMF_HIP(hipEventRecord(t->ev[5], s));
    BMF_HIP(hipStreamSynchronize(s));
    t->timed[2] = true;
    return BMF_OK;
}

int bmf_tape_timing(bmf_tape* t, float* ms) {
    if (!t || !ms) return BMF_EINVAL;
    BMF_HIP(hipSetDevice(t->ctx->device));
    for (int k = 0; k < 3; k++) {
        ms[k] = -1.0f;
        if (t->timed[k]) BMF_HIP(hipEventElapsedTime(&ms[k], t->ev[2 * k], t->ev[2 * k + 1]));
    }
    return BMF_OK;
}

}  // extern "C"
