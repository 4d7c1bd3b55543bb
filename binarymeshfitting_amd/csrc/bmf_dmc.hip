// Quad mode of the extraction path (BMF_MESH_QUADS): dual marching cubes
// over the reference's polygon table (Tables.hpp:96-354) with mass-point or
// QEF vertex placement (qef_simd.h:392-579), quads around the interior
// sign-changing edges, and MeshProcessor<4>/<3> smoothing over per-vertex
// rings.
//
// Per batch (after sample and count, which in this mode count per item the
// polygons of its cells and the quads of its interior sign-changing edges, and
// leave every edge endpoint's density exact):
//   (k_scan)       item bases, arena offsets
//   k_dmc_vertices vertex positions; per surface cell its first vertex id
//                  and mask (cell_tb / cell_mask arenas); for the chunks that
//                  smooth, each vertex's ring (the primitives around it in
//                  ascending id, the reference's order), from the quad ids of
//                  its polygon's edges
//   k_dmc_quads    quad (or two-triangle) indices
//   K x (k_dual_n, k_primal_ring)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bmf_device_tables.h"
#include "bmf_internal.h"
#include "bmf_rows.h"
#include "bmf_words.h"
#include "samplers.h"

namespace bmf {

namespace {

// Per block: polygon count of each mask, and for each mask and local edge
// the polygon holding it (nibbles, 0xF = none).
struct DmcTables {
    uint8_t np[256];
    uint64_t pe[256];
};

__device__ void load_dmc_tables(DmcTables& t) {
    for (int m = threadIdx.x; m < 256; m += blockDim.x) {
        const uint64_t row = c_dmc_table[m];
        const int n = (int)(row >> 60);
        uint64_t pe = ~0ull;
        int p = 0, any = 0;
        for (int s = 0; s < n; s++) {
            const int e = (int)((row >> (4 * s)) & 15ull);
            if (e == 15) {
                p++;
                any = 0;
                continue;
            }
            pe = (pe & ~(15ull << (4 * e))) | ((uint64_t)p << (4 * e));
            any = 1;
        }
        t.np[m] = (uint8_t)(p + any);
        t.pe[m] = pe;
    }
}

// ------------------------------------------------------------------------
// CSG gradient and QEF (FP32, the CPU oracle's operation sequence)
// ------------------------------------------------------------------------
// Gradient of the winning primitive of the max-union (first index on ties),
// zero on the floor.
// The primitives are the chunk's culled list (sphere ids, then box ids, in
// order) when there is one: the others never exceed the floor in the chunk.
__device__ void csg_gradient(const SamplerDev& S, const uint16_t* list, int ns, int nb, float x, float y, float z,
                             float g[3]) {
    float best = kCsgFloor;
    g[0] = g[1] = g[2] = 0.0f;
    if (!list) {
        ns = S.n_spheres;
        nb = S.n_boxes;
    }
    for (int k = 0; k < ns; k++) {
        const float* sp = S.spheres + 4 * (list ? list[k] : k);
        const float dx = x - sp[0], dy = y - sp[1], dz = z - sp[2];
        const float l = sqrtf((dx * dx + dy * dy) + dz * dz);
        const float v = sp[3] - l;
        if (v > best) {
            best = v;
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;
            g[0] = -dx * inv;
            g[1] = -dy * inv;
            g[2] = -dz * inv;
        }
    }
    for (int k = 0; k < nb; k++) {
        const float* b = S.boxes + 6 * (list ? list[ns + k] : k);
        const float px = x - b[0], py = y - b[1], pz = z - b[2];
        const float qx = fabsf(px) - b[3], qy = fabsf(py) - b[4], qz = fabsf(pz) - b[5];
        const float mx = fmaxf(qx, 0.0f), my = fmaxf(qy, 0.0f), mz = fmaxf(qz, 0.0f);
        const float outside = sqrtf((mx * mx + my * my) + mz * mz);
        const float inside = fminf(fmaxf(qx, fmaxf(qy, qz)), 0.0f);
        const float v = -(outside + inside);
        if (v > best) {
            best = v;
            const float sx = px < 0.0f ? -1.0f : 1.0f, sy = py < 0.0f ? -1.0f : 1.0f, sz = pz < 0.0f ? -1.0f : 1.0f;
            if (outside > 0.0f) {
                const float inv = 1.0f / outside;
                g[0] = -mx * sx * inv;
                g[1] = -my * sy * inv;
                g[2] = -mz * sz * inv;
            } else {
                g[0] = g[1] = g[2] = 0.0f;
                if (qx >= qy && qx >= qz) g[0] = -sx;
                else if (qy >= qz) g[1] = -sy;
                else g[2] = -sz;
            }
        }
    }
}

// Gradient of one primitive, as cull_csg writes it.
__device__ __forceinline__ void primitive_gradient(bool sphere, float4 b0, float4 b1, float x, float y, float z,
                                                   float g[3]) {
    g[0] = g[1] = g[2] = 0.0f;
    const float px = x - b0.x, py = y - b0.y, pz = z - b0.z;
    if (sphere) {
        const float l = sqrtf((px * px + py * py) + pz * pz);
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
        g[0] = -px * inv;
        g[1] = -py * inv;
        g[2] = -pz * inv;
        return;
    }
    const float qx = fabsf(px) - b0.w, qy = fabsf(py) - b1.x, qz = fabsf(pz) - b1.y;
    const float mx = fmaxf(qx, 0.0f), my = fmaxf(qy, 0.0f), mz = fmaxf(qz, 0.0f);
    const float outside = sqrtf((mx * mx + my * my) + mz * mz);
    const float sx = px < 0.0f ? -1.0f : 1.0f, sy = py < 0.0f ? -1.0f : 1.0f, sz = pz < 0.0f ? -1.0f : 1.0f;
    if (outside > 0.0f) {
        const float inv = 1.0f / outside;
        g[0] = -mx * sx * inv;
        g[1] = -my * sy * inv;
        g[2] = -mz * sz * inv;
    } else if (qx >= qy && qx >= qz) {
        g[0] = -sx;
    } else if (qy >= qz) {
        g[1] = -sy;
    } else {
        g[2] = -sz;
    }
}

// The same with the item's primitives in LDS (cull_csg's layout): the loop
// finds the winning primitive (first index on ties), whose gradient is then
// formed once, with the same operations as above.
__device__ void csg_gradient_lds(const float4* s_csg, int ns, int nb, float x, float y, float z, float g[3]) {
    float best = kCsgFloor;
    int win = -1;
    for (int k = 0; k < ns; k++) {
        const float4 sp = s_csg[2 * k];
        const float dx = x - sp.x, dy = y - sp.y, dz = z - sp.z;
        const float l = sqrtf((dx * dx + dy * dy) + dz * dz);
        const float v = sp.w - l;
        if (v > best) {
            best = v;
            win = k;
        }
    }
    for (int k = ns; k < ns + nb; k++) {
        const float4 b0 = s_csg[2 * k], b1 = s_csg[2 * k + 1];
        const float px = x - b0.x, py = y - b0.y, pz = z - b0.z;
        const float qx = fabsf(px) - b0.w, qy = fabsf(py) - b1.x, qz = fabsf(pz) - b1.y;
        const float mx = fmaxf(qx, 0.0f), my = fmaxf(qy, 0.0f), mz = fmaxf(qz, 0.0f);
        const float outside = sqrtf((mx * mx + my * my) + mz * mz);
        const float inside = fminf(fmaxf(qx, fmaxf(qy, qz)), 0.0f);
        const float v = -(outside + inside);
        if (v > best) {
            best = v;
            win = k;
        }
    }
    g[0] = g[1] = g[2] = 0.0f;
    if (win < 0) return;  // the floor
    primitive_gradient(win < ns, s_csg[2 * win], s_csg[2 * win + 1], x, y, z, g);
}

// The same over the item's ids (cull_csg_ids).
__device__ void csg_gradient_ids(const SamplerDev& S, const uint16_t* ids, int ns, int nb, float x, float y, float z,
                                 float g[3]) {
    const int b0 = (ns + 3) & ~3;
    float best = kCsgFloor;
    int win = -1;
    for (int k = 0; k < ns; k += 4) {
        float p[4][4];
        csg_fetch<4>(S.spheres, ids, k, ns, p);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (k + u >= ns) break;
            const float dx = x - p[u][0], dy = y - p[u][1], dz = z - p[u][2];
            const float l = sqrtf((dx * dx + dy * dy) + dz * dz);
            const float v = p[u][3] - l;
            win = v > best ? k + u : win;
            best = v > best ? v : best;
        }
    }
    for (int k = 0; k < nb; k += 4) {
        float p[4][6];
        csg_fetch<6>(S.boxes, ids + b0, k, nb, p);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (k + u >= nb) break;
            const float px = x - p[u][0], py = y - p[u][1], pz = z - p[u][2];
            const float qx = fabsf(px) - p[u][3], qy = fabsf(py) - p[u][4], qz = fabsf(pz) - p[u][5];
            const float mx = fmaxf(qx, 0.0f), my = fmaxf(qy, 0.0f), mz = fmaxf(qz, 0.0f);
            const float outside = sqrtf((mx * mx + my * my) + mz * mz);
            const float inside = fminf(fmaxf(qx, fmaxf(qy, qz)), 0.0f);
            const float v = -(outside + inside);
            win = v > best ? b0 + k + u : win;
            best = v > best ? v : best;
        }
    }
    g[0] = g[1] = g[2] = 0.0f;
    if (win < 0) return;  // the floor
    const bool sphere = win < ns;
    const uint32_t id = ids[win];
    const float* q = sphere ? S.spheres + 4 * id : S.boxes + 6 * id;
    const float4 a = make_float4(q[0], q[1], q[2], q[3]);
    const float4 b = sphere ? a : make_float4(q[4], q[5], 0.0f, 0.0f);
    primitive_gradient(sphere, a, b, x, y, z, g);
}

// QEF of `count` (point, unit normal) pairs (qef_simd.h:392-579): normal
// equations about the mass point, 5 Jacobi sweeps over the pairs (0,1),
// (0,2), (1,2) with an exact 1/sqrt Givens cosine, 1/sigma kept when
// min(|sigma|, |1/sigma|) >= tol, residual with the uncentred ATb.
// The sums are accumulated one pair at a time in pair order (qef_add), then
// solved (qef_finish); no pair is kept.
struct QefSums {
    float ata[3][3];
    float atb[3];
    float pa[4];
};

__device__ __forceinline__ void qef_add(QefSums& q, float px, float py, float pz, const float nn[3]) {
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) q.ata[r][c] = q.ata[r][c] + nn[r] * nn[c];
    const float d = (px * nn[0] + py * nn[1]) + pz * nn[2];
#pragma unroll
    for (int r = 0; r < 3; r++) q.atb[r] = q.atb[r] + d * nn[r];
    q.pa[0] = q.pa[0] + px;
    q.pa[1] = q.pa[1] + py;
    q.pa[2] = q.pa[2] + pz;
    q.pa[3] = q.pa[3] + 1.0f;
}

__device__ float qef_finish(const QefSums& q, int count, float tol, float out[3]) {
    if (count < 2 || count > 12) {
        out[0] = out[1] = out[2] = 0.0f;
        return 0.0f;
    }
    const float(&ata)[3][3] = q.ata;
    const float(&atb)[3] = q.atb;
    const float(&pa)[4] = q.pa;
    const float mp[3] = {pa[0] / pa[3], pa[1] / pa[3], pa[2] / pa[3]};
    float rhs[3];
#pragma unroll
    for (int c = 0; c < 3; c++) rhs[c] = atb[c] - ((mp[0] * ata[0][c] + mp[1] * ata[1][c]) + mp[2] * ata[2][c]);
    float a[3][3], v[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) a[r][c] = ata[r][c];
    for (int sw = 0; sw < 5; sw++)
#pragma unroll
        for (int q = 0; q < 3; q++) {
            const int i0 = q == 2 ? 1 : 0, i1 = q == 0 ? 1 : 2;
            if (a[i0][i1] == 0.0f) continue;
            const float pp = a[i0][i0], pq = a[i0][i1], qq = a[i1][i1];
            const float tau = (qq - pp) / (pq * 2.0f);
            const float stt = sqrtf(tau * tau + 1.0f);
            const float tn = 1.0f / (tau >= 0.0f ? tau + stt : tau - stt);
            const float cs = 1.0f / sqrtf(1.0f + tn * tn);
            const float sn = tn * cs;
            const float cc = cs * cs, ss = sn * sn, mx = ((2.0f * cs) * sn) * pq;
            a[i0][i0] = (cc * pp - mx) + ss * qq;
            a[i1][i1] = (ss * pp + mx) + cc * qq;
            const int ua_r = 0, ua_c = 3 - i1, va_r = 1 - i0, va_c = 2;
            const float u3 = a[ua_r][ua_c], v3 = a[va_r][va_c];
#pragma unroll
            for (int r = 0; r < 3; r++) {
                const float vu = v[r][i0], vv = v[r][i1];
                v[r][i0] = cs * vu - sn * vv;
                v[r][i1] = sn * vu + cs * vv;
            }
            a[ua_r][ua_c] = cs * u3 - sn * v3;
            a[va_r][va_c] = sn * u3 + cs * v3;
            a[i0][i1] = 0.0f;
        }
    const float sig[3] = {a[0][0], a[1][1], a[2][2]};
    float inv[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float r1 = 1.0f / sig[k];
        const float ax = sig[k] < 0.0f ? -sig[k] : sig[k], ar = r1 < 0.0f ? -r1 : r1;
        inv[k] = ((ax < ar ? ax : ar) >= tol) ? r1 : 0.0f;
    }
    float pinv[3][3];
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++)
            pinv[r][c] = (v[c][0] * inv[0] * v[r][0] + v[c][1] * inv[1] * v[r][1]) + v[c][2] * inv[2] * v[r][2];
    float x[3];
#pragma unroll
    for (int c = 0; c < 3; c++) x[c] = (rhs[0] * pinv[0][c] + rhs[1] * pinv[1][c]) + rhs[2] * pinv[2][c];
    float e[3];
#pragma unroll
    for (int c = 0; c < 3; c++) e[c] = atb[c] - ((x[0] * ata[0][c] + x[1] * ata[1][c]) + x[2] * ata[2][c]);
    const float err = (e[0] * e[0] + e[1] * e[1]) + e[2] * e[2];
    out[0] = x[0] + mp[0];
    out[1] = x[1] + mp[1];
    out[2] = x[2] + mp[2];
    return err;
}

// Local edge -> offset of its origin sample from the cell origin and axis
// (DMCChunk.cpp:543-565).
__constant__ int8_t c_le[12][4] = {{0, 0, 0, 0}, {0, 0, 1, 0}, {0, 1, 0, 0}, {0, 1, 1, 0},
                                   {0, 0, 0, 1}, {0, 0, 1, 1}, {1, 0, 0, 1}, {1, 0, 1, 1},
                                   {0, 0, 0, 2}, {0, 1, 0, 2}, {1, 0, 0, 2}, {1, 1, 0, 2}};

}  // namespace

// ------------------------------------------------------------------------
// Rings.  Quad ids follow the (x, y, z, axis) order of their lattice edges:
// an item's base plus its interior sign-changing edges before the edge's
// sample (all axes) and before its axis at that sample.  A vertex (a polygon of a cell) lies on the quads of its
// polygon's interior edges, so visiting the cell's local edges in the order of
// their (dx, dy, dz, axis) offsets lists its quads in ascending id.  With
// quads written as triangles (a, b, c), (c, d, a) (MeshProcessor.cpp:74-91) a
// quad's first and last ring cells (corners a and c) are on both triangles,
// the others on one, chosen by the quad's winding.
// ------------------------------------------------------------------------
// For sample row d = 2 dx + dy of the cell at the item's sample `pos`: the
// quad id of the first edge at sample (dx, dy, 0) of the cell, and flag byte
// d: the interior edge bits of axes 0-2 there (bits 0-2) and one sample on
// (bits 3-5), the labels of the two (6, 7).  From the item's windows.
__device__ __forceinline__ void quad_row_at(const ItemWindows& s, const WindowGeom& g, int dim, int pos, int d,
                                            uint32_t& pre, uint32_t& fl) {
    const int dx = d >> 1, dy = d & 1;
    pre = window_edge(s, g, dim, pos, dx, dy, 0, 0);
    const int p = pos + dy * dim + (dx ? g.off : 0);
    uint32_t f = label_pair(s.lab + (dx ? g.n0 : 0), p) << 6;
#pragma unroll
    for (int dz = 0; dz < 2; dz++) {
        const int w = ((p + dz) >> 6) + (dx ? g.n0 : 0), b = (p + dz) & 63;
        f |= (((uint32_t)(s.ex[w] >> b) & 1u) | (((uint32_t)(s.ey[w] >> b) & 1u) << 1) |
              (((uint32_t)(s.ez[w] >> b) & 1u) << 2))
             << (3 * dz);
    }
    fl |= f << (8 * d);
}

// Writes vertex g's ring (polygon p of a cell with polygon-of-edge nibbles
// pe) from the four rows' quad prefixes and flags; returns its size.
__device__ __forceinline__ uint32_t dmc_ring(const Arenas& A, const uint32_t (&pre)[4], uint32_t fl, uint64_t pe,
                                             uint32_t p, int64_t g, bool tris) {
    uint32_t n = 0;
    bool over = false;
    const int64_t cap = A.cap_vertices;
    auto put = [&](uint32_t pid) {
        if (n < (uint32_t)kRingSlots) A.ring[(int64_t)n * cap + g] = pid;
        else over = true;
        n++;
    };
#pragma unroll
    for (int i = 0; i < 12; i++) {
        // local edges in (dx, dy, dz, axis) order: 0, 4, 8, 1, 5, 2, 9, 3, 6, 10, 7, 11
        constexpr int kOrder[12] = {0, 4, 8, 1, 5, 2, 9, 3, 6, 10, 7, 11};
        const int le = kOrder[i];
        if ((uint32_t)((pe >> (4 * le)) & 15ull) != p) continue;
        // c_le[le]: the origin offset and axis (a = le >> 2, the other two
        // offsets bits 1 and 0 of le)
        const int a = le >> 2, b1 = (le >> 1) & 1, b0 = le & 1;
        const int dx = a == 0 ? 0 : b1, dy = a == 0 ? b1 : (a == 2 ? b0 : 0), dz = a == 2 ? 0 : b0;
        const int d = 2 * dx + dy;
        const uint32_t f = fl >> (8 * d);
        const uint32_t cb = dz ? f >> 3 : f;  // interior edge bits of the edge's sample
        if (!((cb >> a) & 1u)) continue;      // on the chunk's boundary: no quad
        const uint32_t qid = pre[d] + (dz ? (f & 1u) + ((f >> 1) & 1u) + ((f >> 2) & 1u) : 0u) +
                             (a >= 1 ? cb & 1u : 0u) + (a == 2 ? (cb >> 1) & 1u : 0u);
        if (!tris) {
            put(qid);
            continue;
        }
        // ring cell r = 3 - (le & 3) of the edge (c_ring order); the quad is
        // (v0, v1, v3, v2), with v1 and v2 swapped when the solid end of the
        // edge is not on the side its axis winds toward
        const int r = 3 - (le & 3);
        const uint32_t prim = 2u * qid;
        if (r == 0 || r == 3) {
            put(prim);
            put(prim + 1u);
        } else {
            const bool solid_origin = ((f >> (6 + dz)) & 1u) == 0u;
            const bool flip = solid_origin != (a != 1);
            put(prim + ((r == 1) == flip ? 1u : 0u));
        }
    }
    if (over) raise_error(A, 10);
    return n;
}

// CSG primitives of one item's edge points: those of the chunk's list that
// can reach the union's surface there (csg_reach).  Up to kItemCsg are staged
// themselves, more as their ids (kCsgIds; more than those: the chunk's list).  A
// larger stage gains a tenth on items of 17 to 64 primitives (98 us instead of
// 108 for 45^3 cells with 90) and costs 118 instead of 115 on thinly spread
// ones (64 chunks of 64^3 cells, 300 primitives).
constexpr int kItemCsg = 16;

struct DmcWave {
    ItemWindows win;
    uint32_t verts[4 * 64];       // a round's vertices: sample | polygon << 10 | corner mask << 12
    float4 csg[2 * kItemCsg];     // cull_csg's layout
    uint16_t ids[kCsgIds] __attribute__((aligned(8)));  // cull_csg_ids'
};

// ------------------------------------------------------------------------
// vertices: one per polygon of each active cell, a wave per item.  Rounds of
// 64 cells: each cell's first vertex id and mask, its polygons compacted into
// a dense list, then a lane per vertex places it (mass point or QEF) and, for
// chunks that smooth, writes its ring.  QEF placement is bound by the
// normals (a pass over the primitives per edge point): the item's own list
// keeps the few that can win.  64 chunks of 64^3 cells, 300 primitives,
// 326,882 vertices: 106 us, with the plane's rows and the chunk's list 169.
// ------------------------------------------------------------------------
__device__ void place_vertex(const Arenas& A, const ChunkMeta& M, const SamplerDev& S, const uint16_t* csg,
                             const float4* s_csg, const uint16_t* ids, int ns, int nb, int x, int y, int z, int p,
                             uint32_t mask, bool qef, float out[3], float& err) {
    const int dim = M.dim;
    const float* __restrict__ D = A.dens + M.dens_off;
    const uint64_t row = c_dmc_table[mask];
    const int nn = (int)(row >> 60);
    // skip to polygon p
    int s = 0;
    for (int q = 0; q < p && s < nn; s++)
        if (((row >> (4 * s)) & 15ull) == 15ull) q++;
    QefSums qs = {{{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, {0, 0, 0}, {0, 0, 0, 0}};
    // the polygon's edges (at most 7; an eighth is an error), their endpoint
    // densities loaded together before any is used; local edge e runs along
    // axis e >> 2 from the corner whose other two offsets are bits 1 and 0
    // of e (the rows of c_le)
    int ee[7], k = 0;
    float d0[7], d1[7];
    const int64_t own = ((int64_t)x * dim + y) * dim + z;
#pragma unroll
    for (int j = 0; j < 7; j++) {
        const int e = s + j < nn ? (int)((row >> (4 * (s + j))) & 15ull) : 15;
        const bool valid = e != 15 && k == j;  // the polygon ends at its first separator
        ee[j] = valid ? e : 0;
        const int a = ee[j] >> 2, b1 = (ee[j] >> 1) & 1, b0 = ee[j] & 1;
        const int ox = a == 0 ? 0 : b1, oy = a == 0 ? b1 : (a == 2 ? b0 : 0), oz = a == 2 ? 0 : b0;
        const int64_t i0 = (((int64_t)(x + ox) * dim) + (y + oy)) * dim + (z + oz);
        const int64_t i1 = i0 + (a == 0 ? (int64_t)dim * dim : (a == 1 ? (int64_t)dim : 1));
        d0[j] = D[valid ? i0 : own];
        d1[j] = D[valid ? i1 : own];
        k += valid ? 1 : 0;
    }
    {
        const int e8 = s + 7 < nn ? (int)((row >> (4 * (s + 7))) & 15ull) : 15;
        if (k == 7 && e8 != 15) k = 8;  // more than 7 edges: reported below
    }
    float ax = 0.0f, ay = 0.0f, az = 0.0f;
#pragma unroll
    for (int j = 0; j < 7; j++) {
        if (j >= k) break;
        const int e = ee[j];
        const int x0 = x + c_le[e][0], y0 = y + c_le[e][1], z0 = z + c_le[e][2], a = c_le[e][3];
        const int x1 = x0 + (a == 0), y1 = y0 + (a == 1), z1 = z0 + (a == 2);
        const float s0 = d0[j], s1 = d1[j];
        // DMCChunk::calculate_isovertex (DMCChunk.cpp:657-674)
        const float mu = (0.0f - s0) / (s1 - s0);
        const float dx = (float)x1 - (float)x0, dy = (float)y1 - (float)y0, dz = (float)z1 - (float)z0;
        const float qx = dx * mu + (float)x0, qy = dy * mu + (float)y0, qz = dz * mu + (float)z0;
        ax = ax + qx;
        ay = ay + qy;
        az = az + qz;
        if (qef) {
            // unit normal of the CSG field at the point (world coordinates)
            const float wx = qx * M.delta + M.opos[0], wy = qy * M.delta + M.opos[1], wz = qz * M.delta + M.opos[2];
            float g[3];
            if (s_csg) csg_gradient_lds(s_csg, ns, nb, wx, wy, wz, g);
            else if (ids) csg_gradient_ids(S, ids, ns, nb, wx, wy, wz, g);
            else csg_gradient(S, csg, ns, nb, wx, wy, wz, g);
            const float len = sqrtf((g[0] * g[0] + g[1] * g[1]) + g[2] * g[2]);
            float nrm[3];
            for (int c = 0; c < 3; c++) nrm[c] = len > 0.0f ? g[c] / len : 0.0f;
            qef_add(qs, qx, qy, qz, nrm);
        }
    }
    err = 0.0f;
    if (k == 0 || k > 7) {
        raise_error(A, 8);
        out[0] = out[1] = out[2] = 0.0f;
        return;
    }
    if (qef) {
        err = qef_finish(qs, k, A.qef_tol, out);
    } else {
        const float fk = (float)k;
        out[0] = ax / fk;
        out[1] = ay / fk;
        out[2] = az / fk;
    }
}

// Few items with QEF placement: kVertexParts waves stage each of them and take
// every kVertexParts-th of its rounds of cells, so that a detailed object in
// one chunk is not left to as many waves as it has items.  Stage times with four
// waves and with one: 33^3 cells with 60 primitives on the surface 119 and
// 260 us, 100^3 with 400 208 and 321, 8 chunks of 45^3 with 90 58 and 104.
// kVertexFew: a wave per SIMD without.  Twice as many still gain where the lists
// are long (128^3 cells with 250: 137 and 223) and lose where they are short and
// staging is most of the work (64 chunks of 64^3, 300 spread thinly: 119 and 115).
constexpr int kVertexParts = 4;
constexpr int kVertexFew = 1024;
__global__ void __launch_bounds__(kRowThreads) k_dmc_vertices(Arenas A, int n) {
    __shared__ DmcTables s_t;
    __shared__ DmcWave s_wave[kWordWaves];
    load_dmc_tables(s_t);
    publish(A, n);
    __syncthreads();
    const SamplerDev* __restrict__ S = A.sampler;
    const int wave = uniform_int(threadIdx.x >> 6), lane = lane_id();
    DmcWave& W = s_wave[wave];
    ItemWindows& s = W.win;
    const bool qef = A.placement == BMF_PLACE_QEF && S->kind == BMF_SAMPLER_CSG;
    const bool tris = A.quad_tris != 0;
    const int total = read_const(&A.ctr->n_work);
    const int parts = qef && total <= kVertexFew ? kVertexParts : 1;
    for (int wu = blockIdx.x * kWordWaves + wave; wu < total * parts; wu += gridDim.x * kWordWaves) {
        const int wi = wu / parts, part = wu - wi * parts;
        const int2 im = read_const(A.work + wi);
        const int chunk = uniform_int(im.x), w0 = uniform_int(im.y) * kItemWords;
        const ChunkMeta M = read_chunk(A.meta, chunk);
        if (M.status != BMF_OK || M.V == 0) continue;
        const int dim = M.dim, d2 = dim * dim;
        const float rd = 1.0f / (float)dim, rd2 = 1.0f / (float)d2;
        const WindowGeom g = stage_windows(A, M, w0, s);
        const int nc = push_bits(s.ac[lane >> 2], s.list);
        wave_sync();
        if (nc <= 64 * part) continue;
        const uint16_t* csg = A.csg_list ? A.csg_list + (int64_t)chunk * A.csg_stride : nullptr;
        int ns = M.csg_ns, nb = M.csg_nb;
        bool staged = false, listed = false;
        if (qef && csg) {
            float lo[3], hi[3];
            sample_box(M, 64 * w0, kItemSamples, 1, lo, hi);  // the cells' far corners too
            const float reach = csg_reach(*S, M.delta, lo, hi);
            int is, ib;
            staged = cull_csg(*S, csg, ns, nb, lo, hi, reach, W.csg, kItemCsg, is, ib);
            if (!staged) listed = cull_csg_ids(*S, csg, ns, nb, lo, hi, reach, W.ids, is, ib);
            if (staged || listed) {
                ns = is;
                nb = ib;
            }
            wave_sync();
        }
        const int64_t vo = M.v_off;
        const uint32_t Vc = (uint32_t)M.V;
        const bool smooth = (M.iters > 0 || A.normals) && M.T > 0;  // the chunk runs the smoothing kernels
        uint32_t vb = A.item_c[M.item_slot + im.y];
        for (int e0 = 0; e0 < nc; e0 += 64) {
            // ---- the round's cells ----
            int pos = 0;
            uint32_t mask = 0, np = 0;
            if (e0 + lane < nc) {
                pos = s.list[e0 + lane];
                mask = window_mask(s, g, dim, pos);
                np = s_t.np[mask];
            }
            uint32_t nv;
            const uint32_t pre = wave_prefix<3>(np, nv);
            if (parts > 1 && (e0 >> 6) % parts != part) {  // another wave's
                vb += nv;
                continue;
            }
            if (np) {
                const int64_t ci = M.dens_off + 64ll * w0 + pos;
                A.cell_tb[ci] = vb + pre;
                A.cell_mask[ci] = (uint8_t)mask;
                for (uint32_t p = 0; p < np; p++) W.verts[pre + p] = (uint32_t)pos | (p << 10) | (mask << 12);
            }
            wave_sync();
            // ---- their vertices ----
            for (uint32_t e = (uint32_t)lane; e < nv; e += 64u) {
                const uint32_t item = W.verts[e];
                const int cpos = (int)(item & 1023u), p = (int)((item >> 10) & 3u);
                const uint32_t cmask = item >> 12, v = vb + e;
                if (v >= Vc) {
                    raise_error(A, 8);
                    continue;
                }
                const uint32_t i = 64u * (uint32_t)w0 + (uint32_t)cpos;
                const int x = (int)udiv24(i, (uint32_t)d2, rd2), r = (int)i - x * d2;
                const int y = (int)udiv24((uint32_t)r, (uint32_t)dim, rd), z = r - y * dim;
                A.boundary[vo + v] =
                    (uint8_t)(x == 0 || y == 0 || z == 0 || x + 1 == dim - 1 || y + 1 == dim - 1 || z + 1 == dim - 1);
                A.vedge[vo + v] = (uint32_t)x | ((uint32_t)y << 8) | ((uint32_t)z << 16) | ((uint32_t)p << 24);
                float o[3], err;
                place_vertex(A, M, *S, csg, staged ? W.csg : nullptr, listed ? W.ids : nullptr, ns, nb, x, y, z, p, cmask, qef,
                             o, err);
                float* P = A.pos + (vo + v) * 3;
                P[0] = o[0];
                P[1] = o[1];
                P[2] = o[2];
                if (smooth) A.pos4[vo + v] = make_float4(o[0], o[1], o[2], 0.0f);
                if (A.qef_err) A.qef_err[vo + v] = err;
                if (A.normals) {  // a vertex with no polygon keeps the zero normal
                    A.nrm4[vo + v] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    float* O = A.nrm + (vo + v) * 3;
                    O[0] = 0.0f;
                    O[1] = 0.0f;
                    O[2] = 0.0f;
                }
                if (smooth) {
                    uint32_t pre4[4], fl = 0u;
#pragma unroll
                    for (int d = 0; d < 4; d++) quad_row_at(s, g, dim, cpos, d, pre4[d], fl);
                    A.ring_n[vo + v] = dmc_ring(A, pre4, fl, s_t.pe[cmask], (uint32_t)p, vo + v, tris);
                }
            }
            vb += nv;
            wave_sync();  // the round's vertices are read
        }
    }
}

// ------------------------------------------------------------------------
// quads around the interior sign-changing edges, a wave per item, a lane per
// sample that owns some (the batch above: 18 us, with a wave per row 71)
// ------------------------------------------------------------------------
__global__ void __launch_bounds__(kRowThreads) k_dmc_quads(Arenas A) {
    __shared__ DmcTables s_t;
    __shared__ ItemWindows s_win[kWordWaves];
    load_dmc_tables(s_t);
    __syncthreads();
    const int wave = uniform_int(threadIdx.x >> 6), lane = lane_id();
    ItemWindows& s = s_win[wave];
    const bool tris = A.quad_tris != 0;
    const int total = read_const(&A.ctr->n_work);
    for (int wi = blockIdx.x * kWordWaves + wave; wi < total; wi += gridDim.x * kWordWaves) {
        const ItemRef R = work_ref(A, wi);
        const ChunkMeta& M = R.M;
        if (M.status != BMF_OK || M.T == 0) continue;
        const int dim = M.dim, d2 = dim * dim;
        const float rd = 1.0f / (float)dim, rd2 = 1.0f / (float)d2;
        (void)stage_windows(A, M, R.w0, s);
        const int k4 = lane >> 2;
        const int nq = push_bits(s.ex[k4] | s.ey[k4] | s.ez[k4], s.list);
        wave_sync();
        const uint32_t Vc = (uint32_t)M.V, Tc = (uint32_t)M.T;
        uint32_t* __restrict__ I = A.idx + M.i_off;
        for (int e = lane; e < nq; e += 64) {
            const int pos = s.list[e], w = pos >> 6;
            const uint64_t bit = 1ull << (pos & 63), lt = bit - 1ull;
            const uint64_t ex = s.ex[w], ey = s.ey[w], ez = s.ez[w];
            const bool f[3] = {(ex & bit) != 0ull, (ey & bit) != 0ull, (ez & bit) != 0ull};
            uint32_t qid = s.pre[w] + (uint32_t)(__popcll(ex & lt) + __popcll(ey & lt) + __popcll(ez & lt));
            const bool solid_origin = (s.lab[w] & bit) == 0ull;
            const uint32_t i = 64u * (uint32_t)R.w0 + (uint32_t)pos;
            const int x = (int)udiv24(i, (uint32_t)d2, rd2), r0 = (int)i - x * d2;
            const int y = (int)udiv24((uint32_t)r0, (uint32_t)dim, rd), z = r0 - y * dim;
            // the rings of the sample's three edges are cells of the 2 x 2 x 2
            // block (x-1 .. x, y-1 .. y, z-1 .. z): its eight first-vertex ids
            // and masks load together (a cell outside the chunk reads cell 0;
            // only the rings of interior edges, all inside, use them)
            uint32_t tb8[8], mk8[8];
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const int cx = x - 1 + (c >> 2), cy = y - 1 + ((c >> 1) & 1), cz = z - 1 + (c & 1);
                const bool in = cx >= 0 && cy >= 0 && cz >= 0 && cx <= dim - 2 && cy <= dim - 2 && cz <= dim - 2;
                const int64_t ci = M.dens_off + (in ? ((int64_t)cx * dim + cy) * dim + cz : 0);
                tb8[c] = A.cell_tb[ci];
                mk8[c] = A.cell_mask[ci];
            }
#pragma unroll
            for (int a = 0; a < 3; a++) {
                if (!f[a]) continue;
                uint32_t v[4];
                bool ok = true;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    // ring cell r of axis a: offsets (c_ring) -1 / 0 per axis -> block cell
                    const int c = ((c_ring[a][r][0] + 1) << 2) | ((c_ring[a][r][1] + 1) << 1) | (c_ring[a][r][2] + 1);
                    const uint32_t le = (uint32_t)c_ring[a][r][3];
                    const uint32_t pi = (uint32_t)((s_t.pe[mk8[c]] >> (4 * le)) & 15ull);
                    v[r] = tb8[c] + pi;
                    if (pi == 15u || v[r] >= Vc) ok = false;
                }
                const uint32_t prim = tris ? 2u * qid : qid;
                if (!ok || prim + (tris ? 1u : 0u) >= Tc) {
                    raise_error(A, 9);
                    qid++;
                    continue;
                }
                // cyclic c0 c1 c3 c2: right-hand normal along -x, +y, -z;
                // flipped so that it points to the solid end of the edge
                const bool toward_origin = a != 1;
                uint32_t o[4] = {v[0], v[1], v[3], v[2]};
                if (solid_origin != toward_origin) {
                    o[1] = v[2];
                    o[3] = v[1];
                }
                if (tris) {  // MeshProcessor::flush_to_tris (MeshProcessor.cpp:74-91)
                    uint32_t* t = I + 3ll * prim;
                    t[0] = o[0];
                    t[1] = o[1];
                    t[2] = o[2];
                    t[3] = o[2];
                    t[4] = o[3];
                    t[5] = o[0];
                } else {
                    uint32_t* t = I + 4ll * prim;
                    t[0] = o[0];
                    t[1] = o[1];
                    t[2] = o[2];
                    t[3] = o[3];
                }
                qid++;
            }
        }
        wave_sync();  // the windows and the list are read
    }
}

// ------------------------------------------------------------------------
// smoothing over the rings (chunks of the smoothing list, XCD-grouped tiles
// as in the triangle path)
// ------------------------------------------------------------------------
// Dual step (MeshProcessor.cpp:130-236) for N-gons (N = 3 or 4, one per
// chunk): ((0 + p0) + p1 ...) / N, the corner ids and then the corners
// loaded together.  Tiles come from the per-frame tile map.
__global__ void __launch_bounds__(kSmoothThreads) k_dual_n(Arenas A, int m) {
    for (SmoothTiles tiles(A.smooth_tmap, A.cap_ttiles, A.ctr->xcd_ttiles); tiles.next();) {
        const SmoothTile& M = tiles.t;
        const int iters = M.iters, N = M.ipp, T = M.T;
        const uint32_t V = (uint32_t)M.V;
        const int64_t i_off = M.i_off, v_off = M.v_off;
        if (iters <= m) continue;
        const int64_t t = (int64_t)M.tile * kSmoothThreads + threadIdx.x;
        if (t >= T) continue;
        const uint32_t* __restrict__ I = A.idx + i_off + (int64_t)N * t;
        const float4* __restrict__ P = A.pos4 + v_off;
        const uint32_t u0 = I[0], u1 = I[1], u2 = I[2], u3 = N == 4 ? I[3] : u0;
        if (u0 >= V || u1 >= V || u2 >= V || u3 >= V) {
            raise_error(A, 11);
            continue;
        }
        const float4 a = P[u0], b = P[u1], c = P[u2], d = P[u3];
        float cx = 0.0f, cy = 0.0f, cz = 0.0f;
        cx = cx + a.x;
        cy = cy + a.y;
        cz = cz + a.z;
        cx = cx + b.x;
        cy = cy + b.y;
        cz = cz + b.z;
        cx = cx + c.x;
        cy = cy + c.y;
        cz = cz + c.z;
        if (N == 4) {
            cx = cx + d.x;
            cy = cy + d.y;
            cz = cz + d.z;
        }
        const float fn = (float)N;
        A.cen4[M.t_off + t] = make_float4(cx / fn, cy / fn, cz / fn, 0.0f);
    }
}

// Primal step (MeshProcessor.cpp:238-306) over the ring (ascending primitive
// id): the centroids summed from +0 in ring order, eight ring slots and then
// their centroids loaded per round.
constexpr int kRingRoundN = 8;
__global__ void __launch_bounds__(kSmoothThreads) k_primal_ring(Arenas A, int m) {
    const int64_t cap = A.cap_vertices;
    for (SmoothTiles tiles(A.smooth_vmap, A.cap_vtiles, A.ctr->xcd_vtiles); tiles.next();) {
        const SmoothTile& M = tiles.t;
        const int K = M.iters, V = M.V, bp = M.bp;
        const int64_t v_off = M.v_off;
        if (K <= m) continue;
        const int64_t v = (int64_t)M.tile * kSmoothThreads + threadIdx.x;
        if (v >= V) continue;
        const int64_t g = v_off + v;
        const uint8_t bnd = A.boundary[g];
        const int n = (int)min(A.ring_n[g], (uint32_t)kRingSlots);
        if ((!bp && bnd) || n == 0) continue;
        const float4* __restrict__ C = A.cen4 + M.t_off;
        float sx = 0.0f, sy = 0.0f, sz = 0.0f;
        for (int i0 = 0; i0 < n; i0 += kRingRoundN) {
            uint32_t id[kRingRoundN];
#pragma unroll
            for (int k = 0; k < kRingRoundN; k++) id[k] = A.ring[(int64_t)(i0 + k < n ? i0 + k : i0) * cap + g];
            float4 q[kRingRoundN];
#pragma unroll
            for (int k = 0; k < kRingRoundN; k++) q[k] = C[id[k]];
#pragma unroll
            for (int k = 0; k < kRingRoundN; k++) {
                const bool ok = i0 + k < n;
                sx = ok ? sx + q[k].x : sx;
                sy = ok ? sy + q[k].y : sy;
                sz = ok ? sz + q[k].z : sz;
            }
        }
        const float fc = (float)n;
        const float px = sx / fc, py = sy / fc, pz = sz / fc;
        A.pos4[g] = make_float4(px, py, pz, 0.0f);
        if (m == K - 1) {
            float* __restrict__ P = A.pos + g * 3;
            P[0] = px;
            P[1] = py;
            P[2] = pz;
        }
    }
}

// With vertex normals (the smooth_normals branch of MeshProcessor<N>,
// MeshProcessor.cpp:159-216, 271-287): every chunk of the list runs max(K, 1)
// steps.  Step m's face normal while m == 0, m < max_norms (min(K/2 - 3, 10))
// or m < 3 is, for a triangle, -cross(normalize(p0 - p1), normalize(p0 - p2));
// for a quad, n1 = cross(normalize(p0 - p1), normalize(p0 - p2)) and
// n2 = cross(normalize(p2 - p3), normalize(p2 - p0)) with the reference's NaN
// fallbacks (a NaN n1.x takes n2, or (0, 1, 0) when n2 is NaN too; a NaN
// n2.x then takes n1), and -normalize((n1 + n2) * 0.5) (:187-205); later
// steps take the sum of the corners' normals.  normalize(v) is
// v / sqrt((x*x + y*y) + z*z).
__device__ __forceinline__ float3 unit_cross(float ux, float uy, float uz, float wx, float wy, float wz) {
    const float lu = sqrtf((ux * ux + uy * uy) + uz * uz), lw = sqrtf((wx * wx + wy * wy) + wz * wz);
    ux = ux / lu;
    uy = uy / lu;
    uz = uz / lu;
    wx = wx / lw;
    wy = wy / lw;
    wz = wz / lw;
    return make_float3(uy * wz - wy * uz, uz * wx - wz * ux, ux * wy - wx * uy);
}

__global__ void __launch_bounds__(kSmoothThreads) k_dual_n_nrm(Arenas A, int m) {
    for (SmoothTiles tiles(A.smooth_tmap, A.cap_ttiles, A.ctr->xcd_ttiles); tiles.next();) {
        const SmoothTile& M = tiles.t;
        const int K = M.iters, N = M.ipp, T = M.T;
        const uint32_t V = (uint32_t)M.V;
        const int64_t i_off = M.i_off, v_off = M.v_off;
        if (max(K, 1) <= m) continue;
        const int64_t t = (int64_t)M.tile * kSmoothThreads + threadIdx.x;
        if (t >= T) continue;
        // N = 3 or 4, one per chunk: the corner ids, then the corners, load
        // together (a triangle's fourth repeats its first)
        const uint32_t* __restrict__ I = A.idx + i_off + (int64_t)N * t;
        const float4* __restrict__ P = A.pos4 + v_off;
        const float4* __restrict__ NV = A.nrm4 + v_off;
        const uint32_t u[4] = {I[0], I[1], I[2], I[N == 4 ? 3 : 0]};
        if (u[0] >= V || u[1] >= V || u[2] >= V || u[3] >= V) {
            raise_error(A, 11);
            continue;
        }
        const float4 q[4] = {P[u[0]], P[u[1]], P[u[2]], P[u[3]]};
        float cx = 0.0f, cy = 0.0f, cz = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            if (c == 3 && N == 3) break;
            cx = cx + q[c].x;
            cy = cy + q[c].y;
            cz = cz + q[c].z;
        }
        const float fN = (float)N;
        const int64_t tt = M.t_off + t;
        A.cen4[tt] = make_float4(cx / fN, cy / fN, cz / fN, 0.0f);
        const int max_norms = min(K / 2 - 3, 10);
        float4 fn;
        if (m == 0 || m < max_norms || m < 3) {
            if (N == 3) {
                const float3 f = unit_cross(q[0].x - q[1].x, q[0].y - q[1].y, q[0].z - q[1].z, q[0].x - q[2].x,
                                            q[0].y - q[2].y, q[0].z - q[2].z);
                fn = make_float4(-f.x, -f.y, -f.z, 0.0f);
            } else {
                float3 n1 = unit_cross(q[0].x - q[1].x, q[0].y - q[1].y, q[0].z - q[1].z, q[0].x - q[2].x,
                                       q[0].y - q[2].y, q[0].z - q[2].z);
                float3 n2 = unit_cross(q[2].x - q[3].x, q[2].y - q[3].y, q[2].z - q[3].z, q[2].x - q[0].x,
                                       q[2].y - q[0].y, q[2].z - q[0].z);
                if (__builtin_isnan(n1.x)) {
                    n1 = n2;
                    if (__builtin_isnan(n1.x)) n1 = make_float3(0.0f, 1.0f, 0.0f);
                }
                if (__builtin_isnan(n2.x)) n2 = n1;
                const float hx = (n1.x + n2.x) * 0.5f, hy = (n1.y + n2.y) * 0.5f, hz = (n1.z + n2.z) * 0.5f;
                const float lh = sqrtf((hx * hx + hy * hy) + hz * hz);
                fn = make_float4(-(hx / lh), -(hy / lh), -(hz / lh), 0.0f);
            }
        } else {
            float sx = 0.0f, sy = 0.0f, sz = 0.0f;
            const float4 nc[4] = {NV[u[0]], NV[u[1]], NV[u[2]], NV[u[3]]};
#pragma unroll
            for (int c = 0; c < 4; c++) {
                if (c == 3 && N == 3) break;
                sx = sx + nc[c].x;
                sy = sy + nc[c].y;
                sz = sz + nc[c].z;
            }
            fn = make_float4(sx, sy, sz, 0.0f);
        }
        A.fn4[tt] = fn;
    }
}

// Primal step with normals over the sorted ring: the ring's centroids and
// face normals summed from +0 in ascending primitive order and divided by
// the ring size; the normal is normalised when m == 3 or (m == 0 and K <= 3)
// and kept when its y is not 0, for every vertex with a ring; positions of
// boundary vertices stay unless boundary processing (K > 0 only); the last
// step writes the unit normal (0 for a zero normal).
__global__ void __launch_bounds__(kSmoothThreads) k_primal_ring_nrm(Arenas A, int m) {
    const int64_t cap = A.cap_vertices;
    for (SmoothTiles tiles(A.smooth_vmap, A.cap_vtiles, A.ctr->xcd_vtiles); tiles.next();) {
        const SmoothTile& M = tiles.t;
        const int K = M.iters, V = M.V, bp = M.bp;
        const int64_t v_off = M.v_off;
        const int steps = max(K, 1);
        if (steps <= m) continue;
        const int64_t v = (int64_t)M.tile * kSmoothThreads + threadIdx.x;
        if (v >= V) continue;
        const int64_t g = v_off + v;
        const uint8_t bnd = A.boundary[g];
        const int n = (int)min(A.ring_n[g], (uint32_t)kRingSlots);
        float4 nv = A.nrm4[g];
        const float4* __restrict__ C = A.cen4 + M.t_off;
        const float4* __restrict__ F = A.fn4 + M.t_off;
        if (n > 0) {
            float sx = 0.0f, sy = 0.0f, sz = 0.0f, nx = 0.0f, ny = 0.0f, nz = 0.0f;
            for (int i0 = 0; i0 < n; i0 += kRingRoundN) {
                uint32_t id[kRingRoundN];
#pragma unroll
                for (int k = 0; k < kRingRoundN; k++) id[k] = A.ring[(int64_t)(i0 + k < n ? i0 + k : i0) * cap + g];
                float4 q[kRingRoundN], f[kRingRoundN];
#pragma unroll
                for (int k = 0; k < kRingRoundN; k++) {
                    q[k] = C[id[k]];
                    f[k] = F[id[k]];
                }
#pragma unroll
                for (int k = 0; k < kRingRoundN; k++) {
                    const bool ok = i0 + k < n;
                    sx = ok ? sx + q[k].x : sx;
                    sy = ok ? sy + q[k].y : sy;
                    sz = ok ? sz + q[k].z : sz;
                    nx = ok ? nx + f[k].x : nx;
                    ny = ok ? ny + f[k].y : ny;
                    nz = ok ? nz + f[k].z : nz;
                }
            }
            const float fc = (float)n;
            float ax = nx / fc, ay = ny / fc, az = nz / fc;
            const bool unit = m != steps - 1 && (m == 3 || (m == 0 && K <= 3));
            if (unit) {
                const float l = sqrtf((ax * ax + ay * ay) + az * az);
                ax = ax / l;
                ay = ay / l;
                az = az / l;
            }
            if (ay != 0.0f) {
                nv = make_float4(ax, ay, az, 0.0f);
                A.nrm4[g] = nv;
            }
            if (K > 0 && (bp || !bnd)) {
                const float px = sx / fc, py = sy / fc, pz = sz / fc;
                A.pos4[g] = make_float4(px, py, pz, 0.0f);
                if (m == K - 1) {
                    float* __restrict__ P = A.pos + g * 3;
                    P[0] = px;
                    P[1] = py;
                    P[2] = pz;
                }
            }
        }
        if (m == steps - 1) {
            const float l = sqrtf((nv.x * nv.x + nv.y * nv.y) + nv.z * nv.z);
            float* __restrict__ O = A.nrm + g * 3;
            O[0] = l > 0.0f ? nv.x / l : 0.0f;
            O[1] = l > 0.0f ? nv.y / l : 0.0f;
            O[2] = l > 0.0f ? nv.z / l : 0.0f;
        }
    }
}

// ------------------------------------------------------------------------
// launch wrappers
// ------------------------------------------------------------------------

hipError_t launch_dmc_emit(const Arenas& A, int n, int blocks, hipStream_t s) {
    // the vertices, then the quads that index them
    // a grid sized to one chunk's items: four times that for their parts, as far as they go
    constexpr int kMost = kVertexParts * kVertexFew / kWordWaves;
    const int vblocks = A.placement == BMF_PLACE_QEF ? std::max(blocks, std::min(kVertexParts * blocks, kMost)) : blocks;
    hipLaunchKernelGGL(k_dmc_vertices, dim3(vblocks), dim3(kRowThreads), 0, s, A, n);
    hipLaunchKernelGGL(k_dmc_quads, dim3(blocks), dim3(kRowThreads), 0, s, A);
    return hipGetLastError();
}

hipError_t launch_dmc_smooth(const Arenas& A, int m, int blocks, hipStream_t s) {
    blocks = blocks < kXcds ? kXcds : blocks - blocks % kXcds;  // whole XCD groups
    if (A.normals) {
        hipLaunchKernelGGL(k_dual_n_nrm, dim3(blocks), dim3(kSmoothThreads), 0, s, A, m);
        hipLaunchKernelGGL(k_primal_ring_nrm, dim3(blocks), dim3(kSmoothThreads), 0, s, A, m);
    } else {
        hipLaunchKernelGGL(k_dual_n, dim3(blocks), dim3(kSmoothThreads), 0, s, A, m);
        hipLaunchKernelGGL(k_primal_ring, dim3(blocks), dim3(kSmoothThreads), 0, s, A, m);
    }
    return hipGetLastError();
}

}  // namespace bmf
