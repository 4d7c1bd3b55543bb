// HIP kernels of the chunk-extraction path (gfx950, wave64).
//
// Per batch:  plan -> sample -> count -> scan -> emit -> smooth
// (the per-chunk results are written by plan for culled or skipped chunks
// and by scan for sampled ones, and go to the host with the emission, so no
// launch and no copy follows the smoothing)
//
// Data layout in HBM (per sampled chunk, offsets from the plan kernel):
//   densities   FP32 [x][y][z]                    (DMCChunk density_block)
//   labels      flat bitmap over the sample index (x*dim + y)*dim + z,
//               u64 word i/64, bit i%64, set when the density is < 0;
//               one word per wave of 64 consecutive samples (one ballot)
//   edges       per label word: bits of its samples' sign-changing edges per
//               axis and of its active cells; word_pre its edges' prefix
//               within its item (16 words), item_e / item_c the items' edge
//               and cell counts, then exclusive bases after the scan
//   cell_tb/    per surface cell (same index as the density): first triangle
//   cell_mask   id and corner mask, written only for chunks that smooth
//   output      positions float3, boundary u8, vertex edge code u32,
//               chunk-local triangle indices
// Cell masks and the reference's u32 label words are never materialised on
// the hot path: the word kernels rebuild them from the bitmap with shifts.
#include <hip/hip_runtime.h>

#include "bmf_device_tables.h"
#include "bmf_internal.h"
#include "bmf_rows.h"
#include "bmf_words.h"
#include "samplers.h"

namespace bmf {

// ------------------------------------------------------------------------
// plan: geometry, culling, arena offsets, counters
// ------------------------------------------------------------------------
constexpr int kPlanThreads = 1024;
// Up to this many descriptors every block of the plan forms all the sums
// itself (one launch); larger batches take three passes, whose extra launches
// cost more than they save below it.
constexpr int kPlanShared = 2 * kPlanThreads;
constexpr int kPlanSlice = 64;  // records that a block then writes

// The host-visible result of chunk j from its final record: written by
// k_plan for the chunks it culls or skips and by k_scan for the sampled ones
// (every field is final there: later kernels report errors through the
// counters, not the chunk records).
__device__ __forceinline__ void write_result(const Arenas& A, int j, const ChunkMeta& M) {
    bmf_chunk_result r;
    const bool ok = M.status == BMF_OK;
    r.vertex_offset = ok ? M.v_off : 0;
    r.index_offset = ok ? M.i_off : 0;
    r.vertex_count = ok ? M.V : 0;
    r.index_count = ok ? M.ipp * M.T : 0;
    r.contains_mesh = M.contains_mesh;
    r.status = M.status;
    r.sampled = M.state == kStateSampled;
    r.delta = M.delta;
    r.overlap_pos[0] = M.opos[0];
    r.overlap_pos[1] = M.opos[1];
    r.overlap_pos[2] = M.opos[2];
    A.results[j] = r;
}

// a[i] of a register array by unrolled selects (a runtime index into a
// register array would place it in scratch memory)
template <int N>
__device__ __forceinline__ int64_t pick(const int64_t (&a)[N], int i) {
    int64_t r = 0;
#pragma unroll
    for (int k = 0; k < N; k++) r = k == i ? a[k] : r;
    return r;
}

// ---- how far k_blocks expands a chunk's noise (see there) ----
// No Hessian of the noise has a larger norm, at any position and for any
// gradients: proven by tests/test_noise_bounds_proof.py (the largest that a
// search finds is 48.21).
constexpr float kNoiseHess = 50.0f;
// FP32 error of two noise values and of a gradient over a block, per unit of
// amplitude: a constant for the kernels' arithmetic (about 76.8 * 4 t^3 g.x
// half-ulps of t, under 1e-5 each) and a part proportional to the lattice
// coordinates, whose rounding (under 8e-7 of their sum) moves the noise by
// its gradient (at most 7.1), twice, and the gradient by kNoiseHess.
constexpr float kNoiseSlack = 2e-4f, kNoiseCoordSlack = 4e-5f;
// Roundings of the sums, of the sign test and of the density from its sum,
// relative to the sum of the amplitudes (32 ulps).
constexpr float kSignSlack = 4e-6f;

constexpr int kExpandOctaves = 4;  // a quad of lanes takes an octave each

// The octaves to expand for samples at squared distance rr (in samples) from
// their centre: the k with the least E_k, which goes out as quad * r^2 + base.
__device__ __forceinline__ int expansion(const SamplerDev& S, float delta, float far, float rr, float& quad,
                                         float& base) {
    float q = 0.0f, b = 0.0f, best = S.reach[0];
    int k = 0;
    quad = 0.0f;
    base = best;
#pragma unroll
    for (int o = 0; o < kExpandOctaves; o++) {
        if (o >= S.octaves) break;
        const float f = S.fo[o] * delta;
        q += S.ao[o] * (0.505f * kNoiseHess) * (f * f);
        b += S.ao[o] * (kNoiseSlack + kNoiseCoordSlack * far * fabsf(S.fo[o]));
        const float e = __builtin_fmaf(q, rr, b) + S.reach[o + 1];
        if (e < best) {
            best = e;
            k = o + 1;
            quad = q;
            base = b + S.reach[o + 1];
        }
    }
    base += kSignSlack * S.reach[0];
    return k;
}


// The plan of a terrain chunk's blocks and sub-blocks: a level that would
// decide hardly more than the one before is left out.
__device__ __forceinline__ BlockPlan plan_blocks(const SamplerDev& S, const ChunkMeta& M) {
    BlockPlan p{0, 0, 0.0f, (1.0f + kSignSlack) * S.reach[0], 0.0f, 0.0f};
    if (!S.expand_ok) return p;
    const float ext = (float)(M.dim - 1) * M.delta;
    float far = 0.0f, q, e;
#pragma unroll
    for (int a = 0; a < 3; a++) far += fmaxf(fabsf(M.opos[a]), fabsf(M.opos[a] + ext));
    const int k = expansion(S, M.delta, far, 3.75f, q, e);
    if (__builtin_fmaf(q, 3.75f, e) < 0.8f * p.base4) {
        p.k4 = k;
        p.quad4 = q;
        p.base4 = e;
    }
    p.k2 = expansion(S, M.delta, far, 0.75f, p.quad2, p.base2);
    if (!(__builtin_fmaf(p.quad2, 0.75f, p.base2) < 0.8f * __builtin_fmaf(p.quad4, 3.75f, p.base4))) p.k2 = 0;
    return p;
}

// Plan record of one descriptor: DMCChunk::label_grid geometry
// (DMCChunk.cpp:94-101) and analytic culling; `add` gets its contributions
// to the arena sums (samples, label words, word items, items of the sampler's
// own pre-pass: k_blocks' or k_columns'), each at most 2^24.
__device__ __forceinline__ ChunkMeta plan_record(const Arenas& A, const SamplerDev* __restrict__ S,
                                                 const bmf_chunk_desc& d, int allow_cull, uint32_t (&add)[4]) {
    ChunkMeta m;
    float t = d.overlap * 2.0f;
    t = 1.0f + t;
    t = d.size * t;
    m.delta = t / (float)(d.dim - 1);
    const float so = d.size * d.overlap;
    m.opos[0] = d.pos[0] - so;
    m.opos[1] = d.pos[1] - so;
    m.opos[2] = d.pos[2] - so;
    m.dim = d.dim;
    m.iters = d.iters;
    m.bp = d.boundary_processing;
    m.state = kStateSampled;
    if (allow_cull) {
        const float ylo = m.opos[1];
        const float yhi = (float)(d.dim - 1) * m.delta + m.opos[1];
        const int sign = band_sign(*S, ylo, yhi);
        if (sign) m.state = sign == 1 ? kStateAir : kStateSolid;
    }
    m.csg_ns = m.csg_nb = 0;  // k_csg_cull fills them
    const uint32_t ns = (uint32_t)d.dim * (uint32_t)d.dim * (uint32_t)d.dim;
    const bool sampled = m.state == kStateSampled;
    m.lab_words = sampled ? (ns + 63u) / 64u : 0;
    m.any_air = m.state == kStateAir;
    m.any_solid = m.state == kStateSolid;
    m.contains_mesh = 0;
    m.status = BMF_OK;
    m.V = 0;
    m.T = 0;
    m.ipp = (A.mesh_mode == BMF_MESH_QUADS && !A.quad_tris) ? 4 : 3;
    m.v_off = 0;
    m.i_off = 0;
    m.dens_off = 0;
    m.lab_off = 0;
    m.item_slot = 0;
    const uint32_t nb = ((uint32_t)d.dim + 3u) >> 2;
    add[0] = sampled ? ns : 0u;
    add[1] = (uint32_t)m.lab_words;
    add[2] = ((uint32_t)m.lab_words + kItemWords - 1) / kItemWords;
    add[3] = !sampled                                              ? 0u
             : S->kind == BMF_SAMPLER_TERRAIN                     ? (nb * nb * nb + kWaveBlocks - 1) / kWaveBlocks
             : S->kind == BMF_SAMPLER_NOISE && S->noise_dims == 2 ? ((uint32_t)d.dim * (uint32_t)d.dim + 63u) / 64u
                                                                  : 0u;
    return m;
}

__device__ __forceinline__ bool plan_overflow(const Arenas& A, const int64_t (&tot)[4]) {
    return tot[0] > A.cap_samples || tot[1] > A.cap_samples / 64 + A.cap_chunks;
}

// A record's final state, `at` the arena sums before it.
__device__ __forceinline__ void plan_finish(const Arenas& A, const SamplerDev* __restrict__ S, int j, ChunkMeta& m,
                                            const int64_t (&at)[4], bool overflow) {
    m.dens_off = at[0];
    m.lab_off = at[1];
    m.item_slot = at[2];
    A.block_prefix[j] = overflow ? 0 : at[3];
    m.blocks = BlockPlan{};
    if (m.state == kStateSampled) {
        if (S->kind == BMF_SAMPLER_TERRAIN) m.blocks = plan_blocks(*S, m);
        if (overflow) {
            m.state = kStateSkipped;
            m.status = BMF_ECAPACITY;
        }
    } else {
        // culled chunks: DMCChunk.cpp:159-162 on uniform labels
        m.contains_mesh = (m.state == kStateAir) && (m.dim % 32 != 0);
    }
    A.meta[j] = m;
    if (m.state != kStateSampled) write_result(A, j, m);  // final: k_scan skips it
}

// The batch counters from the totals: word items, overflow.
__device__ __forceinline__ void plan_counters(const Arenas& A, int n, const int64_t (&tot)[4], bool overflow,
                                              int reset_bumps) {
    A.block_prefix[n] = overflow ? 0 : tot[3];
    Counters* c = A.ctr;
    if (reset_bumps) {
        c->v_bump = 0;
        c->i_bump = 0;
        c->need_v = 0;
        c->need_i = 0;
        c->overflow = 0;
        c->error = 0;
        A.host_ctr->error = 0;
    }
    if (overflow) c->overflow = 1;
    c->total_items = overflow ? 0 : tot[2];
    c->n_smooth = 0;
    c->n_work = 0;
    for (int g = 0; g < kXcds; g++) c->xcd_vtiles[g] = c->xcd_ttiles[g] = 0;
    c->total_samples = tot[0];
}

// Batches of up to kPlanShared descriptors, one launch: every block forms the
// sums over all of them (two descriptors per thread at most, 32-bit wave
// scans) and writes the records of its own kPlanSlice.  One block that wrote
// every record took 14 us for 512 descriptors and 33 for 1,536 (a thread's
// records lie side by side, written and read again across the scan);
// this takes 6.7 and 9.9 (5.4 for one).  A single descriptor may come with the
// launch (`by_value`), which saves its copy to the arena.
__global__ void __launch_bounds__(kPlanThreads) k_plan(Arenas A, int n, int allow_cull, int reset_bumps,
                                                       bmf_chunk_desc one, int by_value) {
    __shared__ uint32_t s_w[4][kPlanThreads / 64];
    const SamplerDev* __restrict__ S = A.sampler;
    const int per = (n + kPlanThreads - 1) / kPlanThreads;  // 1 or 2
    const int j0 = threadIdx.x * per;
    uint32_t sum[4] = {0u, 0u, 0u, 0u};
    for (int i = 0; i < per; i++) {
        if (j0 + i >= n) break;
        uint32_t add[4];
        (void)plan_record(A, S, by_value ? one : A.descs[j0 + i], allow_cull, add);
#pragma unroll
        for (int q = 0; q < 4; q++) sum[q] += add[q];
    }
    int64_t excl[4], tot[4];
    block_scan32<4, kPlanThreads>(sum, excl, tot, s_w);
    const bool overflow = plan_overflow(A, tot);
    // the block's own records, formed again
    for (int i = 0; i < per; i++) {
        const int j = j0 + i;
        if (j >= n || j / kPlanSlice != (int)blockIdx.x) break;  // per divides kPlanSlice
        uint32_t add[4];
        ChunkMeta m = plan_record(A, S, by_value ? one : A.descs[j], allow_cull, add);
        plan_finish(A, S, j, m, excl, overflow);
#pragma unroll
        for (int q = 0; q < 4; q++) excl[q] += add[q];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) plan_counters(A, n, tot, overflow, reset_bumps);
}

// Larger batches, pass 1 of 3 (one descriptor per thread over many blocks):
// each block's totals.
__global__ void __launch_bounds__(kPlanThreads) k_plan_part(Arenas A, int n, int allow_cull) {
    __shared__ uint32_t s_w[4][kPlanThreads / 64];
    const int j = blockIdx.x * kPlanThreads + threadIdx.x;
    uint32_t add[4] = {0u, 0u, 0u, 0u};
    if (j < n) (void)plan_record(A, A.sampler, A.descs[j], allow_cull, add);
    int64_t excl[4], tot[4];
    block_scan32<4, kPlanThreads>(add, excl, tot, s_w);
    if (threadIdx.x < 4) A.plan_part[4 * blockIdx.x + threadIdx.x] = pick<4>(tot, (int)threadIdx.x);
}

// Pass 2 (one block, one thread per pass-1 block, at most kPlanThreads):
// block bases, batch totals, overflow flag, counters.  Bases go to
// plan_part[4 (nb + b) ...], the overflow flag after them.
__global__ void __launch_bounds__(kPlanThreads) k_plan_total(Arenas A, int n, int nb, int reset_bumps) {
    __shared__ int64_t s_w[4][kPlanThreads / 64 + 1];
    const int b = threadIdx.x;
    int64_t v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = b < nb ? A.plan_part[4 * b + q] : 0;
    int64_t excl[4], tot[4];
    block_scan<4, kPlanThreads>(v, excl, tot, s_w);
    const bool overflow = plan_overflow(A, tot);
    if (b < nb)
#pragma unroll
        for (int q = 0; q < 4; q++) A.plan_part[4 * (nb + b) + q] = excl[q];
    if (b == 0) {
        A.plan_part[8 * nb] = overflow;
        plan_counters(A, n, tot, overflow, reset_bumps);
    }
}

// Pass 3: the records with their offsets, the results of culled chunks.
__global__ void __launch_bounds__(kPlanThreads) k_plan_fix(Arenas A, int n, int nb, int allow_cull) {
    __shared__ uint32_t s_w[4][kPlanThreads / 64];
    const int j = blockIdx.x * kPlanThreads + threadIdx.x;
    uint32_t add[4] = {0u, 0u, 0u, 0u};
    ChunkMeta m{};
    if (j < n) m = plan_record(A, A.sampler, A.descs[j], allow_cull, add);
    int64_t at[4], tot[4];
    block_scan32<4, kPlanThreads>(add, at, tot, s_w);
    if (j >= n) return;
#pragma unroll
    for (int q = 0; q < 4; q++) at[q] += A.plan_part[4 * (nb + blockIdx.x) + q];
    plan_finish(A, A.sampler, j, m, at, A.plan_part[8 * nb] != 0);
}

// ------------------------------------------------------------------------
// CSG culling: per chunk, the primitives whose value can exceed the floor
// inside its sample box (spheres within r + |floor| of the box, boxes whose
// box grown by |floor| meets it; 0.5 and the slack of csg_reach cover FP32
// rounding), in
// their original order (sphere ids, then box ids).  Block per chunk; order
// kept by a ballot prefix per 256 primitives.
// ------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_csg_cull(Arenas A, int n) {
    __shared__ uint32_t s_wave[4];
    __shared__ uint32_t s_base;
    const SamplerDev* __restrict__ S = A.sampler;
    const int lane = lane_id(), wave = threadIdx.x >> 6;
    const uint64_t lt = lanemask_lt();
    for (int j = blockIdx.x; j < n; j += gridDim.x) {
        ChunkMeta& M = A.meta[j];
        const float lo[3] = {M.opos[0], M.opos[1], M.opos[2]};
        const float ext = (float)(M.dim - 1) * M.delta;
        float far = 0.0f;
        for (int a = 0; a < 3; a++) far = fmaxf(far, fmaxf(fabsf(lo[a]), fabsf(lo[a] + ext)));
        const float reach = -kCsgFloor + 0.5f + 4e-6f * far + S->csg_slack;
        uint16_t* L = A.csg_list + (int64_t)j * A.csg_stride;
        if (threadIdx.x == 0) s_base = 0;
        __syncthreads();
        for (int pass = 0; pass < 2; pass++) {
            const int np = pass == 0 ? S->n_spheres : S->n_boxes;
            for (int i0 = 0; i0 < np; i0 += 256) {
                const int i = i0 + (int)threadIdx.x;
                bool keep = false;
                if (i < np) {
                    if (pass == 0) {
                        const float* sp = S->spheres + 4 * i;
                        float dd = 0.0f;
                        for (int a = 0; a < 3; a++) {
                            const float t = fmaxf(fmaxf(lo[a] - sp[a], sp[a] - (lo[a] + ext)), 0.0f);
                            dd += t * t;
                        }
                        const float r = sp[3] + reach;
                        keep = dd < r * r;
                    } else {
                        const float* b = S->boxes + 6 * i;
                        keep = true;
                        for (int a = 0; a < 3; a++)
                            keep = keep && (b[a] - b[3 + a] - reach <= lo[a] + ext) && (b[a] + b[3 + a] + reach >= lo[a]);
                    }
                }
                const uint64_t bal = __ballot(keep);
                if (lane == 0) s_wave[wave] = (uint32_t)__popcll(bal);
                __syncthreads();
                uint32_t off = s_base;
                for (int w = 0; w < wave; w++) off += s_wave[w];
                if (keep) L[off + (uint32_t)__popcll(bal & lt)] = (uint16_t)i;
                __syncthreads();
                if (threadIdx.x == 0) s_base += s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
                __syncthreads();
            }
            if (threadIdx.x == 0) {
                if (pass == 0) M.csg_ns = (int32_t)s_base;
                else M.csg_nb = (int32_t)s_base - M.csg_ns;
            }
            __syncthreads();
        }
    }
}

// ------------------------------------------------------------------------
// sampling: the adaptive terrain through k_blocks and k_terrain, adaptive 3D
// noise fields through k_field, every other case through k_sample
// ------------------------------------------------------------------------
// A chunk's sample geometry as values (like TerrainTerms): read once per
// tile, so the loops below never reload them after their own stores.
struct ChunkGeom {
    float ox, oy, oz, delta;
};

__device__ __forceinline__ void sample_index(uint32_t i, uint32_t dim, uint32_t dim2, float rd, float rd2, uint32_t& x,
                                             uint32_t& y, uint32_t& z) {
    x = udiv24(i, dim2, rd2);
    const uint32_t rem = i - x * dim2;
    y = udiv24(rem, dim, rd);
    z = rem - y * dim;
}

// NoiseSampler.cpp:21-27: (float)i * scale + p, two roundings
__device__ __forceinline__ void sample_position(const ChunkGeom& G, uint32_t x, uint32_t y, uint32_t z, float& px,
                                                float& py, float& pz) {
    px = (float)x * G.delta + G.ox;
    py = (float)y * G.delta + G.oy;
    pz = (float)z * G.delta + G.oz;
}

__device__ __forceinline__ void sample_coords(const ChunkGeom& G, uint32_t i, uint32_t dim, uint32_t dim2, float rd,
                                              float rd2, float& px, float& py, float& pz) {
    uint32_t x, y, z;
    sample_index(i, dim, dim2, rd, rd2, x, y, z);
    sample_position(G, x, y, z, px, py, pz);
}

// ------------------------------------------------------------------------
// blocks (adaptive terrain): the sign of most samples from a few evaluations
// per 4 x 4 x 4 block of them.
//
// Simplex noise n is twice differentiable with |n| < 1 (the clamp never
// acts) and a Hessian of norm at most kNoiseHess, so at a sample s of a block
// with centre c
//   |n(f s) - (n(f c) + f grad n(f c) . (s - c))| <= kNoiseHess / 2 (f |s - c|)^2,
// and after k octaves expanded that way the sample's FP32 sum of all octaves
// lies within
//   E_k(r^2) = sum_{o<k} a_o (kNoiseHess / 2 (f_o r)^2 + slack_o) + reach[k]
// of the expansion (reach: the octaves not evaluated, as in decide_label;
// slack_o: FP32 errors of both noise values and the coordinates, see
// kNoiseSlack).  A sample whose expansion is further than that from the sum
// at which its density changes sign is decided.  Two levels: 4^3 blocks (one
// per lane), then the 2^3 sub-blocks that hold undecided samples, compacted;
// at each level the number of octaves with the least E_k.  k_terrain
// evaluates what is left, about a thirteenth of a chunk's samples.
//
// A quad of lanes shares a centre, an octave each, so that a wave's chain is
// one octave long.  Bound by VALU issue: 512 chunks of 64^3 cells, 64 sampled
// (17.6 M samples, 5 octaves) take 43 us here and 61 in k_terrain; evaluating
// every sample's octaves until its sign was certain (1.38 on average) took
// 202, and 23 instead of 13 for the endpoints that it left.
// ------------------------------------------------------------------------
// n and its gradient at (x, y, z): snoise3's corners, without its exact
// operation order.
struct NoiseGrad {
    float n, gx, gy, gz;
};
__device__ __forceinline__ void corner_grad(float x, float y, float z, uint32_t h, NoiseGrad& r) {
    const float4 g = lattice_gradient(lattice_mix(h));
    float t = __builtin_fmaf(-x, x, kNoiseR2);
    t = __builtin_fmaf(-y, y, t);
    t = __builtin_fmaf(-z, z, t);
    t = fmaxf(t, 0.0f);
    const float L = __builtin_fmaf(g.x, x, __builtin_fmaf(g.y, y, g.z * z));
    const float t2 = t * t, t4 = t2 * t2, k = -8.0f * t2 * t * L;
    r.n = __builtin_fmaf(t4, L, r.n);
    r.gx = __builtin_fmaf(t4, g.x, __builtin_fmaf(k, x, r.gx));
    r.gy = __builtin_fmaf(t4, g.y, __builtin_fmaf(k, y, r.gy));
    r.gz = __builtin_fmaf(t4, g.z, __builtin_fmaf(k, z, r.gz));
}
__device__ __forceinline__ NoiseGrad snoise3_grad(float x, float y, float z, uint32_t seed) {
    const float G3 = 1.0f / 6.0f;
    const float s = ((x + y) + z) * (1.0f / 3.0f);
    const float fi = floorf(x + s), fj = floorf(y + s), fk = floorf(z + s);
    const int32_t i = (int32_t)fi, j = (int32_t)fj, k = (int32_t)fk;
    const float t = (float)(i + j + k) * G3;
    const float x0 = x - (fi - t), y0 = y - (fj - t), z0 = z - (fk - t);
    const bool gxy = x0 >= y0, gyz = y0 >= z0, gxz = x0 >= z0;
    const bool i1 = gxy && gxz, j1 = !gxy && gyz, k1 = !gxz && !gyz;
    const bool i2 = gxy || gxz, j2 = !gxy || gyz, k2 = !gxz || !gyz;
    const float xm = x0 - 1.0f, ym = y0 - 1.0f, zm = z0 - 1.0f;
    const uint32_t a0 = mul24((uint32_t)i, kP1), a1 = mul24((uint32_t)(i + 1), kP1);
    const uint32_t b0 = mul24((uint32_t)j, kP2), b1 = mul24((uint32_t)(j + 1), kP2);
    const uint32_t c0 = mul24((uint32_t)k, kP3) ^ seed, c1 = mul24((uint32_t)(k + 1), kP3) ^ seed;
    NoiseGrad r{0.0f, 0.0f, 0.0f, 0.0f};
    corner_grad(x0, y0, z0, xor3(a0, b0, c0), r);
    corner_grad((i1 ? xm : x0) + G3, (j1 ? ym : y0) + G3, (k1 ? zm : z0) + G3,
                xor3(i1 ? a1 : a0, j1 ? b1 : b0, k1 ? c1 : c0), r);
    corner_grad((i2 ? xm : x0) + 2.0f * G3, (j2 ? ym : y0) + 2.0f * G3, (k2 ? zm : z0) + 2.0f * G3,
                xor3(i2 ? a1 : a0, j2 ? b1 : b0, k2 ? c1 : c0), r);
    corner_grad(xm + 0.5f, ym + 0.5f, zm + 0.5f, xor3(a1, b1, c1), r);
    r.n *= kNoiseScale;
    r.gx *= kNoiseScale;
    r.gy *= kNoiseScale;
    r.gz *= kNoiseScale;
    return r;
}

// Sum over the lanes of a quad, in every lane of it.
__device__ __forceinline__ float quad_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));
    return v;
}

// The first k octaves expanded about p, lane `o` of the quad taking octave
// o: the sum and its step per sample, in every lane of the quad.
__device__ __forceinline__ NoiseGrad expand(const SamplerDev& S, int k, int o, float delta, float px, float py,
                                            float pz) {
    NoiseGrad r{0.0f, 0.0f, 0.0f, 0.0f};
    if (o < k) {
        const float f = S.fo[o], a = S.ao[o], af = a * (f * delta);
        const NoiseGrad g = snoise3_grad(px * f, py * f, pz * f, S.seed + (uint32_t)o);
        r = NoiseGrad{a * g.n, af * g.gx, af * g.gy, af * g.gz};
    }
    return NoiseGrad{quad_sum(r.n), quad_sum(r.gx), quad_sum(r.gy), quad_sum(r.gz)};
}

__global__ void __launch_bounds__(kRowThreads) k_blocks(Arenas A, int n) {
    // per block and plane dx of it: undecided samples in the low half, air
    // samples in the high half, bit 4 dy + dz
    __shared__ uint32_t s_block[kWordWaves][4 * kWaveBlocks];
    __shared__ uint8_t s_sub[kWordWaves][8 * kWaveBlocks];
    __shared__ unsigned long long s_evals;
    if (threadIdx.x == 0) s_evals = 0;
    __syncthreads();
    load_gradients();
    const SamplerDev* __restrict__ S = A.sampler;
    const int wave = uniform_int(threadIdx.x >> 6), lane = lane_id(), o = lane & 3;
    unsigned long long evals = 0;  // octaves at the centres of this wave's blocks (uniform)
    const int64_t total = A.block_prefix[n];
    for (int64_t it = (int64_t)blockIdx.x * kWordWaves + wave; it < total; it += (int64_t)gridDim.x * kWordWaves) {
        const int j = find_chunk_wave(A.block_prefix, n, it);
        const ChunkMeta M = read_chunk(A.meta, j);
        const int dim = M.dim, nb = (dim + 3) >> 2, nb2 = nb * nb;
        const int b0 = (int)(it - A.block_prefix[j]) * kWaveBlocks, b = b0 + (lane >> 2);
        const int bx = (int)udiv24((uint32_t)b, (uint32_t)nb2, 1.0f / (float)nb2), br = b - bx * nb2;
        const int by = (int)udiv24((uint32_t)br, (uint32_t)nb, 1.0f / (float)nb), bz = br - by * nb;
        const float delta = M.delta;
        const BlockPlan& bp = M.blocks;
        // the sum at which a sample's density amp * sum * inv_norm - t2 is 0
        // (the clamp to [-1, 1] never acts when no amplitude is negative)
        const float per = S->amp * S->inv_norm, inv = 1.0f / per;
        // ---- the blocks: a quad each, lane dx = o its plane of 16 samples ----
        const int rx = dim - 4 * bx, ry = min(4, dim - 4 * by), rz = min(4, dim - 4 * bz);
        uint32_t und = 0u, lab = 0u;
        if (b < nb2 * nb && o < rx) und = (0x1111u * ((1u << rz) - 1u)) & ((1u << (4 * ry)) - 1u);
        if (S->expand_ok) {
            const NoiseGrad g = expand(*S, bp.k4, o, delta, ((float)(4 * bx) + 1.5f) * delta + M.opos[0],
                                       ((float)(4 * by) + 1.5f) * delta + M.opos[1],
                                       ((float)(4 * bz) + 1.5f) * delta + M.opos[2]);
            const float plane = __builtin_fmaf((float)o - 1.5f, g.gx, g.n);
            const float oo = o == 0 || o == 3 ? 2.0f : 0.0f;
            float e[3];  // by the number of the other axes on which the sample is an outer one
#pragma unroll
            for (int c = 0; c < 3; c++) e[c] = __builtin_fmaf(bp.quad4, 0.75f + 2.0f * (float)c + oo, bp.base4);
            uint32_t dec = 0u, neg = 0u;
#pragma unroll
            for (int dy = 0; dy < 4; dy++) {
                const float t2 = ((float)(4 * by + dy) * delta + M.opos[1]) - S->y0;
                const float row = __builtin_fmaf((float)dy - 1.5f, g.gy, plane) - t2 * inv;
#pragma unroll
                for (int dz = 0; dz < 4; dz++) {
                    const float v = __builtin_fmaf((float)dz - 1.5f, g.gz, row);
                    const int outer = (dy == 0 || dy == 3) + (dz == 0 || dz == 3);
                    dec |= fabsf(v) > e[outer] ? 1u << (4 * dy + dz) : 0u;
                    neg |= v < 0.0f ? 1u << (4 * dy + dz) : 0u;
                }
            }
            if (per < 0.0f) neg = ~neg;  // air below the sign change, for a positive amplitude
            lab = und & dec & neg;
            und &= ~dec;
        } else {  // the band alone
            const TerrainTerms T{S->amp, S->y0, S->inv_norm};
#pragma unroll
            for (int dy = 0; dy < 4; dy++) {
                const float t2 = ((float)(4 * by + dy) * delta + M.opos[1]) - T.y0;
                const int d = decide_label(T, S->reach[0], 0.0f, t2);
                const uint32_t row = 0xFu << (4 * dy);
                lab |= d == 1 ? und & row : 0u;
                und &= d ? ~row : ~0u;
            }
        }
        if (bp.k4) evals += (unsigned long long)(bp.k4 * min(kWaveBlocks, nb2 * nb - b0));
        // ---- their sub-blocks with undecided samples: a quad each ----
        if (bp.k2) {
            const uint32_t pair = und | (uint32_t)__builtin_amdgcn_update_dpp(0, (int)und, 0xB1, 0xF, 0xF, true);
            s_block[wave][lane] = und | (lab << 16);
            uint32_t ns = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) {  // (sy, sz); lanes 0 and 2 of the quad take sx = 0 and 1
                const bool need = !(o & 1) && (pair & (0x33u << (8 * (q >> 1) + 2 * (q & 1)))) != 0u;
                const uint64_t bal = __ballot(need);
                if (need) s_sub[wave][ns + mbcnt64(bal)] = (uint8_t)((lane >> 2) * 8 + (o >> 1) * 4 + q);
                ns += (uint32_t)__popcll(bal);
            }
            wave_sync();
            evals += (unsigned long long)bp.k2 * ns;
            const float e2 = __builtin_fmaf(bp.quad2, 0.75f, bp.base2);
            for (uint32_t i0 = 0; i0 < ns; i0 += kWaveBlocks) {
                const uint32_t i = i0 + (uint32_t)(lane >> 2);
                const uint32_t sub = s_sub[wave][min(i, ns - 1u)];
                const int sx = (int)(sub >> 2) & 1, sy = (int)(sub >> 1) & 1, sz = (int)sub & 1;
                const int at = __shfl(bx | (by << 8) | (bz << 16), (int)(4u * (sub >> 3)));  // its block's quad
                const int x = 4 * (at & 255) + 2 * sx, y = 4 * ((at >> 8) & 255) + 2 * sy, z = 4 * (at >> 16) + 2 * sz;
                const NoiseGrad g = expand(*S, bp.k2, o, delta, ((float)x + 0.5f) * delta + M.opos[0],
                                           ((float)y + 0.5f) * delta + M.opos[1], ((float)z + 0.5f) * delta + M.opos[2]);
                // lane (dx, dy) of the quad: its two samples
                const int dx = o >> 1, dy = o & 1;
                const float t2 = ((float)(y + dy) * delta + M.opos[1]) - S->y0;
                const float row = __builtin_fmaf((float)dx - 0.5f, g.gx, __builtin_fmaf((float)dy - 0.5f, g.gy, g.n)) -
                                  t2 * inv;
                uint32_t dec = 0u, neg = 0u;
#pragma unroll
                for (int dz = 0; dz < 2; dz++) {
                    const float v = __builtin_fmaf((float)dz - 0.5f, g.gz, row);
                    dec |= fabsf(v) > e2 ? 1u << dz : 0u;
                    neg |= v < 0.0f ? 1u << dz : 0u;
                }
                if (per < 0.0f) neg = ~neg;
                if (i < ns) {
                    uint32_t* w = &s_block[wave][4 * (sub >> 3) + 2 * sx + dx];
                    const int sh = 4 * (2 * sy + dy) + 2 * sz;
                    const uint32_t hit = *w & (dec << sh);  // the other bits may be cleared meanwhile
                    atomicAnd(w, ~hit);
                    atomicOr(w, (hit & (neg << sh)) << 16);
                }
            }
            wave_sync();
            const uint32_t w = s_block[wave][lane];
            und = w & 0xFFFFu;
            lab = w >> 16;
            wave_sync();  // before the next item's
        }
        // a byte per four samples of a row: undecided low, air high
        if (b < nb2 * nb && o < rx) {
            uint8_t* __restrict__ N = A.signs + M.dens_off + ((int64_t)(4 * bx + o) * dim + 4 * by) * nb + bz;
            for (int dy = 0; dy < ry; dy++)
                N[dy * nb] = (uint8_t)(((und >> (4 * dy)) & 15u) | (((lab >> (4 * dy)) & 15u) << 4));
        }
    }
    if (lane == 0 && evals) atomicAdd(&s_evals, evals);
    __syncthreads();
    if (threadIdx.x == 0 && (int)blockIdx.x < A.stat_cap) A.stat_blocks[2 * A.stat_cap + blockIdx.x] = s_evals;
}

// ------------------------------------------------------------------------
// terrain (adaptive): labels from k_blocks' decisions, every octave of the
// samples it left open.
//
// A workgroup takes four items of label words, a wave each: a lane reads the
// decisions of 16 consecutive samples (a byte holds four of a row), and the
// open samples of all four items go to one list that the workgroup's lanes
// then share.  While the list is long (a field too rough for the expansions)
// it is evaluated octave by octave and compacted in place: after k octaves
// the FP32 partial sum S_k bounds the final sum, each remaining step being
// fma(a_o, n_o, S) with |n_o| <= 1 and rounding monotone, so that S_O lies in
// [S_k - reach[k], S_k + reach[k]] (reach: sum_{o>=k} |a_o| widened by the
// rounding of those steps and of the two bounds, host side), and the density
// is monotone in S.  Samples that run all octaves get their exact density
// and their bit in the `exact` bitmap; the others only their label (k_count
// finishes the densities of those that are endpoints of a sign-changing
// edge).  Labels and every density that a mesh reads are those of the full
// evaluation, bit for bit.  Bound by VALU issue (61 us on the batch above).
// kTerrainDirect: short lists lose less to octaves that an early decision would
// have spared than to the rounds' barriers.
// ------------------------------------------------------------------------
constexpr int kTerrainSamples = kWordWaves * kItemSamples;
constexpr int kTerrainDirect = 1024;  // open samples up to which all octaves run at once

__global__ void __launch_bounds__(kRowThreads) k_terrain(Arenas A, int n) {
    struct Geom {
        ChunkGeom G;
        int dim, chunk, i0;
        int64_t dens_off;
    };
    __shared__ Geom s_geom[kWordWaves];
    __shared__ uint64_t s_lab[kWordWaves * kItemWords], s_exact[kWordWaves * kItemWords];
    __shared__ uint16_t s_list[kTerrainSamples];
    __shared__ float s_sum[kTerrainSamples];
    __shared__ uint32_t s_n;
    __shared__ unsigned long long s_evals;
    __shared__ float s_oct[3][BMF_MAX_OCTAVES + 1];  // per octave: frequency, amplitude, reach
    load_gradients();
    const SamplerDev* __restrict__ S = A.sampler;
    const TerrainTerms TT{S->amp, S->y0, S->inv_norm};
    const int O = S->octaves;
    const uint32_t seed0 = S->seed;  // octave k uses seed0 + k
    const int tid = threadIdx.x, wave = uniform_int(tid >> 6), lane = lane_id();
    for (int t = tid; t <= O; t += blockDim.x) {
        s_oct[0][t] = t < O ? S->fo[t] : 0.0f;
        s_oct[1][t] = t < O ? S->ao[t] : 0.0f;
        s_oct[2][t] = S->reach[t];
    }
    if (tid == 0) s_evals = 0;
    unsigned long long evals = 0;  // octaves this lane evaluated
    const int64_t total = read_const(&A.ctr->total_items);
    // position and y - y0 of list entry v: wave << 10 | sample of its item
    auto locate = [&](uint32_t v, uint32_t& i, float& px, float& py, float& pz) {
        const Geom& g = s_geom[v >> 10];
        const uint32_t dim = (uint32_t)g.dim, dim2 = dim * dim;
        i = (uint32_t)g.i0 + (v & 1023u);
        sample_coords(g.G, i, dim, dim2, 1.0f / (float)dim, 1.0f / (float)dim2, px, py, pz);
    };
    auto set_bit = [&](uint64_t* words, uint32_t v) {
        atomicOr(reinterpret_cast<uint32_t*>(words) + (v >> 5), 1u << (v & 31u));
    };
    for (int64_t it0 = (int64_t)blockIdx.x * kWordWaves; it0 < total; it0 += (int64_t)gridDim.x * kWordWaves) {
        if (tid == 0) s_n = 0;
        __syncthreads();
        const int64_t it = it0 + wave;
        uint32_t und = 0u, lab = 0u;
        if (it < total) {
            const int j = find_item_wave(A.meta, n, it);
            const ChunkMeta M = read_chunk(A.meta, j);
            const int dim = M.dim, d2 = dim * dim, n3 = d2 * dim, nb = (dim + 3) >> 2;
            const int item = (int)(it - M.item_slot);
            if (lane == 0) {
                A.item_map[it] = make_int2(j, item);
                s_geom[wave] = Geom{{M.opos[0], M.opos[1], M.opos[2], M.delta}, dim, j, item * kItemSamples, M.dens_off};
            }
            // the lane's 16 samples, a run within a row at a time
            int i = item * kItemSamples + 16 * lane;
            if (i < n3) {
                const int x = (int)udiv24((uint32_t)i, (uint32_t)d2, 1.0f / (float)d2);
                const int r = i - x * d2, y = (int)udiv24((uint32_t)r, (uint32_t)dim, 1.0f / (float)dim);
                int z = r - y * dim;
                const uint8_t* __restrict__ N = A.signs + M.dens_off + (int64_t)(x * dim + y) * nb;
                for (int got = 0; got < 16 && i < n3;) {
                    uint64_t w;  // the row's bytes from z on: 5 are used
                    __builtin_memcpy(&w, N + (z >> 2), 8);
                    const int run = min(16 - got, dim - z);
                    const uint32_t m = (1u << run) - 1u;
                    und |= ((low_nibbles(w) >> (z & 3)) & m) << got;
                    lab |= ((low_nibbles(w >> 4) >> (z & 3)) & m) << got;
                    got += run;
                    i += run;
                    z = 0;
                    N += nb;
                }
            }
        }
        reinterpret_cast<uint16_t*>(s_lab)[tid] = (uint16_t)lab;
        reinterpret_cast<uint16_t*>(s_exact)[tid] = 0u;
        {
            uint32_t cnt, b = und;
            uint32_t at = wave_prefix<5>((uint32_t)__popc(b), cnt);
            uint32_t base = 0;
            if (lane == 0 && cnt) base = atomicAdd(&s_n, cnt);
            at += (uint32_t)uniform_int((int)base);
            while (b) {
                s_list[at++] = (uint16_t)(wave << 10 | (16 * lane + __ffs(b) - 1));
                b &= b - 1u;
            }
        }
        __syncthreads();
        uint32_t nq = s_n;
        int k = 0;
        // ---- a long list: an octave at a time, the survivors moved up ----
        while (nq > (uint32_t)kTerrainDirect && k < O - 1) {
            __syncthreads();  // every thread has read s_n
            if (tid == 0) s_n = 0;
            for (uint32_t e0 = 0; e0 < nq; e0 += kRowThreads) {
                const uint32_t e = e0 + (uint32_t)tid;
                const uint32_t v = e < nq ? s_list[e] : 0u;
                float sum = e < nq && k > 0 ? s_sum[e] : 0.0f;
                __syncthreads();  // this part of the list is read: it may be overwritten
                int dec = 2;
                if (e < nq) {
                    uint32_t i;
                    float px, py, pz;
                    locate(v, i, px, py, pz);
                    const float f = s_oct[0][k];
                    sum = __builtin_fmaf(s_oct[1][k], snoise3(px * f, py * f, pz * f, seed0 + (uint32_t)k), sum);
                    dec = decide_label(TT, s_oct[2][k + 1], sum, py - TT.y0);
                    if (dec == 1) set_bit(s_lab, v);
                    evals++;
                }
                const uint64_t push = __ballot(dec == 0);
                if (push) {
                    uint32_t base = 0;
                    if (lane == 0) base = atomicAdd(&s_n, (uint32_t)__popcll(push));
                    const uint32_t at = (uint32_t)uniform_int((int)base) + mbcnt64(push);
                    if (dec == 0) {
                        s_list[at] = (uint16_t)v;
                        s_sum[at] = sum;
                    }
                }
            }
            __syncthreads();
            nq = s_n;
            k++;
        }
        // ---- the rest of the octaves of the open samples ----
        for (uint32_t e = (uint32_t)tid; e < nq; e += kRowThreads) {
            const uint32_t v = s_list[e];
            float sum = k > 0 ? s_sum[e] : 0.0f;
            uint32_t i;
            float px, py, pz;
            locate(v, i, px, py, pz);
            for (int o = k; o < O; o++) {
                const float f = s_oct[0][o];
                sum = __builtin_fmaf(s_oct[1][o], snoise3(px * f, py * f, pz * f, seed0 + (uint32_t)o), sum);
            }
            const float d = density_from_sum(TT, sum, py - TT.y0);
            A.dens[s_geom[v >> 10].dens_off + i] = d;
            if (d < 0.0f) set_bit(s_lab, v);
            set_bit(s_exact, v);
            evals += (unsigned long long)(O - k);
        }
        __syncthreads();
        // ---- the items' words ----
        if (tid < kWordWaves * kItemWords && it0 + tid / kItemWords < total) {
            const Geom& g = s_geom[tid / kItemWords];
            const int i = g.i0 + 64 * (tid % kItemWords), left = g.dim * g.dim * g.dim - i;
            const uint64_t lb = s_lab[tid];
            if (left > 0) {
                const int64_t w = A.meta[g.chunk].lab_off + (i >> 6);
                A.labels[w] = lb;
                A.exact[w] = s_exact[tid];
            }
            const uint64_t have = left > 0 ? ~bits_from(left) : 0ull;
            const uint64_t group = 0xFFFFull << (lane & 48);
            const bool air = (__ballot((lb & have) != 0ull) & group) != 0ull;
            const bool solid = (__ballot((~lb & have) != 0ull) & group) != 0ull;
            if ((lane & 15) == 0) {
                if (air && !A.meta[g.chunk].any_air) atomicOr(&A.meta[g.chunk].any_air, 1u);
                if (solid && !A.meta[g.chunk].any_solid) atomicOr(&A.meta[g.chunk].any_solid, 1u);
            }
        }
        __syncthreads();  // before the next items'
    }
    if (evals) atomicAdd(&s_evals, evals);
    __syncthreads();
    if (tid == 0 && (int)blockIdx.x < A.stat_cap) A.stat_blocks[blockIdx.x] = s_evals;
}

// ------------------------------------------------------------------------
// sample: the other samplers but CSG (k_csg), one wave per WORDS label words
// (all of them in a chunk's first item, and so on): no barrier and no LDS.  The
// words per wave balance the chip's last round against the wave's own set-up.
// Bound by VALU issue where a sampler is evaluated, by HBM where densities only
// pass through.
//   terrain in full  129^3 samples, 5 octaves: 52 us (tiles of 2,048
//                    samples per workgroup, 1,049 of them: 95)
//   external         48 chunks of 41^3: 12 us (tiles: 52)
//   2D noise field   from the columns of k_columns
//   implicit shapes  whole passes of one chunk of 16^3 cells 80 us, of 64^3 83,
//                    64 of 64^3 125 (tiles: 130, 144, 380)
// ------------------------------------------------------------------------
constexpr int kSampleImplicit = 0, kSampleTerrain = 1, kSampleField2 = 2, kSampleField3 = 3, kSampleExternal = 4;

// 2D noise fields: n at every (x, z) column of every chunk, a lane each, into
// the cell arena (free until the emission), from the chunk's first sample on.
// Evaluated per tile of samples instead, the columns filled 96 of a
// workgroup's 256 lanes: 168 chunks of 32^3 took 76 us; this and the pass
// over the samples take 26 + 18.
__global__ void __launch_bounds__(kRowThreads) k_columns(Arenas A, int n) {
    load_gradients();
    const SamplerDev* __restrict__ S = A.sampler;
    const int64_t total = A.block_prefix[n];
    const int lane = lane_id();
    for (int64_t it = (int64_t)blockIdx.x * kWordWaves + (threadIdx.x >> 6); it < total;
         it += (int64_t)gridDim.x * kWordWaves) {
        const int j = find_chunk_wave(A.block_prefix, n, it);
        const ChunkMeta M = read_chunk(A.meta, j);
        const int c = (int)(it - A.block_prefix[j]) * 64 + lane;
        if (c >= M.dim * M.dim) continue;
        const int x = c / M.dim, z = c - x * M.dim;
        const ChunkGeom G{M.opos[0], M.opos[1], M.opos[2], M.delta};
        float px, py, pz;
        sample_position(G, (uint32_t)x, 0u, (uint32_t)z, px, py, pz);
        A.cell_tb[M.dens_off + c] = __float_as_uint(noise_value(*S, px, 0.0f, pz));
    }
}

// ------------------------------------------------------------------------
// 3D noise fields (adaptive): a wave per kFieldWords label words.
//
// The perturbation's frequencies are low, so that a wave's samples mostly lie
// in one simplex of it: then the four corners' gradients are the wave's, formed
// once for all its words, and a lane is left with the corners' falloffs, shared
// by the three fields, and three multiply-adds per corner and field.  The
// fractal's octaves follow one at a time over the samples of the workgroup
// whose sign is still open, compacted into dense lanes: what the rest of the
// octaves can add bounds the density from both sides.  Once that is no more
// than the field changes by over two sample steps (field_end), the open samples
// are mostly ends of sign-changing edges, whose density is wanted: they get all
// the other octaves.  k_count evaluates the ends that are left.
//
// Bound by VALU issue.  108 chunks of 32^3 cells (3.9 M samples, 3 x 3
// perturbation and 8 fractal octaves, a mean of 3.4 of these taken): 161 us
// and 9 more in k_count.  With compares and selects for the noise's gradients
// (see gradient_table) it took 203 and 18, every octave at every sample 320.
// ------------------------------------------------------------------------
constexpr int kFieldWords = 4;
constexpr int kFieldSamples = 64 * kFieldWords;

// The gradients at the corners of a simplex of three noise fields of one
// frequency, the same in every lane.
struct FieldSimplex {
    int i, j, k, rank;  // rank < 0: none yet
    float g[3][4][3];   // field, corner, axis
};

__device__ __forceinline__ float lane_value(float x, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// One octave of the 3D gradient perturbation at (x, y, z): the three fields of
// seeds s, s + 1, s + 2, as snoise3 gives them.  All lanes are active.
__device__ __forceinline__ void warp_octave(float x, float y, float z, uint32_t seed, FieldSimplex& F, float (&w)[3]) {
    const float F3 = 1.0f / 3.0f, G3 = 1.0f / 6.0f, G3x2 = 2.0f * G3;
    const float s = ((x + y) + z) * F3;
    const float fi = floorf(x + s), fj = floorf(y + s), fk = floorf(z + s);
    const int i = (int32_t)fi, j = (int32_t)fj, k = (int32_t)fk;
    const float t = (float)(i + j + k) * G3;
    const float x0 = x - (fi - t), y0 = y - (fj - t), z0 = z - (fk - t);
    const uint64_t gxy = __ballot(x0 >= y0), gyz = __ballot(y0 >= z0), gxz = __ballot(x0 >= z0);
    const int ui = uniform_int(i), uj = uniform_int(j), uk = uniform_int(k);
    const bool one = __ballot((i == ui) & (j == uj) & (k == uk)) == ~0ull && (gxy == 0ull || gxy == ~0ull) &&
                     (gyz == 0ull || gyz == ~0ull) && (gxz == 0ull || gxz == ~0ull);
    if (!one) {
        for (int a = 0; a < 3; a++) w[a] = snoise3(x, y, z, seed + (uint32_t)a);
        return;
    }
    const bool bxy = gxy != 0ull, byz = gyz != 0ull, bxz = gxz != 0ull;
    const bool i1 = bxy && bxz, j1 = !bxy && byz, k1 = !bxz && !byz;
    const bool i2 = bxy || bxz, j2 = !bxy || byz, k2 = !bxz || !byz;
    const int rank = (int)bxy + 2 * (int)byz + 4 * (int)bxz;
    if (F.rank != rank || F.i != ui || F.j != uj || F.k != uk) {
        F.i = ui;
        F.j = uj;
        F.k = uk;
        F.rank = rank;
        // lane 4 a + c: field a's gradient at corner c
        const int lane = lane_id(), c = lane & 3;
        const uint32_t ci = (uint32_t)ui + (uint32_t)(c == 3 || (c == 1 && i1) || (c == 2 && i2));
        const uint32_t cj = (uint32_t)uj + (uint32_t)(c == 3 || (c == 1 && j1) || (c == 2 && j2));
        const uint32_t ck = (uint32_t)uk + (uint32_t)(c == 3 || (c == 1 && k1) || (c == 2 && k2));
        const float4 g = lattice_gradient(lattice_mix(
            xor3(mul24(ci, kP1), mul24(cj, kP2), mul24(ck, kP3) ^ (seed + (uint32_t)(lane >> 2)))));
#pragma unroll
        for (int q = 0; q < 12; q++) {
            F.g[q >> 2][q & 3][0] = lane_value(g.x, q);
            F.g[q >> 2][q & 3][1] = lane_value(g.y, q);
            F.g[q >> 2][q & 3][2] = lane_value(g.z, q);
        }
    }
    const float xm = x0 - 1.0f, ym = y0 - 1.0f, zm = z0 - 1.0f;
    const float cx[4] = {x0, (i1 ? xm : x0) + G3, (i2 ? xm : x0) + G3x2, xm + 0.5f};
    const float cy[4] = {y0, (j1 ? ym : y0) + G3, (j2 ? ym : y0) + G3x2, ym + 0.5f};
    const float cz[4] = {z0, (k1 ? zm : z0) + G3, (k2 ? zm : z0) + G3x2, zm + 0.5f};
    float n[3];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        float q = __builtin_fmaf(-cx[c], cx[c], kNoiseR2);
        q = __builtin_fmaf(-cy[c], cy[c], q);
        q = __builtin_fmaf(-cz[c], cz[c], q);
        q = fmaxf(q, 0.0f);
        q = q * q;
        q = q * q;
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const float dot = __builtin_fmaf(
                F.g[a][c][0], cx[c], __builtin_fmaf(F.g[a][c][1], cy[c], F.g[a][c][2] * cz[c]));
            const float v = q * dot;
            n[a] = c == 0 ? v : n[a] + v;
        }
    }
#pragma unroll
    for (int a = 0; a < 3; a++) w[a] = fminf(fmaxf(kNoiseScale * n[a], -1.0f), 1.0f);
}

// The octave of the fractal from which k_field decides no more signs (see
// there): a sample step changes octave o by about a_o f_o times the step of
// its argument, times a noise gradient of about 2.  Down to one such step,
// two or four, the batch above with its meshing and formatting takes 300, 288
// and 289 us.
__device__ __forceinline__ int field_end(const SamplerDev& S, float delta) {
    float step = 0.0f;
    for (int o = 0; o < S.octaves; o++) step += fabsf(S.ao[o] * S.fo[o]);
    step *= 2.0f * delta * fabsf(S.g_scale);
    int k = 1;
    while (k < S.octaves && S.field_dn[k] + S.field_up[k] > 2.0f * step) k++;
    return k;
}

__global__ void __launch_bounds__(kRowThreads) k_field(Arenas A, int n) {
    constexpr int kParts = kItemWords / kFieldWords;  // waves per item of the word kernels
    constexpr int kList = kWordWaves * kFieldSamples;
    struct Geom {
        int64_t dens_off;  // of the wave's first sample
        int end;           // octaves after which the list is taken to the end
    };
    __shared__ Geom s_geom[kWordWaves];
    // open samples: perturbed position, height, fractal sum, wave << 8 | sample
    __shared__ float s_x[kList], s_y[kList], s_z[kList], s_py[kList], s_sum[kList];
    __shared__ uint16_t s_at[kList];
    __shared__ uint32_t s_n;
    __shared__ uint64_t s_lab[kWordWaves * kFieldWords], s_exact[kWordWaves * kFieldWords];
    load_gradients();
    const SamplerDev& S = *A.sampler;
    const bool rigid = S.noise_fractal == BMF_FRACTAL_RIGID, value = S.noise_basis == BMF_NOISE_VALUE;
    const int tid = threadIdx.x, wave = uniform_int(tid >> 6), lane = lane_id(), O = S.octaves;
    auto octave = [&](float sum, int o, float cx, float cy, float cz) {
        const float f = S.fo[o], a = S.ao[o];
        const float b = value ? value3(cx * f, cy * f, cz * f, S.seed + (uint32_t)o)
                              : snoise3(cx * f, cy * f, cz * f, S.seed + (uint32_t)o);
        if (!rigid) return __builtin_fmaf(a, b, sum);
        const float t = 1.0f - fabsf(b);
        return o == 0 ? t : __builtin_fmaf(-t, a, sum);
    };
    auto density = [&](float sum, float py) {
        return noise_density_from(S, rigid ? sum : fminf(fmaxf(sum * S.inv_norm, -1.0f), 1.0f), py);
    };
    auto set_bit = [&](uint64_t* words, uint32_t at) {
        atomicOr(reinterpret_cast<uint32_t*>(words) + (at >> 5), 1u << (at & 31u));
    };
    const int64_t total = A.ctr->total_items * kParts;
    for (int64_t u0 = (int64_t)blockIdx.x * kWordWaves; u0 < total; u0 += (int64_t)gridDim.x * kWordWaves) {
        // ---- each wave's samples, perturbed, into the list ----
        if (tid == 0) s_n = 0;
        if (tid < kWordWaves * kFieldWords) s_lab[tid] = s_exact[tid] = 0ull;
        __syncthreads();
        const int64_t u = u0 + wave, it = u / kParts;
        int64_t lab_off = 0;
        int j = 0, open = 0;
        if (u < total) {
            const int part = (int)(u - it * kParts);
            j = find_item_wave(A.meta, n, it);
            const ChunkMeta M = read_chunk(A.meta, j);
            const int item = (int)(it - M.item_slot), w0 = item * kItemWords + part * kFieldWords;
            if (part == 0 && lane == 0) A.item_map[it] = make_int2(j, item);  // for the word kernels
            const uint32_t dim = (uint32_t)M.dim, dim2 = dim * dim, ns = dim2 * dim, first = 64u * (uint32_t)w0;
            const float rd = 1.0f / (float)dim, rd2 = 1.0f / (float)dim2;
            const ChunkGeom G{M.opos[0], M.opos[1], M.opos[2], M.delta};
            lab_off = M.lab_off + w0;
            open = first < ns ? (int)min((uint32_t)kFieldSamples, ns - first) : 0;
            // no early decision where a coordinate can leave the range of the bounds
            const float ext = (float)(dim - 1u) * M.delta;
            const bool early = S.early_ok && fmaxf(fmaxf(fabsf(G.ox), fabsf(G.oy)), fabsf(G.oz)) + ext < 1e9f;
            uint32_t base = 0;
            if (lane == 0) {
                s_geom[wave] = Geom{M.dens_off + first, early ? field_end(S, M.delta) : 0};
                base = atomicAdd(&s_n, (uint32_t)open);
            }
            base = (uint32_t)uniform_int((int)base);
            float cx[kFieldWords], cy[kFieldWords], cz[kFieldWords], ph[kFieldWords];
#pragma unroll
            for (int r = 0; r < kFieldWords; r++) {
                float px, pz;
                sample_coords(G, min(first + 64u * r + (uint32_t)lane, ns - 1u), dim, dim2, rd, rd2, px, ph[r], pz);
                if (S.perturb == BMF_PERTURB_GRADIENT) {
                    cx[r] = px * S.g_scale;
                    cy[r] = ph[r] * S.g_scale;
                    cz[r] = pz * S.g_scale;
                } else {
                    noise_warp(S, px, ph[r], pz, cx[r], cy[r], cz[r]);
                }
            }
            if (S.perturb == BMF_PERTURB_GRADIENT) {
                FieldSimplex F;
                for (int k = 0; k < S.perturb_octaves; k++) {
                    const float f = S.pf[k], a = S.pa[k];
                    F.rank = -1;
#pragma unroll
                    for (int r = 0; r < kFieldWords; r++) {
                        float w[3];
                        warp_octave(cx[r] * f, cy[r] * f, cz[r] * f, S.seed + 1000u + 3u * (uint32_t)k, F, w);
                        cx[r] = __builtin_fmaf(a, w[0], cx[r]);
                        cy[r] = __builtin_fmaf(a, w[1], cy[r]);
                        cz[r] = __builtin_fmaf(a, w[2], cz[r]);
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < kFieldWords; r++) {
                const int e = 64 * r + lane;
                if (e < open) {
                    s_x[base + e] = cx[r];
                    s_y[base + e] = cy[r];
                    s_z[base + e] = cz[r];
                    s_py[base + e] = ph[r];
                    s_at[base + e] = (uint16_t)(wave << 8 | e);
                }
            }
        }
        __syncthreads();
        uint32_t nq = s_n;
        int end = O;
        for (int w = 0; w < kWordWaves; w++)
            if (u0 + w < total) end = min(end, s_geom[w].end);
        // ---- an octave at a time, the samples still open moved up ----
        int o = 0;
        for (; o < end && o < O - 1 && nq; o++) {
            const float dn = S.field_dn[o + 1], up = S.field_up[o + 1];
            __syncthreads();  // every thread has read s_n
            if (tid == 0) s_n = 0;
            for (uint32_t e0 = 0; e0 < nq; e0 += kRowThreads) {
                const uint32_t e = e0 + (uint32_t)tid;
                const bool in = e < nq;
                const float cx = s_x[in ? e : 0u], cy = s_y[in ? e : 0u], cz = s_z[in ? e : 0u], py = s_py[in ? e : 0u];
                float sum = o > 0 && in ? s_sum[e] : 0.0f;
                const uint32_t at = s_at[in ? e : 0u];
                __syncthreads();  // this part of the list is read: it may be overwritten
                bool keep = false;
                if (in) {
                    sum = octave(sum, o, cx, cy, cz);
                    const float d0 = density(sum - dn, py), d1 = density(sum + up, py);
                    const bool air = fmaxf(d0, d1) < 0.0f;
                    if (air) set_bit(s_lab, at);
                    keep = !(air || fminf(d0, d1) >= 0.0f);
                }
                const uint64_t push = __ballot(keep);
                if (push) {
                    uint32_t base = 0;
                    if (lane == 0) base = atomicAdd(&s_n, (uint32_t)__popcll(push));
                    const uint32_t k = (uint32_t)uniform_int((int)base) + mbcnt64(push);
                    if (keep) {
                        s_x[k] = cx;
                        s_y[k] = cy;
                        s_z[k] = cz;
                        s_py[k] = py;
                        s_sum[k] = sum;
                        s_at[k] = (uint16_t)at;
                    }
                }
            }
            __syncthreads();
            nq = s_n;
        }
        // ---- the rest of the octaves of the samples still open ----
        for (uint32_t e = (uint32_t)tid; e < nq; e += kRowThreads) {
            const float cx = s_x[e], cy = s_y[e], cz = s_z[e];
            float sum = o > 0 ? s_sum[e] : 0.0f;
            const uint32_t at = s_at[e];
            for (int k = o; k < O; k++) sum = octave(sum, k, cx, cy, cz);
            const float d = density(sum, s_py[e]);
            A.dens[s_geom[at >> 8].dens_off + (at & 255u)] = d;
            if (d < 0.0f) set_bit(s_lab, at);
            set_bit(s_exact, at);
        }
        __syncthreads();
        // ---- the words ----
        const int left = open - 64 * lane;
        const bool mine = lane < kFieldWords && left > 0;
        const uint64_t lb = mine ? s_lab[wave * kFieldWords + lane] : 0ull, have = ~bits_from(left);
        if (mine) {
            A.labels[lab_off + lane] = lb;
            A.exact[lab_off + lane] = s_exact[wave * kFieldWords + lane];
        }
        const bool air = __any(mine && lb != 0ull), solid = __any(mine && (~lb & have) != 0ull);
        if (lane == 0) {
            if (air && !A.meta[j].any_air) atomicOr(&A.meta[j].any_air, 1u);
            if (solid && !A.meta[j].any_solid) atomicOr(&A.meta[j].any_solid, 1u);
        }
        __syncthreads();  // before the next words'
    }
    if (tid == 0 && (int)blockIdx.x < A.stat_cap) A.stat_blocks[blockIdx.x] = 0ull;  // no octaves counted
}

template <int MODE, int WORDS>
__global__ void __launch_bounds__(kRowThreads) k_sample(Arenas A, int n) {
    constexpr int kParts = kItemWords / WORDS;  // waves per item of the word kernels
    if constexpr (MODE == kSampleTerrain || MODE == kSampleField3) load_gradients();
    const SamplerDev* __restrict__ S = A.sampler;
    const int wave = uniform_int(threadIdx.x >> 6), lane = lane_id();
    const int64_t total = A.ctr->total_items * kParts;
    for (int64_t u = (int64_t)blockIdx.x * kWordWaves + wave; u < total; u += (int64_t)gridDim.x * kWordWaves) {
        const int64_t it = u / kParts;
        const int part = (int)(u - it * kParts);
        const int j = find_item_wave(A.meta, n, it);
        const ChunkMeta M = read_chunk(A.meta, j);
        const int item = (int)(it - M.item_slot), w0 = item * kItemWords + part * WORDS;
        if (part == 0 && lane == 0) A.item_map[it] = make_int2(j, item);  // for the word kernels
        if (w0 >= (int)M.lab_words) continue;
        const uint32_t dim = (uint32_t)M.dim, dim2 = dim * dim, ns = dim2 * dim;
        const ChunkGeom G{M.opos[0], M.opos[1], M.opos[2], M.delta};
        float* __restrict__ dens = A.dens + M.dens_off;
        const uint32_t first = 64u * (uint32_t)w0;
        uint64_t mine = 0ull;  // lane r keeps word r
        bool air = false, solid = false;
        auto word = [&](int r, bool valid, bool is_air) {
            const uint64_t bl = __ballot(valid && is_air), vb = __ballot(valid);
            mine = lane == r ? bl : mine;
            air = air || bl != 0ull;
            solid = solid || bl != vb;
        };
        if constexpr (MODE == kSampleExternal) {
            const float* __restrict__ src = (A.ext ? A.ext : S->ext) + A.ext_base + M.dens_off;
            float v[WORDS];
#pragma unroll
            for (int r = 0; r < WORDS; r++) v[r] = src[min(first + 64u * r + (uint32_t)lane, ns - 1u)];
#pragma unroll
            for (int r = 0; r < WORDS; r++) {
                const uint32_t i = first + 64u * r + (uint32_t)lane;
                if (i < ns) dens[i] = v[r];
                word(r, i < ns, v[r] < 0.0f);
            }
        } else {
            // a lane's sample advances by 64 per word: its (y, z) by
            // (64 / dim, 64 % dim) with at most one carry per axis while
            // 64 / dim + 1 < dim; smaller chunks divide
            const float rd = 1.0f / (float)dim, rd2 = 1.0f / (float)dim2;
            const uint32_t step_y = 64u / dim, step_z = 64u - step_y * dim;
            const bool stepping = step_y + 1 < dim;
            uint32_t x, y, z;
            sample_index(first + (uint32_t)lane, dim, dim2, rd, rd2, x, y, z);
#pragma unroll 1
            for (int r = 0; r < WORDS; r++) {
                const uint32_t i = first + 64u * (uint32_t)r + (uint32_t)lane;
                const bool valid = i < ns;
                float d = 0.0f;
                if (valid) {
                    float px, py, pz;
                    sample_position(G, x, y, z, px, py, pz);
                    if constexpr (MODE == kSampleTerrain) d = terrain_density(*S, px, py, pz);
                    else if constexpr (MODE == kSampleField2)
                        d = noise_density_from(*S, __uint_as_float(A.cell_tb[M.dens_off + x * dim + z]), py);
                    else if constexpr (MODE == kSampleField3) d = noise_density_from(*S, noise_value(*S, px, py, pz), py);
                    else d = implicit_density(S->kind, S->world_size, px, py, pz);
                    dens[i] = d;
                }
                word(r, valid, d < 0.0f);
                if (stepping) {
                    z += step_z;
                    y += step_y;
                    if (z >= dim) {
                        z -= dim;
                        y++;
                    }
                    if (y >= dim) {
                        y -= dim;
                        x++;
                    }
                } else {
                    sample_index(min(i + 64u, ns), dim, dim2, rd, rd2, x, y, z);
                }
            }
        }
        if (lane < WORDS && w0 + lane < (int)M.lab_words) {
            const int left = (int)ns - 64 * (w0 + lane);
            A.labels[M.lab_off + w0 + lane] = mine;
            A.exact[M.lab_off + w0 + lane] = ~bits_from(left);
        }
        if (lane == 0) {
            if (air && !A.meta[j].any_air) atomicOr(&A.meta[j].any_air, 1u);
            if (solid && !A.meta[j].any_solid) atomicOr(&A.meta[j].any_solid, 1u);
        }
    }
    if (threadIdx.x == 0 && (int)blockIdx.x < A.stat_cap) A.stat_blocks[blockIdx.x] = 0ull;  // no octaves counted
}

// ------------------------------------------------------------------------
// CSG: a wave per item of label words with the item's own primitives, culled
// from its chunk's list.  full: values are wanted at every sample (stage
// inspection, the tape) and nothing is culled.  Otherwise only signs and the
// densities at the ends of sign-changing edges are read, where the union lies
// within a sample step of 0 (csg_reach): primitives that stay further below it
// everywhere in the item's box cannot win there, and an item without any is air.
// Bound by VALU issue (the square root of each primitive's distance).
// ------------------------------------------------------------------------
// A wave takes its item's words in groups whose samples share a primitive's
// loads; batches of up to kCsgFew items have a wave, and a cull, per group.
// Sampling with a group and with an item per wave: one chunk of 20^3 cells with
// 300 primitives 84 and 314 us, of 64^3 (269 items) 42 and 135, 8 of 45^3 (760)
// 29 and 51 (with 30 primitives 23 and 17), 8 of 64^3 (2,145) 72 and 47.
constexpr int kCsgGroup = 4;
constexpr int kCsgFew = 1024;
__global__ void __launch_bounds__(kRowThreads) k_csg(Arenas A, int n, int full) {
    __shared__ __attribute__((aligned(8))) uint16_t s_ids[kWordWaves][kCsgIds];
    const SamplerDev& S = *A.sampler;
    const int wave = uniform_int(threadIdx.x >> 6), lane = lane_id();
    const int64_t items = read_const(&A.ctr->total_items);
    const int words = items <= kCsgFew ? kCsgGroup : kItemWords, parts = kItemWords / words;
    uint16_t* const ids = s_ids[wave];
    for (int64_t u = (int64_t)blockIdx.x * kWordWaves + wave; u < items * parts; u += (int64_t)gridDim.x * kWordWaves) {
        const int64_t it = u / parts;
        const int part = (int)(u - it * parts);
        const int j = find_item_wave(A.meta, n, it);
        const ChunkMeta M = read_chunk(A.meta, j);
        const int item = (int)(it - M.item_slot), w0 = item * kItemWords + part * words;
        if (part == 0 && lane == 0) A.item_map[it] = make_int2(j, item);  // for the word kernels
        if (w0 >= (int)M.lab_words) continue;
        const uint32_t dim = (uint32_t)M.dim, dim2 = dim * dim, ns = dim2 * dim;
        const float rd = 1.0f / (float)dim, rd2 = 1.0f / (float)dim2;
        const ChunkGeom G{M.opos[0], M.opos[1], M.opos[2], M.delta};
        float* __restrict__ dens = A.dens + M.dens_off;
        const uint32_t first = 64u * (uint32_t)w0;
        const uint16_t* list = A.csg_list ? A.csg_list + (int64_t)j * A.csg_stride : nullptr;
        int cs = M.csg_ns, cb = M.csg_nb;
        bool fits = false;
        if (list) {
            float lo[3], hi[3];
            sample_box(M, (int)first, 64 * words, 0, lo, hi);
            int is, ib;
            fits = cull_csg_ids(S, list, cs, cb, lo, hi, full ? INFINITY : csg_reach(S, M.delta, lo, hi), ids, is, ib);
            if (fits) {
                cs = is;
                cb = ib;
            }
            wave_sync();
        }
        const bool empty = fits && cs + cb == 0 && !full;
        uint64_t mine = 0ull;  // lane r keeps word r
        bool air = false, solid = false;
#pragma unroll 1
        for (int r0 = 0; r0 < words; r0 += kCsgGroup) {
            float px[kCsgGroup], py[kCsgGroup], pz[kCsgGroup], d[kCsgGroup];
            if (empty) {
#pragma unroll
                for (int r = 0; r < kCsgGroup; r++) d[r] = kCsgFloor;
            } else {
#pragma unroll
                for (int r = 0; r < kCsgGroup; r++)
                    sample_coords(G, min(first + 64u * (uint32_t)(r0 + r) + (uint32_t)lane, ns - 1u), dim, dim2, rd, rd2,
                                  px[r], py[r], pz[r]);
                if (fits) {
                    csg_density_ids<kCsgGroup>(S, ids, cs, cb, px, py, pz, d);
                } else {
#pragma unroll
                    for (int r = 0; r < kCsgGroup; r++)
                        d[r] = list ? csg_density_list(S, list, cs, cb, px[r], py[r], pz[r])
                                    : csg_density(S, px[r], py[r], pz[r]);
                }
            }
#pragma unroll
            for (int r = 0; r < kCsgGroup; r++) {
                const uint32_t i = first + 64u * (uint32_t)(r0 + r) + (uint32_t)lane;
                const bool valid = i < ns;
                if (valid && !empty) dens[i] = d[r];
                const uint64_t bl = __ballot(valid && d[r] < 0.0f), vb = __ballot(valid);
                mine = lane == r0 + r ? bl : mine;
                air = air || bl != 0ull;
                solid = solid || bl != vb;
            }
        }
        wave_sync();  // the ids are read
        if (lane < words && w0 + lane < (int)M.lab_words) {
            const int left = (int)ns - 64 * (w0 + lane);
            A.labels[M.lab_off + w0 + lane] = mine;
            A.exact[M.lab_off + w0 + lane] = ~bits_from(left);
        }
        if (lane == 0) {
            if (air && !A.meta[j].any_air) atomicOr(&A.meta[j].any_air, 1u);
            if (solid && !A.meta[j].any_solid) atomicOr(&A.meta[j].any_solid, 1u);
        }
    }
    if (threadIdx.x == 0 && (int)blockIdx.x < A.stat_cap) A.stat_blocks[blockIdx.x] = 0ull;  // no octaves counted
}

// ------------------------------------------------------------------------
// count: one wave per item of kItemWords label words -> the words' edge and
// active-cell bits, their edge prefix, and the item's edges (vertices; quads
// in the quad mode) and cell counts (triangles; polygons in the quad mode).
// With REFINE it also gives every endpoint of a sign-changing edge that
// the adaptive sampling labelled early its full density.
//
// All 64 labels of a word meet their neighbours in a few 64-bit operations,
// so what is left per sample is done only for the few that the surface
// meets, compacted into dense lanes (a terrain item of 1,024 samples holds
// about 40 active cells).  A wave per label row with a lane per sample kept
// 3 % of its lanes busy: 512 chunks of 64^3 cells, 64 sampled, took 70 us
// and 23 more for the refinement as a kernel of its own; this takes 31 us.
// ------------------------------------------------------------------------
template <int REFINE>
__global__ void __launch_bounds__(kRowThreads) k_count(Arenas A) {
    __shared__ uint8_t s_n[256];  // triangles (polygons in the quad mode) of each corner mask
    __shared__ uint64_t s_corner[kWordWaves][kItemWords][8];
    __shared__ uint16_t s_list[kWordWaves][kItemSamples];
    __shared__ unsigned long long s_evals;
    if constexpr (REFINE) load_gradients();
    const bool quads = A.mesh_mode == BMF_MESH_QUADS;
    for (int t = threadIdx.x; t < 256; t += blockDim.x)
        s_n[t] = (uint8_t)(quads ? dmc_polygons(c_dmc_table[t]) : (uint32_t)((c_tri_table[t] >> 60) / 3));
    if (threadIdx.x == 0) s_evals = 0;
    __syncthreads();
    const SamplerDev* __restrict__ S = A.sampler;
    const int wave = uniform_int(threadIdx.x >> 6), lane = lane_id(), q = lane & 3;
    uint16_t* const list = s_list[wave];
    unsigned long long evals = 0;  // octaves of this wave's refined samples (uniform)
    const int64_t total = read_const(&A.ctr->total_items);
    for (int64_t it = (int64_t)blockIdx.x * kWordWaves + wave; it < total; it += (int64_t)gridDim.x * kWordWaves) {
        const ItemRef R = item_ref(A, it);
        const ChunkMeta& M = R.M;
        if (!(M.any_air && M.any_solid)) {  // no surface in this chunk: nothing reads its words
            if (lane == 0) A.item_e[it] = A.item_c[it] = 0u;
            continue;
        }
        const int dim = M.dim, d2 = dim * dim, nw = (int)M.lab_words;
        const int w = R.w0 + (lane >> 2);
        const uint64_t* __restrict__ L = A.labels + M.lab_off;
        uint64_t c[8];
        moved_labels(L, nw, w, 0, c[0], c[1]);
        moved_labels(L, nw, w, dim, c[2], c[3]);
        moved_labels(L, nw, w, d2, c[4], c[5]);
        moved_labels(L, nw, w, d2 + dim, c[6], c[7]);
        uint64_t lz = c[0], ly = c[0], lx = c[0];  // the neighbours below, for the refinement
        if constexpr (REFINE) {
            uint64_t unused;
            moved_labels(L, nw, w, -1, lz, unused);
            moved_labels(L, nw, w, -dim, ly, unused);
            moved_labels(L, nw, w, -d2, lx, unused);
        }
        uint64_t diff = 0;
#pragma unroll
        for (int k = 1; k < 8; k++) diff |= c[0] ^ c[k];
        uint64_t field = 0ull;  // lane q of a word's four keeps its field q
        uint32_t ne = 0u, nc = 0u;
        // items inside one uniform region end here (labels past the bitmap
        // and across row ends only cost the shortcut)
        if (__any((diff | (c[0] ^ lz) | (c[0] ^ ly) | (c[0] ^ lx)) != 0ull)) {
            const WordFaces f = word_faces(64 * w, dim, row_period(dim));
            uint64_t ex = (c[0] ^ c[4]) & f.in & ~f.x1, ey = (c[0] ^ c[2]) & f.in & ~f.y1,
                     ez = (c[0] ^ c[1]) & f.in & ~f.z1;
            const uint64_t ac = diff & f.in & ~(f.x1 | f.y1 | f.z1);
            uint64_t need = 0ull;
            if constexpr (REFINE) {
                const uint64_t ep = ex | ey | ez | ((c[0] ^ lz) & ~f.z0) | ((c[0] ^ ly) & ~f.y0) | ((c[0] ^ lx) & ~f.x0);
                need = ep & f.in & ~(w < nw ? A.exact[M.lab_off + w] : 0ull);
            }
            if (quads) {  // only the edges whose four cells lie in the chunk carry a quad
                const uint64_t x = f.x0 | f.x1, y = f.y0 | f.y1, z = f.z0 | f.z1;
                ex &= ~(y | z);
                ey &= ~(x | z);
                ez &= ~(x | y);
            }
            field = q == 0 ? ex : (q == 1 ? ey : (q == 2 ? ez : ac));
            // edges before each word within the item
            const uint32_t pre = wave_prefix<8>(
                q == 0 ? (uint32_t)(__popcll(ex) + __popcll(ey) + __popcll(ez)) : 0u, ne);
            if (q == 0 && w < nw) A.word_pre[M.lab_off + w] = pre;
            // cells
            s_corner[wave][lane >> 2][2 * q] = q == 0 ? c[0] : (q == 1 ? c[2] : (q == 2 ? c[4] : c[6]));
            s_corner[wave][lane >> 2][2 * q + 1] = q == 0 ? c[1] : (q == 1 ? c[3] : (q == 2 ? c[5] : c[7]));
            const int ncell = push_bits(ac, list);
            wave_sync();
            for (int e0 = 0; e0 < ncell; e0 += 64) {
                uint32_t n = 0;
                if (e0 + lane < ncell) {
                    const uint32_t pos = list[e0 + lane];
                    const uint32_t* cw = reinterpret_cast<const uint32_t*>(s_corner[wave][pos >> 6]) + ((pos >> 5) & 1u);
                    uint32_t mask = 0;
#pragma unroll
                    for (int k = 0; k < 8; k++) mask |= ((cw[2 * k] >> (pos & 31u)) & 1u) << k;
                    n = s_n[mask];
                }
                nc += (uint32_t)__popcll(__ballot(n & 1u)) + 2u * (uint32_t)__popcll(__ballot(n & 2u)) +
                      4u * (uint32_t)__popcll(__ballot(n & 4u));
            }
            if constexpr (REFINE) {
                wave_sync();  // the cells are read
                const int nq = push_bits(need, list);
                wave_sync();
                if constexpr (REFINE == kRefineTerrain) evals += (unsigned long long)nq * (unsigned long long)S->octaves;
                const float rd = 1.0f / (float)dim, rd2 = 1.0f / (float)d2;
                for (int e = lane; e < nq; e += 64) {
                    const uint32_t i = 64u * (uint32_t)R.w0 + list[e];
                    const uint32_t x = udiv24(i, (uint32_t)d2, rd2), r = i - x * (uint32_t)d2;
                    const uint32_t y = udiv24(r, (uint32_t)dim, rd), z = r - y * (uint32_t)dim;
                    const float px = (float)x * M.delta + M.opos[0], py = (float)y * M.delta + M.opos[1],
                                pz = (float)z * M.delta + M.opos[2];
                    if constexpr (REFINE == kRefineTerrain) A.dens[M.dens_off + i] = terrain_density(*S, px, py, pz);
                    else A.dens[M.dens_off + i] = noise_density_from(*S, noise_value(*S, px, py, pz), py);
                }
            }
            wave_sync();  // the next item reuses the list and the corners
        } else if (q == 0 && w < nw) {
            A.word_pre[M.lab_off + w] = 0u;
        }
        if (w < nw) reinterpret_cast<uint64_t*>(A.edges + M.lab_off + w)[q] = field;
        if (lane == 0) {
            A.item_e[it] = ne;
            A.item_c[it] = nc;
        }
    }
    if constexpr (REFINE) {
        if (lane == 0 && evals) atomicAdd(&s_evals, evals);
        __syncthreads();
    }
    if (threadIdx.x == 0 && (int)blockIdx.x < A.stat_cap) A.stat_blocks[A.stat_cap + blockIdx.x] = s_evals;
}

// ------------------------------------------------------------------------
// scan: one block per chunk -> item bases, totals, output reservation, and the
// chunk's entries in the smoothing tile maps: the k-th chunk to get there goes
// to XCD k % 8, so that all its tiles run on one XCD and its positions,
// indices and centroids stay in that XCD's L2 (workgroups are dispatched to
// the 8 XCDs round-robin by block index; a different dispatch order only costs
// locality, and the order of the maps only which block does which tile).  Two
// launches that built the maps from an ordered list of the chunks took 11 us.
// ------------------------------------------------------------------------
// Chunks that run the smoothing kernels (K > 0 or normals, a mesh, fitted).
__device__ __forceinline__ bool smooths(const ChunkMeta& M, int normals) {
    return (M.iters > 0 || normals) && M.V > 0 && M.T > 0 && M.status == BMF_OK && M.state == kStateSampled;
}

constexpr int kScanThreads = 256;

__global__ void __launch_bounds__(kScanThreads) k_scan(Arenas A, int n) {
    constexpr int NW = kScanThreads / 64;
    // a chunk's tiles of 64 items, and the items of each that have edges or cells
    constexpr int kTiles = (BMF_MAX_DIM * BMF_MAX_DIM * BMF_MAX_DIM / kItemSamples + 63) / 64;
    __shared__ uint64_t s_some[kTiles];
    __shared__ uint32_t s_we[NW], s_wc[NW], s_wn[NW];  // wave totals
    __shared__ int s_work;                             // the chunk's first entry of the work list
    __shared__ SmoothTile s_tile;
    __shared__ int s_map[5];  // XCD, first vertex and triangle tile in its maps, their counts
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int j = blockIdx.x; j < n; j += gridDim.x) {
        ChunkMeta& M = A.meta[j];
        if (M.state != kStateSampled) continue;
        const int dim = M.dim;
        const int64_t R = (M.lab_words + kItemWords - 1) / kItemWords;
        uint32_t* re = A.item_e + M.item_slot;
        uint32_t* rc = A.item_c + M.item_slot;
        // exclusive scan of the items: each wave scans a contiguous run of
        // 64-item tiles (coalesced, wave shuffles, a running carry; four tiles'
        // loads issued together), then one exchange of the wave totals and a
        // second pass that adds each wave's base
        const int64_t ntile = (R + 63) / 64;
        const int64_t tpw = (ntile + NW - 1) / NW;
        const int64_t t0 = (int64_t)wave * tpw, t1 = t0 + tpw < ntile ? t0 + tpw : ntile;
        uint32_t we = 0, wc = 0, wn = 0;  // running totals of this wave's run
        for (int64_t tg = t0; tg < t1; tg += 4) {
            uint32_t ae[4], ac[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int64_t r = (tg + k) * 64 + lane;
                const bool in = tg + k < t1 && r < R;
                ae[k] = in ? re[r] : 0u;
                ac[k] = in ? rc[r] : 0u;
            }
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (tg + k >= t1) break;
                const uint32_t se = wave_scan(ae[k]), sc = wave_scan(ac[k]);
                const int64_t r = (tg + k) * 64 + lane;
                if (r < R) {
                    re[r] = we + se - ae[k];
                    rc[r] = wc + sc - ac[k];
                }
                we += (uint32_t)__builtin_amdgcn_readlane((int)se, 63);
                wc += (uint32_t)__builtin_amdgcn_readlane((int)sc, 63);
                const uint64_t some = __ballot((ae[k] | ac[k]) != 0u);
                wn += (uint32_t)__popcll(some);
                if (lane == 0) s_some[tg + k] = some;
            }
        }
        if (lane == 0) {
            s_we[wave] = we;
            s_wc[wave] = wc;
            s_wn[wave] = wn;
        }
        __syncthreads();
        uint32_t be = 0, bc = 0, bn = 0, te = 0, tc = 0, tn = 0;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const uint32_t xe = s_we[w], xc = s_wc[w], xn = s_wn[w];
            if (w < wave) {
                be += xe;
                bc += xc;
                bn += xn;
            }
            te += xe;
            tc += xc;
            tn += xn;
        }
        if (be | bc)
            for (int64_t t = t0; t < t1; t++) {
                const int64_t r = t * 64 + lane;
                if (r < R) {
                    re[r] += be;
                    rc[r] += bc;
                }
            }
        // triangles: a vertex per edge; quads: a vertex per polygon, a
        // quad (or two triangles) per edge
        const bool quads = A.mesh_mode == BMF_MESH_QUADS;
        const uint32_t V = quads ? tc : te, T = quads ? te * (A.quad_tris ? 2u : 1u) : tc;
        if (wave == 0) {
            // the chunk's output range, a lane per counter so that the four
            // additions, the map's turn and the work list's room take one
            // round trip together
            const uint64_t ni = (uint64_t)M.ipp * T;
            unsigned long long got = 0;
            if (V > 0 && lane < 4) {
                unsigned long long* at = lane == 0   ? &A.ctr->v_bump
                                         : lane == 1 ? &A.ctr->i_bump
                                         : lane == 2 ? &A.ctr->need_v
                                                     : &A.ctr->need_i;
                got = atomicAdd(at, lane & 1 ? ni : (unsigned long long)V);
            }
            int g = 0;
            if (V > 0 && T > 0 && lane == 4) g = atomicAdd(&A.ctr->n_smooth, 1) & (kXcds - 1);
            if (lane == 5 && tn) g = atomicAdd(&A.ctr->n_work, (int)tn);
            const int64_t vo = (int64_t)__shfl((long long)got, 0), io = (int64_t)__shfl((long long)got, 1);
            const int work = __shfl(g, 5);
            g = __shfl(g, 4);
            // every lane forms the record's new fields, lane 0 writes them
            ChunkMeta m = M;
            m.V = (int32_t)V;
            m.T = (int32_t)T;
            m.contains_mesh = m.any_air && (m.any_solid || (dim % 32 != 0));
            if (V > 0) {
                if (vo + V > A.cap_vertices || io + (int64_t)ni > A.cap_indices) m.status = BMF_ECAPACITY;
                m.v_off = vo;
                m.i_off = io;
            }
            const bool on = smooths(m, A.normals);
            const int vt = on ? (int)((V + kSmoothThreads - 1) / kSmoothThreads) : 0;
            const int tt = on ? (int)((T + kSmoothThreads - 1) / kSmoothThreads) : 0;
            int at = 0;
            if (on && lane < 2) at = atomicAdd(lane == 0 ? &A.ctr->xcd_vtiles[g] : &A.ctr->xcd_ttiles[g], lane == 0 ? vt : tt);
            if (lane == 0) {
                if (V > 0 && m.status == BMF_ECAPACITY) A.ctr->overflow = 1;
                M.V = m.V;
                M.T = m.T;
                M.contains_mesh = m.contains_mesh;
                M.status = m.status;
                M.v_off = m.v_off;
                M.i_off = m.i_off;
                write_result(A, j, m);
                s_tile = SmoothTile{j,        0, m.V, m.T, m.v_off, m.i_off, m.i_off / m.ipp,
                                    m.iters, (uint8_t)m.bp, (uint8_t)m.ipp, (uint16_t)m.dim};
                s_work = work;
                s_map[0] = g;
                s_map[3] = vt;
                s_map[4] = tt;
            }
            if (lane < 2) s_map[1 + lane] = at;
        }
        __syncthreads();
        int at = s_work + (int)bn;
        for (int64_t t = t0; t < t1; t++) {
            const uint64_t some = s_some[t];
            if ((some >> lane) & 1ull) A.work[at + (int)mbcnt64(some)] = make_int2(j, (int)(t * 64) + lane);
            at += (int)__popcll(some);
        }
        const int vt = s_map[3], tt = s_map[4];
        if (vt) {
            SmoothTile* __restrict__ VM = A.smooth_vmap + (int64_t)s_map[0] * A.cap_vtiles + s_map[1];
            SmoothTile* __restrict__ TM = A.smooth_tmap + (int64_t)s_map[0] * A.cap_ttiles + s_map[2];
            SmoothTile t = s_tile;
            for (int r = tid; r < vt; r += kScanThreads) {
                t.tile = r;
                VM[r] = t;
            }
            for (int r = tid; r < tt; r += kScanThreads) {
                t.tile = r;
                TM[r] = t;
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------
// emit: one wave per item of kItemWords label words.  The label and edge
// words around the item are staged in the wave's LDS windows; the samples
// that own sign-changing edges and the active cells are compacted, and dense
// lanes write them: a lane per sample places its up to three vertices, a
// lane per cell writes its up to five triangles, each corner's vertex id a
// prefix popcount of its word.  For chunks that smooth the cell's first
// triangle and mask are kept.
//
// Bound by the latency of an item's chain (map, record, windows, densities,
// stores), hidden by the waves in flight: 512 chunks of 64^3 cells, 719,423
// vertices and 1,406,794 triangles (29 MB written), took 126 us with a wave
// per row of samples and 3 % of its lanes busy; this takes 42 us.
// ------------------------------------------------------------------------
// Local edge e of a cell (the 12-edge numbering of DMCChunk.cpp:543-565):
// x-edges e = 2 dy + dz, y-edges e = 4 + 2 dx + dz, z-edges e = 8 + 2 dx + dy,
// the edge of axis `ax` starting at corner (dx, dy, dz); 5 bits per edge,
// dx | dy << 1 | dz << 2 | ax << 3.
__host__ __device__ constexpr uint64_t edge_corner_code(int e) {
    return e < 4 ? (uint64_t)(0 | ((e >> 1) << 1) | ((e & 1) << 2) | (0 << 3))
                 : e < 8 ? (uint64_t)(((e - 4) >> 1) | (0 << 1) | ((e & 1) << 2) | (1 << 3))
                         : (uint64_t)(((e - 8) >> 1) | ((e & 1) << 1) | (0 << 2) | (2 << 3));
}
__host__ __device__ constexpr uint64_t edge_corner_table() {
    uint64_t t = 0;
    for (int e = 0; e < 12; e++) t |= edge_corner_code(e) << (5 * e);
    return t;
}
constexpr uint64_t kEdgeCorners = edge_corner_table();

// The vertices of the item's samples (DMCChunk::calculate_isovertex,
// DMCChunk.cpp:657-674; a sample's in x, y, z edge order).
__device__ __forceinline__ void emit_vertices(const Arenas& A, const ChunkMeta& M, ItemWindows& s, int w0) {
    const int lane = lane_id(), k4 = lane >> 2, dim = M.dim, d2 = dim * dim;
    const int ns = push_bits(s.ex[k4] | s.ey[k4] | s.ez[k4], s.list);
    wave_sync();
    const int64_t vo = M.v_off;
    const uint32_t Vc = (uint32_t)M.V;
    const bool cells = M.iters > 0 || A.normals;  // the chunk runs the smoothing kernels
    // with K > 0 the last primal step writes the output position of every
    // vertex it moves (every vertex has a ring; boundary vertices move only
    // with boundary processing), so only the others are written here
    const bool moves = M.iters > 0 && A.smoothing_follows;
    const bool moves_boundary = moves && M.bp;
    float* __restrict__ P = A.pos + vo * 3;
    float4* __restrict__ P4 = cells ? A.pos4 + vo : nullptr;  // smoothing state
    float4* __restrict__ N4 = cells && A.normals ? A.nrm4 + vo : nullptr;
    uint8_t* __restrict__ B = A.boundary + vo;
    uint32_t* __restrict__ E = A.vedge + vo;
    const float* __restrict__ D = A.dens + M.dens_off;
    const float rd = 1.0f / (float)dim, rd2 = 1.0f / (float)d2;
    for (int e = lane; e < ns; e += 64) {
        const int pos = s.list[e], w = pos >> 6;
        const uint64_t bit = 1ull << (pos & 63), lt = bit - 1ull;
        const uint64_t ex = s.ex[w], ey = s.ey[w], ez = s.ez[w];
        const uint32_t fx = (ex & bit) != 0ull, fy = (ey & bit) != 0ull, fz = (ez & bit) != 0ull;
        uint32_t id = s.pre[w] + (uint32_t)(__popcll(ex & lt) + __popcll(ey & lt) + __popcll(ez & lt));
        // the sample and the far ends of its edges load together (an edge
        // that is not set reads the sample again)
        const uint32_t i = 64u * (uint32_t)w0 + (uint32_t)pos;
        const float s0 = D[i];
        const float e1[3] = {D[fx ? i + (uint32_t)d2 : i], D[fy ? i + (uint32_t)dim : i], D[fz ? i + 1u : i]};
        const int x = (int)udiv24(i, (uint32_t)d2, rd2), r = (int)i - x * d2;
        const int y = (int)udiv24((uint32_t)r, (uint32_t)dim, rd), z = r - y * dim;
        if (id + fx + fy + fz > Vc) {
            raise_error(A, 2);  // counts and ids disagree: report, never write past the chunk
            continue;
        }
#pragma unroll
        for (int ax = 0; ax < 3; ax++) {
            const uint32_t f = ax == 0 ? fx : (ax == 1 ? fy : fz);
            if (!f) continue;
            const int xe = x + (ax == 0), ye = y + (ax == 1), ze = z + (ax == 2);
            const float s1 = e1[ax];
            const float mu = (0.0f - s0) / (s1 - s0);
            const float dx = (float)xe - (float)x, dy = (float)ye - (float)y, dz = (float)ze - (float)z;
            const float qx = dx * mu + (float)x, qy = dy * mu + (float)y, qz = dz * mu + (float)z;
            const bool bnd = x == 0 || y == 0 || z == 0 || x == dim - 1 || y == dim - 1 || z == dim - 1 ||
                             xe == dim - 1 || ye == dim - 1 || ze == dim - 1;
            if (!(bnd ? moves_boundary : moves)) {
                P[3 * (int64_t)id + 0] = qx;
                P[3 * (int64_t)id + 1] = qy;
                P[3 * (int64_t)id + 2] = qz;
            }
            if (P4) P4[id] = make_float4(qx, qy, qz, 0.0f);
            if (N4) N4[id] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            B[id] = (uint8_t)bnd;
            E[id] = (uint32_t)x | ((uint32_t)y << 8) | ((uint32_t)z << 16) | ((uint32_t)ax << 24);
            id++;
        }
    }
}

// The triangles of the item's active cells, `tbase` before them.
__device__ __forceinline__ void emit_triangles(const Arenas& A, const ChunkMeta& M, ItemWindows& s,
                                               const WindowGeom& g, const uint8_t* s_ntri, const uint64_t* s_tri,
                                               int w0, uint32_t tbase) {
    const int lane = lane_id(), dim = M.dim;
    const int nc = push_bits(s.ac[lane >> 2], s.list);
    wave_sync();
    const uint32_t Vc = (uint32_t)M.V, Tc = (uint32_t)M.T;
    const bool cells = M.iters > 0 || A.normals;
    for (int e0 = 0; e0 < nc; e0 += 64) {
        int pos = 0;
        uint32_t mask = 0, nt = 0;
        if (e0 + lane < nc) {
            pos = s.list[e0 + lane];
            mask = window_mask(s, g, dim, pos);
            nt = s_ntri[mask];
        }
        uint32_t round;
        const uint32_t tb = tbase + wave_prefix<3>(nt, round);
        tbase += round;
        if (!nt) continue;
        if (tb + nt > Tc) {
            raise_error(A, 3);
            continue;
        }
        const uint64_t row = s_tri[mask];
        // per triangle: the three corner ids read together, written
        // together; an id past the chunk's vertices (counts and ids
        // disagree) is reported, its slot is inside the chunk's range
        uint32_t* __restrict__ I = A.idx + M.i_off + 3ll * tb;
        bool bad = false;
        // at most 5 triangles per cell: unrolled, so each slot's table bits
        // are a constant field of the row
#pragma unroll
        for (int q = 0; q < 5; q++) {
            if (q >= (int)nt) break;
            uint32_t v[3];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const uint32_t le = (uint32_t)(row >> (4 * (3 * q + c))) & 15u;
                const uint32_t code = (uint32_t)(kEdgeCorners >> (5u * le)) & 31u;
                v[c] = window_edge(s, g, dim, pos, (int)(code & 1u), (int)((code >> 1) & 1u), (int)((code >> 2) & 1u),
                                   (int)(code >> 3));
                bad = bad || v[c] >= Vc;
            }
            I[3 * q] = v[0];
            I[3 * q + 1] = v[1];
            I[3 * q + 2] = v[2];
        }
        if (bad) raise_error(A, 4);
        if (cells) {
            const int64_t ci = M.dens_off + 64ll * w0 + pos;
            A.cell_tb[ci] = tb;
            A.cell_mask[ci] = (uint8_t)mask;
        }
    }
}

__global__ void __launch_bounds__(kRowThreads) k_emit(Arenas A, int n) {
    __shared__ ItemWindows s_win[kWordWaves];
    __shared__ uint64_t s_tri[256];  // the triangle table
    __shared__ uint8_t s_ntri[256];
    for (int t = threadIdx.x; t < 256; t += blockDim.x) {
        s_tri[t] = c_tri_table[t];
        s_ntri[t] = (uint8_t)((c_tri_table[t] >> 60) / 3);
    }
    publish(A, n);
    __syncthreads();
    const int wave = uniform_int(threadIdx.x >> 6);
    ItemWindows& s = s_win[wave];
    const int total = read_const(&A.ctr->n_work);
    for (int w = blockIdx.x * kWordWaves + wave; w < total; w += gridDim.x * kWordWaves) {
        const ItemRef R = work_ref(A, w);
        const ChunkMeta& M = R.M;
        if (M.status != BMF_OK || M.V == 0) continue;
        const WindowGeom g = stage_windows(A, M, R.w0, s);
        emit_vertices(A, M, s, R.w0);
        wave_sync();  // the sample list is read
        emit_triangles(A, M, s, g, s_ntri, s_tri, R.w0, A.item_c[R.it]);
        wave_sync();  // the windows are read
    }
}

// ------------------------------------------------------------------------
// smoothing, iteration m of MeshProcessor<3> (MeshProcessor.cpp:130-306 as
// driven by ChunkGenerator.cpp:112-124), over the chunks with K > m:
//   k_dual   per triangle: centroid ((0 + p0) + p1) + p2, then / 3
//   k_primal per vertex: sum of the adjacent centroids from +0 in ascending
//            triangle id, / count; boundary vertices stay unless
//            boundary_processing.  The adjacent triangles come from the ring
//            of cells around the vertex's lattice edge (c_ring) and each
//            cell's table slots, which is ascending id order.
// Positions live in a float4 buffer during the iterations (updated in place
// by k_primal: k_dual has consumed them); the last iteration also writes the
// float3 output.
// ------------------------------------------------------------------------
__global__ void __launch_bounds__(kSmoothThreads) k_dual(Arenas A, int m) {
    for (SmoothTiles tiles(A.smooth_tmap, A.cap_ttiles, A.ctr->xcd_ttiles); tiles.next();) {
        const SmoothTile& M = tiles.t;
        const int64_t T = M.T, i_off = M.i_off, v_off = M.v_off;
        const uint32_t V = (uint32_t)M.V;
        if (M.iters <= m) continue;
        const int64_t t = (int64_t)M.tile * kSmoothThreads + threadIdx.x;
        if (t >= T) continue;
        const uint32_t* __restrict__ I = A.idx + i_off + 3 * t;
        const float4* __restrict__ P = A.pos4 + v_off;
        const uint32_t i0 = I[0], i1 = I[1], i2 = I[2];
        if (i0 >= V || i1 >= V || i2 >= V) {
            raise_error(A, 5);
            continue;
        }
        const float4 a = P[i0], b = P[i1], c = P[i2];
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
        A.cen4[M.t_off + t] = make_float4(cx / 3.0f, cy / 3.0f, cz / 3.0f, 0.0f);
    }
}

// A vertex's ring, packed: word c for ring cell c (the cells around the
// vertex's lattice edge in c_ring order) = the cell's first triangle | the
// bits of its triangles that use the edge << 27.  A chunk holds at most
// 5 * 255^3 < 2^27 triangles.  The first smoothing step packs it (four
// independent cell reads), later steps load it as one 16-byte word.
constexpr uint32_t kRingFirst = (1u << 27) - 1u;
constexpr int kRingRound = 8;  // centroids loaded per round (a ring has about six triangles)

// Ring cell c around an edge along `ax` is the edge origin offset by
// (c >> 1) - 1 and (c & 1) - 1 along the other two axes in x, y, z order,
// with local edge 4 ax + 3 - c: the rows of c_ring.
__device__ __forceinline__ uint4 pack_ring(const uint32_t* __restrict__ CT, const uint8_t* __restrict__ CM,
                                           uint32_t code, int dim, uint32_t T, bool& bad) {
    const int ex = (int)(code & 255u), ey = (int)((code >> 8) & 255u), ez = (int)((code >> 16) & 255u);
    const int ax = (int)(code >> 24);
    int64_t ci[4];
    bool in[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const int u = (c >> 1) - 1, w = (c & 1) - 1;
        const int cx = ex + (ax == 0 ? 0 : u), cy = ey + (ax == 0 ? u : (ax == 1 ? 0 : w)), cz = ez + (ax == 2 ? 0 : w);
        in[c] = cx >= 0 && cy >= 0 && cz >= 0 && cx <= dim - 2 && cy <= dim - 2 && cz <= dim - 2;
        ci[c] = in[c] ? ((int64_t)cx * dim + cy) * dim + cz : 0;
    }
    uint32_t tb[4], mk[4], r[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        tb[c] = CT[ci[c]];
        mk[c] = CM[ci[c]];
    }
#pragma unroll
    for (int c = 0; c < 4; c++) mk[c] = c_edge_tris.m[mk[c]][4 * ax + 3 - c];  // any mask byte is a valid row
#pragma unroll
    for (int c = 0; c < 4; c++) {
        uint32_t tm = in[c] ? mk[c] : 0u;
        if (tm && tb[c] + (uint32_t)(31 - __clz(tm)) >= T) {  // past the chunk's triangles
            bad = true;
            tm = 0u;
        }
        r[c] = (tm ? tb[c] & kRingFirst : 0u) | (tm << 27);
    }
    return make_uint4(r[0], r[1], r[2], r[3]);
}

// Sums of the ring's centroids (and face normals) from +0 in ascending
// triangle id, the order of MeshProcessor<3>'s adjacency lists; returns the
// ring size.  kRingRound centroids are loaded per round, a lane's unused slots
// reading its round's first triangle and adding nothing.
template <bool NRM>
__device__ __forceinline__ uint32_t ring_sums(uint4 r, const float4* __restrict__ C, const float4* __restrict__ F,
                                              float (&s)[6]) {
    uint32_t bits = (r.x >> 27) | ((r.y >> 27) << 5) | ((r.z >> 27) << 10) | ((r.w >> 27) << 15);
    const uint32_t cnt = (uint32_t)__popc(bits);
    // triangle of bit b = 5 c + slot: first(c) + slot = (first(c) - 5 c) + b, modulo 2^32
    const uint32_t f0 = r.x & kRingFirst, f1 = (r.y & kRingFirst) - 5u, f2 = (r.z & kRingFirst) - 10u,
                   f3 = (r.w & kRingFirst) - 15u;
    while (bits) {
        uint32_t t[kRingRound];
        bool ok[kRingRound];
#pragma unroll
        for (int k = 0; k < kRingRound; k++) {
            ok[k] = bits != 0u;
            const uint32_t b = ok[k] ? (uint32_t)(__ffs(bits) - 1) : 0u;
            const uint32_t f = b < 5u ? f0 : (b < 10u ? f1 : (b < 15u ? f2 : f3));
            t[k] = ok[k] ? f + b : (k == 0 ? 0u : t[0]);  // slot 0 is always used
            bits &= bits - 1u;
        }
        float4 q[kRingRound], n[kRingRound];
#pragma unroll
        for (int k = 0; k < kRingRound; k++) {
            q[k] = C[t[k]];
            if (NRM) n[k] = F[t[k]];
        }
#pragma unroll
        for (int k = 0; k < kRingRound; k++) {
            s[0] = ok[k] ? s[0] + q[k].x : s[0];
            s[1] = ok[k] ? s[1] + q[k].y : s[1];
            s[2] = ok[k] ? s[2] + q[k].z : s[2];
            if (NRM) {
                s[3] = ok[k] ? s[3] + n[k].x : s[3];
                s[4] = ok[k] ? s[4] + n[k].y : s[4];
                s[5] = ok[k] ? s[5] + n[k].z : s[5];
            }
        }
    }
    return cnt;
}

__global__ void __launch_bounds__(kSmoothThreads) k_primal(Arenas A, int m) {
    for (SmoothTiles tiles(A.smooth_vmap, A.cap_vtiles, A.ctr->xcd_vtiles); tiles.next();) {
        const SmoothTile& M = tiles.t;
        const int K = M.iters, dim = M.dim, bp = M.bp;
        const int64_t V = M.V, v_off = M.v_off, t_off = M.t_off;
        const uint32_t T = (uint32_t)M.T;
        if (K <= m) continue;
        const int64_t v = (int64_t)M.tile * kSmoothThreads + threadIdx.x;
        if (v >= V) continue;
        const int64_t g = v_off + v;
        // the boundary flag, the lattice edge and the packed ring load together
        const uint8_t bnd = A.boundary[g];
        const uint32_t code = m == 0 ? A.vedge[g] : 0u;
        uint4 r = m == 0 ? make_uint4(0u, 0u, 0u, 0u) : A.vring[g];
        if (!bp && bnd) continue;  // stays at its position in both buffers
        if (m == 0) {
            bool bad = false;
            const int64_t dens_off = A.meta[M.chunk].dens_off;
            r = pack_ring(A.cell_tb + dens_off, A.cell_mask + dens_off, code, dim, T, bad);
            if (bad) raise_error(A, 7);
        }
        float s[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        const uint32_t cnt = ring_sums<false>(r, A.cen4 + t_off, nullptr, s);
        if (m == 0 && K > 1) A.vring[g] = r;  // stored after the loads: a store here is waited for with them
        if (cnt == 0) {  // MeshProcessor.cpp:247: no adjacency, unchanged (the emit kernel left its output to here)
            if (m == K - 1) {
                const float4 q = A.pos4[g];
                float* __restrict__ P = A.pos + g * 3;
                P[0] = q.x;
                P[1] = q.y;
                P[2] = q.z;
            }
            continue;
        }
        const float fc = (float)cnt;
        const float px = s[0] / fc, py = s[1] / fc, pz = s[2] / fc;
        A.pos4[g] = make_float4(px, py, pz, 0.0f);
        if (m == K - 1) {
            float* __restrict__ P = A.pos + g * 3;
            P[0] = px;
            P[1] = py;
            P[2] = pz;
        }
    }
}


// With vertex normals (the smooth_normals branch of MeshProcessor<3>,
// MeshProcessor.cpp:159-216, 271-287, for N = 3): every chunk of the list
// runs max(K, 1) steps; step m's face normal is
// -cross(normalize(p0 - p1), normalize(p0 - p2)) while m == 0, m < max_norms
// (min(K/2 - 3, 10)) or m < 3, else the sum of its corners' normals; the
// primal step averages them over the ring for every vertex with a ring,
// normalises when m == 3 or (m == 0 and K <= 3) and keeps the result when
// its y is not 0; positions move as in k_dual/k_primal (K > 0 only); the
// last step writes the unit normal.
__global__ void __launch_bounds__(kSmoothThreads) k_dual_nrm(Arenas A, int m) {
    for (SmoothTiles tiles(A.smooth_tmap, A.cap_ttiles, A.ctr->xcd_ttiles); tiles.next();) {
        const SmoothTile& M = tiles.t;
        const int K = M.iters;
        if (max(K, 1) <= m) continue;
        const int64_t t = (int64_t)M.tile * kSmoothThreads + threadIdx.x;
        if (t >= M.T) continue;
        const uint32_t* __restrict__ I = A.idx + M.i_off + 3 * t;
        const float4* __restrict__ P = A.pos4 + M.v_off;
        const uint32_t i0 = I[0], i1 = I[1], i2 = I[2];
        if (i0 >= (uint32_t)M.V || i1 >= (uint32_t)M.V || i2 >= (uint32_t)M.V) {
            raise_error(A, 5);
            continue;
        }
        const float4 a = P[i0], b = P[i1], c = P[i2];
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
        const int64_t tt = M.t_off + t;
        A.cen4[tt] = make_float4(cx / 3.0f, cy / 3.0f, cz / 3.0f, 0.0f);
        const int max_norms = min(K / 2 - 3, 10);
        float4 fn;
        if (m == 0 || m < max_norms || m < 3) {
            float ux = a.x - b.x, uy = a.y - b.y, uz = a.z - b.z;
            float wx = a.x - c.x, wy = a.y - c.y, wz = a.z - c.z;
            const float lu = sqrtf((ux * ux + uy * uy) + uz * uz), lw = sqrtf((wx * wx + wy * wy) + wz * wz);
            ux = ux / lu;
            uy = uy / lu;
            uz = uz / lu;
            wx = wx / lw;
            wy = wy / lw;
            wz = wz / lw;
            fn = make_float4(-(uy * wz - wy * uz), -(uz * wx - wz * ux), -(ux * wy - wx * uy), 0.0f);
        } else {
            const float4* __restrict__ N = A.nrm4 + M.v_off;
            const float4 na = N[i0], nb = N[i1], nc = N[i2];
            float sx = 0.0f, sy = 0.0f, sz = 0.0f;
            sx = sx + na.x;
            sy = sy + na.y;
            sz = sz + na.z;
            sx = sx + nb.x;
            sy = sy + nb.y;
            sz = sz + nb.z;
            sx = sx + nc.x;
            sy = sy + nc.y;
            sz = sz + nc.z;
            fn = make_float4(sx, sy, sz, 0.0f);
        }
        A.fn4[tt] = fn;
    }
}

__global__ void __launch_bounds__(kSmoothThreads) k_primal_nrm(Arenas A, int m) {
    for (SmoothTiles tiles(A.smooth_vmap, A.cap_vtiles, A.ctr->xcd_vtiles); tiles.next();) {
        const SmoothTile& M = tiles.t;
        const int K = M.iters;
        const int steps = max(K, 1);
        if (steps <= m) continue;
        const int64_t v = (int64_t)M.tile * kSmoothThreads + threadIdx.x;
        if (v >= M.V) continue;
        const int64_t g = M.v_off + v, t_off = M.t_off;
        const int dim = M.dim, bp = M.bp;
        const uint32_t T = (uint32_t)M.T;
        uint4 r;
        if (m == 0) {
            bool bad = false;
            const int64_t dens_off = A.meta[M.chunk].dens_off;
            r = pack_ring(A.cell_tb + dens_off, A.cell_mask + dens_off, A.vedge[g], dim, T, bad);
            if (bad) raise_error(A, 7);
        } else {
            r = A.vring[g];
        }
        float s[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        const uint32_t cnt = ring_sums<true>(r, A.cen4 + t_off, A.fn4 + t_off, s);
        if (m == 0 && steps > 1) A.vring[g] = r;
        const float sx = s[0], sy = s[1], sz = s[2], nx = s[3], ny = s[4], nz = s[5];
        float4 n = A.nrm4[g];
        if (cnt > 0) {
            const float fc = (float)cnt;
            float ax2 = nx / fc, ay2 = ny / fc, az2 = nz / fc;
            const bool unit = m != steps - 1 && (m == 3 || (m == 0 && K <= 3));
            if (unit) {
                const float l = sqrtf((ax2 * ax2 + ay2 * ay2) + az2 * az2);
                ax2 = ax2 / l;
                ay2 = ay2 / l;
                az2 = az2 / l;
            }
            if (ay2 != 0.0f) {
                n = make_float4(ax2, ay2, az2, 0.0f);
                A.nrm4[g] = n;
            }
            if (K > 0 && (bp || !A.boundary[g])) {
                const float px = sx / fc, py = sy / fc, pz = sz / fc;
                A.pos4[g] = make_float4(px, py, pz, 0.0f);
                if (m == K - 1) {
                    float* __restrict__ P = A.pos + g * 3;
                    P[0] = px;
                    P[1] = py;
                    P[2] = pz;
                }
            }
        } else if (K > 0 && m == K - 1 && (bp || !A.boundary[g])) {
            // no ring: unchanged, and the emit kernel left its output to here
            const float4 q = A.pos4[g];
            float* __restrict__ P = A.pos + g * 3;
            P[0] = q.x;
            P[1] = q.y;
            P[2] = q.z;
        }
        if (m == steps - 1) {
            const float l = sqrtf((n.x * n.x + n.y * n.y) + n.z * n.z);
            float* __restrict__ O = A.nrm + g * 3;
            O[0] = l > 0.0f ? n.x / l : 0.0f;
            O[1] = l > 0.0f ? n.y / l : 0.0f;
            O[2] = l > 0.0f ? n.z / l : 0.0f;
        }
    }
}

__global__ void k_ref_labels(Arenas A, uint32_t* words) {
    const ChunkMeta& M = A.meta[0];
    const int dim = M.dim, zc = (dim + 31) / 32;
    const int64_t nwords = (int64_t)dim * dim * zc;
    for (int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; w < nwords; w += (int64_t)gridDim.x * blockDim.x) {
        const int64_t row = w / zc;
        const int zb = (int)(w - row * zc);
        const int x = (int)(row / dim), y = (int)(row - (int64_t)x * dim);
        uint32_t v = 0;
        if (M.state == kStateSampled) {
            const RowBits<kMaxRowWords> rb = load_row<kMaxRowWords>(A.labels + M.lab_off, M.lab_words, dim, x, y);
            const uint64_t q = word_at<kMaxRowWords>(rb, zb >> 1);
            v = (uint32_t)(q >> (32 * (zb & 1)));
        } else if (M.state == kStateAir) {
            const int nb = min(32, dim - 32 * zb);
            v = nb >= 32 ? 0xFFFFFFFFu : ((1u << nb) - 1u);
        }
        words[w] = v;
    }
}

// DMCChunk::label_edges masks [x][y][ceil(dim/8)], byte z%8 (DMCChunk.cpp:200-438)
__global__ void k_ref_masks(Arenas A, uint64_t* masks) {
    const ChunkMeta& M = A.meta[0];
    const int dim = M.dim, z8 = (dim + 7) / 8;
    const int64_t nwords = (int64_t)dim * dim * z8;
    for (int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; w < nwords; w += (int64_t)gridDim.x * blockDim.x) {
        const int64_t row = w / z8;
        const int zw = (int)(w - row * z8);
        const int x = (int)(row / dim), y = (int)(row - (int64_t)x * dim);
        constexpr int W = kMaxRowWords;
        RowBits<W> r00 = zero_row<W>(), r01 = zero_row<W>(), r10 = zero_row<W>(), r11 = zero_row<W>();
        if (M.state == kStateSampled) {
            const uint64_t* L = A.labels + M.lab_off;
            r00 = load_row<W>(L, M.lab_words, dim, x, y);
            r01 = load_row<W>(L, M.lab_words, dim, x, y + 1);
            r10 = load_row<W>(L, M.lab_words, dim, x + 1, y);
            r11 = load_row<W>(L, M.lab_words, dim, x + 1, y + 1);
        } else if (M.state == kStateAir) {
            RowBits<W> full = zero_row<W>();
            for (int k = 0; k < W; k++) {
                const int nb = dim - 64 * k;
                full.w[k] = nb >= 64 ? ~0ull : (nb > 0 ? (1ull << nb) - 1ull : 0ull);
            }
            r00 = full;
            if (y + 1 < dim) r01 = full;
            if (x + 1 < dim) r10 = full;
            if (x + 1 < dim && y + 1 < dim) r11 = full;
        }
        uint64_t v = 0;
        for (int b = 0; b < 8; b++) {
            const int z = 8 * zw + b;
            if (z >= dim) break;
            v |= (uint64_t)cell_mask<W>(r00, r01, r10, r11, z) << (8 * b);
        }
        masks[w] = v;
    }
}

// ------------------------------------------------------------------------
// launch wrappers
// ------------------------------------------------------------------------
hipError_t launch_plan(const Arenas& A, int n, int allow_cull, int reset_bumps, hipStream_t s,
                       const bmf_chunk_desc* one) {
    if (n <= kPlanShared) {
        hipLaunchKernelGGL(k_plan, dim3((n + kPlanSlice - 1) / kPlanSlice), dim3(kPlanThreads), 0, s, A, n, allow_cull,
                           reset_bumps, one ? *one : bmf_chunk_desc{}, one != nullptr);
    } else {
        const int nb = (n + kPlanThreads - 1) / kPlanThreads;
        if (nb > kPlanThreads) return hipErrorInvalidValue;  // beyond BMF's 2^20 chunks
        hipLaunchKernelGGL(k_plan_part, dim3(nb), dim3(kPlanThreads), 0, s, A, n, allow_cull);
        hipLaunchKernelGGL(k_plan_total, dim3(1), dim3(kPlanThreads), 0, s, A, n, nb, reset_bumps);
        hipLaunchKernelGGL(k_plan_fix, dim3(nb), dim3(kPlanThreads), 0, s, A, n, nb, allow_cull);
    }
    if (A.csg_list) hipLaunchKernelGGL(k_csg_cull, dim3((unsigned)(n < 2048 ? n : 2048)), dim3(256), 0, s, A, n);
    return hipGetLastError();
}
hipError_t launch_sample(const Arenas& A, int n, int blocks, int adaptive, int kind, int slab, hipStream_t s) {
    const dim3 g(blocks), b(kRowThreads);
    if (kind == BMF_SAMPLER_TERRAIN && adaptive) {
        hipLaunchKernelGGL(k_blocks, g, b, 0, s, A, n);
        hipLaunchKernelGGL(k_terrain, g, b, 0, s, A, n);
    } else if (kind == BMF_SAMPLER_TERRAIN) {
        hipLaunchKernelGGL((k_sample<kSampleTerrain, 4>), g, b, 0, s, A, n);
    } else if (kind == BMF_SAMPLER_NOISE && slab) {
        hipLaunchKernelGGL(k_columns, g, b, 0, s, A, n);
        hipLaunchKernelGGL((k_sample<kSampleField2, 16>), g, b, 0, s, A, n);
    } else if (kind == BMF_SAMPLER_NOISE && adaptive) {
        hipLaunchKernelGGL(k_field, g, b, 0, s, A, n);
    } else if (kind == BMF_SAMPLER_NOISE) {
        hipLaunchKernelGGL((k_sample<kSampleField3, 4>), g, b, 0, s, A, n);
    } else if (kind == BMF_SAMPLER_CSG) {
        hipLaunchKernelGGL(k_csg, g, b, 0, s, A, n, !adaptive);
    } else if (kind == BMF_SAMPLER_EXTERNAL) {
        hipLaunchKernelGGL((k_sample<kSampleExternal, 16>), g, b, 0, s, A, n);
    } else {
        hipLaunchKernelGGL((k_sample<kSampleImplicit, 16>), g, b, 0, s, A, n);
    }
    return hipGetLastError();
}
hipError_t launch_count(const Arenas& A, int blocks, int refine, hipStream_t s) {
    if (refine == kRefineTerrain)
        hipLaunchKernelGGL(k_count<kRefineTerrain>, dim3(blocks), dim3(kRowThreads), 0, s, A);
    else if (refine == kRefineField)
        hipLaunchKernelGGL(k_count<kRefineField>, dim3(blocks), dim3(kRowThreads), 0, s, A);
    else hipLaunchKernelGGL(k_count<kRefineNone>, dim3(blocks), dim3(kRowThreads), 0, s, A);
    return hipGetLastError();
}
hipError_t launch_scan(const Arenas& A, int n, int blocks, hipStream_t s) {
    hipLaunchKernelGGL(k_scan, dim3(blocks), dim3(kScanThreads), 0, s, A, n);
    return hipGetLastError();
}
hipError_t launch_emit(const Arenas& A, int n, int blocks, hipStream_t s) {
    hipLaunchKernelGGL(k_emit, dim3(blocks), dim3(kRowThreads), 0, s, A, n);
    return hipGetLastError();
}
hipError_t launch_smooth(const Arenas& A, int m, int blocks, hipStream_t s) {
    blocks = blocks < kXcds ? kXcds : blocks - blocks % kXcds;  // whole XCD groups
    if (A.normals) {
        hipLaunchKernelGGL(k_dual_nrm, dim3(blocks), dim3(kSmoothThreads), 0, s, A, m);
        hipLaunchKernelGGL(k_primal_nrm, dim3(blocks), dim3(kSmoothThreads), 0, s, A, m);
    } else {
        hipLaunchKernelGGL(k_dual, dim3(blocks), dim3(kSmoothThreads), 0, s, A, m);
        hipLaunchKernelGGL(k_primal, dim3(blocks), dim3(kSmoothThreads), 0, s, A, m);
    }
    return hipGetLastError();
}
hipError_t launch_ref_labels(const Arenas& A, uint32_t* words, hipStream_t s) {
    hipLaunchKernelGGL(k_ref_labels, dim3(512), dim3(256), 0, s, A, words);
    return hipGetLastError();
}
hipError_t launch_ref_masks(const Arenas& A, uint64_t* masks, hipStream_t s) {
    hipLaunchKernelGGL(k_ref_masks, dim3(512), dim3(256), 0, s, A, masks);
    return hipGetLastError();
}

}  // namespace bmf
