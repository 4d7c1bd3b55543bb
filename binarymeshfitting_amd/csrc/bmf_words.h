// The word kernels' work items: kItemWords consecutive words of a chunk's
// flat label bitmap (bit i = sample (x * dim + y) * dim + z), one wave per
// item.  Vertex, quad and cell order are the flat sample order, so that every
// prefix is one over words; the few samples and cells that the surface meets
// are compacted into dense lanes by the wave itself (no block barrier).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bmf_internal.h"
#include "bmf_rows.h"

namespace bmf {

constexpr int kWordWaves = kRowThreads / 64;  // items (waves) per workgroup
// A window of label and edge words around an item: the item's own words and
// those of the samples up to dim + 1 after its last one.
constexpr int kWindowWords = kItemWords + BMF_MAX_DIM / 64 + 2;

// Orders the wave's own LDS accesses (lanes exchange data through LDS).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Bits a .. 63 (any a).
__device__ __forceinline__ uint64_t bits_from(int a) { return a <= 0 ? ~0ull : (a >= 64 ? 0ull : ~0ull << a); }

// World box of the chunk's samples a .. a + count - 1, grown by `grow`
// sample steps along x and y (z spans the row): lo and hi per axis.
__device__ __forceinline__ void sample_box(const ChunkMeta& M, int a, int count, int grow, float (&lo)[3],
                                           float (&hi)[3]) {
    const int dim = M.dim, d2 = dim * dim, b = min(a + count, d2 * dim) - 1;
    const int xa = a / d2, xb = b / d2;
    const int ya = (a - xa * d2) / dim, yb = (b - xb * d2) / dim;
    const int c0[3] = {xa, xa == xb ? ya : 0, 0};
    const int c1[3] = {xb + grow, xa == xb ? yb + grow : dim - 1, dim - 1};
#pragma unroll
    for (int k = 0; k < 3; k++) {
        lo[k] = (float)c0[k] * M.delta + M.opos[k];
        hi[k] = (float)c1[k] * M.delta + M.opos[k];
    }
}

// The low four bits of each byte, packed.
__device__ __forceinline__ uint32_t low_nibbles(uint64_t w) {
    w &= 0x0F0F0F0F0F0F0F0Full;
    w = (w | (w >> 4)) & 0x00FF00FF00FF00FFull;
    w = (w | (w >> 8)) & 0x0000FFFF0000FFFFull;
    return (uint32_t)(w | (w >> 16));
}

// Exclusive prefix of a per-lane count below 2^BITS over the wave's lanes
// (bit-sliced ballots), and its total.
template <int BITS>
__device__ __forceinline__ uint32_t wave_prefix(uint32_t c, uint32_t& total) {
    uint32_t pre = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < BITS; i++) {
        const uint64_t b = __ballot((c >> i) & 1u);
        pre += mbcnt64(b) << i;
        tot += (uint32_t)__popcll(b) << i;
    }
    total = tot;
    return pre;
}

// Which of a word's samples lie on the chunk's faces: its last and first
// sample per axis; `in` those that exist.  per: bits 0, dim, 2 dim, ... below 64.
struct WordFaces {
    uint64_t in, x1, y1, z1, x0, y0, z0;
};
__device__ __forceinline__ uint64_t row_period(int dim) {
    uint64_t p = 0;
    for (int b = 0; b < 64; b += dim) p |= 1ull << b;
    return p;
}
__device__ __forceinline__ WordFaces word_faces(int i0, int dim, uint64_t per) {
    const int d2 = dim * dim, n3 = d2 * dim;
    const uint32_t x = udiv24((uint32_t)i0, (uint32_t)d2, 1.0f / (float)d2);
    const int q = i0 - (int)x * d2;  // offset within the x-plane
    const int z = q - (int)udiv24((uint32_t)q, (uint32_t)dim, 1.0f / (float)dim) * dim;
    WordFaces f;
    f.in = ~bits_from(n3 - i0);
    f.x1 = bits_from(n3 - d2 - i0);
    f.x0 = ~bits_from(d2 - i0);
    const int a1 = dim - 1 - z, a0 = z == 0 ? 0 : dim - z;
    f.z1 = a1 < 64 ? per << a1 : 0ull;
    f.z0 = a0 < 64 ? per << a0 : 0ull;
    // a plane's last row is its last dim samples, its first row the first
    f.y1 = f.y0 = 0ull;
    for (int a = d2 - dim - q; a < 64; a += d2) f.y1 |= bits_from(a) & ~bits_from(a + dim);
    for (int a = -q; a < 64; a += d2) f.y0 |= bits_from(a) & ~bits_from(a + dim);
    return f;
}

// The labels of the 64 samples of word w moved by o (c0) and by o + 1 (c1):
// two words of the bitmap, the same shift in every lane.  Samples outside
// the bitmap read 0; callers mask them by the faces.
__device__ __forceinline__ void moved_labels(const uint64_t* __restrict__ L, int nw, int w, int o, uint64_t& c0,
                                             uint64_t& c1) {
    const int q = w + (o >> 6), s = o & 63;
    const uint64_t a = L[min(max(q, 0), nw - 1)], b = L[min(max(q + 1, 0), nw - 1)];
    const uint64_t A = q >= 0 && q < nw ? a : 0ull, B = q + 1 >= 0 && q + 1 < nw ? b : 0ull;
    c0 = s ? (A >> s) | (B << (64 - s)) : A;
    c1 = ((A >> s) >> 1) | (B << (63 - s));
}

// Appends the set bits of the wave's kItemWords words to `list` in order, as
// 64 * word + bit: lane 4 k + q takes 16 bits of word k.  Returns their count.
__device__ __forceinline__ int push_bits(uint64_t word, uint16_t* list) {
    const int lane = lane_id(), k = lane >> 2, q = lane & 3;
    uint32_t b = (uint32_t)(word >> (16 * q)) & 0xFFFFu, total;
    uint32_t at = wave_prefix<5>((uint32_t)__popc(b), total);
    const uint32_t base = (uint32_t)(64 * k + 16 * q);
    while (b) {
        list[at++] = (uint16_t)(base + (uint32_t)(__ffs(b) - 1));
        b &= b - 1u;
    }
    return (int)total;
}

// The windows of one item, staged by its wave: window 0 from the item's
// first word, window 1 the same moved one x-plane on (its first sample is bit
// `off` of its first word).
struct ItemWindows {
    uint64_t ex[2 * kWindowWords], ey[2 * kWindowWords], ez[2 * kWindowWords];
    uint64_t lab[2 * kWindowWords + 1];  // a pad word: pairs are read across words
    uint32_t pre[2 * kWindowWords];      // edges of the chunk before the word
    uint64_t ac[kItemWords];             // the item's active cells
    uint16_t list[kItemSamples];
};
static_assert(2 * kWindowWords <= 64, "a lane per window word");

struct WindowGeom {
    int n0;   // words of window 0; window 1 follows
    int off;  // first bit of window 1
};

__device__ __forceinline__ WindowGeom stage_windows(const Arenas& A, const ChunkMeta& M, int w0, ItemWindows& s) {
    const int lane = lane_id(), dim = M.dim, d2 = dim * dim, nw = (int)M.lab_words;
    WindowGeom g;
    g.off = d2 & 63;
    g.n0 = ((kItemSamples + dim) >> 6) + 1;
    const int n1 = ((g.off + kItemSamples + dim) >> 6) + 1;
    if (lane < g.n0 + n1) {
        const int w = lane < g.n0 ? w0 + lane : w0 + (d2 >> 6) + lane - g.n0;
        EdgeWord e{0ull, 0ull, 0ull, 0ull};
        uint64_t l = 0ull;
        uint32_t p = 0u;
        if (w < nw) {
            e = A.edges[M.lab_off + w];
            l = A.labels[M.lab_off + w];
            p = A.item_e[M.item_slot + w / kItemWords] + A.word_pre[M.lab_off + w];
        }
        s.ex[lane] = e.ex;
        s.ey[lane] = e.ey;
        s.ez[lane] = e.ez;
        s.lab[lane] = l;
        s.pre[lane] = p;
        if (lane < kItemWords) s.ac[lane] = e.ac;
    }
    if (lane == 0) s.lab[g.n0 + n1] = 0ull;
    wave_sync();
    return g;
}

// Labels of samples p and p + 1 (bits of a window from its first word), as
// bits 0 and 1.
__device__ __forceinline__ uint32_t label_pair(const uint64_t* win, int p) {
    const uint32_t* w = reinterpret_cast<const uint32_t*>(win) + (p >> 5);
    return __builtin_amdgcn_alignbit(w[1], w[0], (uint32_t)(p & 31)) & 3u;
}

// Corner mask of the item's cell at sample `pos`: corner bit 4 dx + 2 dy + dz
// (DMCChunk.cpp:200-438).
__device__ __forceinline__ uint32_t window_mask(const ItemWindows& s, const WindowGeom& g, int dim, int pos) {
    const uint64_t* w1 = s.lab + g.n0;
    return label_pair(s.lab, pos) | (label_pair(s.lab, pos + dim) << 2) | (label_pair(w1, g.off + pos) << 4) |
           (label_pair(w1, g.off + pos + dim) << 6);
}

// Edges of the chunk before axis `ax` of the sample dx planes, dy rows and dz
// samples from the item's sample `pos` (a vertex id in the triangle mode, a
// quad id in the quad mode).
__device__ __forceinline__ uint32_t window_edge(const ItemWindows& s, const WindowGeom& g, int dim, int pos, int dx,
                                                int dy, int dz, int ax) {
    const int p = pos + dy * dim + dz + (dx ? g.off : 0);
    const int w = (p >> 6) + (dx ? g.n0 : 0);
    const uint64_t bit = 1ull << (p & 63), lt = bit - 1ull, le = lt | bit;
    return s.pre[w] + (uint32_t)__popcll(s.ex[w] & (ax >= 1 ? le : lt)) +
           (uint32_t)__popcll(s.ey[w] & (ax == 2 ? le : lt)) + (uint32_t)__popcll(s.ez[w] & lt);
}

// (chunk, item within the chunk) of work item `it`, and the chunk's record.
struct ItemRef {
    int64_t it;  // the item
    int w0;      // its first word
    ChunkMeta M;
};
__device__ __forceinline__ ItemRef item_ref(const Arenas& A, int64_t it) {
    const int2 m = read_const(A.item_map + it);
    return ItemRef{it, uniform_int(m.y) * kItemWords, read_chunk(A.meta, m.x)};
}
// Entry w of the list of items with edges or cells.
__device__ __forceinline__ ItemRef work_ref(const Arenas& A, int w) {
    const int2 m = read_const(A.work + w);
    const int item = uniform_int(m.y);
    ItemRef r{0, item * kItemWords, read_chunk(A.meta, m.x)};
    r.it = r.M.item_slot + item;
    return r;
}

}  // namespace bmf
