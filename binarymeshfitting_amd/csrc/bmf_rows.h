// Helpers shared by the kernels: wave and block primitives, the chunk table
// and sample coordinates, and label rows (samples (x, y, 0..dim-1)) as W u64
// words for the stage inspection.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bmf_internal.h"

namespace bmf {

// ------------------------------------------------------------------------
// small helpers
// ------------------------------------------------------------------------
__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63); }

__device__ __forceinline__ int uniform_int(int v) { return __builtin_amdgcn_readfirstlane(v); }

// A record at a wave-uniform address that the kernel itself never writes:
// read through the constant address space, so by scalar loads into scalar
// registers, whose latency is the shorter, and not again after the kernel's
// own stores (which the compiler cannot otherwise tell apart from it).
template <class T>
__device__ __forceinline__ T read_const(const T* p) {
    static_assert(sizeof(T) % 4 == 0, "records are read in 32-bit words");
    constexpr int kWords = (int)(sizeof(T) / 4);
    using ConstWords = const __attribute__((address_space(4))) uint32_t*;
    const ConstWords src = (ConstWords)p;
    uint32_t w[kWords];
#pragma unroll
    for (int i = 0; i < kWords; i++) w[i] = src[i];
    T r;
    __builtin_memcpy(&r, w, sizeof(T));
    return r;
}
// Chunk j of the chunk table.
__device__ __forceinline__ ChunkMeta read_chunk(const ChunkMeta* table, int j) {
    return read_const(table + uniform_int(j));
}

// The smoothing tiles of a block: those of its XCD's map, the record loaded
// beside the map's end.
struct SmoothTiles {
    const SmoothTile* map;
    int tile, step, last, end;
    SmoothTile t;
    __device__ __forceinline__ SmoothTiles(const SmoothTile* maps, int64_t cap, const int32_t* ends) {
        const int xcd = blockIdx.x % kXcds;
        map = maps + (int64_t)xcd * cap;
        tile = blockIdx.x / kXcds;
        step = gridDim.x / kXcds;
        last = (int)cap - 1;
        end = read_const(ends + xcd);
    }
    __device__ __forceinline__ bool next() {
        uint32_t w[sizeof(SmoothTile) / 4];
        const SmoothTile r = read_const(map + min(tile, last));
        __builtin_memcpy(w, &r, sizeof w);
        // all of it at once: left alone, the loads follow the branches that use them
#pragma unroll
        for (int i = 0; i < (int)(sizeof w / 4); i++) asm volatile("" : "+s"(w[i]));
        __builtin_memcpy(&t, w, sizeof w);
        const bool in = tile < end;
        tile += step;
        return in;
    }
};

// Counts and ids disagree, or a map entry is out of range: raised for the
// host, and nothing is written past the chunk.
__device__ __forceinline__ void raise_error(const Arenas& A, int code) {
    A.ctr->error = code;
    A.host_ctr->error = code;
}

// The results of the n chunks and the counters to the host, once the row scan
// is through, by the whole grid (written where they are formed, a lane per
// chunk, they held the plan up: 65,536 chunks 84 us instead of 27).
__device__ __forceinline__ void publish(const Arenas& A, int n) {
    static_assert(sizeof(bmf_chunk_result) % 8 == 0, "results are copied in 64-bit words");
    const int64_t words = (int64_t)n * (int64_t)(sizeof(bmf_chunk_result) / 8);
    const uint64_t* __restrict__ src = reinterpret_cast<const uint64_t*>(A.results);
    uint64_t* __restrict__ dst = reinterpret_cast<uint64_t*>(A.host_results);
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const Counters c = *A.ctr;
    Counters* h = A.host_ctr;
    h->v_bump = c.v_bump;
    h->i_bump = c.i_bump;
    h->need_v = c.need_v;
    h->need_i = c.need_i;
    h->total_samples = c.total_samples;
    h->overflow = c.overflow;
}

// Set bits of a wave mask below this lane.
__device__ __forceinline__ uint32_t mbcnt64(uint64_t w) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(w >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)w, 0u));
}

__device__ __forceinline__ uint64_t lanemask_lt() {
    const int l = lane_id();
    return l == 0 ? 0ull : (~0ull >> (64 - l));
}

// Exclusive prefix and total over a block of NT threads (NT / 64 <= 64
// waves) of N values per thread, one value at a time: lane shuffles inside
// each wave, then wave 0 scans the wave totals.  s_w: N x (NT / 64 + 1)
// scratch in LDS (the last column holds the totals).
template <int N, int NT>
__device__ __forceinline__ void block_scan(const int64_t (&v)[N], int64_t (&excl)[N], int64_t (&tot)[N],
                                           int64_t (*s_w)[NT / 64 + 1]) {
    constexpr int NW = NT / 64;
    const int lane = (int)(threadIdx.x & 63), w = (int)(threadIdx.x >> 6);
    int64_t inc[N];
    for (int q = 0; q < N; q++) {
        int64_t x = v[q];
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int64_t t = __shfl_up(x, off);
            if (lane >= off) x += t;
        }
        inc[q] = x;
        if (lane == 63) s_w[q][w] = x;
    }
    __syncthreads();
    if (w == 0) {
        for (int q = 0; q < N; q++) {
            const int64_t x = lane < NW ? s_w[q][lane] : 0;
            int64_t y = x;
#pragma unroll
            for (int off = 1; off < NW; off <<= 1) {
                const int64_t t = __shfl_up(y, off);
                if (lane >= off) y += t;
            }
            if (lane < NW) s_w[q][lane] = y - x;
            if (lane == NW - 1) s_w[q][NW] = y;
        }
    }
    __syncthreads();
    for (int q = 0; q < N; q++) {
        excl[q] = s_w[q][w] + inc[q] - v[q];
        tot[q] = s_w[q][NW];
    }
    __syncthreads();  // the scratch may be reused
}

// Inclusive prefix over the wave's lanes (row shifts and broadcasts, no LDS).
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false);  // row_shr 1, 2, 4, 8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);  // row_bcast 15, 31
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);
    return v;
}

// block_scan of values whose sum over a wave fits 32 bits: exclusive prefix
// and total as 64-bit values.
template <int N, int NT>
__device__ __forceinline__ void block_scan32(const uint32_t (&v)[N], int64_t (&excl)[N], int64_t (&tot)[N],
                                             uint32_t (*s_w)[NT / 64]) {
    constexpr int NW = NT / 64;
    const int lane = (int)(threadIdx.x & 63), w = (int)(threadIdx.x >> 6);
    uint32_t inc[N];
#pragma unroll
    for (int q = 0; q < N; q++) {
        inc[q] = wave_scan(v[q]);
        if (lane == 63) s_w[q][w] = inc[q];
    }
    __syncthreads();
    // every wave scans the (at most 16) wave totals, in 16-bit halves
    static_assert(NW <= 16, "wave totals in one row of lanes");
    const int uw = uniform_int(w);
#pragma unroll
    for (int q = 0; q < N; q++) {
        const uint32_t x = lane < NW ? s_w[q][lane] : 0u;
        const int lo = (int)wave_scan(x & 0xFFFFu), hi = (int)wave_scan(x >> 16);
        const int bl = uw ? __builtin_amdgcn_readlane(lo, uw - 1) : 0, bh = uw ? __builtin_amdgcn_readlane(hi, uw - 1) : 0;
        excl[q] = ((int64_t)bh << 16) + bl + (int64_t)(inc[q] - v[q]);
        tot[q] = ((int64_t)__builtin_amdgcn_readlane(hi, NW - 1) << 16) + __builtin_amdgcn_readlane(lo, NW - 1);
    }
    __syncthreads();  // the scratch may be reused
}

// The largest j in [0, n) with at(j) <= g, for at non-decreasing and
// at(0) <= g, by one wave: 64 probes a round, two dependent loads up to 4,096
// entries where a binary search has twelve.
template <class F>
__device__ __forceinline__ int find_wave(int n, int64_t g, F at) {
    const int lane = lane_id();
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int step = (hi - lo + 63) >> 6, i = lo + lane * step;
        const uint64_t ok = __ballot(i < hi && at(min(i, hi - 1)) <= g);
        lo += ((int)__popcll(ok) - 1) * step;
        hi = min(hi, lo + step);
    }
    return uniform_int(lo);
}
__device__ __forceinline__ int find_chunk_wave(const int64_t* __restrict__ prefix, int n, int64_t g) {
    return find_wave(n, g, [=](int j) { return prefix[j]; });
}
// The chunk that item `it` of the word kernels belongs to.
__device__ __forceinline__ int find_item_wave(const ChunkMeta* __restrict__ meta, int n, int64_t it) {
    return find_wave(n, it, [=](int j) { return meta[j].item_slot; });
}

// q = n / d for n <= 2^24, 0 < d < 2^24 and a quotient below 2^22, with
// rcp = 1/d correctly rounded.  (float)n is exact and fl(n * rcp) =
// (n/d)(1 + e) with |e| <= 2^-23 + 2^-48, so the estimate is within 0.5 of
// n/d and its truncation is floor(n/d) - 1, floor(n/d) or floor(n/d) + 1:
// one correction step each way, as selects, makes it exact.  (The sample
// coordinates divide by dim and dim^2 with quotients below 256.)
__device__ __forceinline__ uint32_t udiv24(uint32_t n, uint32_t d, float rcp) {
    int32_t q = (int32_t)((float)n * rcp);
    int32_t r = (int32_t)n - q * (int32_t)d;
    const bool lo = r < 0;
    q = lo ? q - 1 : q;
    r = lo ? r + (int32_t)d : r;
    q = r >= (int32_t)d ? q + 1 : q;
    return (uint32_t)q;
}

// A label row: bits z = 0..dim-1 of row (x, y) in W u64 words, W = ceil(dim/64).
template <int W>
struct RowBits {
    uint64_t w[W];
};

template <int W>
__device__ __forceinline__ RowBits<W> zero_row() {
    RowBits<W> r;
#pragma unroll
    for (int k = 0; k < W; k++) r.w[k] = 0ull;
    return r;
}

// Row (x, y) of a chunk's flat label bitmap: bits start at (x*dim + y)*dim.
template <int W>
__device__ __forceinline__ RowBits<W> load_row(const uint64_t* __restrict__ L, int64_t nwords, int dim, int x, int y) {
    RowBits<W> r = zero_row<W>();
    if (x < 0 || y < 0 || x >= dim || y >= dim) return r;
    const int64_t base = ((int64_t)x * dim + y) * dim;
#pragma unroll
    for (int k = 0; k < W; k++) {
        const int nb = dim - 64 * k;  // >= 1 because W = ceil(dim/64)
        const int64_t bit = base + 64 * k;
        const int64_t w = bit >> 6;
        const int sh = (int)(bit & 63);
        uint64_t v = L[w];
        if (sh) {
            const uint64_t hi = (w + 1 < nwords) ? L[w + 1] : 0ull;
            v = (v >> sh) | (hi << (64 - sh));
        }
        if (nb < 64) v &= (1ull << nb) - 1ull;
        r.w[k] = v;
    }
    return r;
}

template <int W>
__device__ __forceinline__ uint64_t word_at(const RowBits<W>& r, int k) {
    uint64_t v = 0ull;
#pragma unroll
    for (int q = 0; q < W; q++) v = k == q ? r.w[q] : v;
    return v;
}

template <int W>
__device__ __forceinline__ uint32_t bit_at(const RowBits<W>& r, int z) {
    return (uint32_t)((word_at<W>(r, z >> 6) >> (z & 63)) & 1ull);
}

// 8-corner mask of cell (x, y, z) from the four rows around it; corner bit
// 4dx + 2dy + dz (DMCChunk.cpp:200-438).
template <int W>
__device__ __forceinline__ uint32_t cell_mask(const RowBits<W>& r00, const RowBits<W>& r01, const RowBits<W>& r10,
                                              const RowBits<W>& r11, int z) {
    return bit_at<W>(r00, z) | (bit_at<W>(r00, z + 1) << 1) | (bit_at<W>(r01, z) << 2) |
           (bit_at<W>(r01, z + 1) << 3) | (bit_at<W>(r10, z) << 4) | (bit_at<W>(r10, z + 1) << 5) |
           (bit_at<W>(r11, z) << 6) | (bit_at<W>(r11, z + 1) << 7);
}

}  // namespace bmf
