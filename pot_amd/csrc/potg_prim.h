// potg_prim.h -- device primitives (scans, radix sort) used by
// the step pipeline.  All launches go to the given stream; none allocates.
#pragma once

#include "potg_dev.h"

namespace potg {

// A scan over many blocks is two launches, each also doing the work around
// it: the first computes its tile's elements and leaves the tile's sum in
// `part`, the second adds up the sums of the tiles before its own
// (sum_before: a load or two per thread below a million elements) and scans
// its tile.  A launch of its own for the scan of the sums costs 4.5 us; adding
// them up in every block costs the square of their number, which from
// SCAN_SUMS tiles on is more: tree and targets of 16M / 32M / 64M / 200M particles
// 3.43 / 7.50 / 16.6 / 91.6 ms without that launch, 3.39 / 7.42 / 17.0 / 82.5 with.
constexpr int SCAN_BT = 256;               // threads of a scanning block
constexpr int SCAN_IPT = 4;                // elements per thread
constexpr int SCAN_TILE = SCAN_BT * SCAN_IPT;
constexpr uint32_t SCAN_SUMS = 65536;
inline uint32_t scan_blocks(uint32_t n) { return n ? (n + SCAN_TILE - 1) / SCAN_TILE : 1; }

// inclusive scan across a wavefront
__device__ inline uint32_t wave_incl_scan(uint32_t v)
{
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        uint32_t o = __shfl_up(v, d, WAVE);
        if ((int)__lane_id() >= d) v += o;
    }
    return v;
}

// exclusive scan of one value per thread over a SCAN_BT-thread block
__device__ inline uint32_t block_excl_scan(uint32_t v, uint32_t* sh_w, uint32_t* total)
{
    const int w = threadIdx.x / WAVE;
    uint32_t inc = wave_incl_scan(v);
    if (__lane_id() == WAVE - 1) sh_w[w] = inc;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < SCAN_BT / WAVE; k++) {
        if (k < w) off += sh_w[k];
        tot += sh_w[k];
    }
    __syncthreads();
    if (total) *total = tot;
    return off + inc - v;
}

// between a scan's two launches over nb tiles, where that pays: part[b] becomes
// the sum of part[0..b), and the result is what sum_before takes as `summed`
int scan_sums(uint32_t* part, uint32_t nb, hipStream_t s);

// the sum of part[0..b), in every thread of the block
__device__ inline uint32_t sum_before(const uint32_t* __restrict__ part, uint32_t b, int summed,
                                      uint32_t* sh_w)
{
    if (summed) return part[b];
    uint32_t v = 0, total;
    for (uint32_t i = threadIdx.x; i < b; i += SCAN_BT) v += part[i];
    block_excl_scan(v, sh_w, &total);
    return total;
}

// exclusive scan of the tile in sh (SCAN_TILE values, sh[j] for element j),
// in place, from `off`; returns the tile's sum.  Barriers on both sides.
__device__ inline uint32_t tile_excl_scan(uint32_t* sh, uint32_t off, uint32_t* sh_w)
{
    __syncthreads();
    uint32_t loc[SCAN_IPT], s = 0, total;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        loc[k] = s;
        s += sh[threadIdx.x * SCAN_IPT + k];
    }
    const uint32_t o = off + block_excl_scan(s, sh_w, &total);
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) sh[threadIdx.x * SCAN_IPT + k] = o + loc[k];
    __syncthreads();
    return total;
}

size_t radix_temp_words(uint32_t n);
// Stable LSD sort of (keys, vals) on bits [0, end_bit); the sorted data end
// up in keys/vals (the pointers are swapped with the _alt buffers as needed).
// ipt: elements per thread of a tile, 8 or 16 (tiles of 2048 or 4096).
void radix_sort_pairs(uint64_t*& keys, uint64_t*& keys_alt, uint32_t*& vals, uint32_t*& vals_alt,
                      uint32_t n, int end_bit, uint32_t* temp, int ipt, hipStream_t s);

// The same order for fewer keys than MERGE_MAX: tiles of MERGE_TILE sorted by
// the kernel that computes the keys (sort_tile), then merged a few at a time.
// The tiles lie in keys/vals if the passes are even in number, else in the
// _alt buffers; the sorted data end up in keys/vals.  Keys and sort, us, at
// 16k / 150k / 300k / 500k / 800k / 1.2M particles: by digits 165 / 172 / 180 /
// 195 / 204 / 236, merging 24 / 42 / 78 / 108 / 170 / 280
constexpr uint32_t MERGE_MAX = 900000;
constexpr int MERGE_TILE = 1024;
// passes and ways of a pass: the fewest passes that `most` ways allow, and the
// fewest ways for them.  Where a pass is its launch and the latency of a
// search, many ways are best; where it is the searches, few: all passes of
// at most 8 / 6 / 4 ways take, us, at 16k 15 / 14 / 18, 60k 16 / 22 / 20, 150k
// 39 / 31 / 33, 300k 60 / 66 / 61, 800k 202 / 156 / 137
inline uint32_t merge_ways(uint32_t n, uint32_t* passes)
{
    const uint32_t most = n <= 65536u ? 8u : (n <= 250000u ? 6u : 4u);
    uint64_t len = MERGE_TILE;
    uint32_t p = 0;
    for (; len < n; len *= most) p++;
    *passes = p;
    for (uint32_t w = 2;; w++) {
        len = MERGE_TILE;
        for (uint32_t k = 0; k < p; k++) len *= w;
        if (len >= n) return w;
    }
}
inline uint32_t merge_passes(uint32_t n)
{
    uint32_t p;
    merge_ways(n, &p);
    return p;
}
void merge_tiles(uint64_t* keys, uint64_t* keys_alt, uint32_t* vals, uint32_t* vals_alt, uint32_t n,
                 hipStream_t s);

struct TileSort {
    uint64_t key[2][MERGE_TILE];
    uint16_t idx[2][MERGE_TILE];
};

// lane ^ X's value, X below 4
template <int X>
__device__ inline uint32_t quad_xor(uint32_t v)
{
    constexpr int P = (0 ^ X) | (1 ^ X) << 2 | (2 ^ X) << 4 | (3 ^ X) << 6;
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, P, 0xf, 0xf, true);
}
template <int X>
__device__ inline uint32_t quad_before(uint64_t key)
{
    const uint64_t o =
        (uint64_t)quad_xor<X>((uint32_t)(key >> 32)) << 32 | quad_xor<X>((uint32_t)key);
    const uint32_t l = threadIdx.x & 3;
    return (o < key) | ((o == key) & ((l ^ X) < l));
}

// A block of MERGE_TILE threads sorts its threads' keys, equal keys in thread
// order: runs of four by comparing all pairs, then four times four runs into
// one, every element searching the three others.  Thread t gets the t-th key
// and the thread it came from.
__device__ inline void sort_tile(TileSort& sh, uint64_t& key, uint32_t& idx)
{
    const uint32_t t = threadIdx.x;
    const uint32_t to4 = (t & ~3u) + quad_before<1>(key) + quad_before<2>(key) + quad_before<3>(key);
    sh.key[0][to4] = key;
    sh.idx[0][to4] = (uint16_t)t;
    __syncthreads();
    int cur = 0;
#pragma unroll
    for (uint32_t len = 4; len < (uint32_t)MERGE_TILE; len *= 4) {
        key = sh.key[cur][t];
        idx = sh.idx[cur][t];
        const uint32_t g0 = t / (4 * len) * (4 * len), own = t / len & 3;
        uint32_t pos[3] = {};
#pragma unroll
        for (uint32_t h = len; h; h >>= 1) {
#pragma unroll
            for (uint32_t k = 0; k < 3; k++) {
                const uint32_t r = k + (k >= own), e = pos[k] + h;
                const uint64_t o = sh.key[cur][g0 + r * len + (e <= len ? e : 1) - 1];
                const bool before = (o < key) | ((o == key) & (r < own));
                pos[k] = (e <= len) & before ? e : pos[k];
            }
        }
        const uint32_t to = g0 + (t & (len - 1)) + pos[0] + pos[1] + pos[2];
        cur ^= 1;
        sh.key[cur][to] = key;
        sh.idx[cur][to] = (uint16_t)idx;
        __syncthreads();
    }
    key = sh.key[cur][t];
    idx = sh.idx[cur][t];
}

}  // namespace potg
