// potg_prim.h -- device primitives (scans, radix sort) used by
// the step pipeline.  All launches go to the given stream; none allocates.
#pragma once

#include "potg_dev.h"

namespace potg {

// A scan over many blocks is two launches, each also doing the work around
// it: the first computes its tile's elements and leaves the tile's sum in
// `part`, the second adds up the sums of the tiles before its own
// (sum_before: a load or two per thread below a million elements) and scans
// its tile.  (A launch of its own for the scan of the sums cost 4.5 us.)
constexpr int SCAN_BT = 256;               // threads of a scanning block
constexpr int SCAN_IPT = 4;                // elements per thread
constexpr int SCAN_TILE = SCAN_BT * SCAN_IPT;
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

// the sum of part[0..b), in every thread of the block
__device__ inline uint32_t sum_before(const uint32_t* __restrict__ part, uint32_t b, uint32_t* sh_w)
{
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

}  // namespace potg
