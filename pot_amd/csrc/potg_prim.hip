// potg_prim.hip -- sorts for gfx950.
//
// Written for wave64: ranks inside a wavefront come from ballots, block
// partials through LDS.  Every routine takes an optional device-resident
// element count so that a captured step never needs a host round trip.
#include "potg_prim.h"

namespace potg {

namespace {

constexpr int BT = SCAN_BT;

__device__ inline uint32_t lane_id() { return __lane_id(); }

__device__ inline uint64_t lanemask_lt() { return (1ull << lane_id()) - 1ull; }

// exclusive scan of the tile sums, one block: 16 of them a thread in turn, so
// that 400000 (400M elements) take 25 turns
__global__ __launch_bounds__(1024) void k_scan_sums(uint32_t* __restrict__ part, uint32_t nb)
{
    constexpr int K = 16;
    __shared__ uint32_t sh_w[1024 / WAVE];
    uint32_t carry = 0;
    for (uint32_t b0 = 0; b0 < nb; b0 += 1024u * K) {
        const uint32_t i0 = b0 + threadIdx.x * K;
        uint32_t v[K], s = 0;
#pragma unroll
        for (int k = 0; k < K; k++) {
            v[k] = i0 + k < nb ? part[i0 + k] : 0u;
            s += v[k];
        }
        const uint32_t inc = wave_incl_scan(s);
        if (lane_id() == WAVE - 1) sh_w[threadIdx.x / WAVE] = inc;
        __syncthreads();
        uint32_t off = carry + inc - s;
        for (uint32_t w = 0; w < 1024 / WAVE; w++) {
            if (w < threadIdx.x / WAVE) off += sh_w[w];
            carry += sh_w[w];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (i0 + k < nb) part[i0 + k] = off;
            off += v[k];
        }
    }
}

// ---- radix sort -------------------------------------------------------
//
// 8-bit digits, three launches per pass: the digit counts of every tile of
// 256 x RS_IPT elements (k_rs_count), a scan of each digit's counts over the
// tiles (k_rs_scan, one block per digit), and k_rs_scatter, which ranks its
// tile stably by digit with wave ballots, stages it in LDS in digit order
// and then stores every digit's run to its global place, so that
// neighbouring lanes store to neighbouring addresses.  The tile is 2048 or
// 4096 elements (RS_IPT 8 or 16, picked by potg_tune): a smaller tile gives
// more blocks, and so fills the device, when the keys are few.

constexpr int RS_WAVES = BT / WAVE;

inline uint32_t rs_blocks(uint32_t n, int ipt) { return (n + BT * ipt - 1) / (BT * ipt); }

template <int RS_IPT>
__global__ __launch_bounds__(BT) void k_rs_count(const uint64_t* __restrict__ keys, uint32_t n,
                                                  int shift, uint32_t nb,
                                                  uint32_t* __restrict__ cnt)
{
    constexpr int RS_TILE = BT * RS_IPT;
    __shared__ uint32_t h[RS_WAVES][256];
#pragma unroll
    for (int k = 0; k < RS_WAVES; k++) h[k][threadIdx.x] = 0;
    __syncthreads();
    const int w = threadIdx.x / WAVE;
    const uint32_t base = blockIdx.x * RS_TILE;
    uint32_t d[RS_IPT];
#pragma unroll
    for (int k = 0; k < RS_IPT; k++) {
        const uint32_t i = base + k * BT + threadIdx.x;
        d[k] = i < n ? (uint32_t)(keys[i] >> shift) & 255u : 256u;
    }
#pragma unroll
    for (int k = 0; k < RS_IPT; k++)
        if (d[k] < 256u) atomicAdd(&h[w][d[k]], 1u);
    __syncthreads();
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < RS_WAVES; k++) c += h[k][threadIdx.x];
    cnt[threadIdx.x * nb + blockIdx.x] = c;
}

// in place: cnt[d][b] becomes the count of digit d in the tiles before b;
// tot[d] = the count of digit d over all tiles
__global__ __launch_bounds__(BT) void k_rs_scan(uint32_t* __restrict__ cnt, uint32_t nb,
                                                 uint32_t* __restrict__ tot)
{
    __shared__ uint32_t sh_w[BT / WAVE];
    uint32_t* c = cnt + (size_t)blockIdx.x * nb;
    uint32_t carry = 0;
    for (uint32_t b0 = 0; b0 < nb; b0 += BT * 4) {
        uint32_t v[4], sum = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t i = b0 + threadIdx.x * 4 + k;
            v[k] = i < nb ? c[i] : 0u;
            sum += v[k];
        }
        uint32_t total;
        uint32_t off = carry + block_excl_scan(sum, sh_w, &total);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t i = b0 + threadIdx.x * 4 + k;
            if (i < nb) c[i] = off;
            off += v[k];
        }
        carry += total;
    }
    if (threadIdx.x == 0) tot[blockIdx.x] = carry;
}

template <int RS_IPT>
__global__ __launch_bounds__(BT) void k_rs_scatter(const uint64_t* __restrict__ kin,
                                                    const uint32_t* __restrict__ vin,
                                                    uint64_t* __restrict__ kout,
                                                    uint32_t* __restrict__ vout, uint32_t n,
                                                    int shift, uint32_t nb,
                                                    const uint32_t* __restrict__ cnt,
                                                    const uint32_t* __restrict__ tot)
{
    constexpr int RS_TILE = BT * RS_IPT;
    constexpr int RS_WTILE = RS_TILE / RS_WAVES;  // contiguous elements per wavefront
    __shared__ uint64_t skey[RS_TILE];
    __shared__ uint32_t sval[RS_TILE];
    __shared__ uint32_t wc[RS_WAVES][256];  // running digit counts per wavefront
    __shared__ uint32_t gdelta[256];        // global index - LDS index, per digit
    __shared__ uint32_t sh_w[BT / WAVE];

    const int w = threadIdx.x / WAVE;
    const uint32_t lane = lane_id();
#pragma unroll
    for (int k = 0; k < RS_WAVES; k++) wc[k][threadIdx.x] = 0;
    // where this tile's run of digit threadIdx.x starts in the output (the
    // scan's barriers also publish the zeroed counts)
    const uint32_t gstart =
        block_excl_scan(tot[threadIdx.x], sh_w, nullptr) + cnt[threadIdx.x * nb + blockIdx.x];

    // wavefront w ranks the elements [base, base + RS_WTILE) in rounds of 64
    const uint32_t base = blockIdx.x * RS_TILE + w * RS_WTILE;
    uint64_t key[RS_IPT];
    uint32_t val[RS_IPT], rnk[RS_IPT];
#pragma unroll
    for (int r = 0; r < RS_IPT; r++) {
        const uint32_t i = base + r * WAVE + lane;
        key[r] = i < n ? kin[i] : 0ull;
        val[r] = i < n ? vin[i] : 0u;
    }
#pragma unroll
    for (int r = 0; r < RS_IPT; r++) {
        const bool valid = base + r * WAVE + lane < n;
        const uint32_t d = (uint32_t)(key[r] >> shift) & 255u;
        uint64_t m = ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const uint64_t bb = ballot((d >> b) & 1u);
            m &= ((d >> b) & 1u) ? bb : ~bb;
        }
        const uint32_t below = __popcll(m & lanemask_lt());
        // every lane reads the count before the lowest lane of its digit
        // adds the round's run to it (one wavefront: LDS accesses in order)
        const uint32_t run = wc[w][d];
        rnk[r] = run + below;
        if (valid && below == 0) wc[w][d] = run + __popcll(m);
    }
    __syncthreads();
    {
        // per digit: start of each wavefront's run in the tile, and of the
        // tile's run in LDS (digit order)
        const uint32_t d = threadIdx.x;
        uint32_t sum = 0;
#pragma unroll
        for (int k = 0; k < RS_WAVES; k++) {
            const uint32_t c = wc[k][d];
            wc[k][d] = sum;
            sum += c;
        }
        const uint32_t lstart = block_excl_scan(sum, sh_w, nullptr);
#pragma unroll
        for (int k = 0; k < RS_WAVES; k++) wc[k][d] += lstart;
        gdelta[d] = gstart - lstart;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_IPT; r++) {
        if (base + r * WAVE + lane < n) {
            const uint32_t p = wc[w][(uint32_t)(key[r] >> shift) & 255u] + rnk[r];
            skey[p] = key[r];
            sval[p] = val[r];
        }
    }
    __syncthreads();
    const uint32_t t0 = blockIdx.x * RS_TILE;
    const uint32_t tile_n = n - t0 < (uint32_t)RS_TILE ? n - t0 : (uint32_t)RS_TILE;
#pragma unroll
    for (int r = 0; r < RS_IPT; r++) {
        const uint32_t p = r * BT + threadIdx.x;
        if (p < tile_n) {
            const uint64_t k = skey[p];
            const uint32_t o = p + gdelta[(uint32_t)(k >> shift) & 255u];
            kout[o] = k;
            vout[o] = sval[p];
        }
    }
}

// ---- merge sort -------------------------------------------------------
//
// For keys too few to fill the device: sorted tiles (sort_tile, by the kernel
// that computes the keys), then passes that each merge a few sorted runs
// into one.  A thread finds its element's place by a binary search in every
// other run of its group, SEARCHES of them in flight together: a pass is bound
// by the latency of one search (16k keys 7 us), and from some 200k keys on by
// the searches' loads (300k 9 to 15 us, four runs to one).
template <int SEARCHES>
__global__ __launch_bounds__(BT) void k_merge(const uint64_t* __restrict__ kin,
                                              const uint32_t* __restrict__ vin,
                                              uint64_t* __restrict__ kout,
                                              uint32_t* __restrict__ vout, uint32_t n, uint32_t len,
                                              uint32_t len_p2, uint32_t ways)
{
    const uint32_t i = blockIdx.x * BT + threadIdx.x;
    if (i >= n) return;
    const uint64_t key = kin[i];
    const uint32_t val = vin[i];
    const uint32_t run = i / len, r0 = run / ways * ways;
    const uint32_t own = run - r0, g0 = r0 * len;  // the group's first element
    const uint32_t left = (n - g0 - 1) / len + 1;  // runs to the end, of which the last may be short
    const uint32_t runs = left < ways ? left : ways;
    uint32_t rank = i - run * len;
    // elements before it: of the runs before its own those not above its
    // key, of the runs behind those below it, so that equal keys keep their order
    for (uint32_t q = 0; q < runs; q += SEARCHES) {
        uint32_t pos[SEARCHES] = {}, beg[SEARCHES], m[SEARCHES];
#pragma unroll
        for (int k = 0; k < SEARCHES; k++) {
            const uint32_t r = q + k;
            beg[k] = r < runs ? g0 + r * len : i;
            m[k] = r < runs && r != own ? (n - beg[k] < len ? n - beg[k] : len) : 0u;
        }
        for (uint32_t h = len_p2; h; h >>= 1) {
            uint64_t o[SEARCHES];
#pragma unroll
            for (int k = 0; k < SEARCHES; k++) {
                const uint32_t e = pos[k] + h;
                o[k] = kin[e <= m[k] ? beg[k] + e - 1 : i];
            }
#pragma unroll
            for (int k = 0; k < SEARCHES; k++) {
                const uint32_t e = pos[k] + h;
                const bool before = (o[k] < key) | ((o[k] == key) & (q + k < own));
                pos[k] = (e <= m[k]) & before ? e : pos[k];
            }
        }
#pragma unroll
        for (int k = 0; k < SEARCHES; k++) rank += pos[k];
    }
    kout[g0 + rank] = key;
    vout[g0 + rank] = val;
}

}  // namespace

int scan_sums(uint32_t* part, uint32_t nb, hipStream_t s)
{
    if (nb < SCAN_SUMS) return 0;
    k_scan_sums<<<1, 1024, 0, s>>>(part, nb);
    return 1;
}

// sized for the smaller tile, which needs more per-tile counts
size_t radix_temp_words(uint32_t n) { return 256ull * (rs_blocks(n, 8) + 1) + 64; }

void radix_sort_pairs(uint64_t*& keys, uint64_t*& keys_alt, uint32_t*& vals, uint32_t*& vals_alt,
                      uint32_t n, int end_bit, uint32_t* temp, int ipt, hipStream_t s)
{
    if (n == 0) return;
    ipt = ipt == 8 ? 8 : 16;
    const uint32_t nb = rs_blocks(n, ipt);
    uint32_t* cnt = temp;
    uint32_t* tot = temp + 256ull * nb;
    for (int shift = 0; shift < end_bit; shift += 8) {
        if (ipt == 8) k_rs_count<8><<<nb, BT, 0, s>>>(keys, n, shift, nb, cnt);
        else k_rs_count<16><<<nb, BT, 0, s>>>(keys, n, shift, nb, cnt);
        k_rs_scan<<<256, BT, 0, s>>>(cnt, nb, tot);
        if (ipt == 8)
            k_rs_scatter<8><<<nb, BT, 0, s>>>(keys, vals, keys_alt, vals_alt, n, shift, nb, cnt, tot);
        else
            k_rs_scatter<16><<<nb, BT, 0, s>>>(keys, vals, keys_alt, vals_alt, n, shift, nb, cnt,
                                                tot);
        uint64_t* tk = keys; keys = keys_alt; keys_alt = tk;
        uint32_t* tv = vals; vals = vals_alt; vals_alt = tv;
    }
}

void merge_tiles(uint64_t* keys, uint64_t* keys_alt, uint32_t* vals, uint32_t* vals_alt, uint32_t n,
                 hipStream_t s)
{
    // the last pass ends in keys
    uint32_t passes;
    const uint32_t ways = merge_ways(n, &passes);
    auto* merge = ways <= 4 ? k_merge<4> : (ways <= 6 ? k_merge<6> : k_merge<8>);
    uint64_t len = MERGE_TILE;
    for (uint32_t p = 0; p < passes; p++, len *= ways) {
        const bool alt = (passes - p) & 1;
        uint32_t p2 = 1;
        while (p2 < len) p2 *= 2;
        merge<<<(n + BT - 1) / BT, BT, 0, s>>>(alt ? keys_alt : keys, alt ? vals_alt : vals,
                                                 alt ? keys : keys_alt, alt ? vals : vals_alt, n,
                                                 (uint32_t)len, p2, ways);
    }
}

}  // namespace potg
