// potg_tree.hip -- octree build on gfx950.
//
// The reference inserts particles one at a time into an octree of leaf
// capacity 1 whose boxes come from the float64 midpoint recurrence
// mid = (x1 + x2) / 2 (build_tree, pot.c:1457-1643).  The node set of such a
// tree depends only on the positions, so it is rebuilt here in parallel:
//
//   1. keys: every particle descends key_levels levels of the same
//      recurrence; the digits (numbered in the reference's child order)
//      form a sort key behind the instance number;
//   2. a merge sort (or an LSD radix sort, of many) orders the particles;
//      runs of equal keys are ordered by descending further (rare);
//   3. lcp[i] = number of leading digits particles i and i+1 share;
//      internal node (a, l) exists for every level l with
//      lcp[a-1] < l <= lcp[a] -- numbering the nodes by (a, l) gives a
//      pre-order; parents come from one binary search over the keys;
//   4. child slots, child counts and a scan lay the children of every node
//      out contiguously for the walk;
//   5. monopole moments are folded bottom-up (by blocks of nodes, or level by
//      level for large trees), children in the reference
//      order (compute_node_values / update_node_moments, pot.c:1290-1402),
//      with the same float64 operations, so every node matches the
//      reference bit for bit.
#include "potg_internal.h"
#include "potg_prim.h"

namespace potg {

namespace {

constexpr int BT = 256;
inline uint32_t grid(uint32_t n) { return n ? (n + BT - 1) / BT : 1; }

__device__ inline int charge_of(uint8_t s, int32_t grain_q)
{
    return s == 0 ? grain_q : (s == 1 ? 1 : -1);
}

// digit of a position at depth `level` (1-based) and the box at that depth
__device__ inline int descend_to(double px, double py, double pz, double root_x2, int level,
                                 double& x1, double& x2)
{
    double y1 = 0.0, y2 = root_x2, z1 = 0.0, z2 = root_x2;
    int d = 0;
    x1 = 0.0;
    x2 = root_x2;
    for (int l = 0; l < level; l++) d = descend1(px, py, pz, x1, x2, y1, y2, z1, z2);
    return d;
}

// first depth at which two positions fall into different children; MAXD
// when they never separate (coincident)
__device__ inline int split_depth(double ax, double ay, double az, double bx, double by, double bz,
                                  double root_x2)
{
    double x1 = 0.0, x2 = root_x2, y1 = 0.0, y2 = root_x2, z1 = 0.0, z2 = root_x2;
    for (int l = 0; l < MAXD; l++) {
        const double mx = (x1 + x2) / 2.0, my = (y1 + y2) / 2.0, mz = (z1 + z2) / 2.0;
        const bool gax = !(ax < mx), gay = !(ay < my), gaz = !(az < mz);
        const bool gbx = !(bx < mx), gby = !(by < my), gbz = !(bz < mz);
        if (gax != gbx || gay != gby || gaz != gbz) return l;
        if (gax) x1 = mx; else x2 = mx;
        if (gay) y1 = my; else y2 = my;
        if (gaz) z1 = mz; else z2 = mz;
    }
    return MAXD;
}

// ---------------------------------------------------------------------
// A new step begins, in the first block of the launch that computes its keys:
// every thread reads the step counter before thread 0 advances it (the
// barrier), however many instances there are.  Nothing else in that launch
// reads what is written here.
__device__ inline void begin_step(const InstParams* __restrict__ P, InstState* __restrict__ S,
                                  Globals* g, uint32_t n_inst)
{
    const uint64_t t = g->t + 1;  // the step being taken (pot.c:4261)
    for (uint32_t k = threadIdx.x; k < n_inst; k += blockDim.x) {
        // first stepped index: the lowest index whose species is due
        // (pot.c:2430-2434); the grain itself is never stepped here
        uint32_t start = NONE;
        for (int s = 1; s < 3; s++)
            if (P[k].first_idx[s] != NONE && (t % P[k].tss[s]) == 0 && P[k].first_idx[s] < start)
                start = P[k].first_idx[s];
        S[k].start = start;
        S[k].acc_q = 0;
        S[k].acc_e = 0;
        S[k].acc_i = 0;
        S[k].n_pushed = 0;
        S[k].n_reinj_abs = 0;
        S[k].n_reinj_out = 0;
        S[k].n_wall_inward = 0;
        for (int c = 0; c < 3; c++) {
            S[k].acc_p_lo[c] = 0ull;
            S[k].acc_p_hi[c] = 0ull;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        g->t = t;
        g->tile_ctr = 0;
        g->tile_ctr2 = 0;
        g->n_reinj = 0;
    }
}

// the low 21 bits of v, two zeros behind each
__device__ inline uint64_t spread3(uint32_t v)
{
    uint64_t x = v & 0x1fffffu;
    x = (x | x << 32) & 0x001f00000000ffffull;
    x = (x | x << 16) & 0x001f0000ff0000ffull;
    x = (x | x << 8) & 0x100f00f00f00f00full;
    x = (x | x << 4) & 0x10c30c30c30c30c3ull;
    return (x | x << 2) & 0x1249249249249249ull;
}

// the key of the particle in slot i
__device__ inline uint64_t key_of(uint32_t i, const InstParams* __restrict__ P, const PState& st,
                                  int levels, Globals* g)
{
    const uint32_t inst = st.inst[i];
    const InstParams& p = P[inst];
    // the analytic spheroid grain stays out of the tree (SPH:1516-1521)
    if (p.geometry != 0 && st.spec[i] == 0) return ~0ull;
    const double px = st.x[i], py = st.y[i], pz = st.z[i];
    const double r2 = p.root_x2;
    if (!(px >= 0.0) || px > r2 || !(py >= 0.0) || py > r2 || !(pz >= 0.0) || pz > r2) {
        raise_err(g, KERR_OUT_OF_BOX, st.ref[i]);
        return (uint64_t)inst << (3 * levels);
    }
    // The position in cells of the last level (at most 2^21 along a side).
    // It carries an error below 2^-30 cells and the recurrence's midpoints
    // one below 2^-27, so further than 2^-20 from a face its whole part holds
    // the recurrence's decisions.  (The recurrence for every particle, 440
    // float64 instructions: 2M keys 38 us instead of 22.)
    const double scale = p.invR * (double)(1u << (levels - 1));
    const double cx = px * scale, cy = py * scale, cz = pz * scale;
    const uint32_t ix = (uint32_t)cx, iy = (uint32_t)cy, iz = (uint32_t)cz;
    const double fx = cx - (double)ix, fy = cy - (double)iy, fz = cz - (double)iz;
    const double lo = fmin(fx, fmin(fy, fz)), hi = fmax(fx, fmax(fy, fz));
    if (lo > 0x1p-20 && hi < 1.0 - 0x1p-20)
        // ref_digit of every level: y, whether x and y agree, z
        return (uint64_t)inst << (3 * levels) | spread3(iy) << 2 |
               spread3(~(ix ^ iy) & ((1u << levels) - 1u)) << 1 | spread3(iz);
    double x1 = 0.0, x2 = r2, y1 = 0.0, y2 = r2, z1 = 0.0, z2 = r2;
    uint64_t k = inst;
    for (int l = 0; l < levels; l++) k = (k << 3) | (uint64_t)descend1(px, py, pz, x1, x2, y1, y2, z1, z2);
    return k;
}

// begins: the instances of the step that begins, or 0
__global__ void k_keys(const InstParams* __restrict__ P, InstState* __restrict__ S, uint32_t begins,
                       PState st, uint32_t n, int levels, uint64_t* __restrict__ key,
                       uint32_t* __restrict__ perm, Globals* g)
{
    if (begins && blockIdx.x == 0) begin_step(P, S, g, begins);
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    perm[i] = i;
    key[i] = key_of(i, P, st, levels, g);
}

// the keys in sorted tiles
__global__ __launch_bounds__(MERGE_TILE) void k_key_tiles(const InstParams* __restrict__ P,
                                                          InstState* __restrict__ S, uint32_t begins,
                                                          PState st, uint32_t n, int levels,
                                                          uint64_t* __restrict__ key,
                                                          uint32_t* __restrict__ perm, Globals* g)
{
    __shared__ TileSort sh;
    if (begins && blockIdx.x == 0) begin_step(P, S, g, begins);
    const uint32_t t0 = blockIdx.x * MERGE_TILE, i = t0 + threadIdx.x;
    // what fills the last tile sorts behind all
    uint64_t k = i < n ? key_of(i, P, st, levels, g) : ~0ull;
    uint32_t idx;
    sort_tile(sh, k, idx);
    if (i < n) {
        key[i] = k;
        perm[i] = t0 + idx;
    }
}

// orders the run of equal keys from slot i by their deeper digits (insertion
// sort); returns its end
__device__ inline uint32_t order_ties(uint32_t i, const uint64_t* __restrict__ key, uint32_t* perm,
                                      const InstParams* __restrict__ P, const PState& st,
                                      uint32_t n_tree, Globals* g)
{
    uint32_t e = i + 1;
    while (e + 1 < n_tree && key[e + 1] == key[i]) e++;
    const double r2 = P[st.inst[perm[i]]].root_x2;
    for (uint32_t a = i + 1; a <= e; a++) {
        const uint32_t pa = perm[a];
        uint32_t b = a;
        while (b > i) {
            const uint32_t pb = perm[b - 1];
            // does pa sort before pb?  compare digits at the first split
            const int d = split_depth(st.x[pa], st.y[pa], st.z[pa], st.x[pb], st.y[pb], st.z[pb], r2);
            if (d >= MAXD) {
                raise_err(g, KERR_COINCIDENT, st.ref[pa]);
                return e + 1;
            }
            double x1, x2;
            const int da = descend_to(st.x[pa], st.y[pa], st.z[pa], r2, d + 1, x1, x2);
            const int db = descend_to(st.x[pb], st.y[pb], st.z[pb], r2, d + 1, x1, x2);
            if (da >= db) break;
            perm[b] = pb;
            b--;
        }
        perm[b] = pa;
    }
    return e + 1;
}

// the particles into sorted order, runs of equal keys (rare) by the thread
// that has the first of them; the grain of each instance notes its slot (the
// potential-energy pass reads the grain's potential there)
__global__ void k_permute(const uint64_t* __restrict__ key, uint32_t* perm, PState src, PState dst,
                          uint32_t n, uint32_t n_tree, const InstParams* __restrict__ P,
                          InstState* __restrict__ S, Globals* g)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t end = i + 1;
    if (i < n_tree) {
        const uint64_t k = key[i];
        if (i > 0 && key[i - 1] == k) return;
        if (end < n_tree && key[end] == k) end = order_ties(i, key, perm, P, src, n_tree, g);
    }
    for (; i < end; i++) {
        const uint32_t j = perm[i];
        dst.x[i] = src.x[j];
        dst.y[i] = src.y[j];
        dst.z[i] = src.z[j];
        dst.vx[i] = src.vx[j];
        dst.vy[i] = src.vy[j];
        dst.vz[i] = src.vz[j];
        const uint32_t r = src.ref[j];
        const uint16_t inst = src.inst[j];
        const uint8_t spec = src.spec[j];
        dst.ref[i] = r;
        dst.inst[i] = inst;
        dst.spec[i] = spec;
        if (spec == 0 && r == P[inst].offset) S[inst].grain_slot = i;
    }
}

// lcp[i] and the tile's count of internal nodes: particle i owns a node for
// every level above lcp[i - 1] up to lcp[i]
__global__ __launch_bounds__(SCAN_BT) void k_lcp(const uint64_t* __restrict__ key, PState st,
                                                 const InstParams* __restrict__ P, uint32_t n_tree,
                                                 int levels, int32_t* __restrict__ lcp,
                                                 uint32_t* __restrict__ part, Globals* g,
                                                 MomentLists ml)
{
    __shared__ int32_t sh[SCAN_TILE + 1];  // lcp from the particle before the tile
    __shared__ uint32_t sh_w[SCAN_BT / WAVE];
    const uint64_t dmask = (levels >= 21) ? ~0ull >> 1 : ((1ull << (3 * levels)) - 1);
    const auto lcp_of = [&](uint32_t i) {
        if (i + 1 >= n_tree || st.inst[i] != st.inst[i + 1]) return -1;
        const uint64_t diff = (key[i] ^ key[i + 1]) & dmask;
        if (diff) return levels - 1 - (63 - (int)__clzll(diff)) / 3;
        const int v = split_depth(st.x[i], st.y[i], st.z[i], st.x[i + 1], st.y[i + 1], st.z[i + 1],
                                  P[st.inst[i]].root_x2);
        if (v >= MAXD - 1) raise_err(g, KERR_COINCIDENT, st.ref[i]);
        return v;
    };
    const uint32_t t0 = blockIdx.x * SCAN_TILE;
    if (threadIdx.x == 0) sh[0] = t0 ? lcp_of(t0 - 1) : -1;
    if (blockIdx.x == 0) {  // the moment pass' lists start empty
        if (threadIdx.x == 0 && ml.n_top) *ml.n_top = 0;
        for (uint32_t k = threadIdx.x; k < ml.n_groups; k += SCAN_BT) ml.n_list[k] = 0;
    }
    int mx = -1;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const uint32_t j = k * SCAN_BT + threadIdx.x, i = t0 + j;
        int v = -1;
        if (i < n_tree) {
            v = lcp_of(i);
            lcp[i] = v;
        }
        sh[j + 1] = v;
        mx = v > mx ? v : mx;
    }
    __syncthreads();
    uint32_t sum = 0, total;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const uint32_t j = k * SCAN_BT + threadIdx.x;
        if (t0 + j < n_tree && sh[j + 1] > sh[j]) sum += (uint32_t)(sh[j + 1] - sh[j]);
    }
    block_excl_scan(sum, sh_w, &total);
    if (threadIdx.x == 0) part[blockIdx.x] = total;
    // deepest internal level + 1: reduced over the block, and the atomic
    // only where it raises the value (it rarely does after the first step)
    uint32_t m = (uint32_t)(mx + 1);
    for (int d = 1; d < WAVE; d <<= 1) {
        const uint32_t o = __shfl_xor(m, d, WAVE);
        m = o > m ? o : m;
    }
    if (__lane_id() == 0) sh_w[threadIdx.x / WAVE] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < SCAN_BT / WAVE; w++) m = sh_w[w] > m ? sh_w[w] : m;
        if (m > *(volatile const uint32_t*)&g->max_depth) atomicMax(&g->max_depth, m);
    }
}

// the internal nodes, numbered by owner and level (a pre-order)
__global__ __launch_bounds__(SCAN_BT) void k_nodes(const int32_t* __restrict__ lcp,
                                                   const uint32_t* __restrict__ part,
                                                   int summed, uint32_t n_tree, uint32_t cap,
                                                   uint32_t* __restrict__ base,
                                                   uint32_t* __restrict__ owner,
                                                   int32_t* __restrict__ level,
                                                   uint32_t* __restrict__ slots, Globals* g)
{
    __shared__ int32_t shl[SCAN_TILE + 1];
    __shared__ uint32_t sh[SCAN_TILE];
    __shared__ uint32_t sh_w[SCAN_BT / WAVE];
    const uint32_t t0 = blockIdx.x * SCAN_TILE;
    const uint32_t off = sum_before(part, blockIdx.x, summed, sh_w);
    if (threadIdx.x == 0) shl[0] = t0 ? lcp[t0 - 1] : -1;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const uint32_t j = k * SCAN_BT + threadIdx.x;
        shl[j + 1] = t0 + j < n_tree ? lcp[t0 + j] : -1;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const uint32_t j = k * SCAN_BT + threadIdx.x;
        sh[j] = t0 + j < n_tree && shl[j + 1] > shl[j] ? (uint32_t)(shl[j + 1] - shl[j]) : 0u;
    }
    const uint32_t total = tile_excl_scan(sh, off, sh_w);
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) g->n_internal = off + total;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const uint32_t j = k * SCAN_BT + threadIdx.x, i = t0 + j;
        if (i >= n_tree) continue;
        uint32_t n = sh[j];
        base[i] = n;
        for (int l = shl[j] + 1; l <= shl[j + 1]; l++, n++) {
            if (n >= cap) {
                raise_err(g, KERR_CAPACITY, n);
                break;
            }
            owner[n] = i;
            level[n] = l;
            const uint4 none = make_uint4(NONE, NONE, NONE, NONE);
            ((uint4*)slots)[2 * (size_t)n] = none;
            ((uint4*)slots)[2 * (size_t)n + 1] = none;
        }
    }
}

__device__ inline uint32_t n_int_of(const Globals* g, uint32_t cap)
{
    const uint32_t n = g->n_internal;
    return n < cap ? n : cap;
}

// start of the level-L node that contains sorted slot p: the first slot in
// [tb, p] whose key is not below p's key prefix.  A backward galloping
// search brackets it, then bisection: the cells of the deep levels, where
// most nodes are, hold few slots.
__device__ inline uint32_t range_start(const uint64_t* key, const int32_t* lcp, uint32_t tb,
                                       uint32_t p, int L, int levels)
{
    if (L <= levels) {
        const int sh = 3 * (levels - L);
        const uint64_t low = (sh >= 64) ? ~0ull : ((1ull << sh) - 1ull);
        const uint64_t pk = key[p] & ~low;
        uint32_t lo = tb, hi = p;
        for (uint64_t step = 1; step <= (uint64_t)(p - tb); step <<= 1) {
            const uint32_t j = p - (uint32_t)step;
            if (key[j] < pk) {
                lo = j + 1;
                break;
            }
            hi = j;
        }
        while (lo < hi) {
            const uint32_t mid = lo + (hi - lo) / 2;
            if (key[mid] < pk) lo = mid + 1; else hi = mid;
        }
        return lo;
    }
    uint32_t j = p;
    while (j > tb && lcp[j - 1] >= L) j--;
    return j;
}

__device__ inline uint32_t node_id(const int32_t* lcp, const uint32_t* base, uint32_t a, int l)
{
    const int lo = (a == 0) ? -1 : lcp[a - 1];
    return base[a] + (uint32_t)(l - lo - 1);
}

__device__ inline int digit_of(const uint64_t* key, PState st, uint32_t i, int l, int levels,
                               double root_x2)
{
    if (l <= levels) return (int)((key[i] >> (3 * (levels - l))) & 7u);
    double x1, x2;
    return descend_to(st.x[i], st.y[i], st.z[i], root_x2, l, x1, x2);
}

// every internal node (k < n_internal) and every leaf (tree slot) enters
// its parent's child slot at its digit; internal nodes also get their box
// size, roots their walk id
__global__ void k_link(const uint64_t* __restrict__ key, const int32_t* __restrict__ lcp,
                       const uint32_t* __restrict__ base, const uint32_t* __restrict__ owner,
                       const int32_t* __restrict__ level, PState st,
                       const InstParams* __restrict__ P, uint32_t n_tree, int levels,
                       uint32_t cap, Globals* g, uint32_t* __restrict__ slots,
                       uint32_t* __restrict__ wid_int, uint32_t* __restrict__ wid_leaf,
                       double* __restrict__ size2)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t nint = n_int_of(g, cap);
    if (k < nint) {
        const uint32_t a = owner[k];
        const int l = level[k];
        const uint32_t inst = st.inst[a];
        const InstParams& p = P[inst];
        double x1, x2;
        const int d = descend_to(st.x[a], st.y[a], st.z[a], p.root_x2, l, x1, x2);
        size2[k] = (x2 - x1) * (x2 - x1);
        if (l == 0) {
            wid_int[k] = inst;
        } else {
            const int lo = (a == 0) ? -1 : lcp[a - 1];
            uint32_t par;
            if (l > lo + 1) {
                par = k - 1;
            } else {
                const uint32_t a2 = range_start(key, lcp, p.tree_begin, a, l - 1, levels);
                par = node_id(lcp, base, a2, l - 1);
            }
            if (par >= nint) raise_err(g, KERR_CAPACITY, k);
            else slots[8 * par + d] = k;
        }
    }
    if (k < n_tree) {
        const uint32_t i = k;
        const uint32_t inst = st.inst[i];
        const InstParams& p = P[inst];
        const int lo = (i == p.tree_begin) ? -1 : lcp[i - 1];
        const int hi = lcp[i];
        const int L = hi > lo ? hi : lo;
        if (L < 0) {
            wid_leaf[i] = inst;  // a one-particle tree: the leaf is the root
        } else {
            uint32_t par;
            if (hi > lo) {
                par = node_id(lcp, base, i, hi);
            } else {
                const uint32_t a2 = range_start(key, lcp, p.tree_begin, i - 1, L, levels);
                par = node_id(lcp, base, a2, L);
            }
            if (par >= nint) {
                raise_err(g, KERR_CAPACITY, i);
                wid_leaf[i] = inst;
            } else {
                slots[8 * par + digit_of(key, st, i, L + 1, levels, p.root_x2)] = LEAF_BIT | i;
            }
        }
    }
}

// child counts, and their sum over the tile
__global__ __launch_bounds__(SCAN_BT) void k_ccount(const uint32_t* __restrict__ slots,
                                                    const Globals* __restrict__ g, uint32_t cap,
                                                    uint32_t* __restrict__ ccount,
                                                    uint32_t* __restrict__ part)
{
    __shared__ uint32_t sh_w[SCAN_BT / WAVE];
    const uint32_t nint = n_int_of(g, cap), t0 = blockIdx.x * SCAN_TILE;
    if (t0 >= nint) return;
    uint32_t sum = 0, total;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const uint32_t n = t0 + k * SCAN_BT + threadIdx.x;
        if (n >= nint) continue;
        const uint4 a = ((const uint4*)slots)[2 * (size_t)n], b = ((const uint4*)slots)[2 * (size_t)n + 1];
        const uint32_t c = (a.x != NONE) + (a.y != NONE) + (a.z != NONE) + (a.w != NONE) +
                           (b.x != NONE) + (b.y != NONE) + (b.z != NONE) + (b.w != NONE);
        ccount[n] = c;
        sum += c;
    }
    block_excl_scan(sum, sh_w, &total);
    if (threadIdx.x == 0) part[blockIdx.x] = total;
}

// the walk's numbering: behind the n_inst roots every node's children in one
// run, the runs in the nodes' order
__global__ __launch_bounds__(SCAN_BT) void k_wids(const uint32_t* __restrict__ slots,
                                                  const uint32_t* __restrict__ ccount,
                                                  const uint32_t* __restrict__ part, int summed,
                                                  Globals* g, uint32_t cap, uint32_t n_inst,
                                                  uint32_t* __restrict__ cfirst,
                                                  uint32_t* __restrict__ wid_int,
                                                  uint32_t* __restrict__ wid_leaf)
{
    __shared__ uint32_t sh[SCAN_TILE];
    __shared__ uint32_t sh_w[SCAN_BT / WAVE];
    const uint32_t nint = n_int_of(g, cap), t0 = blockIdx.x * SCAN_TILE;
    if (nint == 0 && t0 == 0 && threadIdx.x == 0) g->n_children = 0;
    if (t0 >= nint) return;
    const uint32_t off = sum_before(part, blockIdx.x, summed, sh_w);
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const uint32_t j = k * SCAN_BT + threadIdx.x;
        sh[j] = t0 + j < nint ? ccount[t0 + j] : 0u;
    }
    const uint32_t total = tile_excl_scan(sh, n_inst + off, sh_w);
    if (nint - t0 <= (uint32_t)SCAN_TILE && threadIdx.x == 0) g->n_children = off + total;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const uint32_t j = k * SCAN_BT + threadIdx.x, n = t0 + j;
        if (n >= nint) continue;
        uint32_t w = sh[j];
        cfirst[n] = w;
        const uint4 a = ((const uint4*)slots)[2 * (size_t)n], b = ((const uint4*)slots)[2 * (size_t)n + 1];
        const uint32_t c8[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const uint32_t c = c8[q];
            if (c == NONE) continue;
            if (c & LEAF_BIT) wid_leaf[c & ~LEAF_BIT] = w;
            else wid_int[c] = w;
            w++;
        }
    }
}

__device__ inline void put32(NodeRec32* r32, uint32_t w, const InstParams& p, double cx, double cy,
                             double cz, double s2, int q, uint32_t first, uint32_t cnt, uint32_t part)
{
    NodeRec32 f;
    f.cx = (float)((cx - p.R) * p.invR);
    f.cy = (float)((cy - p.R) * p.invR);
    f.cz = (float)((cz - p.R) * p.invR);
    // the opening test of the float32 walks is size2 < d2: the box size
    // squared over theta^2, in units of R^2 (with theta = 0 every cell opens)
    f.size2 = s2 > 0.0 ? (float)(s2 * p.open32) : 0.f;
    f.q = (float)q;
    f.first = first;
    f.cnt = cnt;
    f.part = part;
    r32[w] = f;
}

// a leaf's record: every tree particle is a leaf of charge CHARGE[species]
// (the grain: its current charge, pot.c:1318-1328) and no dipole moment
__device__ inline void put_leaf(uint32_t w, uint32_t i, double x, double y, double z, int q,
                                const InstParams& p, NodeRec64* __restrict__ r64,
                                NodeRec32* __restrict__ r32, double* __restrict__ dip64,
                                float4* __restrict__ dip32)
{
    NodeRec64 e;
    e.cx = x;
    e.cy = y;
    e.cz = z;
    e.size2 = 0.0;
    e.q = q;
    e.first = 0;
    e.cnt = LEAF;
    e.part = i;
    r64[w] = e;
    if (r32) put32(r32, w, p, x, y, z, 0.0, q, 0, LEAF, i);
    if (dip64) {
        dip64[3 * (size_t)w] = 0.0;
        dip64[3 * (size_t)w + 1] = 0.0;
        dip64[3 * (size_t)w + 2] = 0.0;
    }
    if (dip32) dip32[w] = make_float4(0.f, 0.f, 0.f, 0.f);
}

__device__ inline void leaf_record(uint32_t i, const PState& st, const InstParams* __restrict__ P,
                                   const InstState* __restrict__ S, uint32_t n_rec,
                                   const uint32_t* __restrict__ wid_leaf,
                                   NodeRec64* __restrict__ r64, NodeRec32* __restrict__ r32,
                                   double* __restrict__ dip64, float4* __restrict__ dip32)
{
    const uint32_t inst = st.inst[i], w = wid_leaf[i];
    if (w < n_rec)
        put_leaf(w, i, st.x[i], st.y[i], st.z[i], charge_of(st.spec[i], S[inst].grain_q), P[inst], r64,
                 r32, dip64, dip32);
}

__global__ void k_leaf_records(PState st, const InstParams* __restrict__ P,
                               const InstState* __restrict__ S, uint32_t n_tree, uint32_t n_rec,
                               const uint32_t* __restrict__ wid_leaf, NodeRec64* __restrict__ r64,
                               NodeRec32* __restrict__ r32, double* __restrict__ dip64,
                               float4* __restrict__ dip32)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_tree) leaf_record(i, st, P, S, n_rec, wid_leaf, r64, r32, dip64, dip32);
}

// roots of trees without internal nodes: an empty cell, or the one leaf
__global__ void k_bare_roots(const InstParams* __restrict__ P, const InstState* __restrict__ S,
                             PState st, uint32_t n_inst, NodeRec64* __restrict__ r64,
                             NodeRec32* __restrict__ r32, double* __restrict__ dip64,
                             float4* __restrict__ dip32)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n_inst || P[k].tree_n > 1) return;
    if (P[k].tree_n == 1) {
        const uint32_t i = P[k].tree_begin;
        put_leaf(k, i, st.x[i], st.y[i], st.z[i], charge_of(st.spec[i], S[k].grain_q), P[k], r64, r32,
                 dip64, dip32);
        return;
    }
    NodeRec64 e;
    e.cx = e.cy = e.cz = 0.0;
    e.size2 = 0.0;
    e.q = 0;
    e.first = 0;
    e.cnt = 0;
    e.part = 0;
    r64[k] = e;
    if (r32) {
        NodeRec32 f;
        f.cx = f.cy = f.cz = 0.f;
        f.size2 = 0.f;
        f.q = 0.f;
        f.first = 0;
        f.cnt = 0;
        f.part = 0;
        r32[k] = f;
    }
}

// A node's moments while its children are folded in (update_node_moments,
// pot.c:1290-1310): charge, |charge|, centre of |charge| and, for DIPOLES
// instances, the dipole moment about that centre.  A lane folds one of the
// three coordinates.
struct Moments {
    double c = 0.0, p = 0.0;
    int q = 0;
    uint32_t aq = 0;

    // the reference's float64 operations; a child without charge, or none,
    // changes nothing.  The division's own steps -- the reciprocal refined
    // twice, the quotient corrected by its remainder -- stand here without the
    // scaling that they need near the subnormal numbers only: a lone
    // wavefront's folds are a serial chain of ~10 cycles an instruction.
    __device__ inline void add(bool dip, int qc, uint32_t aqc, double x, double d)
    {
        const bool on = aqc != 0u;
        const double o = c;
        const double den = on ? (double)(aq + aqc) : 1.0;
        const double num = (double)aq * c + (double)aqc * x;
        double r = __builtin_amdgcn_rcp(den);
        r = __builtin_fma(r, __builtin_fma(-den, r, 1.0), r);
        r = __builtin_fma(r, __builtin_fma(-den, r, 1.0), r);
        double v = num * r;
        v = __builtin_fma(__builtin_fma(-den, v, num), r, v);
        const uint32_t e = (uint32_t)(__double_as_longlong(num) >> 52) & 0x7ffu;
        if (ballot((e - 123u >= 1800u) & (num != 0.0))) v = num / den;
        c = on ? v : c;
        if (dip && on) {
            // shift the dipole to the new centre, then add the child's
            // (zero for a leaf)
            p -= (c - o) * (double)q;
            p += d - (c - x) * (double)qc;
        }
        q += on ? qc : 0;
        aq += aqc;
    }
};

// a cell's record
__device__ inline void put_cell(uint32_t w, const InstParams& ip, double cx, double cy, double cz,
                                double px, double py, double pz, double s2, int q, uint32_t first,
                                uint32_t cnt, uint32_t aq, NodeRec64* __restrict__ r64,
                                NodeRec32* __restrict__ r32, double* __restrict__ dip64,
                                float4* __restrict__ dip32)
{
    NodeRec64 e;
    e.cx = cx;
    e.cy = cy;
    e.cz = cz;
    e.size2 = s2;
    e.q = q;
    e.first = first;
    e.cnt = cnt;
    e.part = aq;
    r64[w] = e;
    if (r32) put32(r32, w, ip, cx, cy, cz, s2, q, first, cnt, aq);
    if (dip64) {
        dip64[3 * (size_t)w] = px;
        dip64[3 * (size_t)w + 1] = py;
        dip64[3 * (size_t)w + 2] = pz;
    }
    // the float32 walk works in units of R: p / R
    if (dip32)
        dip32[w] = make_float4((float)(px * ip.invR), (float)(py * ip.invR), (float)(pz * ip.invR), 0.f);
}

// the moments of a block's nodes, by slot: how a cell's reach its parent's
template <int N, bool DIP>
struct CellsLds {
    double c[3][N];
    double p[DIP ? 3 : 1][DIP ? N : 1];
    int32_t q[N];
    uint32_t aq[N];

    __device__ inline void put(uint32_t i, uint32_t axis, const Moments& m)
    {
        if (axis > 2) return;
        c[axis][i] = m.c;
        if constexpr (DIP) p[axis][i] = m.p;
        q[i] = m.q;
        aq[i] = m.aq;
    }

    __device__ inline void record(uint32_t i, uint32_t w, const InstParams& ip, double s2, uint32_t first,
                                  uint32_t cnt, NodeRec64* __restrict__ r64,
                                  NodeRec32* __restrict__ r32, double* __restrict__ dip64,
                                  float4* __restrict__ dip32) const
    {
        double px = 0.0, py = 0.0, pz = 0.0;
        if constexpr (DIP) {
            px = p[0][i];
            py = p[1][i];
            pz = p[2][i];
        }
        put_cell(w, ip, c[0][i], c[1][i], c[2][i], px, py, pz, s2, q[i], first, cnt, aq[i], r64, r32,
                 dip64, dip32);
    }
};

// a node of the moment pass in the registers of its four lanes: its children
// (without gaps), of which the lane holds one coordinate.  `src` says where a
// child's moments are: LEAF_BIT, in `v` already; else the slot of a cell of
// this block.
template <bool DIP>
struct MomentNode {
    uint32_t cnt;
    double v[8];
    double p[DIP ? 8 : 1];
    int q[8];
    uint32_t aq[8], src[8];
};

// node k's children's ids in order, without the gaps between; s_child is the
// thread's column of the block's scratch
template <int BT_>
__device__ inline uint32_t children_of(const uint32_t* __restrict__ slots, uint32_t k,
                                       uint32_t (*s_child)[BT_], uint32_t col, uint32_t c8[8])
{
    const uint4 a = ((const uint4*)slots)[2 * (size_t)k], b = ((const uint4*)slots)[2 * (size_t)k + 1];
    const uint32_t d8[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t n = 0;
#pragma unroll
    for (int j = 0; j < 8; j++)
        if (d8[j] != NONE) s_child[n++][col] = d8[j];
#pragma unroll
    for (int j = 0; j < 8; j++) c8[j] = j < (int)n ? s_child[j][col] : NONE;
    return n;
}

// folds the node's children; the cells' moments come from LDS
template <int N, bool DIP>
__device__ inline Moments fold_children(MomentNode<DIP>& d, bool dip, uint32_t axis,
                                        const CellsLds<N, DIP>& cells)
{
    const uint32_t ax = axis < 3 ? axis : 2;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const uint32_t c = d.src[j];
        if (c < (uint32_t)N) {
            d.v[j] = cells.c[ax][c];
            d.q[j] = cells.q[c];
            d.aq[j] = cells.aq[c];
            if constexpr (DIP) d.p[j] = cells.p[ax][c];
        }
    }
    Moments m;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        if (!ballot(j < (int)d.cnt)) break;
        m.add(dip, d.q[j], d.aq[j], d.v[j], DIP ? d.p[DIP ? j : 0] : 0.0);
    }
    return m;
}

// the record of a node that waits in a list, at `pos`
constexpr uint32_t LISTED = 0xFFFFFFFEu;
__device__ inline void put_listed(NodeRec64* __restrict__ r64, uint32_t n_rec, uint32_t w, uint32_t pos)
{
    if (w >= n_rec) return;
    r64[w].cnt = LISTED;
    r64[w].part = pos;
}

// The records: moments bottom up (compute_node_values, pot.c:1312-1402) in
// two or three launches whatever the depth.  Nodes are numbered in pre-order,
// so a subtree is a run of nodes: a block takes MOM_NODES consecutive ones
// (and an even share of the leaves, whose records it writes) and goes up the
// levels with a barrier between, a cell's moments passing to its parent
// through LDS.  A node has four lanes, a coordinate each and one idle, and
// the nodes are dealt to the wavefronts by level, so that few work on one.
// The ancestors of the next block's first node (a node is one if every node
// after it, up to that one, is deeper) are left in a list to k_moments_up,
// some five a block.  Bound by the serial folds: 16k particles 17 us (and 21
// in k_moments_up), 300k 46 us.
template <bool DIP>
__global__ __launch_bounds__(MOM_BT) void k_moments(
    const int32_t* __restrict__ level, const uint32_t* __restrict__ slots, PState st,
    const InstParams* __restrict__ P, const InstState* __restrict__ S, const Globals* __restrict__ g,
    uint32_t n_tree, uint32_t cap, const uint32_t* __restrict__ owner,
    const uint32_t* __restrict__ ccount, const uint32_t* __restrict__ cfirst,
    const uint32_t* __restrict__ wid_int, const uint32_t* __restrict__ wid_leaf,
    const double* __restrict__ size2, NodeRec64* __restrict__ r64, NodeRec32* __restrict__ r32,
    double* __restrict__ dip64, float4* __restrict__ dip32, uint32_t n_rec, MomentLists ml)
{
    constexpr int NW = MOM_NODES / WAVE;
    __shared__ CellsLds<MOM_NODES, DIP> cells;
    __shared__ uint32_t s_child[8][MOM_NODES];
    __shared__ uint16_t s_order[MOM_NODES];
    __shared__ int32_t s_min[NW];
    __shared__ uint32_t s_cnt[WAVE];  // nodes per level; [WAVE - 1]: those left to the list
    __shared__ unsigned long long s_present;
    const uint32_t nint = n_int_of(g, cap), k0 = blockIdx.x * MOM_NODES;
    if (k0 >= nint) return;
    const uint32_t t = threadIdx.x, lane = __lane_id(), wv = t / WAVE;
    const uint32_t nk = nint - k0 < (uint32_t)MOM_NODES ? nint - k0 : (uint32_t)MOM_NODES;
    const uint32_t kt = k0 + t;
    const bool has = t < nk;  // of the first MOM_NODES threads, one a node
    if (t < WAVE) s_cnt[t] = 0;
    const int lv = has ? level[kt] : 0x7fffffff;
    // the lowest level after this node, up to the next block's first
    int lo = __shfl_down(lv, 1, WAVE);
    if (lane == WAVE - 1) lo = 0x7fffffff;
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const int o = __shfl_down(lo, d, WAVE);
        if (lane + d < WAVE && o < lo) lo = o;
    }
    const int wlo = lv < lo ? lv : lo;
    if (lane == 0 && wv < NW) s_min[wv] = wlo;
    __syncthreads();
    for (uint32_t v = wv + 1; v < NW; v++) lo = s_min[v] < lo ? s_min[v] : lo;
    if (t == 0) ml.block_min[blockIdx.x] = lo < wlo ? lo : wlo;
    const int next = k0 + nk < nint ? level[k0 + nk] : -1;
    const bool listed = has && (next < lo ? next : lo) > lv;
    if (listed) {
        const uint32_t grp = blockIdx.x / ml.group;
        const uint32_t pos = atomicAdd(&ml.n_list[grp], 1u);
        MomentItem it;
        it.k = kt;
        it.w = wid_int[kt];
        it.first = cfirst[kt];
        it.cnt = (uint16_t)ccount[kt];
        it.level = (int16_t)lv;
        it.inst = st.inst[owner[kt]];
        it.pad = 0;
        it.size2 = size2[kt];
        ml.list[(size_t)grp * ml.group * MOM_LIST + pos] = it;
        put_listed(r64, n_rec, it.w, pos);
    }
    // counting sort by level, the deepest first, the listed last
    const int bin = listed ? WAVE - 1 : lv;
    uint32_t rank = 0;
    for (uint64_t left = ballot(has); left;) {
        const int b = __builtin_amdgcn_readlane(bin, __ffsll((unsigned long long)left) - 1);
        const uint64_t same = ballot(has && bin == b);
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(&s_cnt[b & (WAVE - 1)], (uint32_t)__popcll(same));
        base = __builtin_amdgcn_readfirstlane(base);
        if (bin == b) rank = base + __popcll(same & ((1ull << lane) - 1ull));
        left &= ~same;
    }
    __syncthreads();
    if (t < WAVE) {
        // lane b: bin MAXD - b, then the list's
        const int b = (int)lane <= MAXD ? MAXD - (int)lane : WAVE - 1;
        const uint32_t c = (int)lane <= MAXD + 1 ? s_cnt[b] : 0u;
        const uint64_t some = ballot(c != 0u && b <= MAXD);
        const uint32_t off = wave_incl_scan(c) - c;
        if ((int)lane <= MAXD + 1) s_cnt[b] = off;
        if (lane == 0) s_present = some;
    }
    __syncthreads();
    if (has) s_order[s_cnt[bin & (WAVE - 1)] + rank] = (uint16_t)t;
    __syncthreads();
    // the four lanes' node and its leaf children
    const uint32_t slot = t / 4, axis = t & 3;
    uint32_t own = 0;
    int my = -1;
    bool dip = false;
    MomentNode<DIP> d;
    if (slot < s_cnt[WAVE - 1]) {
        own = s_order[slot];
        const uint32_t k = k0 + own;
        uint32_t c8[8];
        d.cnt = children_of<MOM_NODES>(slots, k, s_child, slot, c8);
        my = level[k];
        const uint32_t inst = st.inst[owner[k]];
        const int gq = S[inst].grain_q;
        if (DIP) dip = P[inst].dipoles != 0;
        const double* coord = axis == 0 ? st.x : (axis == 1 ? st.y : st.z);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t i = c8[j] & ~LEAF_BIT;
            d.v[j] = 0.0;
            if constexpr (DIP) d.p[j] = 0.0;
            d.q[j] = 0;
            d.aq[j] = 0u;
            d.src[j] = c8[j] & LEAF_BIT ? LEAF_BIT : c8[j] - k0;
            if (j < (int)d.cnt && (c8[j] & LEAF_BIT) && i < n_tree) {
                d.v[j] = coord[i];
                d.q[j] = charge_of(st.spec[i], gq);
                d.aq[j] = (uint32_t)abs(d.q[j]);
            }
        }
    }
    // the block's share of the leaf records
    const uint32_t share = (n_tree - 1) / ((nint - 1) / MOM_NODES + 1) + 1;
    const uint64_t i0 = (uint64_t)blockIdx.x * share;
    for (uint32_t j = t; j < share && i0 + j < n_tree; j += MOM_BT)
        leaf_record((uint32_t)i0 + j, st, P, S, n_rec, wid_leaf, r64, r32, dip64, dip32);
    for (unsigned long long m = s_present; m;) {
        const int L = MAXD - (__ffsll(m) - 1);
        m &= m - 1;
        if (my == L) cells.put(own, axis, fold_children(d, dip, axis, cells));
        __syncthreads();
    }
    if (has && !listed && wid_int[kt] < n_rec)
        cells.record(t, wid_int[kt], P[st.inst[owner[kt]]], size2[kt], cfirst[kt], ccount[kt], r64, r32,
                     dip64, dip32);
}

// The nodes k_moments listed, a group of its blocks a block here: a child's
// finished record is in registers before the first level, a listed child's
// moments come from LDS.  Ancestors of the next group's first node go to the
// next list, which `last` takes in one block.  A block has seldom more nodes
// than lanes for them; those beyond are loaded at their level, and those
// beyond the LDS slots reach their parents through their records.  Bound by
// latency: the loads before the first level, then the folds.
template <bool DIP>
__global__ __launch_bounds__(MOM_BT) void k_moments_up(
    int last, const int32_t* __restrict__ level, const InstParams* __restrict__ P,
    const Globals* __restrict__ g, uint32_t cap, NodeRec64* __restrict__ r64,
    NodeRec32* __restrict__ r32, double* __restrict__ dip64, float4* __restrict__ dip32, uint32_t n_rec,
    MomentLists ml)
{
    constexpr uint32_t SLOTS = 768, LV = 4096;
    __shared__ CellsLds<SLOTS, DIP> cells;
    __shared__ int8_t s_level[LV];
    __shared__ int32_t s_after[WAVE];  // lowest level of the group's later blocks
    __shared__ unsigned long long s_present;
    const uint32_t t = threadIdx.x, slot = t / 4, axis = t & 3;
    const uint32_t b0 = blockIdx.x * ml.group;  // the group's first block
    const uint32_t n = last ? *ml.n_top : ml.n_list[blockIdx.x];
    const MomentItem* list = last ? ml.top : ml.list + (size_t)b0 * MOM_LIST;
    if (n == 0) return;
    if (t == 0) s_present = 0ull;
    if (!last && t < WAVE) {
        const uint32_t nint = n_int_of(g, cap);
        // a group that ends the nodes passes nothing on
        const uint64_t end = (uint64_t)(b0 + ml.group) * MOM_NODES;
        int m = end < nint ? level[end] : -1;
        if (ml.group <= WAVE) {
            // lane b: the blocks after b
            const uint32_t b = b0 + t + 1;
            const int own =
                t + 1 < ml.group && (uint64_t)b * MOM_NODES < nint ? ml.block_min[b] : 0x7fffffff;
            m = own < m ? own : m;
            for (int d = 1; d < WAVE; d <<= 1) {
                const int o = __shfl_down(m, d, WAVE);
                if (t + d < WAVE && o < m) m = o;
            }
        }
        s_after[t] = m;
    }
    const auto load = [&](const MomentItem& it, MomentNode<DIP>& d) {
        bool late = false;  // a child's record is not there before the level
        d.cnt = it.cnt;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            d.src[j] = LEAF_BIT;
            d.v[j] = 0.0;
            if constexpr (DIP) d.p[j] = 0.0;
            d.q[j] = 0;
            d.aq[j] = 0u;
            const uint32_t w = it.first + j;
            if (j >= (int)d.cnt || w >= n_rec) continue;
            const NodeRec64& r = r64[w];
            d.v[j] = axis == 0 ? r.cx : (axis == 1 ? r.cy : r.cz);
            d.q[j] = r.q;
            d.aq[j] = r.cnt == LEAF ? (uint32_t)abs(r.q) : r.part;
            if constexpr (DIP) d.p[j] = dip64[3 * (size_t)w + (axis < 3 ? axis : 2)];
            if (r.cnt == LISTED) {
                if (r.part < SLOTS) d.src[j] = r.part;
                else late = true;
            }
        }
        return late;
    };
    __syncthreads();
    // the levels; nodes to be passed on have none here
    unsigned long long has = 0ull;
    for (uint32_t i = t; i < n; i += MOM_BT) {
        int l = list[i].level;
        if (!last) {
            const MomentItem o = list[i];
            const uint32_t c = ml.group <= WAVE ? o.k / MOM_NODES - b0 : 0u;
            if (s_after[c & (WAVE - 1)] > l) {
                const uint32_t to = atomicAdd(ml.n_top, 1u);
                ml.top[to] = o;
                put_listed(r64, n_rec, o.w, to);
                l = -1;
            }
        }
        if (i < LV) s_level[i] = (int8_t)l;
        if (l >= 0) has |= 1ull << l;
    }
    if (has) atomicOr(&s_present, has);
    __syncthreads();
    const auto level_of = [&](uint32_t i) {
        if (i < LV) return (int)s_level[i];
        const MomentItem o = list[i];
        const uint32_t c = last || ml.group > WAVE ? 0u : o.k / MOM_NODES - b0;
        return !last && s_after[c & (WAVE - 1)] > o.level ? -1 : (int)o.level;
    };
    // the lanes' node, loaded before its level unless it waits for a record
    MomentNode<DIP> d;
    MomentItem it = {};
    uint32_t held = NONE;
    int L = -1;
    for (unsigned long long m = s_present;;) {
        for (uint32_t i = slot; i < n; i += MOM_NODES) {
            if (L >= 0 ? level_of(i) != L : i != slot) continue;
            if (held != i) {
                it = list[i];
                held = load(it, d) ? NONE : i;
            }
            if (L < 0) continue;
            const Moments mo = fold_children(d, DIP && P[it.inst].dipoles, axis, cells);
            if (i < SLOTS) {
                cells.put(i, axis, mo);
                continue;
            }
            const double cx = __shfl(mo.c, 0, 4), cy = __shfl(mo.c, 1, 4), cz = __shfl(mo.c, 2, 4);
            const double px = __shfl(mo.p, 0, 4), py = __shfl(mo.p, 1, 4), pz = __shfl(mo.p, 2, 4);
            if (axis == 0 && it.w < n_rec)
                put_cell(it.w, P[it.inst], cx, cy, cz, px, py, pz, it.size2, mo.q, it.first, it.cnt, mo.aq,
                         r64, r32, dip64, dip32);
        }
        __syncthreads();
        if (!m) break;
        L = 63 - __clzll(m);
        m &= ~(1ull << L);
    }
    for (uint32_t i = t; i < n && i < SLOTS; i += MOM_BT) {
        const MomentItem o = list[i];
        if (level_of(i) >= 0 && o.w < n_rec)
            cells.record(i, o.w, P[o.inst], o.size2, o.first, o.cnt, r64, r32, dip64, dip32);
    }
}

// Internal nodes bucketed by depth, so that each level's moment pass visits
// only that level's nodes: a counting sort without atomics.  Block b owns a
// contiguous chunk of the node ids; per-block level histograms are scanned
// level-major, then each block writes its nodes at its offsets.  Order
// within a level is free (the nodes of one level are independent).
__device__ inline void level_chunk(const Globals* g, uint32_t cap, uint32_t& lo, uint32_t& hi)
{
    const uint32_t nint = n_int_of(g, cap);
    const uint32_t chunk = (nint + LVL_BLOCKS - 1) / LVL_BLOCKS;
    lo = blockIdx.x * chunk;
    hi = lo + chunk < nint ? lo + chunk : nint;
    if (lo > hi) lo = hi;
}

__global__ __launch_bounds__(BT) void k_level_count(const int32_t* __restrict__ level,
                                                    const Globals* __restrict__ g, uint32_t cap,
                                                    uint32_t* __restrict__ hist)
{
    __shared__ uint32_t h[MAXD];
    if (threadIdx.x < MAXD) h[threadIdx.x] = 0;
    __syncthreads();
    uint32_t lo, hi;
    level_chunk(g, cap, lo, hi);
    for (uint32_t k = lo + threadIdx.x; k < hi; k += BT) {
        const int32_t L = level[k];
        if (L >= 0 && L < MAXD) atomicAdd(&h[L], 1u);
    }
    __syncthreads();
    if (threadIdx.x < MAXD) hist[threadIdx.x * LVL_BLOCKS + blockIdx.x] = h[threadIdx.x];
}

// exclusive scan of the MAXD x LVL_BLOCKS histogram in level-major order;
// lstart[L] = first slot of level L, lstart[MAXD] = all internal nodes
__global__ __launch_bounds__(1024) void k_level_offsets(const uint32_t* __restrict__ hist,
                                                        uint32_t* __restrict__ off,
                                                        uint32_t* __restrict__ lstart)
{
    constexpr uint32_t N = MAXD * LVL_BLOCKS;
    constexpr uint32_t PER = (N + 1023) / 1024;
    __shared__ uint32_t part[1024];
    const uint32_t t = threadIdx.x;
    uint32_t sum = 0;
    for (uint32_t j = 0; j < PER; j++) {
        const uint32_t i = t * PER + j;
        if (i < N) sum += hist[i];
    }
    part[t] = sum;
    __syncthreads();
    for (uint32_t d = 1; d < 1024; d <<= 1) {
        const uint32_t v = t >= d ? part[t - d] : 0u;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    uint32_t run = part[t] - sum;  // exclusive prefix of this thread's run
    for (uint32_t j = 0; j < PER; j++) {
        const uint32_t i = t * PER + j;
        if (i < N) {
            off[i] = run;
            if (i % LVL_BLOCKS == 0) lstart[i / LVL_BLOCKS] = run;
            run += hist[i];
        }
    }
    if (t == 1023) lstart[MAXD] = part[1023];
}

__global__ __launch_bounds__(BT) void k_level_scatter(const int32_t* __restrict__ level,
                                                      const Globals* __restrict__ g, uint32_t cap,
                                                      const uint32_t* __restrict__ off,
                                                      uint32_t* __restrict__ by_level)
{
    __shared__ uint32_t h[MAXD], base[MAXD];
    uint32_t lo, hi;
    level_chunk(g, cap, lo, hi);
    if (threadIdx.x < MAXD) base[threadIdx.x] = off[threadIdx.x * LVL_BLOCKS + blockIdx.x];
    for (uint32_t k0 = lo; k0 < hi; k0 += BT) {
        if (threadIdx.x < MAXD) h[threadIdx.x] = 0;
        __syncthreads();
        const uint32_t k = k0 + threadIdx.x;
        int32_t L = -1;
        uint32_t rank = 0;
        if (k < hi) {
            L = level[k];
            if (L >= 0 && L < MAXD) rank = atomicAdd(&h[L], 1u);
            else L = -1;
        }
        __syncthreads();
        if (L >= 0) {
            const uint32_t pos = base[L] + rank;
            if (pos < cap) by_level[pos] = k;
        }
        __syncthreads();
        if (threadIdx.x < MAXD) base[threadIdx.x] += h[threadIdx.x];
    }
}

// the moments of internal node k, its children folded in the reference
// order (compute_node_values / update_node_moments, pot.c:1290-1402):
// charge, |charge|, centre of |charge| and, for DIPOLES instances, the
// dipole moment about that centre.  The children are read from their
// records, contiguous in that order and finished before this level: the
// leaves by k_leaf_records, internal children by the deeper levels.
__device__ void level_node_moments(uint32_t k, PState st, const InstParams* __restrict__ P,
                                   uint32_t cap, const uint32_t* __restrict__ owner,
                                   const uint32_t* __restrict__ ccount,
                                   const uint32_t* __restrict__ cfirst,
                                   const uint32_t* __restrict__ wid_int,
                                   const double* __restrict__ size2,
                                   NodeRec64* __restrict__ r64, NodeRec32* __restrict__ r32,
                                   double* __restrict__ dip64, float4* __restrict__ dip32,
                                   uint32_t n_rec)
{
    if (k >= cap) return;
    const uint32_t w = wid_int[k];
    if (w >= n_rec) return;
    const uint32_t first = cfirst[k];
    const uint32_t end = first + ccount[k] < n_rec ? first + ccount[k] : n_rec;
    const uint32_t inst = st.inst[owner[k]];
    const bool dip = dip64 && P[inst].dipoles;
    double cx = 0.0, cy = 0.0, cz = 0.0, px = 0.0, py = 0.0, pz = 0.0;
    int q = 0;
    uint32_t aq = 0;
    // every child's record in flight at once, then the serial fold
    NodeRec64 ch[8];
#pragma unroll
    for (uint32_t j = 0; j < 8; j++)
        if (first + j < end) ch[j] = r64[first + j];
#pragma unroll
    for (uint32_t jj = 0; jj < 8; jj++) {
        if (first + jj >= end) break;
        const uint32_t j = first + jj;
        const NodeRec64& c = ch[jj];
        const int qc = c.q;
        const uint32_t aqc = c.cnt == LEAF ? (uint32_t)abs(qc) : c.part;
        if (aqc) {
            // update_node_moments (pot.c:1290-1310), same float64 operations
            const double ox = cx, oy = cy, oz = cz;
            const double den = (double)(aq + aqc);
            cx = ((double)aq * cx + (double)aqc * c.cx) / den;
            cy = ((double)aq * cy + (double)aqc * c.cy) / den;
            cz = ((double)aq * cz + (double)aqc * c.cz) / den;
            if (dip) {
                // shift the dipole to the new centre, then add the child's
                // (zero for a leaf)
                px -= (cx - ox) * (double)q;
                py -= (cy - oy) * (double)q;
                pz -= (cz - oz) * (double)q;
                px += dip64[3 * (size_t)j] - (cx - c.cx) * (double)qc;
                py += dip64[3 * (size_t)j + 1] - (cy - c.cy) * (double)qc;
                pz += dip64[3 * (size_t)j + 2] - (cz - c.cz) * (double)qc;
            }
            q += qc;
            aq += aqc;
        }
    }
    NodeRec64 e;
    e.cx = cx;
    e.cy = cy;
    e.cz = cz;
    e.size2 = size2[k];
    e.q = q;
    e.first = first;
    e.cnt = ccount[k];
    e.part = aq;
    r64[w] = e;
    if (r32) put32(r32, w, P[inst], cx, cy, cz, e.size2, q, e.first, e.cnt, aq);
    if (dip64) {
        dip64[3 * (size_t)w] = px;
        dip64[3 * (size_t)w + 1] = py;
        dip64[3 * (size_t)w + 2] = pz;
    }
    // the float32 walk works in units of R: p / R
    if (dip32)
        dip32[w] = make_float4((float)(px * P[inst].invR), (float)(py * P[inst].invR),
                               (float)(pz * P[inst].invR), 0.f);
}

// the moments of the internal nodes at depth L; the deeper levels were
// finished by earlier launches
__global__ void k_level_moments(int L, PState st, const InstParams* __restrict__ P,
                                const Globals* __restrict__ g, uint32_t cap,
                                const uint32_t* __restrict__ owner,
                                const uint32_t* __restrict__ ccount,
                                const uint32_t* __restrict__ cfirst,
                                const uint32_t* __restrict__ wid_int,
                                const double* __restrict__ size2, NodeRec64* __restrict__ r64,
                                NodeRec32* __restrict__ r32, double* __restrict__ dip64,
                                float4* __restrict__ dip32, uint32_t n_rec,
                                const uint32_t* __restrict__ lstart,
                                const uint32_t* __restrict__ by_level)
{
    if ((uint32_t)L + 1 > g->max_depth) return;  // no internal node this deep
    const uint32_t lo = lstart[L], hi = lstart[L + 1];
    for (uint32_t idx = lo + blockIdx.x * blockDim.x + threadIdx.x; idx < hi;
         idx += gridDim.x * blockDim.x)
        level_node_moments(by_level[idx], st, P, cap, owner, ccount, cfirst, wid_int, size2, r64,
                           r32, dip64, dip32, n_rec);
}

// levels Lhi down to Llo by one block, a barrier between levels: for the
// thinly populated deep and shallow levels, where a launch per level would
// cost more than the work
__global__ __launch_bounds__(1024) void k_level_moments_block(
    int Lhi, int Llo, PState st, const InstParams* __restrict__ P, const Globals* __restrict__ g,
    uint32_t cap, const uint32_t* __restrict__ owner, const uint32_t* __restrict__ ccount,
    const uint32_t* __restrict__ cfirst, const uint32_t* __restrict__ wid_int,
    const double* __restrict__ size2, NodeRec64* __restrict__ r64, NodeRec32* __restrict__ r32,
    double* __restrict__ dip64, float4* __restrict__ dip32, uint32_t n_rec,
    const uint32_t* __restrict__ lstart, const uint32_t* __restrict__ by_level)
{
    const uint32_t depth = g->max_depth;
    for (int L = Lhi; L >= Llo; L--) {
        if ((uint32_t)L + 1 > depth) continue;  // uniform over the block
        const uint32_t lo = lstart[L], hi = lstart[L + 1];
        for (uint32_t idx = lo + threadIdx.x; idx < hi; idx += blockDim.x)
            level_node_moments(by_level[idx], st, P, cap, owner, ccount, cfirst, wid_int, size2,
                               r64, r32, dip64, dip32, n_rec);
        // the next level up reads what this one wrote
        __syncthreads();
    }
}

}  // namespace

// the leaf records again, from the current state: between the two fields
// of velocity Verlet / Euler-Richardson the reference's walk reads its leaves
// from the live array, which then holds the intermediate state, while the
// cells keep the moments of the step's build (pot.c:1785-1804, 2557-2613)
void launch_leaf_refresh(Bufs& b, hipStream_t s)
{
    const uint32_t n = b.n_tree;
    if (!n) return;
    k_leaf_records<<<grid(n), BT, 0, s>>>(b.st, b.P, b.S, n, b.n_rec, b.wid_leaf, b.rec64,
                                          b.precision ? b.rec32 : nullptr, b.dip64,
                                          b.precision ? b.dip32 : nullptr);
}

void launch_keys_sort_permute(Bufs& b, bool begin, hipStream_t s)
{
    const uint32_t n = b.n_total, begins = begin ? b.n_inst : 0u;
    if (n < MERGE_MAX) {
        const bool alt = merge_passes(n) & 1;
        k_key_tiles<<<(n + MERGE_TILE - 1) / MERGE_TILE, MERGE_TILE, 0, s>>>(
            b.P, b.S, begins, b.st, n, b.key_levels, alt ? b.key_alt : b.key,
            alt ? b.perm_alt : b.perm, b.g);
        merge_tiles(b.key, b.key_alt, b.perm, b.perm_alt, n, s);
    } else {
        k_keys<<<grid(n), BT, 0, s>>>(b.P, b.S, begins, b.st, n, b.key_levels, b.key, b.perm, b.g);
        radix_sort_pairs(b.key, b.key_alt, b.perm, b.perm_alt, n, b.key_bits, b.sort_tmp,
                         (int)b.sort_ipt, s);
    }
    k_permute<<<grid(n), BT, 0, s>>>(b.key, b.perm, b.st, b.alt, n, b.n_tree, b.P, b.S, b.g);
    PState t = b.st;
    b.st = b.alt;
    b.alt = t;
}

void launch_tree(Bufs& b, hipStream_t s)
{
    const uint32_t n = b.n_tree;
    NodeRec32* r32 = b.precision ? b.rec32 : nullptr;
    float4* d32 = b.precision ? b.dip32 : nullptr;
    if (b.any_bare)
        k_bare_roots<<<grid(b.n_inst), BT, 0, s>>>(b.P, b.S, b.st, b.n_inst, b.rec64, r32, b.dip64, d32);
    if (!n) return;
    const uint32_t cap = b.cap_int;
    k_lcp<<<scan_blocks(n), SCAN_BT, 0, s>>>(b.key, b.st, b.P, n, b.key_levels, b.lcp, b.scan_tmp,
                                             b.g, b.ml);
    int summed = scan_sums(b.scan_tmp, scan_blocks(n), s);
    k_nodes<<<scan_blocks(n), SCAN_BT, 0, s>>>(b.lcp, b.scan_tmp, summed, n, cap, b.base, b.owner,
                                               b.level, b.slots, b.g);
    k_link<<<grid(cap > n ? cap : n), BT, 0, s>>>(b.key, b.lcp, b.base, b.owner, b.level, b.st, b.P,
                                                   n, b.key_levels, cap, b.g, b.slots, b.wid_int,
                                                   b.wid_leaf, b.size2);
    k_ccount<<<scan_blocks(cap), SCAN_BT, 0, s>>>(b.slots, b.g, cap, b.ccount, b.scan_tmp);
    // (the sums of tiles past the nodes there are, are never read)
    summed = scan_sums(b.scan_tmp, scan_blocks(cap), s);
    k_wids<<<scan_blocks(cap), SCAN_BT, 0, s>>>(b.slots, b.ccount, b.scan_tmp, summed, b.g, cap,
                                                b.n_inst, b.cfirst, b.wid_int, b.wid_leaf);
    if (!b.ml.group) {
        k_leaf_records<<<grid(n), BT, 0, s>>>(b.st, b.P, b.S, n, b.n_rec, b.wid_leaf, b.rec64, r32,
                                              b.dip64, d32);
        const uint32_t gb = grid(cap) < 2048u ? grid(cap) : 2048u;
        k_level_count<<<LVL_BLOCKS, BT, 0, s>>>(b.level, b.g, cap, b.lvl_hist);
        k_level_offsets<<<1, 1024, 0, s>>>(b.lvl_hist, b.lvl_off, b.lvl_start);
        k_level_scatter<<<LVL_BLOCKS, BT, 0, s>>>(b.level, b.g, cap, b.lvl_off, b.by_level);
        // deepest level first.  Levels below LVL_WIDE_LO hold few nodes in
        // any plasma (their cells are a few mean spacings wide or less), as
        // do the top ones, at most 8^L n_inst: one block each; the levels
        // between get a launch of their own.  (16 trees' four top levels in
        // one block took 177 us, three and a launch 40.)
        int hi = LVL_WIDE_HI;
        while (hi >= 0 && ((uint64_t)b.n_inst << (3 * hi)) > 1024u) hi--;
        k_level_moments_block<<<1, 1024, 0, s>>>(MAXD - 1, LVL_WIDE_LO, b.st, b.P, b.g, cap, b.owner,
                                                 b.ccount, b.cfirst, b.wid_int, b.size2, b.rec64, r32,
                                                 b.dip64, d32, b.n_rec, b.lvl_start, b.by_level);
        for (int L = LVL_WIDE_LO - 1; L > hi; L--)
            k_level_moments<<<gb, BT, 0, s>>>(L, b.st, b.P, b.g, cap, b.owner, b.ccount, b.cfirst,
                                              b.wid_int, b.size2, b.rec64, r32, b.dip64, d32, b.n_rec,
                                              b.lvl_start, b.by_level);
        if (hi < 0) return;
        k_level_moments_block<<<1, 1024, 0, s>>>(hi, 0, b.st, b.P, b.g, cap, b.owner,
                                                 b.ccount, b.cfirst, b.wid_int, b.size2, b.rec64, r32,
                                                 b.dip64, d32, b.n_rec, b.lvl_start, b.by_level);
        return;
    }
    const uint32_t nb = moment_blocks(cap), ng = b.ml.n_groups;
    auto* moments = b.dip64 ? k_moments<true> : k_moments<false>;
    auto* up = b.dip64 ? k_moments_up<true> : k_moments_up<false>;
    moments<<<nb, MOM_BT, 0, s>>>(b.level, b.slots, b.st, b.P, b.S, b.g, n, cap, b.owner, b.ccount,
                                  b.cfirst, b.wid_int, b.wid_leaf, b.size2, b.rec64, r32, b.dip64, d32,
                                  b.n_rec, b.ml);
    for (int last = 0; last < (ng > 1 ? 2 : 1); last++)
        up<<<last ? 1 : ng, MOM_BT, 0, s>>>(last, b.level, b.P, b.g, cap, b.rec64, r32, b.dip64, d32,
                                            b.n_rec, b.ml);
}

}  // namespace potg
