// Octree build on the device (replaces BHTree::make, src/bhtree.cpp:55-107).
//
// The reference builds a pointer octree top-down, serially: the root cube
// is the bounding box (centre, largest extent) or the periodic box
// (src/bhtree.cpp:19-31, 59-94); a particle goes to child slot
// sum_k [x_k > c_k] << k (src/bhtree.cpp:168-175); a child's centre is the
// parent's +-edge/4 and its edge half the parent's (src/bhtree.cpp:188-196);
// a child at level L is split when it holds more than leafParticleNumber
// particles and L-1 < maxTreeLevel (src/bhtree.cpp:154-158; root level 1).
//
// Here every particle replays that descent once, with the same FP64
// comparisons and centre updates, to get a key of maxTreeLevel D-bit slot
// groups (most significant = first split).  Sorting the keys puts each
// cell's particles in one contiguous range and the cells in depth-first
// pre-order, with children in slot order -- the reference's visiting order.
// The cells that exist, and which of them are leaves, follow from counts of
// equal key prefixes; a node starting at particle b exists at level L iff
// b begins a level-L cell whose parent holds more than leafParticleNumber
// particles.  Each particle emits the nodes that start at it, so an
// exclusive scan of those counts is the pre-order numbering.  Mass moments
// are reduced bottom-up, in slices of consecutive nodes by one workgroup each
// and then, for the few cells that span slices, by a single workgroup.  The
// root keeps zero mass and centre of mass, as the reference never
// accumulates them (include/bhtree.hpp:46-53).
#include <cstring>

#include "ctx.hpp"

#include <rocprim/rocprim.hpp>

namespace sphgpu {

// ------------------------------------------------------------ bounding box
// One block per CU; the last one to finish reduces the blocks' extents.
constexpr int BBOX_THREADS = 1024;
template <int D> __global__ void __launch_bounds__(BBOX_THREADS) bbox_kernel(State s, int n, double *partial, int *ticket, double *scal)
{
#pragma clang fp contract(off)
    double lo[D], hi[D];
#pragma unroll
    for(int k = 0; k < D; ++k) { lo[k] = 1.7976931348623157e308; hi[k] = -1.7976931348623157e308; }
    for(int i = blockIdx.x * BBOX_THREADS + threadIdx.x; i < n; i += gridDim.x * BBOX_THREADS)
#pragma unroll
        for(int k = 0; k < D; ++k) {
            const double x = s.f[F_X + k][i];
            lo[k] = x < lo[k] ? x : lo[k];
            hi[k] = x > hi[k] ? x : hi[k];
        }
    __shared__ double sh[2 * D][BBOX_THREADS / WAVE];
#pragma unroll
    for(int k = 0; k < D; ++k) {
        lo[k] = wave_minv(lo[k]);
        hi[k] = wave_maxv(hi[k]);
    }
    const int w = threadIdx.x / WAVE;
    if(wave_lane() == 0)
#pragma unroll
        for(int k = 0; k < D; ++k) { sh[k][w] = lo[k]; sh[D + k][w] = hi[k]; }
    __syncthreads();
    if(threadIdx.x == 0) {
#pragma unroll
        for(int k = 0; k < D; ++k) {
            double a = sh[k][0], b = sh[D + k][0];
            for(int j = 1; j < BBOX_THREADS / WAVE; ++j) {
                a = sh[k][j] < a ? sh[k][j] : a;
                b = sh[D + k][j] > b ? sh[D + k][j] : b;
            }
            put(partial + blockIdx.x * 2 * D + k, a);
            put(partial + blockIdx.x * 2 * D + D + k, b);
        }
    }
    if(!last_block(ticket) || threadIdx.x >= WAVE) return;
    // Root cube: centre (max+min)/2, edge = largest extent (src/bhtree.cpp:80-94).
    // One wave: lanes stride over the block partials, then a wave min/max
    // (exact, so the result does not depend on the order).
    for(int k = 0; k < D; ++k) { lo[k] = 1.7976931348623157e308; hi[k] = -1.7976931348623157e308; }
    for(int b = threadIdx.x; b < (int)gridDim.x; b += WAVE)
        for(int k = 0; k < D; ++k) {
            const double a = get(partial + b * 2 * D + k), c = get(partial + b * 2 * D + D + k);
            lo[k] = a < lo[k] ? a : lo[k];
            hi[k] = c > hi[k] ? c : hi[k];
        }
    for(int k = 0; k < D; ++k) {
        lo[k] = wave_minv(lo[k]);
        hi[k] = wave_maxv(hi[k]);
    }
    if(threadIdx.x != 0) return;
    double edge = 0.0;
    for(int k = 0; k < D; ++k) {
        scal[S_ROOT_CX + k] = (hi[k] + lo[k]) * 0.5;
        const double r = hi[k] - lo[k];
        if(edge < r) edge = r;
    }
    scal[S_ROOT_EDGE] = edge;
}

// Levels of the tree (> deepest level: max_level + 1 <= 65).
constexpr int NLEVEL = 72;

// Layout of lvl, all cleared by the keys' kernel: the number of search
// groups, the sort's flag and the number of nodes (one copy takes them to the
// host), the scans' tickets, and the number of slice-spanning cells of each
// level.
constexpr int LVL_GROUPS = 0, LVL_SORT = 1, LVL_NODES = 2, LVL_HOST = 3, LVL_TICKET = 3, LVL_SPAN = 5, LVL_SIZE = LVL_SPAN + NLEVEL;

// ------------------------------------------------------------------- scan
// Exclusive scans by tiles: a block scans its tile and publishes the tile's
// sum; the block that publishes last replaces the sums by their own scan
// (their total at [gridDim.x]).  An element's prefix is its place in the
// tile plus the tile's, two loads instead of a second pass; one launch.
constexpr int SCAN_THREADS = 1024;

// Exclusive scan over a block of SCAN_THREADS.
__device__ __forceinline__ int block_scan(int v, int *sh, int &total)
{
    constexpr int NWAVE = SCAN_THREADS / WAVE;
    const int lane = wave_lane(), w = threadIdx.x / WAVE;
    int inc = v;
#pragma unroll
    for(int d = 1; d < WAVE; d *= 2) {
        const int u = __shfl_up(inc, d, WAVE);
        if(lane >= d) inc += u;
    }
    __syncthreads();  // sh is free
    if(lane == WAVE - 1) sh[w] = inc;
    __syncthreads();
    int before = 0;
    total = 0;
#pragma unroll
    for(int k = 0; k < NWAVE; ++k) {
        const int x = sh[k];
        before += k < w ? x : 0;
        total += x;
    }
    return before + inc - v;
}

__device__ __forceinline__ void scan_publish(int sum, int *base, int *ticket, int *sh)
{
    const int nb = gridDim.x;
    if(threadIdx.x == 0) put(base + blockIdx.x, sum);
    if(!last_block(ticket)) return;
    int carry = 0;
    for(int k0 = 0; k0 < nb; k0 += SCAN_THREADS) {
        const int k = k0 + threadIdx.x;
        const int v = k < nb ? get(base + k) : 0;
        int total;
        const int ex = block_scan(v, sh, total);
        if(k < nb) base[k] = carry + ex;
        carry += total;
    }
    if(threadIdx.x == 0) base[nb] = carry;
}

// ------------------------------------------------------------------- keys
// The keys' sort.  The particles of one cell of an upper level (a bucket: the
// cells numbered by the leading bucket_bits of the key, at most twice as many
// as there are particles) are counted as the keys are made, the counts
// scanned, the particles moved to their bucket's range, and each finds its
// place there by counting the smaller (key, index) pairs: the order of a
// stable sort by key, whatever order the counting took.  What bounds it is
// launch latency and one pass over keys and indices each; with some ten
// particles to a bucket the comparisons are few (reorder included 99 us at
// 1M particles, 24 us at 393k).  Steps against the library's merge sort (up
// to 1M keys) and radix sort: 2D KHI at 393k 0.863 -> 0.766 ms, the blast at
// 2M 5.31 -> 5.05, Evrard at 20k 0.470 -> 0.445 and at 1M 4.92 -> 4.82; at
// 400 and 4,096 particles the launches are as many and the time the same.
// A bucket of more than BUCKET_MOST particles would make the counting
// quadratic: the build is then done again with the library's sort, which is
// kept for the next BUCKET_WAIT builds.
constexpr int BUCKET_MOST = 512;
constexpr int BUCKET_WAIT = 16;

// The reference's descent, one level per slot group (src/bhtree.cpp:163-204).
// With cnt, also each particle's rank in its bucket, in idx (otherwise idx
// receives the index).
template <int D>
__global__ void __launch_bounds__(BLOCK) keys_kernel(State s, int n, const double *scal, int levels, uint64_t *keys, int *idx,
                                                     int *cnt, int shift, int *lvl)
{
#pragma clang fp contract(off)
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if(i < LVL_SIZE) lvl[i] = 0;  // the first block has them all
    if(i >= n) return;
    double c[D], x[D];
#pragma unroll
    for(int k = 0; k < D; ++k) { c[k] = scal[S_ROOT_CX + k]; x[k] = s.f[F_X + k][i]; }
    double e = scal[S_ROOT_EDGE];
    uint64_t key = 0;
    for(int L = 0; L < levels; ++L) {
        uint64_t slot = 0;
#pragma unroll
        for(int k = 0; k < D; ++k) {
            const bool up = x[k] > c[k];
            slot |= (uint64_t)up << k;
            c[k] = c[k] + (up ? 1.0 : -1.0) * e * 0.25;
        }
        e = e * 0.5;
        key = (key << D) | slot;
    }
    keys[i] = key;
    if(!cnt) {
        idx[i] = i;
        return;
    }
    // Neighbouring lanes are mostly in one bucket (the particles are nearly
    // in key order): the first lane of each run counts for the run, as many
    // updates of one counter would run one after the other.
    const int b = (int)(key >> shift);
    const int lane = wave_lane();
    const int before = __shfl_up(b, 1, WAVE);  // by every lane: lane 1 reads lane 0
    const bool head = lane == 0 || before != b;
    const uint64_t heads = ballot(head), here = ballot(true);
    const int first = 63 - __clzll((long long)(heads & (~0ull >> (63 - lane))));
    const uint64_t later = lane == 63 ? 0 : heads >> (lane + 1) << (lane + 1);
    const int end = later ? (int)__builtin_ctzll(later) : __popcll(here);
    int base = 0;
    if(head) base = atomicAdd(cnt + b, end - lane);
    idx[i] = __shfl(base, first, WAVE) + (lane - first);
}

static_assert(LVL_SIZE <= BLOCK, "one block of the keys' kernel clears lvl");

// The buckets' starts; clears their counts.
constexpr int BUCKET_TILE = 4 * SCAN_THREADS;
struct BucketOff {
    const int *off, *base;
    __device__ __forceinline__ int operator()(int b) const { return off[b] + base[b / BUCKET_TILE]; }
};

__global__ void __launch_bounds__(SCAN_THREADS) bucket_scan_kernel(int4 *cnt, int nbucket, int4 *off, int *base, int *ticket)
{
    __shared__ int sh[SCAN_THREADS / WAVE];
    const int i = blockIdx.x * SCAN_THREADS + threadIdx.x;
    int4 v = make_int4(0, 0, 0, 0);
    if(i < nbucket / 4) {
        v = cnt[i];
        cnt[i] = make_int4(0, 0, 0, 0);
    }
    int total;
    const int ex = block_scan(v.x + v.y + v.z + v.w, sh, total);
    if(i < nbucket / 4) off[i] = make_int4(ex, ex + v.x, ex + v.x + v.y, ex + v.x + v.y + v.z);
    scan_publish(total, base, ticket, sh);
}

// Keys and indices into their buckets' ranges.
__global__ void __launch_bounds__(BLOCK) bucket_scatter_kernel(const uint64_t *keys, const int *rank, int n, int shift, BucketOff off,
                                                               uint64_t *bkeys, int *bidx)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if(i >= n) return;
    const uint64_t key = keys[i];
    const int p = off((int)(key >> shift)) + rank[i];
    bkeys[p] = key;
    bidx[p] = i;
}

// --------------------------------------------------------------- reorder
constexpr int PACK_BESIDE = 1 << 19;  // with gravity, more particles than this have their records packed later (Reorder::pm)

struct Reorder {
    const double *src[NF];
    double *dst[NF];
    const int *isrc[2];
    int *idst[2];
    // with sml set: the gather search radius of every particle in the new
    // order, from its mass and density (the combined search's radius)
    double *sml;
    const double *mass, *dens;
    double nngb, ratio;
    // the pre-interaction's records (pm null: none; rec is PreRec<float> with
    // mixed), written here where their fields pass through anyway: a launch
    // and a pass less (steps: 1D, 1,600 particles 0.171 -> 0.160 ms, 2D KHI at
    // 393k 0.687 -> 0.679, FP64 Evrard at 131k 1.195 -> 1.186).  In large runs
    // with gravity the separate pass goes beside the gravity walk and costs
    // less (2^20 particles: 4.594 ms, with the records here 4.611).
    State old;
    double4 *pm;
    void *rec;
    bool mixed;
    // sort by buckets: the keys in their buckets' ranges, the buckets' starts
    // and the sorted keys (bkeys null: perm is sorted)
    const uint64_t *bkeys;
    BucketOff off;
    int shift, nbucket;
    uint64_t *keys;
    int *sort_flag;
};

template <int D> __global__ void __launch_bounds__(BLOCK) reorder_kernel(Reorder r, const int *perm, int n, int nfields)
{
    const int p = blockIdx.x * BLOCK + threadIdx.x;
    if(p >= n) return;
    const int j = perm[p];
    int i = p;  // the particle's place
    if(r.bkeys) {
        const uint64_t key = r.bkeys[p];
        const int b = (int)(key >> r.shift);
        const int lo = r.off(b), hi = b + 1 < r.nbucket ? r.off(b + 1) : n;
        if(hi - lo <= BUCKET_MOST) {
            i = lo;
#pragma unroll 4
            for(int q = lo; q < hi; ++q) {
                const uint64_t k = r.bkeys[q];
                i += k < key || (k == key && perm[q] < j);
            }
        } else {
            *r.sort_flag = 1;
        }
        r.keys[i] = key;
    }
    for(int f = 0; f < nfields; ++f) r.dst[f][i] = r.src[f][j];
    r.idst[0][i] = r.isrc[0][j];
    if(r.isrc[1]) r.idst[1][i] = r.isrc[1][j];
    if(r.sml) r.sml[i] = sml_guess<D>(r.mass[j], r.dens[j], r.nngb, r.ratio);
    if(r.pm) {
        double4 pm;
        if(r.mixed) ((PreRec<float> *)r.rec)[i] = make_pre_rec<D, float>(r.old, j, pm);
        else ((PreRec<double> *)r.rec)[i] = make_pre_rec<D, double>(r.old, j, pm);
        r.pm[i] = pm;
    }
}

// ----------------------------------------------------------------- delta
// delta[i] = number of equal leading slot groups of keys i-1 and i: the two
// particles share the cells of levels 1 .. delta+1.
__device__ __forceinline__ int key_delta(const uint64_t *k, int i, int G, int D)
{
    if(i == 0) return 0;
    const uint64_t x = k[i - 1] ^ k[i];
    if(x == 0) return G;
    const int lz = __clzll((long long)x) - (64 - G * D);
    return lz / D;
}

// Search groups: compact sets of at most 64 key-consecutive particles.
// Every cell holding more than 64 particles packs its children that hold at
// most 64 (cells the tree does not split further, or leaves) into groups,
// consecutive children filling a group until the next would take it past
// 64; a child holding more than 64 is packed by its own children, and a
// leaf holding more than 64 is cut into runs of 64.  A group then lies in
// one parent cell, so its box is compact, and it is as full as siblings
// allow (46.7 particles on average at the Evrard benchmark's density
// profile, against 15.6 for single cells; runs of 64 key-consecutive
// particles fill the waves but can straddle a jump of the key order across
// the domain).  In 1D and 2D a stretch of consecutive small children is
// instead cut into equal groups of at most 64 (still inside the parent).
constexpr int GROUP = 64;

struct TreeShape {
    int n, G, D, leaf, max_level;
};

// First level at which particle b begins a cell, from its delta.
__device__ __forceinline__ int first_level(int delta_b, int b) { return b == 0 ? 2 : delta_b + 2; }

// Level-L cells are the runs of sorted keys that share their top L-1 levels
// (the prefix cell_end compares).  The two helpers below find a run's ends
// within leaf positions of b by binary search over the keys, so every lane
// takes the same few steps (a scan of the key-difference bytes took up to
// 2 leaf steps, different for each lane).
__device__ __forceinline__ uint64_t cell_prefix(uint64_t k, int shift) { return shift >= 64 ? 0 : k >> shift; }

// Size of the level-L cell that begins at b, or leaf+1 if it is larger.
__device__ __forceinline__ int cell_count_bounded(const uint64_t *keys, const TreeShape &ts, int b, int L)
{
    const int shift = (ts.G - (L - 1)) * ts.D;
    const uint64_t pre = cell_prefix(keys[b], shift);
    // last member of the run in [b, b + leaf]
    int lo = b, hi = min(ts.n - 1, b + ts.leaf);
    while(lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if(cell_prefix(keys[mid], shift) > pre) hi = mid - 1;
        else lo = mid;
    }
    return lo - b + 1;  // leaf + 1 when the run reaches b + leaf
}

// Does the level-P cell containing b hold more than leaf particles?  Its
// members within leaf positions on either side of b number more than leaf
// exactly when the whole cell does.
__device__ __forceinline__ bool parent_split(const uint64_t *keys, const TreeShape &ts, int b, int P)
{
    const int shift = (ts.G - (P - 1)) * ts.D;
    const uint64_t pre = cell_prefix(keys[b], shift);
    int lo = max(0, b - ts.leaf), hi = b;  // first member in [b - leaf, b]
    while(lo < hi) {
        const int mid = (lo + hi) >> 1;
        if(cell_prefix(keys[mid], shift) < pre) lo = mid + 1;
        else hi = mid;
    }
    const int first = lo;
    lo = b;
    hi = min(ts.n - 1, b + ts.leaf);  // last member in [b, b + leaf]
    while(lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if(cell_prefix(keys[mid], shift) > pre) hi = mid - 1;
        else lo = mid;
    }
    return lo - first + 1 > ts.leaf;
}

// Number of nodes that begin at particle b (all at consecutive levels).
__device__ __forceinline__ int nodes_at(const uint64_t *keys, int delta_b, const TreeShape &ts, int b)
{
    if(b > 0 && delta_b >= ts.G) return 0;  // same deepest cell as b-1
    const int lvl0 = first_level(delta_b, b);
    if(lvl0 > 2 && !parent_split(keys, ts, b, lvl0 - 1)) return 0;
    int k = 0;
    for(int L = lvl0;; ++L) {
        ++k;
        const int cnt = cell_count_bounded(keys, ts, b, L);
        if(!(cnt > ts.leaf && L <= ts.max_level)) break;
    }
    return k;
}

// Nodes beginning at each particle, scanned by tiles of SCAN_THREADS, and
// the deltas for emit_nodes_kernel.  None where the sort has given up: the
// keys are then in no order, and the host builds again.
__global__ void __launch_bounds__(SCAN_THREADS) count_nodes_kernel(const uint64_t *keys, TreeShape ts, uint8_t *delta, int *nn, int *noff,
                                                                int *base, int *lvl)
{
    __shared__ int sh[SCAN_THREADS / WAVE];
    const int b = blockIdx.x * SCAN_THREADS + threadIdx.x;
    int k = 0;
    if(b < ts.n && !lvl[LVL_SORT]) {
        const int d = key_delta(keys, b, ts.G, ts.D);
        delta[b] = (uint8_t)d;
        k = nodes_at(keys, d, ts, b);
    }
    int total;
    const int ex = block_scan(k, sh, total);
    if(b < ts.n) {
        nn[b] = k;
        noff[b] = ex;
    }
    scan_publish(total, base, lvl + LVL_TICKET + 1, sh);
}

// End (exclusive) of the level-L cell that begins at b: first particle
// whose key differs in the first L-1 slot groups.  Most cells are small, so
// steps of 16, 64, ... look for a stretch that holds the end first.
__device__ __forceinline__ int cell_end(const uint64_t *keys, const TreeShape &ts, int b, int L)
{
    const int shift = (ts.G - (L - 1)) * ts.D;
    const uint64_t pre = cell_prefix(keys[b], shift);
    int in = b, step = 16;
    while(step < ts.n - in && cell_prefix(keys[in + step], shift) == pre) {
        in += step;
        step = step < 1 << 28 ? step * 4 : step;
    }
    int lo = in + 1, hi = step < ts.n - in ? in + step : ts.n;
    while(lo < hi) {
        const int mid = (lo + hi) >> 1;
        if(cell_prefix(keys[mid], shift) > pre) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}

// Mass and centre of mass of a node from its sums.  The root's stay zero.
__device__ __forceinline__ void store_mom(const TreeDev &t, int p, const double4 &acc)
{
    if(p == 0) t.mom[0] = make_double4(0.0, 0.0, 0.0, 0.0);
    else t.mom[p] = make_double4(acc.x / acc.w, acc.y / acc.w, acc.z / acc.w, acc.w);
}

template <int D> __device__ __forceinline__ void leaf_moments(const State &s, const TreeDev &t, int p, int begin, int end, double4 *msum)
{
    double4 acc = make_double4(0.0, 0.0, 0.0, 0.0);
    double mx[3] = {0.0, 0.0, 0.0};
    for(int j = begin; j < end; ++j) {
        const double mj = s.f[F_MASS][j];
        acc.w += mj;
#pragma unroll
        for(int q = 0; q < D; ++q) mx[q] += s.f[F_X + q][j] * mj;
    }
    acc.x = mx[0];
    acc.y = mx[1];
    acc.z = mx[2];
    msum[p] = acc;
    store_mom(t, p, acc);
}

// The nodes that begin at a block's particles: a node per lane (they are
// consecutive; the particle by bisection in LDS), so that no lane walks a
// chain of searches for a particle where many cells begin.  Also the search
// group of a root that holds at most GROUP particles, and the leaves' moments
// (their particles in order).  At 400 particles (11
// levels) 13 us, without the leaves' moments and with a particle per lane 26;
// in 2D at 393k 15 (39), in 3D at 2M 109 (126).
template <int D>
__global__ void __launch_bounds__(BLOCK) emit_nodes_kernel(const uint64_t *keys, const uint8_t *delta, TreeShape ts, const int *nn,
                                                        const int *noff, const int *base, const double *scal, State s, TreeDev t, double4 *msum,
                                                        int64_t node_cap, int64_t *counters, int2 *groups, int *num_groups, int *nodes_out)
{
#pragma clang fp contract(off)
    __shared__ int first[BLOCK + 1];  // first node of each particle
    const int b0 = blockIdx.x * BLOCK, nb = min(BLOCK, ts.n - b0);
    const int total = 1 + base[(ts.n + SCAN_THREADS - 1) / SCAN_THREADS];
    const auto node_of = [&](int b) { return 1 + noff[b] + base[b / SCAN_THREADS]; };
    if((int)threadIdx.x < nb) {
        const int b = b0 + threadIdx.x;
        const int f = node_of(b);
        first[threadIdx.x] = f;
        if((int)threadIdx.x == nb - 1) first[nb] = f + nn[b];
        if(b == 0) {
            *t.num_nodes = *nodes_out = total <= node_cap ? total : (int)node_cap;
            if(total > node_cap) atomicAdd((unsigned long long *)&counters[C_TREE_ERR], 1ull);
            t.geo[0] = make_double4(scal[S_ROOT_CX], D > 1 ? scal[S_ROOT_CY] : 0.0, D > 2 ? scal[S_ROOT_CZ] : 0.0, scal[S_ROOT_EDGE]);
            t.rng[0] = make_int4(0, ts.n, total, 1);
            if(ts.n <= GROUP) {
                groups[0] = make_int2(0, ts.n);
                *num_groups = 1;
            }
        }
    }
    __syncthreads();
    const uint64_t mask = (1ull << D) - 1ull;
    const int end_node = min((int64_t)first[nb], node_cap);
    for(int node = first[0] + threadIdx.x; node < end_node; node += BLOCK) {
        int lo = 0, hi = nb - 1;  // last particle whose first node is not past this one
        while(lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if(first[mid] <= node) lo = mid;
            else hi = mid - 1;
        }
        const int b = b0 + lo;
        const int L = first_level((int)delta[b], b) + node - first[lo];
        const bool leaf = node == first[lo + 1] - 1;
        const uint64_t key = keys[b];
        const int end = leaf && L <= ts.max_level ? b + cell_count_bounded(keys, ts, b, L) : cell_end(keys, ts, b, L);
        const int skip = end < ts.n ? node_of(end) : total;
        // replay the descent down to level L
        double c[D];
#pragma unroll
        for(int k = 0; k < D; ++k) c[k] = scal[S_ROOT_CX + k];
        double e = scal[S_ROOT_EDGE];
        for(int g = 0; g < L - 1; ++g) {
            const uint64_t slot = (key >> ((ts.G - 1 - g) * D)) & mask;
#pragma unroll
            for(int k = 0; k < D; ++k) c[k] = c[k] + (((slot >> k) & 1) ? 1.0 : -1.0) * e * 0.25;
            e = e * 0.5;
        }
        t.geo[node] = make_double4(c[0], D > 1 ? c[D > 1 ? 1 : 0] : 0.0, D > 2 ? c[D > 2 ? 2 : 0] : 0.0, e);
        t.rng[node] = make_int4(b, end, skip, L | (leaf ? 256 : 0));
        if(leaf) leaf_moments<D>(s, t, node, b, end, msum);
    }
}

// ---------------------------------------------------- moments and groups
__device__ __forceinline__ int node_level(const int4 &r) { return (r.w & 255) < NLEVEL ? (r.w & 255) : NLEVEL - 1; }

// The search groups of a packing cell (range rq, first child q + 1):
// emit(begin, end) for each.  small(c) is the number of particles of node c
// if it is at most GROUP, otherwise -1; next(c) the node after its subtree.
template <class Small, class Next, class Emit>
__device__ __forceinline__ void pack_groups(const int4 *rng, int q, const int4 &rq, int total, bool runs, Small &&small, Next &&next, Emit &&emit)
{
    // runs: a stretch [b, e) of consecutive small children is cut into
    // ceil((e - b) / GROUP) groups of equal size, which fills the waves
    // but does not keep whole cells together
    auto cut = [&](int b, int e) {
        const int k = runs ? (e - b + GROUP - 1) / GROUP : 1;
        for(int j = 0; j < k; ++j) emit(b + (e - b) * j / k, b + (e - b) * (j + 1) / k);  // at most 8 GROUP particles
    };
    const int end = min(rq.z, total);
    int cb = -1, ce = rq.x;  // the open stretch; the children cover the cell in order
    for(int c = q + 1; c < end; c = next(c)) {
        const int cnt = small(c);
        if(cnt < 0) {
            if(cb >= 0) cut(cb, ce);
            cb = -1;
            const int4 rc = rng[c];
            if(rc.w & 256)
                for(int b = rc.x; b < rc.y; b += GROUP) emit(b, b + GROUP < rc.y ? b + GROUP : rc.y);
            ce = rc.y;
        } else {
            if(!runs && cb >= 0 && ce + cnt - cb > GROUP) {
                cut(cb, ce);
                cb = -1;
            }
            if(cb < 0) cb = ce;
            ce += cnt;
        }
    }
    if(cb >= 0) cut(cb, ce);
}

// Moments of the internal cells and search groups of SLICE consecutive
// nodes.  A cell sums its children, in child order: the cells whose whole
// subtree lies in the slice, level after level in LDS.  For those that reach
// past it (one to a level at most) the children are listed for
// spanning_kernel, and the sums that these need go to msum.  What bounds it
// is latency (about eight dependent LDS reads per cell and level); one
// launch takes the place of node lists by level and a launch for each
// level: 29 us (with the moments of leaves 61) in 2D at 393k
// particles, 39 (153) at 1M and 105 (400) at 2M in 3D.
constexpr int SLICE = 2048;  // the larger, the fewer cells span slices; 74 KB of LDS
constexpr int NO_CHILD = -1;  // a child c that spans slices itself is listed as -2 - c
constexpr int SLICE_PER = SLICE / SCAN_THREADS;
__global__ void __launch_bounds__(SCAN_THREADS) slice_kernel(TreeDev t, double4 *msum, int *span_cnt, int *span, int4 *span_child, int span_cap,
                                                          int2 *groups, int *num_groups, int64_t group_cap, int runs)
{
    __shared__ double4 m[SLICE];
    __shared__ uint16_t skip[SLICE];   // of the cells within the slice: the node after the subtree
    __shared__ uint8_t count[SLICE];   // particles, or 255 (more than GROUP)
    __shared__ uint8_t used[SLICE];    // internal cells: summed into the parent
    __shared__ int deepest, ngroups, group0;
    const int total = *t.num_nodes;
    for(int v0 = blockIdx.x * SLICE; v0 < total; v0 += gridDim.x * SLICE) {
        const int nloc = min(SLICE, total - v0), v1 = v0 + nloc;
        if(threadIdx.x == 0) {
            deepest = 0;
            ngroups = 0;
        }
        __syncthreads();
        int4 r[SLICE_PER];
        int level[SLICE_PER];  // of an internal cell within the slice, otherwise -1
#pragma unroll
        for(int k = 0; k < SLICE_PER; ++k) {
            const int i = threadIdx.x + k * SCAN_THREADS;
            r[k] = i < nloc ? t.rng[v0 + i] : make_int4(0, 0, 0, 0);
        }
#pragma unroll
        for(int k = 0; k < SLICE_PER; ++k) {
            const int i = threadIdx.x + k * SCAN_THREADS;
            level[k] = -1;
            if(i >= nloc) continue;
            skip[i] = (uint16_t)min(r[k].z - v0, SLICE);
            count[i] = (uint8_t)(r[k].y - r[k].x <= GROUP ? r[k].y - r[k].x : 255);
            used[i] = 0;
            if(r[k].w & 256) {
                m[i] = msum[v0 + i];
            } else if(r[k].z <= v1) {
                level[k] = node_level(r[k]);
                atomicMax(&deepest, level[k]);
            }
        }
        __syncthreads();
        for(int L = deepest; L >= 1; --L) {
#pragma unroll
            for(int k = 0; k < SLICE_PER; ++k) {
                if(level[k] != L) continue;
                const int i = threadIdx.x + k * SCAN_THREADS;
                const int end = r[k].z - v0;
                double4 acc = make_double4(0.0, 0.0, 0.0, 0.0);
                int guard = 0;
                for(int c = i + 1; c < end && guard < 8; c = skip[c], ++guard) {
                    const double4 v = m[c];
                    acc.x += v.x; acc.y += v.y; acc.z += v.z; acc.w += v.w;
                    used[c] = 1;
                }
                m[i] = acc;
            }
            __syncthreads();
        }
        const auto small = [&](int c) {
            if(c < v1) return count[c - v0] <= GROUP ? (int)count[c - v0] : -1;
            const int4 rc = t.rng[c];
            return rc.y - rc.x <= GROUP ? rc.y - rc.x : -1;
        };
        const auto next = [&](int c) { return c < v1 && skip[c - v0] < SLICE ? v0 + skip[c - v0] : t.rng[c].z; };
        int ng[SLICE_PER], at0[SLICE_PER];
#pragma unroll
        for(int k = 0; k < SLICE_PER; ++k) {
            const int i = threadIdx.x + k * SCAN_THREADS;
            ng[k] = at0[k] = 0;
            if(i >= nloc) continue;
            if(r[k].w & 256) continue;
            if(level[k] >= 0) {
                const double4 acc = m[i];
                store_mom(t, v0 + i, acc);
                if(!used[i]) msum[v0 + i] = acc;
            } else {
                const int L = node_level(r[k]), slot = atomicAdd(span_cnt + L, 1);
                int child[8], c = v0 + i + 1;
                const int end = min(r[k].z, total);
#pragma unroll
                for(int q = 0; q < 8; ++q) {
                    child[q] = NO_CHILD;
                    if(c >= end) continue;
                    const int4 rc = t.rng[c];
                    const bool spans = !(rc.w & 256) && rc.z > (c / SLICE + 1) * SLICE && rc.z > c;
                    child[q] = spans ? -2 - c : c;
                    c = rc.z > c ? rc.z : c + 1;
                }
                if(slot < span_cap) {
                    const int64_t at = (int64_t)L * span_cap + slot;
                    span[at] = v0 + i;
                    span_child[2 * at] = make_int4(child[0], child[1], child[2], child[3]);
                    span_child[2 * at + 1] = make_int4(child[4], child[5], child[6], child[7]);
                }
            }
            if(r[k].y - r[k].x > GROUP) {
                pack_groups(t.rng, v0 + i, r[k], total, runs, small, next, [&](int, int) { ++ng[k]; });
                if(ng[k]) at0[k] = atomicAdd(&ngroups, ng[k]);
            }
        }
        __syncthreads();
        if(threadIdx.x == 0 && ngroups) group0 = atomicAdd(num_groups, ngroups);
        __syncthreads();
#pragma unroll
        for(int k = 0; k < SLICE_PER; ++k) {
            if(!ng[k]) continue;
            int64_t g = (int64_t)group0 + at0[k];
            pack_groups(t.rng, v0 + (int)threadIdx.x + k * SCAN_THREADS, r[k], total, runs, small, next, [&](int b, int e) {
                if(g < group_cap) groups[g] = make_int2(b, e);
                ++g;
            });
        }
        __syncthreads();  // the slice's LDS is free
    }
}

// Moments of the cells that span slices, in one workgroup: the children
// within slices are fetched for all cells at once, then level after level
// bottom-up those that span slices themselves; a barrier between levels
// orders the children's results before their parents read them (one
// workgroup runs on one CU, whose waves see each other's stores once past
// the barrier).  Two chunks of cells take 84 us at
// 2M particles, one 10 to 18 at 393k and 1M.
__global__ void __launch_bounds__(SCAN_THREADS) spanning_kernel(TreeDev t, double4 *msum, const int *span_cnt, const int *span,
                                                             const int4 *span_child, int span_cap, int *work, int nwork)
{
    // the task counters of the search that follows
    for(int k = threadIdx.x; k < nwork; k += SCAN_THREADS) work[k] = 0;
    __shared__ int sh[SCAN_THREADS / WAVE];
    __shared__ int off[NLEVEL];  // of the level NLEVEL - 1 - e: deepest first
    if(*t.num_nodes <= SLICE) return;  // one slice: none spans
    int total;
    const int ex = block_scan((int)threadIdx.x < NLEVEL ? span_cnt[NLEVEL - 1 - threadIdx.x] : 0, sh, total);
    if((int)threadIdx.x < NLEVEL) off[threadIdx.x] = ex;
    __syncthreads();
    const auto entry = [&](int k) {  // the last e with off[e] <= k
        int lo = 0, hi = NLEVEL - 1;
        while(lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if(off[mid] <= k) lo = mid;
            else hi = mid - 1;
        }
        return lo;
    };
    for(int k0 = 0; k0 < total; k0 += SCAN_THREADS) {
        const int k = k0 + threadIdx.x;
        int e = -1, p = 0;
        int child[8];
        double4 v[8];
        if(k < total) {
            e = entry(k);
            const int64_t at = (int64_t)(NLEVEL - 1 - e) * span_cap + k - off[e];
            p = span[at];
            const int4 a = span_child[2 * at], b = span_child[2 * at + 1];
            child[0] = a.x; child[1] = a.y; child[2] = a.z; child[3] = a.w;
            child[4] = b.x; child[5] = b.y; child[6] = b.z; child[7] = b.w;
#pragma unroll
            for(int q = 0; q < 8; ++q)
                if(child[q] >= 0) v[q] = msum[child[q]];
        }
        const int e1 = entry(min(k0 + SCAN_THREADS, total) - 1);
        for(int x = entry(k0); x <= e1; ++x) {
            if(e == x) {
                double4 acc = make_double4(0.0, 0.0, 0.0, 0.0);
#pragma unroll
                for(int q = 0; q < 8; ++q) {
                    if(child[q] == NO_CHILD) continue;
                    if(child[q] < NO_CHILD) v[q] = msum[-2 - child[q]];
                    acc.x += v[q].x; acc.y += v[q].y; acc.z += v[q].z; acc.w += v[q].w;
                }
                msum[p] = acc;
                store_mom(t, p, acc);
            }
            __syncthreads();
        }
    }
}

// One level of them, the deepest first, by many blocks: the single workgroup
// handles about a thousand cells in some 20 us, one batch after the other, a
// launch for each level takes 3 us.  How many cells span slices follows the
// nodes, so the line is drawn there, not at a number of particles (whose nodes
// differ by a factor of ten with leafParticleNumber).  Tree build, batches
// against launches, us: 1.90M nodes (1.5M particles, one to a leaf) 457 and 461,
// 2.10M (1D) 398 and 391, 2.33M (4.2M particles, eight to a leaf) 918 and 914,
// 2.40M (2.1M, one) 580 and 562, 5.8M (4.2M, one) 1,320 and 1,087; but 299k nodes
// (4.2M particles, 32 to a leaf) 761 and 822.
constexpr int SPAN_BATCHES = 2000000;
__global__ void __launch_bounds__(BLOCK) spanning_level_kernel(TreeDev t, double4 *msum, const int *span_cnt, const int *span,
                                                            const int4 *span_child, int span_cap, int L, int *work, int nwork)
{
    const int first = blockIdx.x * BLOCK + threadIdx.x;
    if(first < nwork) work[first] = 0;
    for(int k = first; k < span_cnt[L]; k += gridDim.x * BLOCK) {
        const int64_t at = (int64_t)L * span_cap + k;
        const int p = span[at];
        const int4 a = span_child[2 * at], b = span_child[2 * at + 1];
        const int child[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        double4 v[8];
#pragma unroll
        for(int q = 0; q < 8; ++q)
            if(child[q] != NO_CHILD) v[q] = msum[child[q] < NO_CHILD ? -2 - child[q] : child[q]];
        double4 acc = make_double4(0.0, 0.0, 0.0, 0.0);
#pragma unroll
        for(int q = 0; q < 8; ++q) {
            if(child[q] == NO_CHILD) continue;
            acc.x += v[q].x; acc.y += v[q].y; acc.z += v[q].z; acc.w += v[q].w;
        }
        msum[p] = acc;
        store_mom(t, p, acc);
    }
}

// ------------------------------------------------------------------ host
int tree_alloc(Ctx &c)
{
    const int64_t n = c.cap_n;
    c.node_cap = 5 * n + 1;  // BHTree::resize: 5 nodes per particle (+ root)
    SPHGPU_HIP(hipMalloc(&c.keys, n * sizeof(uint64_t)));
    SPHGPU_HIP(hipMalloc(&c.keys_sorted, n * sizeof(uint64_t)));
    SPHGPU_HIP(hipMalloc(&c.idx, n * sizeof(int)));
    SPHGPU_HIP(hipMalloc(&c.perm, n * sizeof(int)));
    SPHGPU_HIP(hipMalloc(&c.delta, n));
    SPHGPU_HIP(hipMalloc(&c.nn, n * sizeof(int)));
    SPHGPU_HIP(hipMalloc(&c.noff, n * sizeof(int)));
    SPHGPU_HIP(hipMalloc(&c.nbase, (grid_for(n, SCAN_THREADS) + 1) * sizeof(int)));
    SPHGPU_HIP(hipMalloc(&c.t.geo, c.node_cap * sizeof(double4)));
    SPHGPU_HIP(hipMalloc(&c.t.mom, c.node_cap * sizeof(double4)));
    SPHGPU_HIP(hipMalloc(&c.t.rng, c.node_cap * sizeof(int4)));
    SPHGPU_HIP(hipMalloc(&c.t.num_nodes, sizeof(int)));
    c.span_cap = (int)grid_for(c.node_cap, SLICE);
    SPHGPU_HIP(hipMalloc(&c.span, (size_t)NLEVEL * c.span_cap * sizeof(int)));
    SPHGPU_HIP(hipMalloc(&c.span_child, (size_t)NLEVEL * c.span_cap * 2 * sizeof(int4)));
    SPHGPU_HIP(hipMalloc(&c.msum, c.node_cap * sizeof(double4)));
    if(c.p.gravity_is_valid) {
        SPHGPU_HIP(hipMalloc(&c.gnode, c.node_cap * sizeof(GravNode)));
        // one spare record: a scalar load may fetch a whole record past the last
        SPHGPU_HIP(hipMalloc(&c.gpart, (n + 1) * sizeof(GravPart<double>)));
        SPHGPU_HIP(hipMalloc(&c.gacc, (size_t)c.D * n * sizeof(double)));
        // one record list per wave: a wave per 64 particles in blocks of
        // four, or several
        const size_t waves = (size_t)grid_for(n) * (BLOCK / WAVE) * gravity_parts(n, c.num_cu);
        SPHGPU_HIP(hipMalloc(&c.leafhit, waves * LEAFHIT_CAP * sizeof(LeafHit)));
        SPHGPU_HIP(hipMalloc(&c.leafcnt, waves * sizeof(int)));
    }
    if(!c.lvl) SPHGPU_HIP(hipMalloc(&c.lvl, LVL_SIZE * sizeof(int)));
    c.num_groups = c.lvl + LVL_GROUPS;
    if(!c.lvl_host) SPHGPU_HIP(hipHostMalloc(&c.lvl_host, LVL_HOST * sizeof(int), hipHostMallocDefault));
    for(int k = 0; k < LVL_HOST; ++k) c.lvl_host[k] = 0;
    // buckets: the cells of the deepest level that has at most twice as many
    // cells as there are particles
    int levels = 0;
    while(levels < c.p.tree_max_level && (levels + 1) * c.D <= 30 && ((int64_t)1 << ((levels + 1) * c.D)) <= 2 * (int64_t)n) ++levels;
    c.bucket_bits = levels * c.D;
    c.bucket_clear = false;
    c.bucket_wait = 0;
    c.tree_nodes = 0;
    const int64_t nbucket = std::max<int64_t>((int64_t)1 << c.bucket_bits, 4);  // scanned by fours
    SPHGPU_HIP(hipMalloc(&c.bucket_cnt, nbucket * sizeof(int)));
    SPHGPU_HIP(hipMalloc(&c.bucket_off, nbucket * sizeof(int)));
    SPHGPU_HIP(hipMalloc(&c.bucket_base, (grid_for(nbucket, BUCKET_TILE) + 1) * sizeof(int)));
    c.group_cap = c.node_cap + n / 64 + 1;
    SPHGPU_HIP(hipMalloc(&c.groups, c.group_cap * sizeof(int2)));
    size_t bytes = 0;
    const unsigned key_bits = (unsigned)(c.p.tree_max_level * c.D);
    SPHGPU_HIP(rocprim::radix_sort_pairs(nullptr, bytes, c.keys, c.keys_sorted, c.idx, c.perm, (unsigned)n, 0, key_bits, c.stream));
    c.sort_tmp_bytes = bytes;
    SPHGPU_HIP(hipMalloc(&c.sort_tmp, bytes));
    return SPHGPU_OK;
}

// Fields that a sphgpu_integrate step writes after its tree build before
// any kernel reads them: acc and du/dt (force pass), pressure, h and 1/h
// (pre-interaction; h is first the search radius the guess writes),
// grad-h (SSPH, DISPH), the Balsara switch where the pre-interaction sets it,
// and phi (gravity walk).
static bool rewritten_in_step(const Ctx &c, int f)
{
    if(f >= F_A && f < F_A + 3) return true;
    if(f == F_DENE || f == F_PRES || f == F_SML || f == F_HINV) return true;
    if(f == F_GRADH) return c.p.sph_type != SPHGPU_GSPH;
    if(f == F_BAL) return c.p.av_use_balsara_switch && c.D != 1 && c.p.sph_type != SPHGPU_GSPH;
    if(f == F_PHI) return c.p.gravity_is_valid != 0;
    return false;
}

__global__ void __launch_bounds__(BLOCK) clear_kernel(int *p, int n)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if(i < n) p[i] = 0;
}

template <int D> static int tree_build_d(Ctx &c)
{
    const int n = (int)c.n;
    const int G = c.p.tree_max_level;
    c.radius_ready = c.pre_packed = false;
    const bool buckets = c.bucket_wait == 0;
    if(!buckets) --c.bucket_wait;
    const int nbucket = 1 << c.bucket_bits, nscan = std::max(nbucket, 4), shift = G * D - c.bucket_bits;
    // root geometry
    if(!c.p.periodic_is_valid) {
        hipLaunchKernelGGL(bbox_kernel<D>, dim3(std::min(grid_for(n, BBOX_THREADS), c.num_cu)), dim3(BBOX_THREADS), 0, c.stream, c.s, n, c.partial,
                           c.ticket, c.scal);
    }
    if(buckets && !c.bucket_clear)
        hipLaunchKernelGGL(clear_kernel, dim3(grid_for(nscan)), dim3(BLOCK), 0, c.stream, c.bucket_cnt, nscan);
    c.bucket_clear = false;
    hipLaunchKernelGGL(keys_kernel<D>, dim3(grid_for(n)), dim3(BLOCK), 0, c.stream, c.s, n, c.scal, G, c.keys, c.idx,
                       buckets ? c.bucket_cnt : nullptr, shift, c.lvl);
    const BucketOff off{c.bucket_off, c.bucket_base};
    if(buckets) {
        hipLaunchKernelGGL(bucket_scan_kernel, dim3(grid_for(nscan, BUCKET_TILE)), dim3(SCAN_THREADS), 0, c.stream, (int4 *)c.bucket_cnt, nscan,
                           (int4 *)c.bucket_off, c.bucket_base, c.lvl + LVL_TICKET);
        hipLaunchKernelGGL(bucket_scatter_kernel, dim3(grid_for(n)), dim3(BLOCK), 0, c.stream, c.keys, c.idx, n, shift, off, c.keys_sorted, c.perm);
        c.bucket_clear = true;
        // the keys in bucket order are read, the sorted ones written
        std::swap(c.keys, c.keys_sorted);
    } else {
        size_t bytes = c.sort_tmp_bytes;
        SPHGPU_HIP(rocprim::radix_sort_pairs(c.sort_tmp, bytes, c.keys, c.keys_sorted, c.idx, c.perm, (unsigned)n, 0, (unsigned)(G * D), c.stream));
    }
    // gather the state into key order (in sphgpu_integrate, without the
    // fields that the step rewrites before anything reads them)
    Reorder r{};
    int nf = 0;
    for(int f = 0; f < NF; ++f) {
        if(!c.s.f[f]) continue;
        if(c.reorder_light && rewritten_in_step(c, f)) continue;
        r.src[nf] = c.s.f[f];
        r.dst[nf] = c.alt.f[f];
        ++nf;
    }
    r.isrc[0] = c.s.id; r.idst[0] = c.alt.id;
    r.isrc[1] = c.reorder_light ? nullptr : c.s.nb; r.idst[1] = c.alt.nb;
    // sphgpu_integrate's combined search needs the radii h_guess * ratio, set
    // here by the reorder, and its records and boxes
    const bool radius = c.reorder_light;
    const bool packed = radius && (!c.p.gravity_is_valid || n <= PACK_BESIDE);
    if(radius) {
        if(packed) {
            r.old = c.s;
            r.pm = c.posrec;
            r.rec = c.pair_rec;
            r.mixed = c.p.precision == SPHGPU_MIXED;
        }
        r.sml = c.alt.f[F_SML];
        r.mass = c.s.f[F_MASS];
        r.dens = c.s.f[F_DENS];
        r.nngb = (double)c.p.neighbor_number;
        r.ratio = c.p.iterative_sml ? 1.2 : 1.0;
    }
    if(buckets) {
        r.bkeys = c.keys;
        r.off = off;
        r.shift = shift;
        r.nbucket = nbucket;
        r.keys = c.keys_sorted;
        r.sort_flag = c.lvl + LVL_SORT;
    }
    hipLaunchKernelGGL(reorder_kernel<D>, dim3(grid_for(n)), dim3(BLOCK), 0, c.stream, r, c.perm, n, nf);
    const auto swap_state = [&c] {
        for(int f = 0; f < NF; ++f) std::swap(c.s.f[f], c.alt.f[f]);
        std::swap(c.s.id, c.alt.id);
        std::swap(c.s.nb, c.alt.nb);
    };
    swap_state();
    if(radius) {
        int rc = search_boxes(c, c.s.f[F_SML]);
        if(rc) return rc;
    }

    const TreeShape ts{n, G, D, c.p.tree_leaf_particle_num, c.p.tree_max_level};
    hipLaunchKernelGGL(count_nodes_kernel, dim3(grid_for(n, SCAN_THREADS)), dim3(SCAN_THREADS), 0, c.stream, c.keys_sorted, ts, c.delta, c.nn,
                       c.noff, c.nbase, c.lvl);
    hipLaunchKernelGGL(emit_nodes_kernel<D>, dim3(grid_for(n)), dim3(BLOCK), 0, c.stream, c.keys_sorted, c.delta, ts, c.nn, c.noff, c.nbase,
                       c.scal, c.s, c.t, c.msum, c.node_cap, c.counters, c.groups, c.num_groups, c.lvl + LVL_NODES);
    // in 1D and 2D the waves are filled from runs of small cells (2D KHI
    // step 2 % faster); in 3D whole cells stay together (the Evrard step
    // was 6 % slower with runs: less compact groups keep more candidates.
    // Both were measured when the search walked the octree, which took about
    // twice the box search's time, and not since)
    hipLaunchKernelGGL(slice_kernel, dim3(std::min(c.span_cap, 2 * c.num_cu)), dim3(SCAN_THREADS), 0, c.stream, c.t, c.msum, c.lvl + LVL_SPAN, c.span,
                       c.span_child, c.span_cap, c.groups, c.num_groups, c.group_cap, D < 3 ? 1 : 0);
    SPHGPU_HIP(hipMemcpyAsync(c.lvl_host, c.lvl, LVL_HOST * sizeof(int), hipMemcpyDeviceToHost, c.stream));
    SPHGPU_HIP(hipEventRecord(c.ev_tree, c.stream));
    // (by the last build's nodes; before the first, about as many as a lattice has)
    if((c.tree_nodes > 0 ? c.tree_nodes : 1.3 * n / ts.leaf) > SPAN_BATCHES) {
        for(int L = std::min(G + 1, NLEVEL - 1); L >= 1; --L)
            hipLaunchKernelGGL(spanning_level_kernel, dim3(c.num_cu), dim3(BLOCK), 0, c.stream, c.t, c.msum, c.lvl + LVL_SPAN, c.span,
                               c.span_child, c.span_cap, L, c.work, NUM_XCD * WORK_STRIDE);
    } else {
        hipLaunchKernelGGL(spanning_kernel, dim3(1), dim3(SCAN_THREADS), 0, c.stream, c.t, c.msum, c.lvl + LVL_SPAN, c.span, c.span_child,
                           c.span_cap, c.work, NUM_XCD * WORK_STRIDE);
    }
    SPHGPU_HIP(hipEventSynchronize(c.ev_tree));
    if(buckets && c.lvl_host[LVL_SORT]) {
        // a bucket was too full to be sorted: build again from the state as
        // it was, with the library's sort
        swap_state();
        c.bucket_wait = BUCKET_WAIT;
        return tree_build_d<D>(c);
    }
    c.tree_nodes = c.lvl_host[LVL_NODES];
    c.ngroups = c.lvl_host[LVL_GROUPS];
    if(c.ngroups < 1 || c.ngroups > c.group_cap) return set_error(SPHGPU_E_TREE, "search groups out of range");
    SPHGPU_HIP(hipGetLastError());
    c.radius_ready = radius;
    c.pre_packed = packed;
    return search_alloc(c);
}

int tree_build(Ctx &c)
{
    switch(c.D) {
    case 1: return tree_build_d<1>(c);
    case 2: return tree_build_d<2>(c);
    default: return tree_build_d<3>(c);
    }
}

}  // namespace sphgpu
