// Neighbour search (BHTree::neighbor_search, src/bhtree.cpp:114-126,
// 234-270) for the particles of one search group (at most 64
// key-consecutive particles) per wave, in three phases:
//
//  1. Boxes.  The key-sorted particles are cut into chunks of 32; every
//     chunk has a bounding box with the largest candidate radius in it, 64
//     chunks make a box of the second level and 64 of those one of the
//     third.  The wave tests 64 boxes at a time, one per lane, against the
//     group's own box, from the third level down, and keeps the chunks
//     whose box lies within reach: (distance of the two boxes)^2 <= H^2,
//     H the larger of the group's largest search radius and (symmetric
//     search) the box's largest radius.  Every pair that the reference's
//     test accepts is closer than that, so no candidate of any lane is lost.
//  2. Candidate staging.  The kept chunks' particles are read two chunks at
//     a time with coalesced loads; those within reach of the group box by
//     their own radius are kept, in key order, in the wave's staging buffer.
//  3. Candidate tiles.  With nc kept candidates and T = ceil(nc / 64)
//     tiles, tile t takes candidates t, t + T, t + 2T, ... (lane k of the
//     tile holds candidate t + kT).  The reference's leaf test
//     |x_i - x_j|^2 < H_i^2 with H_i = h_guess * kernel_ratio (gather,
//     src/pre_interaction.cpp:61-70) or max(h_i, leaf's largest h)
//     (symmetric, src/bhtree.cpp:237, 256) is applied by every lane to its
//     candidate for one particle i of the group after the other.  The
//     compare's result is then particle i's 64-bit hit mask of the tile; it
//     is moved to lane i and written with the tile's candidate indices to
//     the group's slab (layout: Ctx::tile_cand).
//
// What bounds it: vector issue in phase 3 (8 FP64 operations, 1-2 compares
// and 2 lane writes per particle and tile; vector ALUs 84 % busy on 2^21
// particles in 3D), and the latency of the dependent box and candidate loads
// in the first two.  Particle i's record is read with one scalar load for
// two tiles, so a test costs no LDS read and no instruction that builds
// bits, and the loop runs over the group's particles (47 on average in 3D)
// with every lane busy, not over 64 candidates with a lane per particle.
// The boxes replace a walk of the octree: their cost does not depend on
// leafParticleNumber, where a tree with one particle per leaf has about 1.4
// nodes per candidate to visit.  Combined search, before and after: 2D KHI,
// 393,160 particles, 515 -> 128 us; 3D periodic, 2^21 particles, leaf 1,
// 3,480 -> 800 us; Evrard, 2^20 particles, leaf 32, alone 1,440 -> 780 us
// (vector instructions 4.0e8 -> 2.5e8).
//
// The sets are the reference's (in mixed precision but for pairs across a
// periodic face that are closer to the cut than the rounding of a position);
// the reference then sorts each list by distance (src/bhtree.cpp:120-124) and
// stops at the first r >= h, whereas the pair passes here test r < h on the
// unsorted set -- the same set.
//
// The combined search takes H_ij = max(R_i, R_j) with the gather radii R,
// so that one search serves both the pre-interaction (which keeps the pairs
// with r < R_i) and the force stage.
#include "tiles.hpp"

#include <type_traits>

namespace sphgpu {

// What a hit is: r < R_i (gather), r < max(R_i, R_j) (combined), or
// r < max(h_i, largest h of j's leaf) (symmetric).
enum SearchMode : int { M_GATHER, M_COMBINED, M_SYMMETRIC };

struct SearchArgs {
    int n;
    const double4 *srec;  // position and squared candidate radius per particle
    const double *own;    // M_SYMMETRIC: h per particle (otherwise srec's radius)
    const double *origin; // of the boxes: the root cube's centre
    const ChunkBox *lev[3];
    int cnt[3];           // boxes per level
    const int2 *groups;
    const int *num_groups;
    int *cand;           // group slabs of candidate tiles (Ctx::tile_cand)
    uint64_t *ma;        // hit masks per (tile, lane)
    int *gnc;            // candidates per group, with the GNC_ flags
    int exact;           // FP64 pairs
    int wcap;            // slots per group slab and per staging buffer
    int *ws_j;           // staging buffers, one per persistent wave
    int cap;             // per-particle capacity (the reference's list size)
    int64_t *counters;
    int stats;            // add to the statistics counters (errors are always counted)
    int *work;           // per-XCD task counters, zeroed before the launch
};

constexpr int SW = BLOCK / WAVE;  // waves per block
constexpr int CHUNKCAP = 256;     // kept chunks collected per flush

// Minimum-image separation of one axis (include/periodic.hpp:34-59).
__device__ __forceinline__ double min_image1(const BoxDev &b, int k, double d)
{
    if(!b.on) return d;
    const double d2 = d + b.len[k], d3 = d - b.len[k];
    const double a1 = fabs(d), a2 = fabs(d2), a3 = fabs(d3);
    double r = d3;
    if(a2 <= a3 && a2 <= a1) r = d2;
    if(a1 <= a2 && a1 <= a3) r = d;
    return r;
}

// Axis k of the boxes' origin (zero where a particle has gone to infinity).
__device__ __forceinline__ double box_origin(const double *origin, int k)
{
    const double o = origin[k];
    return fabs(o) < __builtin_huge_val() ? o : 0.0;
}

// Does box b come within reach of the group's box (centre go from the boxes'
// origin, half extents ge, largest radius squared hmax2)?
template <int D, bool IJ>
__device__ __forceinline__ bool box_near(const BoxDev &box, const ChunkBox &b, const double go[D], const double ge[D], double hmax2)
{
    double d2 = 0.0;
#pragma unroll
    for(int k = 0; k < D; ++k) {
        const double c = 0.5 * ((double)b.lo[k] + (double)b.hi[k]), e = 0.5 * ((double)b.hi[k] - (double)b.lo[k]);
        const double ex = fabs(min_image1(box, k, go[k] - c)) - (ge[k] + e);
        d2 += ex > 0.0 ? ex * ex : 0.0;
    }
    double H2 = hmax2;
    if constexpr(IJ) {
        const double r2 = (double)b.r * (double)b.r;
        H2 = r2 > H2 ? r2 : H2;
    }
    return d2 <= H2 * (1.0 + 1e-6);
}

// Axis k of a candidate's image code (two signed bits to an axis).
__device__ __forceinline__ int image_sign(int code, int k) { return code << (30 - 2 * k) >> 30; }

// A particle's search record through the scalar cache (i wave-uniform; the
// records are not written by this kernel).
__device__ __forceinline__ double4 srec_at(const double4 *p, int i) { return load_ro(p + i); }

// NW waves take a group together: 1, or the block's four.  Each of the four
// tests all the boxes, stages every fourth pair of chunks in a buffer of its
// own and tests every fourth pair of tiles.
template <int D, int MODE, int NW>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(OCC_SEARCH))) search_kernel(BoxDev box, SearchArgs a)
{
    constexpr bool IJ = MODE != M_GATHER;
    static_assert(NW == 1 || NW == SW, "one wave or the whole block per group");
    __shared__ int l_chunk[SW][CHUNKCAP];
    __shared__ int l_kept[NW > 1 ? SW : 1], l_hits[NW > 1 ? SW : 1][NW > 1 ? WAVE : 1];
    __shared__ double l_reach[NW > 1 ? SW : 1];
    __shared__ int l_shift[NW > 1 ? SW : 1];

    const int w = uniform(threadIdx.x / WAVE);
    const int part = NW > 1 ? w : 0;  // this wave's part of the group
    const int lane = wave_lane();
    const int ngroups = uniform(*a.num_groups);
    // this wave's staging buffer
    const size_t wbase = (size_t)(blockIdx.x * SW + w) * (size_t)a.wcap;
    // persistent waves: groups are taken one at a time from this XCD's
    // contiguous share of the Morton curve (a whole block: in turn)
    TaskShare share(a.work, ngroups);
    int turn = NW > 1 ? xcd_block() : 0;
    auto next = [&]() -> int {
        if constexpr(NW == 1) return share.next();
        const int t = turn < ngroups ? turn : -1;
        turn += (int)gridDim.x;
        return t;
    };
    for(int grp = next(); grp >= 0; grp = next()) {
    const int2 gr = make_int2(uniform(a.groups[grp].x), uniform(a.groups[grp].y));
    const int cnt = gr.y - gr.x;
    const bool valid = lane < cnt;
    const size_t gbase = (size_t)grp * (size_t)a.wcap;

    // group box: centre (go: from the boxes' origin), half extent, largest
    // radius squared (wave-uniform).  A particle with a NaN coordinate is at
    // no distance from any other: it hits nothing and stays out of the box,
    // which would otherwise be near everything or leave out the particles
    // whose extremes met it in the reduction.
    double gc[D], go[D], ge[D], hmax2;
    uint64_t live;
    {
        const int i = gr.x + (valid ? lane : 0);
        const double4 me = a.srec[i];
        const double x[3] = {me.x, me.y, me.z};
        bool in = true;
#pragma unroll
        for(int k = 0; k < D; ++k) in = in && x[k] == x[k];
        live = ballot(in);
#pragma unroll
        for(int k = 0; k < D; ++k) {
            const double lo = wave_minv(in ? x[k] : 1.7976931348623157e308);
            const double hi = wave_maxv(in ? x[k] : -1.7976931348623157e308);
            gc[k] = uniform_d(0.5 * (lo + hi));
            go[k] = uniform_d(gc[k] - box_origin(a.origin, k));
            ge[k] = uniform_d(0.5 * (hi - lo) * (1.0 + 1e-12) + 1e-300);
        }
        double h2 = me.w;
        if constexpr(MODE == M_SYMMETRIC) h2 = a.own[i] * a.own[i];
        hmax2 = uniform_d(wave_maxv(in && h2 == h2 ? h2 : 0.0));
    }

    int nkept = 0;               // staged candidates (may pass wcap: overflow)
    double reach2 = hmax2;       // largest squared radius among the kept candidates (per lane)
    int64_t visited = 0, tested = 0;

    // ---- phase 2: stage the particles of the collected chunks, two chunks
    // at a time; the next two are loaded before the current ones are tested
    int nchunk = 0;
    auto flush = [&]() {
        wave_lds_sync();
        auto fetch = [&](int p, int &j, double4 &q) {
            const int s = p + (lane >> 5);
            j = s < nchunk ? l_chunk[w][s] * CHUNK + (lane & (CHUNK - 1)) : a.n;
            if(j < a.n) q = a.srec[j];
        };
        int c_j = a.n;
        double4 c_q = make_double4(0.0, 0.0, 0.0, 0.0);
        fetch(2 * part, c_j, c_q);
        for(int p = 2 * part; p < nchunk; p += 2 * NW) {
            int n_j = a.n;
            double4 n_q = make_double4(0.0, 0.0, 0.0, 0.0);
            if(p + 2 * NW < nchunk) fetch(p + 2 * NW, n_j, n_q);
            bool keep = false;
            if(c_j < a.n) {
                // keep a candidate only if it lies within reach of the group
                // box (the box contains every x_i, so each lane's own test
                // implies this)
                const double x[3] = {c_q.x, c_q.y, c_q.z};
                double d2b = 0.0;
                keep = true;
#pragma unroll
                for(int k = 0; k < D; ++k) {
                    const double ex = fabs(min_image1(box, k, x[k] - gc[k])) - ge[k];
                    d2b += ex > 0.0 ? ex * ex : 0.0;
                    keep = keep && x[k] == x[k];
                }
                double H2 = hmax2;
                if constexpr(IJ) H2 = c_q.w > H2 ? c_q.w : H2;
                keep = keep && d2b <= H2 * (1.0 + 1e-9);
                if constexpr(IJ) reach2 = keep && H2 > reach2 ? H2 : reach2;
            }
            const uint64_t kept = ballot(keep);
            if(keep) {
                const int at = nkept + __popcll(kept & ((1ull << lane) - 1ull));
                if(at < a.wcap) a.ws_j[wbase + at] = c_j;
            }
            const int m = uniform(__popcll(kept));
            nkept += m;
            tested += m;
            c_j = n_j;
            c_q = n_q;
        }
        nchunk = 0;
        wave_lds_sync();
    };

    // ---- phase 1: boxes near the group's box, 64 per window
    auto window = [&](int level, int base) -> uint64_t {
        const int v = base + lane;
        bool hit = false;
        if(v < a.cnt[level]) hit = box_near<D, IJ>(box, a.lev[level][v], go, ge, hmax2);
        visited += min(WAVE, a.cnt[level] - base);
        return ballot(hit);
    };
    for(int b3 = 0; b3 < (live ? a.cnt[2] : 0); b3 += WAVE) {
        // a level with one box is not tested
        uint64_t m3 = a.cnt[2] > 1 ? window(2, b3) : 1ull;
        while(m3) {
            const int k3 = (int)__builtin_ctzll(m3);
            m3 &= m3 - 1ull;
            const int b2 = (b3 + k3) * WAVE;
            uint64_t m2 = a.cnt[1] > 1 ? window(1, b2) : 1ull;
            while(m2) {
                const int k2 = (int)__builtin_ctzll(m2);
                m2 &= m2 - 1ull;
                const int b1 = (b2 + k2) * WAVE;
                const uint64_t m1 = window(0, b1);
                if((m1 >> lane) & 1) l_chunk[w][nchunk + __popcll(m1 & ((1ull << lane) - 1ull))] = b1 + lane;
                nchunk += uniform(__popcll(m1));
                if(nchunk > CHUNKCAP - WAVE) flush();
            }
        }
    }
    if(nchunk) flush();

    // ---- phase 3: strided tiles of the kept candidates, the next tile's
    // records loaded while the current one is tested
    // the staging writes of all lanes before their reads by other lanes
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    double reach = box.on ? wave_maxv(reach2) : 0.0;
    int before[NW];  // candidates staged by the parts before each
    before[0] = 0;
    if constexpr(NW > 1) {
        if(lane == 0) {
            l_kept[w] = nkept;
            l_reach[w] = reach;
        }
        __syncthreads();
        nkept = 0;
#pragma unroll
        for(int k = 0; k < NW; ++k) {
            before[k] = nkept;
            nkept += uniform(l_kept[k]);
            reach = l_reach[k] > reach ? l_reach[k] : reach;
        }
    }
    const int nc = nkept < a.wcap ? nkept : a.wcap;
    const int T = (nc + WAVE - 1) / WAVE;
    // Periodic box: every lane's minimum image of a candidate that can be a
    // hit is the one nearest to the group's centre, if the group and its
    // reach span less than half the box; its shift by L, 0 or -L is then
    // settled once: with FP64 pairs it is added to the pairs' differences, as
    // a minimum image does, with mixed ones the candidate is moved, as their
    // passes do.  Otherwise every pair takes its own minimum image.  The
    // passes read which of it was so from the flags beside the count.
    bool wrap = false;
    if(box.on) {
        const double H = sqrt(uniform_d(reach));
#pragma unroll
        for(int k = 0; k < D; ++k) wrap = wrap || !(2.0 * ge[k] + H < 0.499 * box.len[k]);
    }
    auto fetch_c = [&](int c, int &j, double4 &q) {
        j = -1;
        // past the tile's end: at no finite distance
        q = make_double4(1e200, 1e200, 1e200, 0.0);
        if(c < nc) {
            if constexpr(NW == 1) {
                j = a.ws_j[wbase + c];
            } else {
                int k = 0, b = 0;
#pragma unroll
                for(int u = 1; u < NW; ++u)
                    if(c >= before[u]) {
                        k = u;
                        b = before[u];
                    }
                j = a.ws_j[(size_t)(blockIdx.x * SW + k) * (size_t)a.wcap + (c - b)];
            }
            q = a.srec[j];
        }
    };
    int count = 0;  // hits of particle `lane`
    int shift = 0;  // GNC_SHIFT bits: some candidate is nearest by a shifted image
    using Zero = std::integral_constant<int, 0>;
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    // V consecutive tiles from tt on, the candidates' records in p_j and p_q
    int p_j[2] = {-1, -1};
    double4 p_q[2];
    auto tiles = [&](int tt, auto pairwise, auto width) {
        constexpr bool PER = decltype(pairwise)::value;
        constexpr int V = decltype(width)::value;
        constexpr int U = PER ? 1 : 4;  // particles per pass
        int j[V], code[V];
        double x[V][3], cw[V];
        int moved = 0;
#pragma unroll
        for(int v = 0; v < V; ++v) {
            j[v] = p_j[v];
            x[v][0] = p_q[v].x;
            x[v][1] = p_q[v].y;
            x[v][2] = p_q[v].z;
            cw[v] = p_q[v].w;
            stream_st(a.cand + gbase + (size_t)(tt + v) * WAVE + lane, j[v]);
            code[v] = 0;
            if(!PER && box.on) {
                if(j[v] >= 0) {
#pragma unroll
                    for(int k = 0; k < D; ++k) code[v] |= (near_image(box, k, gc[k], x[v][k]) & 3) << (2 * k);
                }
                moved |= code[v];
            }
        }
        bool any = wave_any(moved != 0);
        if(any) {
#pragma unroll
            for(int k = 0; k < D; ++k) shift |= wave_any((moved >> (2 * k) & 3) != 0) ? GNC_SHIFT_AXIS << k : 0;
            if(!a.exact) {
                // mixed precision: the pairs subtract moved coordinates (GroupImage)
#pragma unroll
                for(int v = 0; v < V; ++v)
#pragma unroll
                    for(int k = 0; k < D; ++k) x[v][k] = near_position(box, k, gc[k], x[v][k]);
                any = false;
            }
        }
        // the next tiles' records, while these are tested
        constexpr int S = V * NW;
        if(tt + S < T) fetch_c(tt + S + lane * T, p_j[0], p_q[0]);
        if(V > 1 && tt + S + 1 < T) fetch_c(tt + S + 1 + lane * T, p_j[1], p_q[1]);
        // particle after particle: the lanes' compares are its hit mask
        int lo[V] = {}, hi[V] = {};
        auto sweep = [&](auto shifted, auto first, auto number) {
            constexpr int V0 = decltype(first)::value, N = decltype(number)::value;
            double s[N][D];
            if constexpr(decltype(shifted)::value) {
#pragma unroll
                for(int v = 0; v < N; ++v)
#pragma unroll
                    for(int k = 0; k < D; ++k) s[v][k] = image_sign(code[V0 + v], k) * box.len[k];
            }
            for(int i0 = 0; i0 < cnt; i0 += U) {
#pragma clang fp contract(off)
                // records past the group's last particle (srec has a spare
                // tile of them) fill lanes that are masked off below
                double4 q[U];
                double o2[U];
#pragma unroll
                for(int u = 0; u < U; ++u) {
                    q[u] = srec_at(a.srec, gr.x + i0 + u);
                    o2[u] = q[u].w;
                }
                if constexpr(MODE == M_SYMMETRIC) {
#pragma unroll
                    for(int u = 0; u < U; ++u) {
                        const double h = a.own[gr.x + min(i0 + u, cnt - 1)];
                        o2[u] = h * h;
                    }
                }
#pragma unroll
                for(int u = 0; u < U; ++u) {
#pragma unroll
                    for(int v = 0; v < N; ++v) {
                        double d[D];
                        d[0] = q[u].x - x[V0 + v][0];
                        if constexpr(D > 1) d[1] = q[u].y - x[V0 + v][1];
                        if constexpr(D > 2) d[2] = q[u].z - x[V0 + v][2];
                        if constexpr(PER) min_image<D>(box, d);
                        if constexpr(decltype(shifted)::value) {
#pragma unroll
                            for(int k = 0; k < D; ++k) d[k] = d[k] + s[v][k];
                        }
                        double r2 = d[0] * d[0];
#pragma unroll
                        for(int k = 1; k < D; ++k) r2 = r2 + d[k] * d[k];
                        uint64_t m = ballot(r2 < o2[u]);
                        if constexpr(IJ) m |= ballot(r2 < cw[V0 + v]);
                        lo[V0 + v] = write_lane((int)(uint32_t)m, i0 + u, lo[V0 + v]);
                        hi[V0 + v] = write_lane((int)(uint32_t)(m >> 32), i0 + u, hi[V0 + v]);
                    }
                }
            }
        };
        if(!any) {
            sweep(std::false_type{}, Zero{}, width);
        } else {
            // one tile after the other (the shifts take the registers of the second)
            sweep(std::true_type{}, Zero{}, One{});
            if constexpr(V > 1) sweep(std::true_type{}, One{}, One{});
        }
#pragma unroll
        for(int v = 0; v < V; ++v) {
            uint64_t mine = valid ? ((uint64_t)(uint32_t)hi[v] << 32) | (uint32_t)lo[v] : 0ull;
            if constexpr(PER) mine &= ballot(j[v] >= 0);  // a wrapped distance is always finite
            stream_st(a.ma + gbase + (size_t)(tt + v) * WAVE + lane, mine);
            count += __popcll(mine);
        }
    };
    if(wrap) {
        int tt = part;
        if(tt < T) fetch_c(tt + lane * T, p_j[0], p_q[0]);
        for(; tt < T; tt += NW) tiles(tt, std::true_type{}, One{});
    } else {
        int tt = 2 * part;
        if(tt < T) fetch_c(tt + lane * T, p_j[0], p_q[0]);
        if(tt + 1 < T) fetch_c(tt + 1 + lane * T, p_j[1], p_q[1]);
        for(; tt + 1 < T; tt += 2 * NW) tiles(tt, std::false_type{}, Two{});
        if(tt < T) tiles(tt, std::false_type{}, One{});
    }
    if constexpr(NW > 1) {
        l_hits[w][lane] = count;
        if(lane == 0) l_shift[w] = shift;
        __syncthreads();
        count = 0;
        shift = 0;
#pragma unroll
        for(int k = 0; k < NW; ++k) {
            count += l_hits[k][lane];
            shift |= l_shift[k];
        }
        // (the next group's first barrier comes after these reads)
        tested = part == 0 ? nkept : 0;
    }
    if(part != 0) continue;
    if(lane == 0) a.gnc[grp] = nc | (wrap ? GNC_WRAP : shift);

    // past the reference's list capacity (its unchecked write,
    // src/bhtree.cpp:257-258) the search reports an overflow
    const int over = wave_sum(count > a.cap ? 1 : 0);
    const int len = wave_maxv(count);
    if(lane == 0) {
        if(a.stats) {
            stat_add(a.counters, grp, C_SEARCH_NODES, visited);
            stat_add(a.counters, grp, C_SEARCH_CAND, tested);
            stat_max(a.counters, grp, C_MAXLIST, len);
        }
        if(over) atomicAdd((unsigned long long *)&a.counters[C_OVERFLOW], (unsigned long long)over);
        if(nkept > a.wcap) atomicAdd((unsigned long long *)&a.counters[C_TILE_OVER], 1ull);
    }
    }  // groups
}

// ------------------------------------------------------------------- boxes
// Search records (position, squared candidate radius) and the boxes of the
// first two levels: a workgroup takes the 2,048 particles of one
// second-level box.  The boxes are FP32 and count from the root cube's centre
// (origin), so that they are as tight for a domain far from zero.
constexpr int BOX_THREADS = 1024;
constexpr int SUPER = CHUNK * WAVE;  // particles per second-level box

__device__ __forceinline__ void box_join(ChunkBox &a, const ChunkBox &b)
{
#pragma unroll
    for(int k = 0; k < 3; ++k) {
        a.lo[k] = b.lo[k] < a.lo[k] ? b.lo[k] : a.lo[k];
        a.hi[k] = b.hi[k] > a.hi[k] ? b.hi[k] : a.hi[k];
    }
    a.r = b.r > a.r ? b.r : a.r;
}

__device__ __forceinline__ ChunkBox box_none()
{
    ChunkBox b;
#pragma unroll
    for(int k = 0; k < 3; ++k) {
        b.lo[k] = 3.4028234e38f;
        b.hi[k] = -3.4028234e38f;
    }
    b.r = 0.0f;
    b.pad = 0.0f;
    return b;
}

// box of W consecutive lanes' boxes, in every one of them
template <int W> __device__ __forceinline__ ChunkBox box_lanes(ChunkBox b)
{
#pragma unroll
    for(int off = W / 2; off > 0; off >>= 1) {
        ChunkBox o;
#pragma unroll
        for(int k = 0; k < 3; ++k) {
            o.lo[k] = __shfl_xor(b.lo[k], off, WAVE);
            o.hi[k] = __shfl_xor(b.hi[k], off, WAVE);
        }
        o.r = __shfl_xor(b.r, off, WAVE);
        box_join(b, o);
    }
    return b;
}

template <int D>
__global__ void __launch_bounds__(BOX_THREADS) chunk_boxes_kernel(State s, const double *rad, const double *origin, int n, double4 *srec,
                                                                   ChunkBox *l1, ChunkBox *l2)
{
    __shared__ ChunkBox sh[WAVE];
    for(int r = 0; r < SUPER / BOX_THREADS; ++r) {
        const int slot = r * BOX_THREADS + threadIdx.x;
        const int64_t i = (int64_t)blockIdx.x * SUPER + slot;
        ChunkBox b = box_none();
        if(i < n) {
            double4 q;
            q.x = s.f[F_X][i];
            q.y = D > 1 ? s.f[F_X + 1][i] : 0.0;
            q.z = D > 2 ? s.f[F_X + 2][i] : 0.0;
            const double h = rad[i];
            q.w = h * h;
            srec[i] = q;
            const double x[3] = {q.x, q.y, q.z};
            bool in = true;
#pragma unroll
            for(int k = 0; k < D; ++k) in = in && x[k] == x[k];
            // FP32, rounded outwards (a particle with a NaN coordinate stays
            // out of the box; a coordinate past FP32's range makes it
            // boundless)
            if(in) {
#pragma unroll
                for(int k = 0; k < 3; ++k) {
                    const float f = k < D ? (float)(x[k] - box_origin(origin, k)) : 0.0f, e = fabsf(f) * 1.2e-7f + 1e-37f;
                    b.lo[k] = e < __builtin_huge_valf() ? f - e : -__builtin_huge_valf();
                    b.hi[k] = e < __builtin_huge_valf() ? f + e : __builtin_huge_valf();
                }
                const float f = (float)h;
                b.r = f == f ? f + f * 1.2e-7f + 1e-37f : 0.0f;
            }
        }
        b = box_lanes<CHUNK>(b);
        if((slot & (CHUNK - 1)) == 0) sh[slot / CHUNK] = b;
    }
    __syncthreads();
    if(threadIdx.x < WAVE) {
        const ChunkBox b = sh[threadIdx.x];
        const int64_t at = (int64_t)blockIdx.x * WAVE + threadIdx.x;
        if(at * CHUNK < n) l1[at] = b;
        const ChunkBox t = box_lanes<WAVE>(b);
        if(threadIdx.x == 0) l2[blockIdx.x] = t;
    }
}

// third level: one box per 64 of the second
__global__ void __launch_bounds__(BLOCK) upper_boxes_kernel(const ChunkBox *l2, int n2, ChunkBox *l3)
{
    const int b = (int)(blockIdx.x * (BLOCK / WAVE) + threadIdx.x / WAVE);
    const int v = b * WAVE + wave_lane();
    if(b * WAVE >= n2) return;
    const ChunkBox t = box_lanes<WAVE>(v < n2 ? l2[v] : box_none());
    if(wave_lane() == 0) l3[b] = t;
}

// Records and boxes of the current particles with candidate radii `rad`.
int search_boxes(Ctx &c, const double *rad)
{
    const int n = (int)c.n, n2 = grid_for(n, SUPER), n3 = grid_for(n2, WAVE);
    ChunkBox *l1 = c.boxes, *l2 = l1 + grid_for(c.cap_n, CHUNK), *l3 = l2 + grid_for(c.cap_n, SUPER);
    switch(c.D) {
    case 1: hipLaunchKernelGGL(chunk_boxes_kernel<1>, dim3(n2), dim3(BOX_THREADS), 0, c.stream, c.s, rad, c.scal + S_ROOT_CX, n, c.srec, l1, l2); break;
    case 2: hipLaunchKernelGGL(chunk_boxes_kernel<2>, dim3(n2), dim3(BOX_THREADS), 0, c.stream, c.s, rad, c.scal + S_ROOT_CX, n, c.srec, l1, l2); break;
    default: hipLaunchKernelGGL(chunk_boxes_kernel<3>, dim3(n2), dim3(BOX_THREADS), 0, c.stream, c.s, rad, c.scal + S_ROOT_CX, n, c.srec, l1, l2); break;
    }
    // with one third-level box the search starts at the second
    if(n3 > 1) hipLaunchKernelGGL(upper_boxes_kernel, dim3(grid_for(n3, SW)), dim3(BLOCK), 0, c.stream, l2, n2, l3);
    SPHGPU_HIP(hipGetLastError());
    return SPHGPU_OK;
}

template <int D, int MODE> static void launch_search(Ctx &c, const SearchArgs &a, bool work_ready, int blocks_per_cu)
{
    if(group_waves(c, GROUP_SEARCH) > 1) {
        const int blocks = std::min(c.ngroups, 8 * c.num_cu);
        hipLaunchKernelGGL((search_kernel<D, MODE, SW>), dim3(blocks), dim3(BLOCK), 0, c.stream, make_box(c), a);
        return;
    }
    const BoxDev box = make_box(c);
    // blocks_per_cu blocks of 4 waves per CU (8 fill every CU), a multiple
    // of the XCD count; blocks beyond what the CUs hold find no task and leave
    const int blocks = std::max(NUM_XCD, std::min(grid_for(c.n, WAVE) / SW, blocks_per_cu * c.num_cu) / NUM_XCD * NUM_XCD);
    if(!work_ready) reset_work(c, 0);
    SearchArgs aw = a;
    aw.work = c.work;
    hipLaunchKernelGGL((search_kernel<D, MODE, 1>), dim3(blocks), dim3(BLOCK), 0, c.stream, box, aw);
}

template <int MODE> static int search_dispatch(Ctx &c, const SearchArgs &a, bool work_ready, int blocks_per_cu)
{
    switch(c.D) {
    case 1: launch_search<1, MODE>(c, a, work_ready, blocks_per_cu); break;
    case 2: launch_search<2, MODE>(c, a, work_ready, blocks_per_cu); break;
    default: launch_search<3, MODE>(c, a, work_ready, blocks_per_cu); break;
    }
    SPHGPU_HIP(hipGetLastError());
    return SPHGPU_OK;
}

// sml = h_guess * ratio (src/pre_interaction.cpp:61-64), the gather search
// radius
template <int D> __global__ void __launch_bounds__(BLOCK) guess_kernel(State s, int n, double nngb, double ratio)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if(i >= n) return;
    s.f[F_SML][i] = sml_guess<D>(s.f[F_MASS][i], s.f[F_DENS][i], nngb, ratio);
}

static int guess(Ctx &c, double ratio)
{
    const double nngb = (double)c.p.neighbor_number;
    switch(c.D) {
    case 1: hipLaunchKernelGGL(guess_kernel<1>, dim3(grid_for(c.n)), dim3(BLOCK), 0, c.stream, c.s, (int)c.n, nngb, ratio); break;
    case 2: hipLaunchKernelGGL(guess_kernel<2>, dim3(grid_for(c.n)), dim3(BLOCK), 0, c.stream, c.s, (int)c.n, nngb, ratio); break;
    default: hipLaunchKernelGGL(guess_kernel<3>, dim3(grid_for(c.n)), dim3(BLOCK), 0, c.stream, c.s, (int)c.n, nngb, ratio); break;
    }
    SPHGPU_HIP(hipGetLastError());
    return search_boxes(c, c.s.f[F_SML]);
}

int search_guess(Ctx &c) { return guess(c, c.p.iterative_sml ? 1.2 : 1.0); }

// The largest h of every particle's leaf (BHTree::set_kernel's value for it,
// src/bhtree.cpp:206-232): the symmetric search's candidate radius.
__global__ void __launch_bounds__(BLOCK) leaf_radius_kernel(TreeDev t, const double *sml, int64_t cap, double *out)
{
    const int total = *t.num_nodes;
    for(int64_t v = (int64_t)blockIdx.x * BLOCK + threadIdx.x; v < total && v < cap; v += (int64_t)gridDim.x * BLOCK) {
        const int4 r = t.rng[v];
        if(!(r.w & 256)) continue;
        double h = 0.0;
        for(int i = r.x; i < r.y; ++i) h = sml[i] > h ? sml[i] : h;
        for(int i = r.x; i < r.y; ++i) out[i] = h;
    }
}

// Blocks of four persistent waves per CU.  More waves hide the dependent
// loads of the first two phases; fewer leave the scalar cache (which holds
// the groups' records) and L2 to each.  Beside the gravity walk, which is
// bound by instruction issue, the step is shortest with two (mixed Evrard
// step, 2^20 particles: 4.62 ms, against 4.63, 4.66 and 4.75 with three,
// four and six).  Alone: 2D KHI, 393,160 particles: 128 us with four (137
// with two, 143 with six); 3D, 2^21 particles: 800 us with six (1,122 with
// two, 865 with four, 824 with eight).
int search_blocks(const Ctx &c, bool beside_walk) { return beside_walk ? 2 : c.D < 3 ? 4 : 6; }

static SearchArgs base_args(Ctx &c)
{
    SearchArgs a{};
    a.n = (int)c.n;
    a.srec = c.srec;
    a.own = c.s.f[F_SML];
    a.origin = c.scal + S_ROOT_CX;
    a.lev[0] = c.boxes;
    a.lev[1] = c.boxes + grid_for(c.cap_n, CHUNK);
    a.lev[2] = a.lev[1] + grid_for(c.cap_n, SUPER);
    a.cnt[0] = grid_for(c.n, CHUNK);
    a.cnt[1] = grid_for(c.n, SUPER);
    a.cnt[2] = grid_for(a.cnt[1], WAVE);
    a.groups = c.groups;
    a.num_groups = c.num_groups;
    a.cand = c.tile_cand;
    a.ma = c.tile_ma;
    a.exact = c.p.precision == SPHGPU_FP64;
    a.gnc = c.tile_nc;
    a.wcap = c.tile_wcap;
    a.ws_j = c.ws_j;
    a.cap = c.cap;
    a.counters = c.counters;
    a.stats = c.stats_on ? 1 : 0;
    return a;
}

// One search for both sets: with the records' radii h_guess * ratio, the
// test r < max(R_i, R_j) finds every gather candidate (r < R_i) and every
// pair with r < max(h_i, h_j) for the final h, as long as no final h exceeds
// its search radius (the caller checks the truncation counter).  With
// `work_ready` the task counters are clear already (the tree build's last
// launch); `blocks_per_cu` sets how many blocks of four
// persistent waves each CU gets.
int search_combined(Ctx &c, bool work_ready, int blocks_per_cu)
{
    return search_dispatch<M_COMBINED>(c, base_args(c), work_ready, blocks_per_cu);
}

int search_gather(Ctx &c, bool initial)
{
    int rc = guess(c, initial ? 1.0 : (c.p.iterative_sml ? 1.2 : 1.0));  // src/pre_interaction.cpp:31-35
    if(rc) return rc;
    return search_dispatch<M_GATHER>(c, base_args(c), false, search_blocks(c, false));
}

int search_symmetric(Ctx &c)
{
    hipLaunchKernelGGL(leaf_radius_kernel, dim3(std::min<int64_t>(grid_for(c.node_cap), 2048)), dim3(BLOCK), 0, c.stream, c.t,
                       c.s.f[F_SML], c.node_cap, c.leaf_rad);
    SPHGPU_HIP(hipGetLastError());
    int rc = search_boxes(c, c.leaf_rad);
    if(rc) return rc;
    return search_dispatch<M_SYMMETRIC>(c, base_args(c), false, search_blocks(c, false));
}

// Search records and boxes of up to n particles, and the symmetric search's
// radii.  The records have a spare tile behind the last particle (the search
// reads a group's records four at a time).
int search_alloc_particles(Ctx &c)
{
    const int64_t n = c.cap_n;
    SPHGPU_HIP(hipMalloc(&c.srec, (n + WAVE) * sizeof(double4)));
    const int64_t nb = grid_for(n, CHUNK) + grid_for(n, SUPER) + grid_for(grid_for(n, SUPER), WAVE);
    SPHGPU_HIP(hipMalloc(&c.boxes, nb * sizeof(ChunkBox)));
    SPHGPU_HIP(hipMalloc(&c.leaf_rad, n * sizeof(double)));
    return SPHGPU_OK;
}

// Slabs of candidate tiles for the c.ngroups groups of the last tree, and
// the staging buffers of the search's persistent waves.  A slab holds
// tile_wcap candidates: the larger of eight times the per-particle capacity
// and 48 times neighborNumber.  A group of 64 particles keeps about 11
// times neighborNumber in 3D (690 at 64 neighbours in the Evrard
// benchmark).
int search_alloc(Ctx &c)
{
    const int64_t want = std::max<int64_t>({(int64_t)8 * c.cap, (int64_t)48 * c.p.neighbor_number, 1024});
    const int wcap = (int)std::min<int64_t>((want + WAVE - 1) / WAVE * WAVE, 1 << 22);
    const int64_t waves = (int64_t)8 * c.num_cu * SW + SW;
    // (the capacities are zero until all of a set's buffers are there, so that
    // a failed allocation is not taken for one later)
    if(wcap != c.tile_wcap || waves > c.ws_waves) {
        c.ws_waves = 0;
        if(c.ws_j) (void)hipFree(c.ws_j);
        c.ws_j = nullptr;
        SPHGPU_HIP(hipMalloc(&c.ws_j, (size_t)waves * wcap * sizeof(int)));
        c.ws_waves = waves;
    }
    if(wcap != c.tile_wcap || c.ngroups > c.tile_groups_cap) {
        // grow with headroom: the group count changes a little every step
        const int64_t groups = std::max<int64_t>((int64_t)c.ngroups + c.ngroups / 4 + 64, c.tile_groups_cap);
        c.tile_groups_cap = 0;
        if(c.tile_cand) (void)hipFree(c.tile_cand);
        if(c.tile_ma) (void)hipFree(c.tile_ma);
        if(c.tile_mn) (void)hipFree(c.tile_mn);
        if(c.tile_nc) (void)hipFree(c.tile_nc);
        c.tile_cand = nullptr;
        c.tile_ma = c.tile_mn = nullptr;
        c.tile_nc = nullptr;
        const size_t slots = (size_t)groups * wcap;
        SPHGPU_HIP(hipMalloc(&c.tile_cand, slots * sizeof(int)));
        SPHGPU_HIP(hipMalloc(&c.tile_ma, slots * sizeof(uint64_t)));
        SPHGPU_HIP(hipMalloc(&c.tile_mn, slots * sizeof(uint64_t)));
        SPHGPU_HIP(hipMalloc(&c.tile_nc, groups * sizeof(int)));
        c.tile_groups_cap = groups;
    }
    c.tile_wcap = wcap;
    return SPHGPU_OK;
}

// The gather sets (r < R_i, sml before the pre-interaction) or with FORCE the
// force sets (r < max(h_i, h_j), r != 0, as the force pass of pair type T
// tests it) as lists in list_at layout, from the tiles of the last search
// (debug): lane l of a group appends its hits in staging order (candidate
// c = t + kT is bit k of tile t).  Entries past cap are dropped (the search
// reports them).  The force pass also records how many pairs each particle
// summed, and sphgpu_neighbor_sets compares.
template <int D, class T, bool FORCE>
__global__ void __launch_bounds__(BLOCK) record_kernel(State s, BoxDev box, const int2 *groups, int ngroups, const int *gnc,
                                                       const int *cand, const uint64_t *ma, int wcap, int cap,
                                                       int *list, int *cnt)
{
    const int grp = xcd_block() * (BLOCK / WAVE) + (int)(threadIdx.x / WAVE);
    if(grp >= ngroups) return;
    const int lane = wave_lane();
    const int2 gr = groups[grp];
    const int i = gr.x + lane;
    if(i >= gr.y) return;
    const size_t gbase = (size_t)grp * wcap;
    const int nc = gnc[grp] & GNC_COUNT;
    const int ntile = (nc + WAVE - 1) / WAVE;
    const size_t lb = list_base(i, cap);
    double xi[D];
#pragma unroll
    for(int k = 0; k < D; ++k) xi[k] = s.f[F_X + k][i];
    const GroupImage<D, T> img(box, gnc[grp], xi);
    const double h = s.f[F_SML][i], h2 = h * h;
    int wf = 0;  // entries written (at most cap)
    for(int k = 0; k < WAVE; ++k) {
        for(int t = 0; t < ntile; ++t) {
            if(t + k * ntile >= nc) break;
            const size_t o = gbase + (size_t)t * WAVE;
            if(!((ma[o + lane] >> k) & 1ull)) continue;
            const int j = cand[o + k];
            double xj[D], d[D];
#pragma unroll
            for(int q = 0; q < D; ++q) xj[q] = img.at(q, s.f[F_X + q][j]);
            const double r2 = img.sep2(xi, xj, d);
            if constexpr(!FORCE) {
                if(!(r2 < h2)) continue;
            } else {
                const double hj = s.f[F_SML][j];
                const double hmax = h < hj ? hj : h;
                if constexpr(sizeof(T) == 8) {
                    const double r = sqrt(r2);
                    if(r >= hmax || r == 0.0) continue;
                } else if(!(r2 < hmax * hmax) || r2 == 0.0) {
                    continue;
                }
            }
            if(wf < cap) list[lb + list_off(wf++)] = j;
        }
    }
    cnt[i] = wf;
}

template <int D, class T> static void launch_record_t(Ctx &c, int *list, int *cnt, bool force)
{
    const auto kernel = force ? record_kernel<D, T, true> : record_kernel<D, T, false>;
    hipLaunchKernelGGL(kernel, dim3(group_grid(c)), dim3(BLOCK), 0, c.stream, c.s, make_box(c), c.groups, c.ngroups,
                       c.tile_nc, c.tile_cand, c.tile_ma, c.tile_wcap, c.cap, list, cnt);
}

template <int D> static void launch_record(Ctx &c, int *list, int *cnt, bool force)
{
    if(c.p.precision == SPHGPU_FP64) launch_record_t<D, double>(c, list, cnt, force);
    else launch_record_t<D, float>(c, list, cnt, force);
}

int search_record(Ctx &c, int *list, int *cnt, bool force)
{
    switch(c.D) {
    case 1: launch_record<1>(c, list, cnt, force); break;
    case 2: launch_record<2>(c, list, cnt, force); break;
    default: launch_record<3>(c, list, cnt, force); break;
    }
    SPHGPU_HIP(hipGetLastError());
    return SPHGPU_OK;
}

}  // namespace sphgpu
