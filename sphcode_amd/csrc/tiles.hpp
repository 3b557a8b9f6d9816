// Sweep of a search group's candidate tiles by its wave, one lane per
// particle (the pair passes of the pre-interaction and the force stage).
//
// stage(t) loads tile t's neighbour records into the wave's LDS slot (every
// lane loads the record of the candidate in its own position) and returns
// this lane's hit mask of the tile; refine(m), optional, narrows the mask
// to the candidates that pass a cheap test (a cut-off the pair applies
// first anyway), each lane testing its own bits once the tile is visible
// to the whole wave; pair(k) handles candidate k of the tile for this lane.
// Each lane then walks the set bits of its mask, as a divergent loop, and
// the wave moves to the next tile when every lane is done.  With NW waves
// per group, wave `part` takes every NW-th tile.
//
// Refining pays where the search radius holds many more candidates than
// the pair's cut-off keeps: in 3D a candidate within 1.2 h_guess passes
// r < h about 60 % of the time, so the pair loop (which runs for as long
// as any lane has bits left) would otherwise spend 40 % of its passes on a
// distance test alone; in 2D (70 %) the extra loop costs more than it saves.
// A variant that kept two tiles resident, so that lanes waited at a tile
// boundary only when one ran a whole tile ahead, needed 8-15 more registers
// and twice the LDS; it was as fast on the 3D Evrard benchmark and 7-10 %
// slower where the pair kernels run alone (2D KHI, 3D Sedov).
#pragma once

#include "ctx.hpp"

namespace sphgpu {

// Periodic images of a group's candidates.  Unless the group's entry in
// Ctx::tile_nc carries GNC_WRAP, every pair's minimum image of a candidate
// is the image nearest to any one particle of the group (the search checked
// that the group and its reach span less than half the box), so a candidate
// is moved there once, when it is staged, and the pairs subtract plain
// coordinates: `pairs` is the box that sep2 gets, switched off then.  The
// three minimum images of a pair cost some 30 FP64 operations and compares.
template <int D> struct GroupImage {
    const BoxDev &box;
    BoxDev pairs;
    bool move;
    double x0[D];
    __device__ __forceinline__ GroupImage(const BoxDev &b, int gnc, const double xi[D]) : box(b), pairs(b)
    {
        pairs.on = b.on && (gnc & GNC_WRAP);
        move = b.on && !(gnc & GNC_WRAP);
        // the first particle with no NaN coordinate (those that have one hit nothing)
        bool in = true;
#pragma unroll
        for(int k = 0; k < D; ++k) in = in && xi[k] == xi[k];
        const uint64_t live = ballot(in);
        const int first = live ? (int)__builtin_ctzll(live) : 0;
#pragma unroll
        for(int k = 0; k < D; ++k) x0[k] = uniform_d(__shfl(xi[k], first, WAVE));
    }
    // axis k of a staged candidate's position
    __device__ __forceinline__ double at(int k, double x) const { return move ? near_image(box, k, x0[k], x) : x; }
};

struct NoRefine {
    __device__ __forceinline__ uint64_t operator()(uint64_t m) const { return m; }
};

template <int NW, class Stage, class Refine, class Pair>
__device__ __forceinline__ void tile_sweep(int part, int ntile, Stage &&stage, Refine &&refine, Pair &&pair)
{
    for(int t = part; t < ntile; t += NW) {
        uint64_t m = stage(t);
        wave_lds_sync();
        m = refine(m);
        while(m) {
            const int k = (int)__builtin_ctzll(m);
            m &= m - 1ull;
            pair(k);
        }
        wave_lds_sync();  // every read of the slot is done before it is restaged
    }
}

template <int NW, class Stage, class Pair>
__device__ __forceinline__ void tile_sweep(int part, int ntile, Stage &&stage, Pair &&pair)
{
    tile_sweep<NW>(part, ntile, stage, NoRefine{}, pair);
}

// A sweep that also narrows: pair(k) says whether candidate k is to be kept,
// and keep(t, m) receives this lane's kept hits of tile t.
template <int NW, class Stage, class Pair, class Keep>
__device__ __forceinline__ void tile_sweep_keep(int part, int ntile, Stage &&stage, Pair &&pair, Keep &&keep)
{
    for(int t = part; t < ntile; t += NW) {
        uint64_t m = stage(t);
        wave_lds_sync();
        uint64_t kept = 0;
        while(m) {
            const int k = (int)__builtin_ctzll(m);
            const uint64_t rest = m & (m - 1ull);
            if(pair(k)) kept |= m ^ rest;
            m = rest;
        }
        keep(t, kept);
        wave_lds_sync();
    }
}

// Sums of the parts' values, lane by lane and part after part (a fixed
// order), in every part: N values at a time through `red`, which all the
// block's waves share.  Nothing to do with one wave per group.
template <int NW> struct PartsLds {
    double v[NW > 1 ? 4 : 1][NW][NW > 1 ? WAVE : 1];
};

template <int NW, int N>
__device__ __forceinline__ void parts_sum(PartsLds<NW> &red, int part, double *const (&v)[N])
{
    static_assert(N <= 4, "four values at a time");
    if constexpr(NW > 1) {
        const int lane = wave_lane();
        __syncthreads();  // the previous values have been read
#pragma unroll
        for(int k = 0; k < N; ++k) red.v[k][part][lane] = *v[k];
        __syncthreads();
#pragma unroll
        for(int k = 0; k < N; ++k) {
            double s = red.v[k][0][lane];
#pragma unroll
            for(int p = 1; p < NW; ++p) s += red.v[k][p][lane];
            *v[k] = s;
        }
    }
}

// The bits of m whose candidate passes keep(k), tested by this lane.
template <class Keep>
__device__ __forceinline__ uint64_t refine_bits(uint64_t m, Keep &&keep)
{
    uint64_t out = 0;
    while(m) {
        const int k = (int)__builtin_ctzll(m);
        m &= m - 1ull;
        if(keep(k)) out |= 1ull << k;
    }
    return out;
}

}  // namespace sphgpu
