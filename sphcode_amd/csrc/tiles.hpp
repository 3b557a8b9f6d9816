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
// slower where the pair kernels run alone (2D KHI, 3D Sedov), measured before
// the Newton sweep narrowed the hits and four waves shared small groups.
#pragma once

#include "ctx.hpp"

namespace sphgpu {

// Periodic images of a group's candidates.  A group's entry in Ctx::tile_nc
// says what they need: every pair its three images compared (GNC_WRAP: the
// group's reach spans half the box; some 30 FP64 operations and compares), or
// on some axes a shift by L for some candidates (GNC_SHIFT), or nothing (no
// face of the box comes near).
//
// With GNC_SHIFT a pair's minimum image is closer than half the box if it is a
// hit, so that the shift is L times the rounded quotient, minus.  FP64 pairs
// take x_i - x_j and then add it, which rounds as the reference does: the sets
// are the reference's to the last bit and the sums no further from 64-bit
// values (a coordinate moved by L first is rounded before the subtraction, and
// doubled that error).  Mixed pairs, whose separations are rounded to FP32
// next, subtract a coordinate that was moved when it was staged, to the image
// nearest to any one particle of the group: it is the same one for all of its
// pairs (rollout gradient of 262,144 particles 34.0 ms, with a shift in each
// pair 36.3).
template <int D, class T> struct GroupImage {
    static constexpr bool EXACT = sizeof(T) == 8;
    const BoxDev &box;
    int flags;     // GNC_WRAP, or GNC_SHIFT's bits, or none
    BoxDev pairs;  // mixed: the box, on with GNC_WRAP only
    bool move;     // mixed: some candidates are moved
    double x0[D];  // to beside this particle, the first with no NaN coordinate (those that have one hit nothing)
    __device__ __forceinline__ GroupImage(const BoxDev &b, int gnc, const double xi[D]) : box(b), pairs(b)
    {
        flags = b.on ? gnc & (GNC_WRAP | GNC_SHIFT) : 0;
        pairs.on = b.on && (gnc & GNC_WRAP);
        move = b.on && (gnc & GNC_SHIFT);
        if constexpr(!EXACT) {
            bool in = true;
#pragma unroll
            for(int k = 0; k < D; ++k) in = in && xi[k] == xi[k];
            const uint64_t live = ballot(in);
            const int first = live ? (int)__builtin_ctzll(live) : 0;
#pragma unroll
            for(int k = 0; k < D; ++k) x0[k] = uniform_d(__shfl(xi[k], first, WAVE));
        }
    }
    // axis k of a candidate's position, as it is staged
    __device__ __forceinline__ double at(int k, double x) const
    {
        if constexpr(EXACT) return x;
        else return move ? near_position(box, k, x0[k], x) : x;
    }
    // r_ij and its square of a pair, the position of j as it was staged
    __device__ __forceinline__ double sep2(const double xi[D], const double xj[D], double d[D]) const
    {
#pragma clang fp contract(off)
#pragma unroll
        for(int k = 0; k < D; ++k) d[k] = xi[k] - xj[k];
        if constexpr(!EXACT) {
            min_image<D>(pairs, d);
        } else if(flags) {
            if(flags & GNC_WRAP) {
                min_image<D>(box, d);
            } else {
#pragma unroll
                for(int k = 0; k < D; ++k)
                    if(flags & GNC_SHIFT_AXIS << k) d[k] = __builtin_fma(-rint(d[k] * box.inv[k]), box.len[k], d[k]);
            }
        }
        double r2 = d[0] * d[0];
#pragma unroll
        for(int k = 1; k < D; ++k) r2 = r2 + d[k] * d[k];
        return r2;
    }
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
