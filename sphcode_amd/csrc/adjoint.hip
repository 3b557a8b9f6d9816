// Adjoint of the SSPH step for the differentiable rollout (a capability the
// reference does not have).  The forward map of one step with a fixed dt is
//
//   v_p = v + a dt/2,  u_p = u + du dt/2                 (src/solver.cpp:431-456)
//   x'  = x + v_p dt,  v~ = v + a dt,  u~ = u + du dt,  c~ = sqrt(g(g-1) u~)
//   (a', du') = F(x', v~, u~)      PreInteraction + FluidForce
//                                  (src/pre_interaction.cpp:39-169, src/fluid_force.cpp:26-116)
//   v'  = v_p + a' dt/2,  u' = u_p + du' dt/2           (src/solver.cpp:458-474)
//
// and Solver::initialize evaluates F once at the initial state.  F is
// differentiated with the neighbour lists of the forward evaluation held
// fixed (the kernels vanish with their first derivatives at the support
// edge, so F is continuous across list changes), and h enters through the
// implicit function theorem on G(h, x) = rho(h, x) h^D - m N_ngb / A_D = 0,
// which the Newton iteration solves (src/pre_interaction.cpp:227-283).
//
// All pair sums of the adjoint are gathers over the search's candidate tiles,
// whose hits hold every force pair (r < max(h_i, h_j)) and with them every
// pair of the gather sets (r < h_i) in either direction: particle k collects the derivative of every
// pair term with respect to its own variables, so no atomics are needed.
// Three passes per force evaluation:
//   1. force pairs  -> adjoints of x, v (direct), h, rho, A = P Omega / rho^2,
//                      Balsara switch, sound speed
//   2. gather sums  -> chain through P, Omega, Balsara, h (IFT) to seeds on
//                      the sums rho, d rho/dh, div v, curl v
//   3. gather pairs -> adjoints of x and v through those sums
// The pair arithmetic follows the context's precision (FP64, or FP32 with
// FP64 accumulation); the per-particle chain rule and the IFT are FP64.
//
// Each pass runs as the forward pair passes do (tiles.hpp): a wave or four
// per search group, the neighbours' records staged through LDS once per
// group.  They are bound by vector issue.  Reading per-particle neighbour
// lists expanded from the tiles instead, one global load per field and pair,
// they were bound by those scattered loads and by the expansion (mixed,
// 262,144 particles: lists 574 us and passes 426, 124 and 344 us, now 170,
// 97 and 171 us; FP64, 29,791 particles: 243, 146, 81 and 124 us, now 55, 34
// and 53 us).  The records' sizes are no multiple of 64 bytes: lanes reading
// different records of a tile would meet in a few LDS banks.
#include <vector>

#include "tiles.hpp"

#include "kderiv.hpp"

namespace sphgpu {

// work arrays (device order), W(k, i) = work[k * n + i]
enum Work : int {
    W_AF = 0,      // seed on a (3)
    W_DUF = 3,     // seed on du
    W_XB = 4,      // adjoint of x (3)
    W_VB = 7,      // adjoint of v (3)
    W_HB = 10,     // partial adjoint of h
    W_RHOB = 11,   // partial adjoint of rho
    W_AB = 12,     // adjoint of A = P Omega / rho^2
    W_BB = 13,     // adjoint of the Balsara switch
    W_CB = 14,     // adjoint of the sound speed
    W_UB = 15,     // adjoint of u
    NWORK = 16
};

// checkpointed fields: what one step or Solver::initialize reads
static int ck_fields(int D, int *f)
{
    int k = 0;
    for(int a = 0; a < D; ++a) f[k++] = F_X + a;
    for(int a = 0; a < D; ++a) f[k++] = F_V + a;
    for(int a = 0; a < D; ++a) f[k++] = F_A + a;
    const int s[] = {F_MASS, F_ENE, F_DENE, F_SML, F_DENS, F_ALPHA, F_BAL, F_SOUND};
    for(int v : s) f[k++] = v;
    return k;
}

// Neighbour records: the fields of j read by passes 1 and 2 ...
template <class T> struct __align__(16) AdjRec {
    T hinv, rho, A, bal, c, alpha, m, duf;  // A = P Omega / rho^2
    T v[3], af[3];
    T pad[sizeof(T) == 4 ? 6 : 4];
};
static_assert(sizeof(AdjRec<float>) == 80 && sizeof(AdjRec<double>) == 144, "AdjRec size");
// ... and by pass 3, written by pass 2
template <class T> struct __align__(16) SeedRec {
    T h, hinv, m, srho, srhop, sdv;
    T v[3], srv[3];
    T pad[sizeof(T) == 4 ? 8 : 2];
};
static_assert(sizeof(SeedRec<float>) == 80 && sizeof(SeedRec<double>) == 112, "SeedRec size");

struct AdjArgs {
    const int2 *groups;
    int ngroups;
    const int *cand;     // candidate tiles (Ctx::tile_cand)
    const uint64_t *ma;
    const int *gnc;
    int wcap;
    double4 *pos;        // x, y, z, h
    void *rec;           // AdjRec<T>
    void *seed;          // SeedRec<T>
    double *w;       // work arrays
    int64_t n;       // their stride
    double *adj;     // adjoint state, caller order
    double gamma;
    double nngb;     // neighbor_number (for b in the IFT)
    int balsara;
    double dt;
    int kick;
};

__device__ __forceinline__ double &W(const AdjArgs &a, int k, int i) { return a.w[(int64_t)k * a.n + i]; }

// layout of the adjoint state (caller order): x (D), v (D), u, a (D), du
template <int D> __device__ __forceinline__ double &ADJ(const AdjArgs &a, int comp, int id)
{
    return a.adj[(int64_t)comp * a.n + id];
}
template <int D> struct AdjLayout {
    static constexpr int X = 0, V = D, U = 2 * D, A = 2 * D + 1, DU = 3 * D + 1, N = 3 * D + 2;
};

// Seeds of F from the adjoint of the step's output state, and the records
// of passes 1 and 2.
template <int D, class T> __global__ void __launch_bounds__(BLOCK) adj_seed_kernel(State s, int n, AdjArgs a)
{
    using L = AdjLayout<D>;
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if(i >= n) return;
    const int id = s.id[i];
    const double half = a.kick ? 0.5 * a.dt : 0.0;
    AdjRec<T> r{};
#pragma unroll
    for(int k = 0; k < D; ++k) {
        const double af = ADJ<D>(a, L::A + k, id) + half * ADJ<D>(a, L::V + k, id);
        W(a, W_AF + k, i) = af;
        r.af[k] = (T)af;
        r.v[k] = (T)s.f[F_V + k][i];
    }
    const double duf = ADJ<D>(a, L::DU, id) + half * ADJ<D>(a, L::U, id);
    W(a, W_DUF, i) = duf;
    r.duf = (T)duf;
    r.hinv = T(1) / (T)s.f[F_SML][i];
    r.rho = (T)s.f[F_DENS][i];
    r.A = (T)s.f[F_PRES][i] * (T)s.f[F_GRADH][i] / (r.rho * r.rho);
    r.bal = (T)s.f[F_BAL][i];
    r.c = (T)s.f[F_SOUND][i];
    r.alpha = (T)s.f[F_ALPHA][i];
    r.m = (T)s.f[F_MASS][i];
    ((AdjRec<T> *)a.rec)[i] = r;
    a.pos[i] = make_double4(s.f[F_X][i], D > 1 ? s.f[F_X + 1][i] : 0.0, D > 2 ? s.f[F_X + 2][i] : 0.0, s.f[F_SML][i]);
}

// Pair arithmetic of the passes: T = double, or float in mixed precision
// (separations taken in FP64 and rounded, fields of j rounded to
// FP32, terms accumulated in FP64 by Acc<T>); the pair-set tests are
// those of the forward stages in the same precision.
template <class T> __device__ __forceinline__ T pair_r(double r2)
{
    if constexpr(sizeof(T) == 8) return sqrt(r2);
    else return gather_r_f32(r2);
}

// One wave's view of its group: particle, tiles, and the staging of the
// candidates' positions (and a record each) in LDS.
constexpr int ASW = BLOCK / WAVE;
template <int D, int NW> struct AdjGroup {
    int w, lane, part, grp, i;
    bool have, valid;
    size_t gbase;
    int gnc, ntile;
    __device__ __forceinline__ explicit AdjGroup(const AdjArgs &a)
    {
        w = threadIdx.x / WAVE;
        lane = wave_lane();
        part = w % NW;
        grp = xcd_block() * (ASW / NW) + w / NW;
        have = grp < a.ngroups;
        const int2 gr = have ? a.groups[grp] : make_int2(0, 0);
        i = gr.x + lane;
        valid = have && i < gr.y;
        if(!valid) i = gr.x;
        gbase = (size_t)(have ? grp : 0) * a.wcap;
        gnc = have ? uniform(a.gnc[grp]) : 0;
        ntile = ((gnc & GNC_COUNT) + WAVE - 1) / WAVE;
    }
    template <class T, class R>
    __device__ __forceinline__ uint64_t stage(const AdjArgs &a, const GroupImage<D, T> &img, int tt, double4 *l_p, R *l_r, const R *rec) const
    {
        const size_t o = gbase + (size_t)tt * WAVE;
        const int jl = stream_ld(a.cand + o + lane);
        if(jl >= 0) {
            double4 q = a.pos[jl];
            q.x = img.at(0, q.x);
            if constexpr(D > 1) q.y = img.at(1, q.y);
            if constexpr(D > 2) q.z = img.at(2, q.z);
            l_p[lane] = q;
            l_r[lane] = rec[jl];
        }
        return valid ? stream_ld(a.ma + o + lane) : 0ull;
    }
};

template <int D, class T> __device__ __forceinline__ double pair_sep2(const GroupImage<D, T> &img, const double xi[D], const double4 &q, double d[D])
{
    double xj[D];
    xj[0] = q.x;
    if constexpr(D > 1) xj[1] = q.y;
    if constexpr(D > 2) xj[2] = q.z;
    return img.sep2(xi, xj, d);
}

// The sweep of a pass: in 3D each lane's hits are first narrowed to those
// that `keep` accepts (see tiles.hpp).
template <int D, int NW, class Stage, class Keep, class Pair>
__device__ __forceinline__ void adj_sweep(const AdjGroup<D, NW> &g, Stage &&stage, Keep &&keep, Pair &&pair)
{
    if constexpr(D == 3) {
        auto refine = [&](uint64_t m) { return refine_bits(m, keep); };
        tile_sweep<NW>(g.part, g.ntile, stage, refine, pair);
    } else {
        tile_sweep<NW>(g.part, g.ntile, stage, [&](int k) {
            if(keep(k)) pair(k);
        });
    }
}

// pass 1: force pairs (src/fluid_force.cpp:26-106)
template <int D, int K, class T, int NW>
__global__ void __launch_bounds__(BLOCK) adj_force_kernel(State s, BoxDev box, AdjArgs a)
{
    constexpr bool FP64 = sizeof(T) == 8;
    __shared__ double4 l_p[ASW][WAVE];
    __shared__ AdjRec<T> l_r[ASW][WAVE];
    __shared__ PartsLds<NW> red;
    const AdjGroup<D, NW> g(a);
    if(!g.have) return;  // (one wave per group only)
    const int i = g.i, w = g.w;
    double xi[D];
    T vi[D], afi[D];
#pragma unroll
    for(int k = 0; k < D; ++k) {
        xi[k] = s.f[F_X + k][i];
        vi[k] = (T)s.f[F_V + k][i];
        afi[k] = (T)W(a, W_AF + k, i);
    }
    const GroupImage<D, T> img(box, g.gnc, xi);
    const double hi_d = s.f[F_SML][i];
    const T hi_inv = T(1) / (T)hi_d, rhoi = (T)s.f[F_DENS][i], pi_ = (T)s.f[F_PRES][i], omi = (T)s.f[F_GRADH][i];
    const T bi = (T)s.f[F_BAL][i], ci = (T)s.f[F_SOUND][i], ali = (T)s.f[F_ALPHA][i], mi = (T)s.f[F_MASS][i];
    const T dufi = (T)W(a, W_DUF, i);
    const T Ai = pi_ * omi / (rhoi * rhoi);

    Acc<T> xb[D], vb[D], hb, rhob, Ab, Bb, cb;
    auto keep = [&](int kc) -> bool {
        const double4 q = l_p[w][kc];
        double dd[D];
        const double r2 = pair_sep2<D, T>(img, xi, q, dd);
        const double hmax = hi_d < q.w ? q.w : hi_d;
        if constexpr(FP64) {
            const double r = sqrt(r2);
            return !(r >= hmax || r == 0.0);
        } else {
            return r2 < hmax * hmax && r2 != 0.0;
        }
    };
    auto pair = [&](int kc) {
        const AdjRec<T> &j = l_r[w][kc];
        double dd[D];
        const double r2 = pair_sep2<D, T>(img, xi, l_p[w][kc], dd);
        T r;
        if constexpr(FP64) r = sqrt(r2);
        else r = sqrtf((float)r2);
        T d[D];
#pragma unroll
        for(int k = 0; k < D; ++k) d[k] = (T)dd[k];
        const T rhoj = j.rho, bj = j.bal, cj = j.c, alj = j.alpha, mj = j.m, dufj = j.duf, Aj = j.A;
        const KernelDerivs<T> ki = kernel_derivs_inv<D, K, T>(r, hi_inv);
        const KernelDerivs<T> kj = kernel_derivs_inv<D, K, T>(r, j.hinv);
        const T gi = ki.f, gj = kj.f, gb = T(0.5) * (gi + gj);
        T v[D], beta[D];
        T sv = T(0), b = T(0);
#pragma unroll
        for(int k = 0; k < D; ++k) {
            v[k] = vi[k] - j.v[k];
            beta[k] = mi * j.af[k] - mj * afi[k];
            sv += v[k] * d[k];
            b += beta[k] * d[k];
        }
        const T psii = mj * dufi, psij = mi * dufj, psis = psii + psij;
        // Monaghan viscosity Pi = K (C - 3 w) w for w = v.r / r < 0
        T Pi = T(0), Kv = T(0), wv = T(0);
        const T Cs = ci + cj, rhos = rhoi + rhoj, al2 = ali + alj;
        if(sv < T(0)) {
            wv = sv / r;
            Kv = T(-0.25) * (bi + bj) * al2 / rhos;
            Pi = Kv * (Cs - T(3) * wv) * wv;
        }
        const T Phi = Ai * gi + Aj * gj + Pi * gb;
        const T EPi = (b + T(0.5) * sv * psis) * gb;
        const T Egi = b * (Ai + T(0.5) * Pi) + sv * (psii * Ai + T(0.25) * psis * Pi);
        const T Egj = b * (Aj + T(0.5) * Pi) + sv * (psij * Aj + T(0.25) * psis * Pi);
        T Es = psii * Ai * gi + psij * Aj * gj + T(0.5) * psis * Pi * gb;
        T Er = Egi * ki.fr + Egj * kj.fr;
        if(sv < T(0)) {
            const T Piw = Kv * (Cs - T(6) * wv);
            Es += EPi * Piw / r;
            Er -= EPi * Piw * wv / r;
            rhob.add(-(EPi * Pi / rhos));
            cb.add(EPi * Kv * wv);
            Bb.add(EPi * (Cs - T(3) * wv) * wv * (T(-0.25) * al2 / rhos));
        }
        const T er = Er / r;
#pragma unroll
        for(int k = 0; k < D; ++k) {
            xb[k].add(beta[k] * Phi + v[k] * Es + d[k] * er);
            vb[k].add(d[k] * Es);
        }
        hb.add(Egi * ki.fh);
        Ab.add((b + sv * psii) * gi);
    };
    const AdjRec<T> *rec = (const AdjRec<T> *)a.rec;
    adj_sweep<D, NW>(g, [&](int tt) { return g.stage(a, img, tt, l_p[w], l_r[w], rec); }, keep, pair);
#pragma unroll
    for(int k = 0; k < D; ++k) parts_sum<NW, 2>(red, g.part, {&xb[k].s, &vb[k].s});
    parts_sum<NW, 4>(red, g.part, {&hb.s, &rhob.s, &Ab.s, &Bb.s});
    parts_sum<NW, 1>(red, g.part, {&cb.s});
    if(!g.valid || g.part != 0) return;
#pragma unroll
    for(int k = 0; k < D; ++k) {
        W(a, W_XB + k, i) = xb[k].val();
        W(a, W_VB + k, i) = vb[k].val();
    }
    W(a, W_HB, i) = hb.val();
    W(a, W_RHOB, i) = rhob.val();
    W(a, W_AB, i) = Ab.val();
    W(a, W_BB, i) = Bb.val();
    W(a, W_CB, i) = cb.val();
}

// v x r for D = 3 (3 components) and D = 2 (z only, stored in slot 2)
template <int D, class T> __device__ __forceinline__ void cross_vr(const T v[D], const T d[D], T o[3])
{
    o[0] = o[1] = o[2] = T(0);
    if constexpr(D == 3) {
        o[0] = v[1] * d[2] - v[2] * d[1];
        o[1] = v[2] * d[0] - v[0] * d[2];
        o[2] = v[0] * d[1] - v[1] * d[0];
    } else if constexpr(D == 2) {
        o[2] = v[0] * d[1] - v[1] * d[0];
    }
}

// pass 2: gather sums of particle i and the chain rule through its
// derived quantities (src/pre_interaction.cpp:66-169), the latter in FP64
template <int D, int K, class T, int NW>
__global__ void __launch_bounds__(BLOCK) adj_pre_kernel(State s, BoxDev box, AdjArgs a)
{
    __shared__ double4 l_p[ASW][WAVE];
    __shared__ AdjRec<T> l_r[ASW][WAVE];
    __shared__ PartsLds<NW> red;
    const AdjGroup<D, NW> gp(a);
    if(!gp.have) return;  // (one wave per group only)
    const int i = gp.i, w = gp.w;
    double xi[D];
    T vi[D];
#pragma unroll
    for(int k = 0; k < D; ++k) {
        xi[k] = s.f[F_X + k][i];
        vi[k] = (T)s.f[F_V + k][i];
    }
    const GroupImage<D, T> img(box, gp.gnc, xi);
    const double h = s.f[F_SML][i];
    const T ht = (T)h, ht_inv = T(1) / ht;
    Acc<T> rho_a, rhop_a, rhopp_a, Dv_a, Dvh_a, Rv_a[3], Rvh_a[3];
    auto keep = [&](int kc) -> bool {
        double dd[D];
        return pair_r<T>(pair_sep2<D, T>(img, xi, l_p[w][kc], dd)) < ht;
    };
    auto pair = [&](int kc) {
        const AdjRec<T> &j = l_r[w][kc];
        double dd[D];
        const double r2 = pair_sep2<D, T>(img, xi, l_p[w][kc], dd);
        const T r = pair_r<T>(r2);
        const T mj = j.m;
        const KernelDerivs<T> kd = kernel_derivs_inv<D, K, T>(r, ht_inv);
        rho_a.add(mj * kd.w);
        rhop_a.add(mj * kd.wh);
        rhopp_a.add(mj * kd.whh);
        // (particle i itself adds nothing to the sums over v_ij)
        if(a.balsara && D > 1) {
            T v[D], d[D], sv = T(0);
#pragma unroll
            for(int k = 0; k < D; ++k) {
                d[k] = (T)dd[k];
                v[k] = vi[k] - j.v[k];
                sv += v[k] * d[k];
            }
            T cr[3];
            cross_vr<D, T>(v, d, cr);
            Dv_a.add(mj * sv * kd.f);
            Dvh_a.add(mj * sv * kd.fh);
#pragma unroll
            for(int k = 0; k < 3; ++k) {
                Rv_a[k].add(mj * cr[k] * kd.f);
                Rvh_a[k].add(mj * cr[k] * kd.fh);
            }
        }
    };
    const AdjRec<T> *rec = (const AdjRec<T> *)a.rec;
    adj_sweep<D, NW>(gp, [&](int tt) { return gp.stage(a, img, tt, l_p[w], l_r[w], rec); }, keep, pair);
    parts_sum<NW, 3>(red, gp.part, {&rho_a.s, &rhop_a.s, &rhopp_a.s});
    if(a.balsara && D > 1) {
        parts_sum<NW, 4>(red, gp.part, {&Dv_a.s, &Rv_a[0].s, &Rv_a[1].s, &Rv_a[2].s});
        parts_sum<NW, 4>(red, gp.part, {&Dvh_a.s, &Rvh_a[0].s, &Rvh_a[1].s, &Rvh_a[2].s});
    }
    if(!gp.valid || gp.part != 0) return;
    const double rho = rho_a.val(), rhop = rhop_a.val(), rhopp = rhopp_a.val(), Dv = Dv_a.val(), Dvh = Dvh_a.val();
    const double Rv[3] = {Rv_a[0].val(), Rv_a[1].val(), Rv_a[2].val()};
    const double Rvh[3] = {Rvh_a[0].val(), Rvh_a[1].val(), Rvh_a[2].val()};

    const double gm1 = a.gamma - 1.0;
    const double rho_f = s.f[F_DENS][i], pres = s.f[F_PRES][i], om = s.f[F_GRADH][i];
    const double ci = s.f[F_SOUND][i], ui = s.f[F_ENE][i];
    const double Ab = W(a, W_AB, i);
    const double A = pres * om / (rho_f * rho_f);
    // A = P Omega / rho^2
    const double Pb = Ab * om / (rho_f * rho_f);
    const double Omb = Ab * pres / (rho_f * rho_f);
    double rhob = W(a, W_RHOB, i) - 2.0 * Ab * A / rho_f;
    double hb = W(a, W_HB, i);
    double cb = W(a, W_CB, i);
    // P = (gamma - 1) rho u
    double ub = gm1 * rho_f * Pb;
    rhob += gm1 * ui * Pb;
    // Omega = 1 / (1 + X), X = h rho' / (D rho)
    const double X = h * rhop / (D * rho);
    const double Xb = -om * om * Omb;
    hb += Xb * rhop / (D * rho);
    const double rhopb = Xb * h / (D * rho);
    rhob -= Xb * X / rho;
    // Balsara switch B = |div| / (|div| + |rot| + 1e-4 c / h)
    double Dvb = 0.0, Rvb[3] = {0.0, 0.0, 0.0};
    if(a.balsara && D > 1) {
        const double Bb = W(a, W_BB, i);
        const double div = -Dv / rho;
        const double R = sqrt(Rv[0] * Rv[0] + Rv[1] * Rv[1] + Rv[2] * Rv[2]);
        const double rot = R / rho;
        const double ad = fabs(div);
        const double ec = 1e-4 * ci / h;
        const double den = ad + rot + ec;
        const double den2 = den * den;
        const double adb = Bb * (rot + ec) / den2;
        const double rotb = -Bb * ad / den2;
        cb -= Bb * ad * (1e-4 / h) / den2;
        hb += Bb * ad * ec / (h * den2);
        const double divb = div > 0.0 ? adb : div < 0.0 ? -adb : 0.0;
        Dvb = -divb / rho;
        rhob -= divb * div / rho;
        if(R > 0.0) {
#pragma unroll
            for(int k = 0; k < 3; ++k) Rvb[k] = rotb * Rv[k] / (R * rho);
            rhob -= rotb * rot / rho;
        }
    }
    // every h dependence of the sums, then h through G(h, x) = rho h^D - b
    hb += rhob * rhop + rhopb * rhopp + Dvb * Dvh + Rvb[0] * Rvh[0] + Rvb[1] * Rvh[1] + Rvb[2] * Rvh[2];
    const double hD1 = ipow<double, D - 1>(h);
    const double Gh = rhop * hD1 * h + D * rho * hD1;
    const double g = -hb / Gh;
    SeedRec<T> o{};
    o.h = (T)s.f[F_SML][i];
    o.hinv = T(1) / o.h;
    o.m = (T)s.f[F_MASS][i];
    o.srho = (T)(rhob + g * hD1 * h);
    o.srhop = (T)rhopb;
    o.sdv = (T)Dvb;
#pragma unroll
    for(int k = 0; k < D; ++k) o.v[k] = (T)s.f[F_V + k][i];
#pragma unroll
    for(int k = 0; k < 3; ++k) o.srv[k] = (T)Rvb[k];
    ((SeedRec<T> *)a.seed)[i] = o;
    // c = sqrt(gamma (gamma - 1) u)
    if(ci > 0.0) ub += cb * a.gamma * gm1 / (2.0 * ci);
    W(a, W_UB, i) = ub;
}

// derivative of the seeded sum terms of one pair with respect to r_ij and
// v_ij; the terms are even in (r_ij, v_ij), so both ends use the same form
template <int D, int K, class T>
__device__ __forceinline__ void sum_term(T r, const T d[D], const T v[D], T sv, T m, T hinv, T srho, T srhop, T sdv,
                                         const T srv[3], Acc<T> xb[D], Acc<T> vb[D])
{
    const KernelDerivs<T> kd = kernel_derivs_inv<D, K, T>(r, hinv);
    T gQd[D], gQv[D], Q = T(0);
    if constexpr(D == 3) {
        // Q = srv . (v x r):  dQ/dr = srv x v,  dQ/dv = r x srv
        gQd[0] = srv[1] * v[2] - srv[2] * v[1];
        gQd[1] = srv[2] * v[0] - srv[0] * v[2];
        gQd[2] = srv[0] * v[1] - srv[1] * v[0];
        gQv[0] = d[1] * srv[2] - d[2] * srv[1];
        gQv[1] = d[2] * srv[0] - d[0] * srv[2];
        gQv[2] = d[0] * srv[1] - d[1] * srv[0];
        Q = gQd[0] * d[0] + gQd[1] * d[1] + gQd[2] * d[2];
    } else if constexpr(D == 2) {
        gQd[0] = -srv[2] * v[1];
        gQd[1] = srv[2] * v[0];
        gQv[0] = srv[2] * d[1];
        gQv[1] = -srv[2] * d[0];
        Q = gQd[0] * d[0] + gQd[1] * d[1];
    } else {
        gQd[0] = gQv[0] = T(0);
    }
    const T radial = m * (srho * kd.f * r + srhop * kd.whr + (sdv * sv + Q) * kd.fr) / r;
    const T mf = m * kd.f;
#pragma unroll
    for(int k = 0; k < D; ++k) {
        xb[k].add(radial * d[k] + mf * (sdv * v[k] + gQd[k]));
        vb[k].add(mf * (sdv * d[k] + gQv[k]));
    }
}

// pass 3: adjoint of x and v through the seeded gather sums of i (pairs
// with r < h_i) and of its neighbours j (pairs with r < h_j)
template <int D, int K, class T, int NW>
__global__ void __launch_bounds__(BLOCK) adj_sum_kernel(State s, BoxDev box, AdjArgs a)
{
    __shared__ double4 l_p[ASW][WAVE];
    __shared__ SeedRec<T> l_r[ASW][WAVE];
    __shared__ PartsLds<NW> red;
    const AdjGroup<D, NW> g(a);
    if(!g.have) return;  // (one wave per group only)
    const int i = g.i, w = g.w;
    double xi[D];
    T vi[D];
#pragma unroll
    for(int k = 0; k < D; ++k) {
        xi[k] = s.f[F_X + k][i];
        vi[k] = (T)s.f[F_V + k][i];
    }
    const GroupImage<D, T> img(box, g.gnc, xi);
    const SeedRec<T> *rec = (const SeedRec<T> *)a.seed;
    const SeedRec<T> me = rec[i];
    Acc<T> xb[D], vb[D];
    auto keep = [&](int kc) -> bool {
        double dd[D];
        const T r = pair_r<T>(pair_sep2<D, T>(img, xi, l_p[w][kc], dd));
        return r != T(0) && (r < me.h || r < l_r[w][kc].h);
    };
    auto pair = [&](int kc) {
        const SeedRec<T> &j = l_r[w][kc];
        double dd[D];
        const T r = pair_r<T>(pair_sep2<D, T>(img, xi, l_p[w][kc], dd));
        T v[D], d[D], sv = T(0);
#pragma unroll
        for(int k = 0; k < D; ++k) {
            d[k] = (T)dd[k];
            v[k] = vi[k] - j.v[k];
            sv += v[k] * d[k];
        }
        if(r < me.h) sum_term<D, K, T>(r, d, v, sv, j.m, me.hinv, me.srho, me.srhop, me.sdv, me.srv, xb, vb);
        if(r < j.h) sum_term<D, K, T>(r, d, v, sv, me.m, j.hinv, j.srho, j.srhop, j.sdv, j.srv, xb, vb);
    };
    adj_sweep<D, NW>(g, [&](int tt) { return g.stage(a, img, tt, l_p[w], l_r[w], rec); }, keep, pair);
#pragma unroll
    for(int k = 0; k < D; ++k) parts_sum<NW, 2>(red, g.part, {&xb[k].s, &vb[k].s});
    if(!g.valid || g.part != 0) return;
#pragma unroll
    for(int k = 0; k < D; ++k) {
        W(a, W_XB + k, i) += xb[k].val();
        W(a, W_VB + k, i) += vb[k].val();
    }
}

// kick-drift adjoint and write-back in caller order
template <int D> __global__ void __launch_bounds__(BLOCK) adj_state_kernel(State s, int n, AdjArgs a)
{
    using L = AdjLayout<D>;
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if(i >= n) return;
    const int id = s.id[i];
    const double dt = a.dt;
    const double ubF = W(a, W_UB, i);
    if(a.kick) {
#pragma unroll
        for(int k = 0; k < D; ++k) {
            const double xbar = ADJ<D>(a, L::X + k, id) + W(a, W_XB + k, i);
            const double vtb = W(a, W_VB + k, i);
            const double vpb = ADJ<D>(a, L::V + k, id) + xbar * dt;
            ADJ<D>(a, L::X + k, id) = xbar;
            ADJ<D>(a, L::V + k, id) = vtb + vpb;
            ADJ<D>(a, L::A + k, id) = vtb * dt + vpb * 0.5 * dt;
        }
        const double upb = ADJ<D>(a, L::U, id);
        ADJ<D>(a, L::U, id) = ubF + upb;
        ADJ<D>(a, L::DU, id) = ubF * dt + upb * 0.5 * dt;
    } else {
#pragma unroll
        for(int k = 0; k < D; ++k) {
            ADJ<D>(a, L::X + k, id) += W(a, W_XB + k, i);
            ADJ<D>(a, L::V + k, id) += W(a, W_VB + k, i);
            ADJ<D>(a, L::A + k, id) = 0.0;
        }
        ADJ<D>(a, L::U, id) += ubF;
        ADJ<D>(a, L::DU, id) = 0.0;
    }
}

template <int D, int K, class T, int NW> static void launch_pairs(Ctx &c, const AdjArgs &a, const BoxDev &box)
{
    const int g = NW > 1 ? c.ngroups : group_grid(c);
    hipLaunchKernelGGL((adj_force_kernel<D, K, T, NW>), dim3(g), dim3(BLOCK), 0, c.stream, c.s, box, a);
    hipLaunchKernelGGL((adj_pre_kernel<D, K, T, NW>), dim3(g), dim3(BLOCK), 0, c.stream, c.s, box, a);
    hipLaunchKernelGGL((adj_sum_kernel<D, K, T, NW>), dim3(g), dim3(BLOCK), 0, c.stream, c.s, box, a);
}

template <int D, int K, class T> static void launch_passes_t(Ctx &c, const AdjArgs &a, const BoxDev &box)
{
    const int g = grid_for(c.n);
    hipLaunchKernelGGL((adj_seed_kernel<D, T>), dim3(g), dim3(BLOCK), 0, c.stream, c.s, (int)c.n, a);
    if(group_waves(c, GROUP_PAIRS) > 1) launch_pairs<D, K, T, ASW>(c, a, box);
    else launch_pairs<D, K, T, 1>(c, a, box);
    hipLaunchKernelGGL((adj_state_kernel<D>), dim3(g), dim3(BLOCK), 0, c.stream, c.s, (int)c.n, a);
}

template <int D, int K> static void launch_passes(Ctx &c, const AdjArgs &a, const BoxDev &box)
{
    if(c.p.precision == SPHGPU_MIXED) launch_passes_t<D, K, float>(c, a, box);
    else launch_passes_t<D, K, double>(c, a, box);
}

int adjoint_step(Ctx &c, bool kick)
{
    AdjArgs a{};
    a.groups = c.groups;
    a.ngroups = c.ngroups;
    a.cand = c.tile_cand;
    a.ma = c.tile_ma;
    a.gnc = c.tile_nc;
    a.wcap = c.tile_wcap;
    a.pos = c.posrec;  // free after the force pass
    a.rec = c.ro.rec;
    a.seed = c.ro.seed;
    a.w = c.ro.work;
    a.n = c.ro.n;
    a.adj = c.ro.adj;
    a.gamma = c.p.gamma;
    a.nngb = c.p.neighbor_number;
    a.balsara = c.p.av_use_balsara_switch;
    a.dt = c.ro.dt;
    a.kick = kick ? 1 : 0;
    const BoxDev box = make_box(c);
    const bool wend = c.p.kernel == SPHGPU_WENDLAND;
    switch(c.D) {
    case 1: launch_passes<1, 0>(c, a, box); break;
    case 2: wend ? launch_passes<2, 1>(c, a, box) : launch_passes<2, 0>(c, a, box); break;
    default: wend ? launch_passes<3, 1>(c, a, box) : launch_passes<3, 0>(c, a, box); break;
    }
    SPHGPU_HIP(hipGetLastError());
    return SPHGPU_OK;
}

void adjoint_free(Ctx &c)
{
    if(c.ro.ck) (void)hipFree(c.ro.ck);
    if(c.ro.ck_id) (void)hipFree(c.ro.ck_id);
    if(c.ro.adj) (void)hipFree(c.ro.adj);
    if(c.ro.work) (void)hipFree(c.ro.work);
    if(c.ro.rec) (void)hipFree(c.ro.rec);
    if(c.ro.seed) (void)hipFree(c.ro.seed);
    c.ro = Ctx::Rollout{};
}

// slots: 0 = state before Solver::initialize, 1..K = state at the start of
// step 0..K-1, K+1 = final state
int adjoint_alloc(Ctx &c, int steps)
{
    const int slots = steps + 2;
    if(c.ro.ck && c.ro.n == c.n && c.ro.slots >= slots) {
        c.ro.steps = 0;
        return SPHGPU_OK;
    }
    adjoint_free(c);
    int f[32];
    const int nck = ck_fields(c.D, f);
    const size_t n = (size_t)c.n;
    SPHGPU_HIP(hipMalloc(&c.ro.ck, (size_t)slots * nck * n * sizeof(double)));
    SPHGPU_HIP(hipMalloc(&c.ro.ck_id, (size_t)slots * n * sizeof(int)));
    SPHGPU_HIP(hipMalloc(&c.ro.adj, (size_t)(3 * c.D + 2) * n * sizeof(double)));
    SPHGPU_HIP(hipMalloc(&c.ro.work, (size_t)NWORK * n * sizeof(double)));
    const bool mixed = c.p.precision == SPHGPU_MIXED;
    SPHGPU_HIP(hipMalloc(&c.ro.rec, n * (mixed ? sizeof(AdjRec<float>) : sizeof(AdjRec<double>))));
    SPHGPU_HIP(hipMalloc(&c.ro.seed, n * (mixed ? sizeof(SeedRec<float>) : sizeof(SeedRec<double>))));
    c.ro.n = c.n;
    c.ro.slots = slots;
    c.ro.steps = 0;
    return SPHGPU_OK;
}

// Copies of a slot's fields and ids in one launch (the state's arrays are
// separate allocations; a copy call for each took 18 launches of 5 us).
struct SlotCopy {
    const double *src[20];
    double *dst[20];
    const int *isrc;
    int *idst;
    int nf;
};

__global__ void __launch_bounds__(BLOCK) slot_copy_kernel(SlotCopy c, int n)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if(i >= n) return;
    for(int k = 0; k < c.nf; ++k) c.dst[k][i] = c.src[k][i];
    c.idst[i] = c.isrc[i];
}

static int slot_copy(Ctx &c, int slot, bool save)
{
    int f[32];
    const int nck = ck_fields(c.D, f);
    const size_t n = (size_t)c.n;
    SlotCopy s{};
    s.nf = nck;
    for(int k = 0; k < nck; ++k) {
        double *ck = c.ro.ck + ((size_t)slot * nck + k) * n;
        s.src[k] = save ? c.s.f[f[k]] : ck;
        s.dst[k] = save ? ck : c.s.f[f[k]];
    }
    int *id = c.ro.ck_id + (size_t)slot * n;
    s.isrc = save ? c.s.id : id;
    s.idst = save ? id : c.s.id;
    hipLaunchKernelGGL(slot_copy_kernel, dim3(grid_for(c.n)), dim3(BLOCK), 0, c.stream, s, (int)c.n);
    SPHGPU_HIP(hipGetLastError());
    return SPHGPU_OK;
}

int adjoint_save(Ctx &c, int slot) { return slot_copy(c, slot, true); }
int adjoint_restore(Ctx &c, int slot) { return slot_copy(c, slot, false); }

// host seeds (caller order, n*D for vectors; NULL = 0) into the adjoint state
int adjoint_seed(Ctx &c, const double *dx, const double *dv, const double *du)
{
    const int D = c.D;
    const int64_t n = c.n;
    Xfer x;
    auto put = [&](const double *src, int comps, int row) {
        const int off = src ? x.add(const_cast<double *>(src), comps) : -1;
        for(int k = 0; k < comps; ++k) x.field(c.ro.adj + (row + k) * n, off, comps, k);
    };
    // the rows of AdjLayout: x, v, u, a, du
    put(dx, D, 0);
    put(dv, D, D);
    put(du, 1, 2 * D);
    put(nullptr, D, 2 * D + 1);
    put(nullptr, 1, 3 * D + 1);
    return xfer_upload(c, x, n);
}

int adjoint_fetch(Ctx &c, double *dx, double *dv, double *du)
{
    const int D = c.D;
    const int64_t n = c.n;
    Xfer x;
    auto get = [&](double *dst, int comps, int row) {
        if(!dst) return;
        const int off = x.add(dst, comps);
        for(int k = 0; k < comps; ++k) x.field(c.ro.adj + (row + k) * n, off, comps, k);
    };
    get(dx, D, 0);
    get(dv, D, D);
    get(du, 1, 2 * D);
    return xfer_download(c, x, n);
}

}  // namespace sphgpu
