// A call that runs out of memory must leave nothing that a later call takes
// for capacity: every buffer is there, in its size, whenever a call succeeds.
#include <cstdio>
#include <cstdlib>

#include "../sphcode_amd/csrc/ctx.hpp"

extern "C" {
void fake_fail_after(long n);
int fake_failed();
size_t fake_room(const void *p);
}

using namespace sphgpu;

static int bad = 0;
static void need(const void *p, size_t bytes, const char *what, long k)
{
    const size_t room = fake_room(p);
    if(p && room >= bytes) return;
    std::printf("%s: %zu bytes where %zu are needed (after failure %ld)\n", what, p ? room : 0, bytes, k);
    ++bad;
}

static void slabs(Ctx &c, long k)
{
    const size_t slots = (size_t)c.ngroups * c.tile_wcap;
    need(c.tile_cand, slots * sizeof(int), "tile_cand", k);
    need(c.tile_ma, slots * sizeof(uint64_t), "tile_ma", k);
    need(c.tile_mn, slots * sizeof(uint64_t), "tile_mn", k);
    need(c.tile_nc, c.ngroups * sizeof(int), "tile_nc", k);
    need(c.ws_j, (size_t)8 * c.num_cu * (BLOCK / WAVE) * c.tile_wcap * sizeof(int), "ws_j", k);
}

int main()
{
    // the search's slabs: few groups, then more than fit, then few again
    for(long k = 0;; ++k) {
        Ctx c;
        c.num_cu = 4;
        c.cap = 256;
        c.p.neighbor_number = 32;
        c.ngroups = 10;
        if(search_alloc(c) != SPHGPU_OK) return 2;
        slabs(c, -1);
        c.ngroups = 1000;
        fake_fail_after(k);
        const int rc = search_alloc(c);
        const bool failed = fake_failed();
        fake_fail_after(-1);
        if(failed == (rc == SPHGPU_OK)) return 3;
        if(rc == SPHGPU_OK) slabs(c, k);
        c.ngroups = 10;
        if(search_alloc(c) != SPHGPU_OK) return 4;
        slabs(c, k);
        if(!failed) break;  // every allocation has failed once
    }
    // an upload: small, then one that does not fit, then the small one again
    sphgpu_params p;
    sphgpu_params_default(&p);
    p.dim = 3;
    p.gamma = 5.0 / 3.0;
    p.neighbor_number = 32;
    p.time_end = 1.0;
    p.gravity_is_valid = 1;
    p.gravity_constant = 1.0;
    static double x[3 * 4096], m[4096];
    for(long k = 0;; ++k) {
        void *ctx = nullptr;
        if(sphgpu_create(&p, &ctx) != SPHGPU_OK) return 5;
        Ctx &c = *static_cast<Ctx *>(ctx);
        sphgpu_particles h{};
        h.pos = x;
        h.mass = m;
        h.n = 300;
        if(sphgpu_upload(ctx, &h) != SPHGPU_OK) return 6;
        h.n = 4000;
        fake_fail_after(k);
        const int rc = sphgpu_upload(ctx, &h);
        const bool failed = fake_failed();
        fake_fail_after(-1);
        if(failed == (rc == SPHGPU_OK)) return 7;
        if(failed && sphgpu_make_tree(ctx) != SPHGPU_E_STATE) {
            std::printf("a state whose upload failed (at %ld) is taken for one\n", k);
            ++bad;
        }
        if(failed) {
            h.n = 300;
            if(sphgpu_upload(ctx, &h) != SPHGPU_OK) return 8;
        }
        const size_t n = h.n;
        for(int f : {F_X, F_V, F_MASS, F_SML, F_PHI}) {
            need(c.s.f[f], n * sizeof(double), "field", k);
            need(c.alt.f[f], n * sizeof(double), "sorted field", k);
        }
        need(c.s.id, n * sizeof(int), "id", k);
        need(c.posrec, n * sizeof(double4), "posrec", k);
        need(c.srec, (n + WAVE) * sizeof(double4), "srec", k);
        need(c.leaf_rad, n * sizeof(double), "leaf_rad", k);
        need(c.keys, n * sizeof(uint64_t), "keys", k);
        need(c.t.rng, (5 * n + 1) * sizeof(int4), "nodes", k);
        need(c.gpart, n * sizeof(GravPart<float>), "gravity records", k);
        need(c.partial, 1024 * sizeof(double), "partials", k);
        sphgpu_destroy(ctx);
        if(!failed) break;
    }
    // recorded sets, switched on twice
    for(long k = 0;; ++k) {
        void *ctx = nullptr;
        if(sphgpu_create(&p, &ctx) != SPHGPU_OK) return 9;
        Ctx &c = *static_cast<Ctx *>(ctx);
        sphgpu_particles h{};
        h.pos = x;
        h.mass = m;
        h.n = 300;
        if(sphgpu_upload(ctx, &h) != SPHGPU_OK) return 10;
        fake_fail_after(k);
        const int rc = sphgpu_set_record_sets(ctx, 1);
        const bool failed = fake_failed();
        fake_fail_after(-1);
        if(failed == (rc == SPHGPU_OK)) return 11;
        if(failed && sphgpu_set_record_sets(ctx, 1) != SPHGPU_OK) return 12;
        for(int *q : {c.rec_gather, c.rec_force}) need(q, (size_t)h.n * c.cap * sizeof(int), "recorded sets", k);
        for(int *q : {c.rec_gather_cnt, c.rec_force_cnt, c.rec_used}) need(q, h.n * sizeof(int), "recorded counts", k);
        sphgpu_destroy(ctx);
        if(!failed) break;
    }
    std::printf("%d faults\n", bad);
    return bad ? 1 : 0;
}
