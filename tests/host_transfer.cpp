// Particle transfers on the CPU, with the kernels' work done here: every byte
// of the caller's arrays arrives, up and down, at sizes around the pieces,
// slots and blocks; several engines at once; pinned memory stays small, is
// handed on and is given back with the last engine.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../sphcode_amd/csrc/transfer.hip"

extern "C" {
extern void (*fake_kernel)(const void *kernel, dim3 grid, dim3 block, void **args);
extern size_t fake_args_bytes;
void fake_fail_after(long n);
int fake_failed();
size_t fake_host_bytes();
size_t fake_host_most();
}

using namespace sphgpu;

static void kernel(const void *f, dim3, dim3, void **args)
{
    // (the inverse permutation is the test's own)
    if(f != (const void *)unpack_kernel && f != (const void *)pack_kernel) return;
    const XferArgs &a = *static_cast<const XferArgs *>(args[0]);
    double *st = reinterpret_cast<double *>(a.stage);
    for(int i = 0; i < a.m; ++i) {
        if(f == (const void *)unpack_kernel) {
            const int64_t j = a.j0 + i;
            for(int k = 0; k < a.nf; ++k) {
                const Xfer::Field &q = a.f[k];
                q.dev[j] = q.off < 0 ? 0.0 : st[(int64_t)q.off * a.m + (int64_t)i * q.stride + q.comp];
            }
            if(a.ints) a.ints[j] = a.int_off < 0 ? 0 : reinterpret_cast<const int *>(a.stage + (int64_t)a.int_off * a.m)[i];
            if(a.id) a.id[j] = (int)j;
        } else {
            const int64_t j = a.inv ? a.inv[a.j0 + i] : a.j0 + i;
            for(int k = 0; k < a.nf; ++k) {
                const Xfer::Field &q = a.f[k];
                st[(int64_t)q.off * a.m + (int64_t)i * q.stride + q.comp] = q.dev ? q.dev[j] : 0.0;
            }
            if(a.ints) reinterpret_cast<int *>(a.stage + (int64_t)a.int_off * a.m)[i] = a.ints[j];
        }
    }
}

#define NEED(x)                                                \
    do {                                                       \
        if(!(x)) {                                             \
            std::printf("line %d: %s (%s)\n", __LINE__, #x, at); \
            std::exit(1);                                      \
        }                                                      \
    } while(0)

// one engine's part: a field of three components, `scalars` scalar ones and an
// int, through a stage of `room` bytes a particle
static void round_trip(int64_t n, int scalars, int64_t room, unsigned seed)
{
    char at[120];
    std::snprintf(at, sizeof at, "n=%lld scalars=%d room=%lld", (long long)n, scalars, (long long)room);
    Ctx c;
    NEED(hipStreamCreateWithFlags(&c.stream, 0) == hipSuccess);
    c.node_cap = n * room / sizeof(double4) + 1;
    NEED(hipMalloc((void **)&c.msum, c.node_cap * sizeof(double4)) == hipSuccess);
    std::mt19937 rng(seed);
    std::vector<double> v(3 * n), vback(3 * n, -1.0);
    for(double &x : v) x = rng();
    std::vector<std::vector<double>> s(scalars, std::vector<double>(n)), sback(scalars, std::vector<double>(n, -1.0));
    for(auto &a : s)
        for(double &x : a) x = rng();
    std::vector<int> nb(n), nbback(n, -1), dev_nb(n), id(n, -1);
    for(int &x : nb) x = rng();
    std::vector<std::vector<double>> dev(3 + scalars + 1, std::vector<double>(n, -2.0));
    xfer_attach();
    {
        Xfer x;
        int off = x.add(v.data(), 3);
        for(int k = 0; k < 3; ++k) x.field(dev[k].data(), off, 3, k);
        for(int k = 0; k < scalars; ++k) x.field(dev[3 + k].data(), x.add(s[k].data(), 1), 1, 0);
        x.field(dev[3 + scalars].data(), -1, 1, 0);
        x.user_ints = nb.data();
        x.dev_ints = dev_nb.data();
        x.dev_id = id.data();
        NEED(xfer_upload(c, x, n) == SPHGPU_OK);
        for(int64_t i = 0; i < n; ++i) {
            for(int k = 0; k < 3; ++k) NEED(dev[k][i] == v[3 * i + k]);
            for(int k = 0; k < scalars; ++k) NEED(dev[3 + k][i] == s[k][i]);
            NEED(dev[3 + scalars][i] == 0.0 && dev_nb[i] == nb[i] && id[i] == i);
        }
    }
    {
        // down in another order
        c.idx = dev_nb.data();
        std::vector<int> inv(n), ints(n);
        for(int64_t i = 0; i < n; ++i) inv[i] = (int)(n - 1 - i);
        c.idx = inv.data();
        for(int64_t i = 0; i < n; ++i) ints[i] = nb[i];
        Xfer x;
        int off = x.add(vback.data(), 3);
        for(int k = 0; k < 3; ++k) x.field(dev[k].data(), off, 3, k);
        for(int k = 0; k < scalars; ++k) x.field(dev[3 + k].data(), x.add(sback[k].data(), 1), 1, 0);
        x.user_ints = nbback.data();
        x.dev_ints = ints.data();
        x.dev_id = id.data();
        NEED(xfer_download(c, x, n) == SPHGPU_OK);
        for(int64_t i = 0; i < n; ++i) {
            const int64_t j = n - 1 - i;
            for(int k = 0; k < 3; ++k) NEED(vback[3 * i + k] == v[3 * j + k]);
            for(int k = 0; k < scalars; ++k) NEED(sback[k][i] == s[k][j]);
            NEED(nbback[i] == nb[j]);
        }
    }
    // a ring that cannot be had is reported, and nothing is left behind
    if(seed == 0) {
        xfer_detach();
        xfer_attach();
        for(int k = 0; k < 2; ++k) {
            Xfer x;
            x.field(dev[0].data(), x.add(v.data(), 1), 1, 0);
            fake_fail_after(k == 0 ? 0 : -1);
            NEED((xfer_upload(c, x, n) == SPHGPU_OK) == (k == 1));
            fake_fail_after(-1);
        }
    }
    xfer_free(c);
    xfer_detach();
    (void)hipFree(c.msum);
    (void)hipStreamDestroy(c.stream);
}

int main()
{
    const char *at = "main";
    fake_kernel = kernel;
    fake_args_bytes = sizeof(XferArgs);
    const int64_t most = 2 * XFER_SLOTS * XFER_SLOT;
    for(int64_t n : {1, 2, 63, 64, 65, 1000, 6553, 6554, 26214, 26215, 100000, 131073})
        for(int scalars : {0, 7, 14}) {
            round_trip(n, scalars, 160, 0);
            NEED(fake_host_bytes() == 0);  // with the last engine
        }
    // stages of less than the particles: blocks of some, of 64
    for(int64_t n : {100, 1000, 40001, 200003}) {
        round_trip(n, 14, 65, 0);
        round_trip(n, 14, n > 5000 ? 1 : 20, 0);
    }
    round_trip(900001, 14, 160, 0);  // 126 MB: every slot several times
    NEED(fake_host_most() <= (size_t)most);
    // engines made one after the other: the ring is handed on
    xfer_attach();
    round_trip(300000, 7, 160, 1);
    const size_t kept = fake_host_bytes();
    NEED(kept > 0 && kept <= (size_t)(XFER_SLOTS * XFER_SLOT));
    round_trip(300000, 7, 160, 1);
    NEED(fake_host_bytes() == kept);
    // and at once
    std::vector<std::thread> t;
    for(unsigned k = 1; k <= 4; ++k) t.emplace_back([=] { round_trip(50000 * k + 1, 7, 160, k); });
    for(std::thread &x : t) x.join();
    NEED(fake_host_bytes() <= (size_t)most);
    xfer_detach();
    NEED(fake_host_bytes() == 0);
    std::printf("ok, at most %zu bytes pinned\n", fake_host_most());
    return 0;
}
