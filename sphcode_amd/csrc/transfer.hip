// Particle arrays between the caller's memory (one array per field, vectors
// as [i*dim + k], caller order) and the device (one array per component, in
// Morton order): the staging copies go over the bus in the caller's layout
// and a kernel does the rest, the transposition and, on the way back, the
// gather into caller order.
//
// What bounds it: the first touch of freshly allocated caller pages (one
// thread fills 128 MB of them in 34 ms, eight in 6.5 ms, against 2.4 ms for
// the copy from the device), then the bus (57 GB/s from pinned memory).  So
// the arrays pass through two pinned buffers of at most XFER_HALF bytes: one
// is on the bus while up to XFER_THREADS threads copy the other.  2^21
// particles' pos, vel, density and energy (128 MB) download in 4.4 ms and an
// initial condition of ten doubles each uploads in 3.7 ms; with the
// transposition and permutation by one host thread, a copy call per
// component, they took 40.2 and 15.4 ms (1,800 particles: 0.06 and 0.06 ms,
// before 0.13 and 0.20 ms).
#include <cstring>
#include <thread>
#include <vector>

#include "ctx.hpp"

namespace sphgpu {

constexpr int64_t XFER_HALF = 32 << 20;  // bytes of a staging buffer, at most
constexpr int64_t XFER_GRAIN = 1 << 20;  // bytes worth a thread of their own
constexpr int XFER_THREADS = 8;

struct XferArgs {
    Xfer::Field f[Xfer::MAX_FIELDS];
    int nf;
    int64_t j0;     // first particle of the chunk (caller order)
    int m;          // particles in the chunk
    char *stage;
    int *ints;      // device int field, or null
    int int_off;    // its offset in the stage in bytes per particle, -1: zeros
    int *id;        // upload: receives the caller's index
    const int *inv; // download: slot of each caller index (null: the index)
};

__global__ void __launch_bounds__(BLOCK) unpack_kernel(XferArgs a)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if(i >= a.m) return;
    const int64_t j = a.j0 + i;
    const double *st = reinterpret_cast<const double *>(a.stage);
    for(int k = 0; k < a.nf; ++k) {
        const Xfer::Field f = a.f[k];
        f.dev[j] = f.off < 0 ? 0.0 : st[(int64_t)f.off * a.m + (int64_t)i * f.stride + f.comp];
    }
    if(a.ints) a.ints[j] = a.int_off < 0 ? 0 : reinterpret_cast<const int *>(a.stage + (int64_t)a.int_off * a.m)[i];
    if(a.id) a.id[j] = (int)j;
}

__global__ void __launch_bounds__(BLOCK) pack_kernel(XferArgs a)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if(i >= a.m) return;
    const int64_t j = a.inv ? a.inv[a.j0 + i] : a.j0 + i;
    double *st = reinterpret_cast<double *>(a.stage);
    for(int k = 0; k < a.nf; ++k) {
        const Xfer::Field f = a.f[k];
        st[(int64_t)f.off * a.m + (int64_t)i * f.stride + f.comp] = f.dev ? f.dev[j] : 0.0;
    }
    if(a.ints) reinterpret_cast<int *>(a.stage + (int64_t)a.int_off * a.m)[i] = a.ints[j];
}

__global__ void __launch_bounds__(BLOCK) inverse_kernel(const int *id, int n, int *inv)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if(i < n) inv[id[i]] = i;
}

struct Piece {
    char *dst;
    const char *src;
    size_t bytes;
};

// The pieces' copies, split over threads by bytes.
static void copy_pieces(const std::vector<Piece> &pieces)
{
    size_t total = 0;
    for(const Piece &p : pieces) total += p.bytes;
    auto part = [&](size_t from, size_t to) {
        size_t at = 0;
        for(const Piece &p : pieces) {
            const size_t b = std::max(from, at), e = std::min(to, at + p.bytes);
            if(b < e) std::memcpy(p.dst + (b - at), p.src + (b - at), e - b);
            at += p.bytes;
        }
    };
    const int hw = (int)std::max(1u, std::thread::hardware_concurrency());
    const int T = (int)std::min<size_t>({(size_t)XFER_THREADS, (size_t)hw, total / XFER_GRAIN});
    if(T < 2) {
        part(0, total);
        return;
    }
    std::vector<std::thread> workers;
    int started = 1;  // part 0 is this thread's
    try {
        workers.reserve(T - 1);
        for(; started < T; ++started)
            workers.emplace_back(part, total * started / T, total * (started + 1) / T);
    } catch(...) {
        // no more threads: the rest of the parts is done here
    }
    part(0, total / T);
    for(int k = started; k < T; ++k) part(total * k / T, total * (k + 1) / T);
    for(std::thread &t : workers) t.join();
}

int Xfer::add(void *user, int comps)
{
    arrays[narrays++] = {static_cast<char *>(user), (int)sizeof(double) * comps};
    const int off = doubles;
    doubles += comps;
    return off;
}

void Xfer::field(double *dev, int off, int stride, int comp)
{
    f[nf++] = {dev, off, stride, comp};
}

// Two staging buffers of `half` bytes on the host and on the device.
static int xfer_buffers(Ctx &c, int64_t half)
{
    if(half > c.xfer_half) {
        if(c.xfer_dev) (void)hipFree(c.xfer_dev);
        if(c.xfer_host) (void)hipHostFree(c.xfer_host);
        c.xfer_dev = c.xfer_host = nullptr;
        c.xfer_half = 0;
        SPHGPU_HIP(hipMalloc(&c.xfer_dev, 2 * half));
        SPHGPU_HIP(hipHostMalloc(&c.xfer_host, 2 * half, hipHostMallocDefault));
        c.xfer_half = half;
    }
    for(hipEvent_t &e : c.ev_xfer)
        if(!e) SPHGPU_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    return SPHGPU_OK;
}

void xfer_free(Ctx &c)
{
    if(c.xfer_dev) (void)hipFree(c.xfer_dev);
    if(c.xfer_host) (void)hipHostFree(c.xfer_host);
    c.xfer_dev = c.xfer_host = nullptr;
    c.xfer_half = 0;
    for(hipEvent_t &e : c.ev_xfer) {
        if(e) (void)hipEventDestroy(e);
        e = nullptr;
    }
}

static int xfer_run(Ctx &c, const Xfer &x, int64_t n, bool up)
{
    const int64_t dbytes = (int64_t)x.doubles * sizeof(double);
    const int64_t per = dbytes + (x.user_ints ? sizeof(int) : 0);  // staged bytes per particle
    // whole 256-byte lines per array and chunk
    const int64_t chunk = per == 0 ? n : std::min<int64_t>((n + 63) / 64 * 64, std::max<int64_t>(64, XFER_HALF / per / 64 * 64));
    int rc = xfer_buffers(c, std::max<int64_t>(per * chunk, 256));
    if(rc) return rc;
    XferArgs a{};
    for(int k = 0; k < x.nf; ++k) a.f[k] = x.f[k];
    a.nf = x.nf;
    a.ints = x.dev_ints;
    a.int_off = x.user_ints ? (int)dbytes : -1;
    if(!up && !x.user_ints) a.ints = nullptr;
    a.id = up ? x.dev_id : nullptr;
    if(!up && x.dev_id) {
        // (idx is the tree build's scratch)
        hipLaunchKernelGGL(inverse_kernel, dim3(grid_for(n)), dim3(BLOCK), 0, c.stream, x.dev_id, (int)n, c.idx);
        a.inv = c.idx;
    }
    auto pieces = [&](int64_t j0, int64_t m, char *host) {
        std::vector<Piece> p;
        int64_t off = 0;
        auto piece = [&](char *user, int64_t bytes) {
            char *u = user + j0 * bytes;
            p.push_back(up ? Piece{host + off * m, u, (size_t)(bytes * m)} : Piece{u, host + off * m, (size_t)(bytes * m)});
            off += bytes;
        };
        for(int k = 0; k < x.narrays; ++k) piece(x.arrays[k].user, x.arrays[k].bytes);
        if(x.user_ints) piece(reinterpret_cast<char *>(x.user_ints), sizeof(int));
        return p;
    };
    std::vector<Piece> pending;  // download: the chunk in flight
    int half = 0;
    for(int64_t j0 = 0; j0 < n; j0 += chunk, half ^= 1) {
        const int64_t m = std::min(chunk, n - j0);
        char *host = static_cast<char *>(c.xfer_host) + half * c.xfer_half;
        a.stage = static_cast<char *>(c.xfer_dev) + half * c.xfer_half;
        a.j0 = j0;
        a.m = (int)m;
        if(up) {
            if(j0 >= 2 * chunk) SPHGPU_HIP(hipEventSynchronize(c.ev_xfer[half]));  // its previous copy has left
            if(per) {
                copy_pieces(pieces(j0, m, host));
                SPHGPU_HIP(hipMemcpyAsync(a.stage, host, per * m, hipMemcpyHostToDevice, c.stream));
                SPHGPU_HIP(hipEventRecord(c.ev_xfer[half], c.stream));
            }
            hipLaunchKernelGGL(unpack_kernel, dim3(grid_for(m)), dim3(BLOCK), 0, c.stream, a);
        } else {
            hipLaunchKernelGGL(pack_kernel, dim3(grid_for(m)), dim3(BLOCK), 0, c.stream, a);
            SPHGPU_HIP(hipMemcpyAsync(host, a.stage, per * m, hipMemcpyDeviceToHost, c.stream));
            SPHGPU_HIP(hipEventRecord(c.ev_xfer[half], c.stream));
            if(!pending.empty()) {
                SPHGPU_HIP(hipEventSynchronize(c.ev_xfer[half ^ 1]));
                copy_pieces(pending);
            }
            pending = pieces(j0, m, host);
        }
    }
    SPHGPU_HIP(hipGetLastError());
    SPHGPU_HIP(hipStreamSynchronize(c.stream));
    if(!up) copy_pieces(pending);
    return SPHGPU_OK;
}

int xfer_upload(Ctx &c, const Xfer &x, int64_t n) { return xfer_run(c, x, n, true); }

int xfer_download(Ctx &c, const Xfer &x, int64_t n)
{
    if(x.narrays == 0 && !x.user_ints) return SPHGPU_OK;
    return xfer_run(c, x, n, false);
}

}  // namespace sphgpu
