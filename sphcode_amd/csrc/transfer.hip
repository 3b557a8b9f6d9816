// Particle arrays between the caller's memory (one array per field, vectors
// as [i*dim + k], caller order) and the device (one array per component, in
// Morton order): the staging copies go over the bus in the caller's layout
// and a kernel does the rest, the transposition and, on the way back, the
// gather into caller order.
//
// What bounds it: the first touch of freshly allocated caller pages (one
// thread fills 128 MB of them in 34 ms, eight in a tenth of that), then the bus
// (57 GB/s from pinned memory).  So the arrays pass through a ring of pinned
// slots: up to XFER_THREADS threads copy pieces of some slots while the others
// are on the bus.  A copy command costs some 15 us beside its bytes, so that
// large transfers take large slots (172 MB up and 134 MB down: 5.7 and 4.4 ms
// with eight slots of 1 MB, 3.9 and 3.1 with four of 4 MB, 3.6 and 2.9 with four
// of 8 MB, 3.5 and 3.2 with two of 32 MB).
//
// Fresh pinned memory is dear: 0.5 ms to allocate, 0.3 ms to free, and 1.5 us
// for the first touch of each page.  With two slots of 32 MB of its own every
// engine's first transfers took 2 ms (110,592 particles) to 10 ms (10^6) longer
// than later ones.  Rings are therefore small, and handed from engine to
// engine (PinnedPool).  On the device a transfer is staged in the tree build's
// moment sums, which nothing reads between builds.
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "ctx.hpp"

namespace sphgpu {

constexpr int XFER_SLOTS = 4;
constexpr int64_t XFER_SLOT = 4 << 20;   // bytes of a slot, at most
constexpr int64_t XFER_PIECE = 1 << 20;  // bytes that a thread copies at once; worth a thread of their own
constexpr int XFER_THREADS = 8;

// ------------------------------------------------------------ pinned memory
// Rings that no transfer holds at the moment: at most two, of at most
// XFER_SLOTS XFER_SLOT bytes each, kept for the next transfer of any engine
// while there is one.  A transfer holds a ring by itself, so that engines in
// several threads do not wait for each other.
struct PinnedPool {
    struct Ring {
        char *p = nullptr;
        int64_t bytes = 0;
    };
    std::mutex mu;
    Ring idle[2];
    int engines = 0;

    // a ring of at least `bytes`
    int take(int64_t bytes, Ring &r)
    {
        {
            std::lock_guard<std::mutex> lock(mu);
            for(Ring &k : idle)
                if(k.bytes >= bytes) {
                    std::swap(r, k);
                    return SPHGPU_OK;
                }
        }
        SPHGPU_HIP(hipHostMalloc(reinterpret_cast<void **>(&r.p), bytes, hipHostMallocPortable));
        r.bytes = bytes;
        return SPHGPU_OK;
    }
    // (the larger rings are kept)
    void give(Ring r)
    {
        {
            std::lock_guard<std::mutex> lock(mu);
            if(engines > 0)
                for(Ring &k : idle)
                    if(r.bytes > k.bytes) std::swap(r, k);
        }
        if(r.p) (void)hipHostFree(r.p);
    }
    void attach()
    {
        std::lock_guard<std::mutex> lock(mu);
        ++engines;
    }
    void detach()
    {
        Ring gone[2];
        {
            std::lock_guard<std::mutex> lock(mu);
            if(--engines > 0) return;
            for(int k = 0; k < 2; ++k) std::swap(gone[k], idle[k]);
        }
        for(Ring &r : gone)
            if(r.p) (void)hipHostFree(r.p);
    }
};
static PinnedPool pool;

void xfer_attach() { pool.attach(); }
void xfer_detach() { pool.detach(); }

struct XferArgs {
    Xfer::Field f[Xfer::MAX_FIELDS];
    int nf;
    int64_t j0;     // first particle of the block (caller order)
    int m;          // particles in the block
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

// A stretch of the stage, and where the caller has it.
struct Stretch {
    char *user;
    int64_t bytes;
};

// Bytes [from, from + n) of the stage between a slot and the caller's arrays.
static void move_bytes(const Stretch *st, int count, bool up, char *slot, int64_t from, int64_t n)
{
    int64_t at = 0;
    for(int k = 0; k < count && at < from + n; at += st[k].bytes, ++k) {
        const int64_t b = std::max(from, at), e = std::min(from + n, at + st[k].bytes);
        if(b >= e) continue;
        char *user = st[k].user + (b - at), *pin = slot + (b - from);
        if(up) std::memcpy(pin, user, e - b);
        else std::memcpy(user, pin, e - b);
    }
}

// `total` bytes between the caller's stretches and the device stage, through
// the ring: in slots of `slot` bytes, which threads fill or empty in pieces.
// Slot c % XFER_SLOTS holds chunk c; pieces are taken in order, and those below
// `open` may be.  The calling thread makes the copies, and lends a hand where
// it would wait for pieces (it does all of them if there is no other thread).
static int xfer_stream(Ctx &c, const Stretch *st, int count, bool up, char *ring, int64_t slot, char *stage, int64_t total)
{
    const int64_t piece = std::min(slot, XFER_PIECE);
    const int64_t P = (slot + piece - 1) / piece;  // pieces of a whole slot
    const int64_t chunks = (total + slot - 1) / slot;
    auto chunk_bytes = [&](int64_t k) { return std::min(slot, total - k * slot); };
    auto chunk_pieces = [&](int64_t k) { return (chunk_bytes(k) + piece - 1) / piece; };
    const int64_t pieces = (chunks - 1) * P + chunk_pieces(chunks - 1);

    std::atomic<int64_t> next{0}, open{up ? XFER_SLOTS * P : 0};
    std::atomic<int64_t> done[XFER_SLOTS];  // pieces of the slot's chunk
    for(auto &d : done) d.store(0);
    std::atomic<bool> stop{false};
    auto run = [&](int64_t q) {
        const int64_t k = q / P, off = (q % P) * piece;
        move_bytes(st, count, up, ring + (k % XFER_SLOTS) * slot + off, k * slot + off, std::min(piece, chunk_bytes(k) - off));
        done[k % XFER_SLOTS].fetch_add(1, std::memory_order_release);
    };
    auto work = [&] {
        for(;;) {
            const int64_t q = next.fetch_add(1);
            if(q >= pieces) return;
            while(q >= open.load(std::memory_order_acquire)) {
                if(stop.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
            }
            run(q);
        }
    };
    // all the pieces of chunk k, by any thread
    auto finish = [&](int64_t k) {
        while(done[k % XFER_SLOTS].load(std::memory_order_acquire) != chunk_pieces(k)) {
            int64_t q = next.load();
            if(q < pieces && q < open.load() && next.compare_exchange_strong(q, q + 1)) run(q);
            else std::this_thread::yield();
        }
    };
    std::vector<std::thread> workers;
    const int hw = (int)std::max(1u, std::thread::hardware_concurrency());
    const int threads = (int)std::min<int64_t>({(int64_t)XFER_THREADS, (int64_t)hw, total / XFER_PIECE});
    try {
        workers.reserve(std::max(0, threads - 1));
        for(int k = 1; k < threads; ++k) workers.emplace_back(work);
    } catch(...) {
        // no more threads: this one does the rest
    }
    auto copies = [&]() -> int {
        constexpr int AHEAD = XFER_SLOTS / 2;  // slots on the bus
        if(up) {
            for(int64_t k = 0; k < chunks; ++k) {
                if(k >= AHEAD) {
                    // the copy of chunk k - AHEAD has left its slot
                    SPHGPU_HIP(hipEventSynchronize(c.ev_xfer[(k - AHEAD) % XFER_SLOTS]));
                    done[(k - AHEAD) % XFER_SLOTS].store(0);
                    open.store((k - AHEAD + 1 + XFER_SLOTS) * P, std::memory_order_release);
                }
                finish(k);
                SPHGPU_HIP(hipMemcpyAsync(stage + k * slot, ring + (k % XFER_SLOTS) * slot, chunk_bytes(k), hipMemcpyHostToDevice, c.stream));
                SPHGPU_HIP(hipEventRecord(c.ev_xfer[k % XFER_SLOTS], c.stream));
            }
        } else {
            for(int64_t k = 0; k < chunks + AHEAD; ++k) {
                if(k < chunks) {
                    if(k >= XFER_SLOTS) finish(k - XFER_SLOTS);
                    done[k % XFER_SLOTS].store(0);
                    SPHGPU_HIP(hipMemcpyAsync(ring + (k % XFER_SLOTS) * slot, stage + k * slot, chunk_bytes(k), hipMemcpyDeviceToHost, c.stream));
                    SPHGPU_HIP(hipEventRecord(c.ev_xfer[k % XFER_SLOTS], c.stream));
                }
                const int64_t here = k - AHEAD;
                if(here >= 0 && here < chunks) {
                    SPHGPU_HIP(hipEventSynchronize(c.ev_xfer[here % XFER_SLOTS]));
                    open.store((here + 1) * P, std::memory_order_release);
                }
            }
            for(int64_t k = std::max<int64_t>(0, chunks - XFER_SLOTS); k < chunks; ++k) finish(k);
        }
        return SPHGPU_OK;
    };
    const int rc = copies();
    stop.store(true);
    for(std::thread &t : workers) t.join();
    return rc;
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

void xfer_free(Ctx &c)
{
    for(hipEvent_t &e : c.ev_xfer) {
        if(e) (void)hipEventDestroy(e);
        e = nullptr;
    }
}

static int xfer_run(Ctx &c, const Xfer &x, int64_t n, bool up)
{
    const int64_t dbytes = (int64_t)x.doubles * sizeof(double);
    const int64_t per = dbytes + (x.user_ints ? sizeof(int) : 0);  // staged bytes per particle
    // a block of particles at a time, as many as the stage holds (all of them
    // up to 160 bytes each), whole 256-byte lines per array if they are many
    char *const stage = reinterpret_cast<char *>(c.msum);
    const int64_t room = c.node_cap * (int64_t)sizeof(double4);
    int64_t block = n;
    if(per * n > room) {
        block = room / per;
        if(block >= 64) block = block / 64 * 64;
    }
    if(block < 1) return set_error(SPHGPU_E_INVALID, "transfer: no room for a particle");
    static_assert(sizeof(c.ev_xfer) == XFER_SLOTS * sizeof(hipEvent_t), "an event per slot");
    for(hipEvent_t &e : c.ev_xfer)
        if(!e) SPHGPU_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    XferArgs a{};
    for(int k = 0; k < x.nf; ++k) a.f[k] = x.f[k];
    a.nf = x.nf;
    a.ints = x.dev_ints;
    a.int_off = x.user_ints ? (int)dbytes : -1;
    if(!up && !x.user_ints) a.ints = nullptr;
    a.id = up ? x.dev_id : nullptr;
    a.stage = stage;
    if(!up && x.dev_id) {
        // (idx is the tree build's scratch)
        hipLaunchKernelGGL(inverse_kernel, dim3(grid_for(n)), dim3(BLOCK), 0, c.stream, x.dev_id, (int)n, c.idx);
        a.inv = c.idx;
    }
    // one slot up to half of the largest (a copy command costs more than the
    // overlap gives), then slots of that size for up to four of the largest
    const int64_t total = per * block;
    const int64_t slot = total <= XFER_SLOT / 2 ? std::max<int64_t>((total + 255) / 256 * 256, 256)
                       : total <= XFER_SLOTS * XFER_SLOT ? XFER_SLOT / 2 : XFER_SLOT;
    PinnedPool::Ring ring;
    if(per) {
        int rc = pool.take(std::min<int64_t>(XFER_SLOTS, (total + slot - 1) / slot) * slot, ring);
        if(rc) return rc;
    }
    auto blocks = [&]() -> int {
        for(int64_t j0 = 0; j0 < n; j0 += block) {
            const int64_t m = std::min(block, n - j0);
            Stretch st[Xfer::MAX_ARRAYS + 1];
            int count = 0;
            for(int k = 0; k < x.narrays; ++k, ++count)
                st[count] = {x.arrays[k].user + j0 * x.arrays[k].bytes, m * x.arrays[k].bytes};
            if(x.user_ints) st[count++] = {reinterpret_cast<char *>(x.user_ints + j0), m * (int64_t)sizeof(int)};
            a.j0 = j0;
            a.m = (int)m;
            if(!up) hipLaunchKernelGGL(pack_kernel, dim3(grid_for(m)), dim3(BLOCK), 0, c.stream, a);
            if(per) {
                int rc = xfer_stream(c, st, count, up, ring.p, slot, stage, per * m);
                if(rc) return rc;
            }
            if(up) {
                hipLaunchKernelGGL(unpack_kernel, dim3(grid_for(m)), dim3(BLOCK), 0, c.stream, a);
                // (the next block's pieces may be written to slots whose copies are still queued)
                if(j0 + block < n) SPHGPU_HIP(hipStreamSynchronize(c.stream));
            }
        }
        SPHGPU_HIP(hipGetLastError());
        return SPHGPU_OK;
    };
    int rc = blocks();
    // the ring is free once nothing is queued on it
    const hipError_t e = hipStreamSynchronize(c.stream);
    pool.give(ring);
    if(!rc && e != hipSuccess) rc = hip_fail(e, "hipStreamSynchronize");
    return rc;
}

int xfer_upload(Ctx &c, const Xfer &x, int64_t n) { return xfer_run(c, x, n, true); }

int xfer_download(Ctx &c, const Xfer &x, int64_t n)
{
    if(x.narrays == 0 && !x.user_ints) return SPHGPU_OK;
    return xfer_run(c, x, n, false);
}

}  // namespace sphgpu
