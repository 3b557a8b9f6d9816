// A HIP runtime without a GPU, for host-side tests of the library's memory
// and transfers: device memory is host memory.  What is queued on a stream is
// done as late as it may be, when the host waits for the stream or for an
// event behind it, so that a buffer reused too early shows.  Kernels are
// handed to a function of the test (or not run).  Allocations are tracked, and
// one of them can be made to fail.
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <vector>

static std::mutex mu;
static std::map<const char *, size_t> live;
static long to_fail = -1;   // allocations until one fails; < 0: none does
static size_t host_bytes = 0, host_most = 0;
static std::map<const char *, size_t> host_live;

// per stream: what is queued, and how many entries have been done
struct Queue {
    std::recursive_mutex mu;
    std::deque<std::function<void()>> work;
    long done = 0;
};
struct Event {
    Queue *q = nullptr;
    long at = 0;  // entries before it
};
static std::map<hipStream_t, Queue *> queues;
static Queue &queue(hipStream_t s)
{
    std::lock_guard<std::mutex> lock(mu);
    Queue *&q = queues[s];
    if(!q) q = new Queue;
    return *q;
}
static void push(hipStream_t s, std::function<void()> f)
{
    Queue &q = queue(s);
    std::lock_guard<std::recursive_mutex> lock(q.mu);
    q.work.push_back(std::move(f));
}
static void drain(Queue &q, long upto)
{
    std::lock_guard<std::recursive_mutex> lock(q.mu);
    while(!q.work.empty() && (upto < 0 || q.done < upto)) {
        q.work.front()();
        q.work.pop_front();
        ++q.done;
    }
}

extern "C" {

// called for every kernel launch, in stream order (the test's own, or null)
void (*fake_kernel)(const void *kernel, dim3 grid, dim3 block, void **args) = nullptr;
size_t fake_args_bytes = 0;  // of a kernel's first argument, which is kept until it runs

void fake_fail_after(long n) { to_fail = n; }
// did the failure happen?
int fake_failed() { return to_fail == -2; }
// bytes from p to the end of its allocation, 0 if it is in none
size_t fake_room(const void *p)
{
    std::lock_guard<std::mutex> lock(mu);
    auto it = live.upper_bound(static_cast<const char *>(p));
    if(it == live.begin()) return 0;
    --it;
    const size_t off = static_cast<const char *>(p) - it->first;
    return off < it->second ? it->second - off : 0;
}
size_t fake_host_bytes() { return host_bytes; }
size_t fake_host_most() { return host_most; }

static bool fails()
{
    if(to_fail < 0) return false;
    if(to_fail-- > 0) return false;
    to_fail = -2;
    return true;
}

hipError_t hipMalloc(void **p, size_t n)
{
    std::lock_guard<std::mutex> lock(mu);
    if(fails()) return hipErrorOutOfMemory;
    *p = calloc(n ? n : 1, 1);
    live[static_cast<char *>(*p)] = n;
    return hipSuccess;
}
static void drain_all()
{
    std::map<hipStream_t, Queue *> all;
    {
        std::lock_guard<std::mutex> lock(mu);
        all = queues;
    }
    for(auto &q : all) drain(*q.second, -1);
}
hipError_t hipFree(void *p)
{
    drain_all();
    std::lock_guard<std::mutex> lock(mu);
    if(p && !live.erase(static_cast<char *>(p))) abort();  // not allocated, or freed before
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> lock(mu);
    if(fails()) return hipErrorOutOfMemory;
    *p = calloc(n ? n : 1, 1);
    host_live[static_cast<char *>(*p)] = n;
    host_bytes += n;
    if(host_bytes > host_most) host_most = host_bytes;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    drain_all();
    std::lock_guard<std::mutex> lock(mu);
    auto it = host_live.find(static_cast<char *>(p));
    if(p && it == host_live.end()) abort();
    if(p) {
        host_bytes -= it->second;
        host_live.erase(it);
    }
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st)
{
    push(st, [=] { memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n)
{
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st)
{
    push(st, [=] { memset(d, v, n); });
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 4; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 4;
    p->warpSize = 64;
    return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    static std::atomic<long> next{1};
    *s = reinterpret_cast<hipStream_t>(next++);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { drain(queue(s), -1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return hipStreamSynchronize(s); }
hipError_t hipEventCreate(hipEvent_t *e) { *e = reinterpret_cast<hipEvent_t>(new Event); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<Event *>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    Queue &q = queue(s);
    std::lock_guard<std::recursive_mutex> lock(q.mu);
    *reinterpret_cast<Event *>(e) = Event{&q, q.done + (long)q.work.size()};
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    const Event v = *reinterpret_cast<Event *>(e);
    if(v.q) drain(*v.q, v.at);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t e, unsigned) { return hipEventSynchronize(e); }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { *p = nullptr; return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t st)
{
    if(!fake_kernel) return hipSuccess;
    std::vector<char> first(static_cast<char *>(args[0]), static_cast<char *>(args[0]) + fake_args_bytes);
    push(st, [=]() mutable {
        void *a[1] = {first.data()};
        fake_kernel(f, g, b, a);
    });
    return hipSuccess;
}
static thread_local hipStream_t launch_stream;
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t s)
{
    launch_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s)
{
    *g = dim3(1), *b = dim3(1), *n = 0, *s = launch_stream;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

}  // extern "C"
