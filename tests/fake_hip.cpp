// A HIP runtime without a GPU, for host-side tests of the library's memory
// and transfers: device memory is host memory, copies are made at once,
// kernels are not run.  Allocations are tracked, and one of them can be made
// to fail.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

static std::mutex mu;
static std::map<const char *, size_t> live;
static long to_fail = -1;   // allocations until one fails; < 0: none does
static size_t host_bytes = 0, host_most = 0;
static std::map<const char *, size_t> host_live;

extern "C" {

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
hipError_t hipFree(void *p)
{
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
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n)
{
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    memset(d, v, n);
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
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = reinterpret_cast<hipStream_t>(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = reinterpret_cast<hipEvent_t>(1); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = reinterpret_cast<hipEvent_t>(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { *p = nullptr; return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s)
{
    *g = dim3(1), *b = dim3(1), *n = 0, *s = nullptr;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

}  // extern "C"
