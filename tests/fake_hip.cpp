// A HIP runtime on the host for tests of the library's host code: device memory
// is host memory (zeroed when allocated), copies are memcpy, kernels do not run
// but are counted by name.  Loaded with RTLD_GLOBAL before the library, its
// functions take the place of libamdhip64's.
#include <hip/hip_runtime_api.h>

#include <stdlib.h>
#include <string.h>

#include <map>
#include <mutex>
#include <string>

namespace {
std::mutex lock;
std::map<const void *, std::string> names;
std::map<std::string, long> launches;
long fail_at = 0, allocations = 0;   // the fail_at'th allocation from now on fails
std::map<void *, size_t> sizes;
size_t most_lds = 0, live = 0;
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
thread_local Config config;
}  // namespace

extern "C" {
// For the tests.
void fake_fail_at(long n) { std::lock_guard<std::mutex> l(lock); fail_at = n; allocations = 0; }
long fake_allocations() { return allocations; }
size_t fake_most_lds() { return most_lds; }
size_t fake_live_bytes() { return live; }
long fake_launches(const char *part)   // of kernels whose mangled name holds `part`
{
    std::lock_guard<std::mutex> l(lock);
    long n = 0;
    for (auto &k : launches)
        if (k.first.find(part) != std::string::npos) n += k.second;
    return n;
}
void fake_forget_launches() { std::lock_guard<std::mutex> l(lock); launches.clear(); }

hipError_t hipMalloc(void **p, size_t n)
{
    std::lock_guard<std::mutex> l(lock);
    *p = nullptr;
    if (++allocations == fail_at) return hipErrorOutOfMemory;
    *p = calloc(n ? n : 1, 1);
    if (!*p) return hipErrorOutOfMemory;
    live += sizes[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::lock_guard<std::mutex> l(lock);
    live -= sizes[p];
    sizes.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    if (!d || !s) return hipErrorInvalidValue;
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    if (!d) return hipErrorInvalidValue;
    if (v || n < (size_t)1 << 28) memset(d, v, n);   // (large arrays are cleared once, when new)
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = *t = (size_t)288 << 30; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int)
{
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "an error"; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 4; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidValue; }

hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t lds, hipStream_t)
{
    std::lock_guard<std::mutex> l(lock);
    ++launches[names[f]];
    if (lds > most_lds) most_lds = lds;
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    config = {g, b, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
{
    *g = config.grid; *b = config.block; *lds = config.lds; *s = config.stream;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *device, unsigned, void *, void *, void *, void *, int *)
{
    names[host] = device;
}
}  // extern "C"
