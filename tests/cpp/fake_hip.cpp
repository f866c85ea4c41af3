// A stand-in for the HIP runtime on the host: memory is host memory, copies
// are memcpy, kernels are not run.  Loaded in front of the runtime, it lets
// the library's host code run without a GPU and records what that code asks
// for: allocations (with a budget that can run out), and each launch's kernel
// and stream (one kernel can be told to fail).  Errors are kept as the runtime
// keeps them: the last one stays until hipGetLastError takes it.
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>
#include <hip/hip_runtime_api.h>

namespace {
struct Launch {
    std::string kernel;
    long stream;
};
std::map<const void*, std::string> names;
std::vector<Launch> launches;
std::map<void*, size_t> blocks;
size_t held = 0, budget = (size_t)-1;
long nmalloc = 0, nstream = 0;
std::string failing;
bool query_fails = false, host_fails = false;
hipError_t last = hipSuccess;
hipError_t give(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
struct Config {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
} config;
}  // namespace

extern "C" {
// what the tests ask
long fake_nmalloc() { return nmalloc; }
long fake_held() { return (long)held; }
void fake_budget(long b) { budget = b < 0 ? (size_t)-1 : (size_t)b; }
void fake_fail_kernel(const char* part) { failing = part; }
void fake_fail_query(int on) { query_fails = on != 0; }
void fake_fail_host_malloc(int on) { host_fails = on != 0; }
void fake_clear() { launches.clear(); }
long fake_nlaunch() { return (long)launches.size(); }
const char* fake_kernel(long i) { return launches[i].kernel.c_str(); }
long fake_stream(long i) { return launches[i].stream; }

// kernels
void** __hipRegisterFatBinary(const void*) {
    static void* h;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
    names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) {
    config = {g, b, s, st};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
    *g = config.grid, *b = config.block, *s = config.shmem, *st = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3, void**, size_t, hipStream_t st) {
    launches.push_back({names[f], (long)(intptr_t)st});
    if (g.x == 0 || g.y == 0 || g.z == 0) return give(hipErrorInvalidConfiguration);
    if (!failing.empty() && names[f].find(failing) != std::string::npos) return give(hipErrorLaunchFailure);
    return hipSuccess;
}

// memory
hipError_t hipMalloc(void** p, size_t n) {
    ++nmalloc;
    if (n > budget || held > budget - n) return give(hipErrorOutOfMemory);
    *p = calloc(1, n);
    blocks[*p] = n;
    held += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    held -= blocks[p];
    blocks.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (host_fails) return give(hipErrorOutOfMemory);
    *p = calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* a, size_t* b) {
    *a = *b = (size_t)1 << 34;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static char scratch[64];
    *p = scratch;
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t) {
    for (size_t i = 0; i < h; ++i) memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
    if (query_fails) return give(hipErrorInvalidValue);
    a->type = hipMemoryTypeUnregistered;
    return hipSuccess;
}

// devices, streams, events
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipStreamCreate(hipStream_t* s) {
    *s = reinterpret_cast<hipStream_t>((intptr_t)++nstream);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = reinterpret_cast<hipEvent_t>((intptr_t)1);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}
}
