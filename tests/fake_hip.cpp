// A stand-in for the HIP runtime on machines without a device, for tests of
// the library's host paths.  Loaded with RTLD_GLOBAL before libglp.so, its
// functions are the ones the library calls: device memory is host memory
// (zeroed), copies are immediate, and a kernel launch only records the
// kernel's name.  Allocations can be made to fail.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>

namespace {
std::mutex mu;
std::map<const void*, std::string>& kernels() {
    static auto* m = new std::map<const void*, std::string>;
    return *m;
}
std::string& log_text() {
    static auto* s = new std::string;
    return *s;
}
// operator new of the arming thread throws once this many more were made
thread_local long news_left = -1;
struct Spared {  // what the stand-in itself allocates does not count
    long saved = news_left;
    Spared() { news_left = -1; }
    ~Spared() { news_left = saved; }
};
void note(const char* what) {
    Spared own;
    std::lock_guard<std::mutex> lk(mu);
    log_text() += what;
    log_text() += '\n';
}
std::map<void*, size_t>& sizes() {
    static auto* m = new std::map<void*, size_t>;
    return *m;
}
size_t device_bytes = 0;       // held now
size_t device_limit = ~0ull;   // hipMalloc fails beyond it
long host_allocs_left = -1;    // hipHostMalloc fails at 0 (-1: never)
long events_left = -1;         // event creation fails at 0 (-1: never)
thread_local struct {
    dim3 grid, block;
    size_t lds;
    hipStream_t s;
} config;

hipError_t give(void** p, size_t n) {
    *p = std::calloc(1, n ? n : 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
}  // namespace

void* operator new(size_t n) {
    if (news_left >= 0 && news_left-- == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
// ---- control (ctypes) ----
const char* fake_log() {  // what was recorded since the last call
    static std::string out;
    std::lock_guard<std::mutex> lk(mu);
    out.swap(log_text());
    log_text().clear();
    return out.c_str();
}
size_t fake_device_bytes() { return device_bytes; }
void fake_limit_device(size_t more) { device_limit = more == ~0ull ? more : device_bytes + more; }
void fake_fail_host_alloc(long after) { host_allocs_left = after; }
void fake_fail_events(long after) { events_left = after; }
void fake_fail_new(long after) { news_left = after; }

// ---- the runtime ----
hipError_t hipMalloc(void** p, size_t n) {
    Spared own;
    std::lock_guard<std::mutex> lk(mu);
    if (n > device_limit || device_bytes > device_limit - n) return hipErrorOutOfMemory;
    const hipError_t e = give(p, n);
    if (e == hipSuccess) {
        sizes()[*p] = n;
        device_bytes += n;
    }
    return e;
}
hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    note("hipFree");
    std::lock_guard<std::mutex> lk(mu);
    device_bytes -= sizes()[p];
    sizes().erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    {
        Spared own;
        note(("hipHostMalloc:" + std::to_string(n)).c_str());
    }
    if (host_allocs_left >= 0 && host_allocs_left-- <= 0) {
        host_allocs_left = 0;
        return hipErrorOutOfMemory;
    }
    return give(p, n);
}
hipError_t hipHostFree(void* p) {
    if (p) note("hipHostFree");
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    note("hipMemcpyAsync");
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    void* p;
    const hipError_t e = give(&p, 8);
    *s = static_cast<hipStream_t>(p);
    return e;
}
hipError_t hipExtStreamCreateWithCUMask(hipStream_t* s, uint32_t, const uint32_t*) {
    return hipStreamCreateWithFlags(s, 0);
}
hipError_t hipStreamDestroy(hipStream_t s) {
    note("hipStreamDestroy");
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    note("hipStreamSynchronize");
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (events_left >= 0 && events_left-- <= 0) {
        events_left = 0;
        return hipErrorOutOfMemory;
    }
    void* p;
    const hipError_t r = give(&p, 8);
    *e = static_cast<hipEvent_t>(p);
    return r;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
    note("hipEventDestroy");
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 0.f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    *g = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* g, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    static int any;
    *g = reinterpret_cast<hipGraphExec_t>(&any);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
    note("hipGraphLaunch");
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
    *p = nullptr;
    return hipErrorNotSupported;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "refused by the test"; }

hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
    note(kernels()[f].c_str());
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    config = {grid, block, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
    *grid = config.grid;
    *block = config.block;
    *lds = config.lds;
    *s = config.s;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
    static void* any;
    return &any;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, dim3*, dim3*,
                           int*) {
    kernels()[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
}
