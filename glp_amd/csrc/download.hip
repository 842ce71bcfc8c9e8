// Device-to-host copies of results into the caller's pageable memory.

#include "device.h"
#include "download.h"

#include <algorithm>
#include <cstring>
#include <pthread.h>

namespace glp {

// A plain copy to pageable memory moves 11-14 GB/s: one thread takes the page
// faults and the copy out of the runtime's own buffer while the link, good
// for 50 GB/s, waits.  Through pinned slots, one thread up to kCopyLarge, four
// above (numpy arrays, plain / slots): 2 MB 161 / 127 us, 4 MB 297 / 232 us, 8
// MB 606 / 449 us, 32 MB 3.1 / 1.1 ms, 128 MB 12.5 / 3.5 ms.  More threads or
// smaller chunks above were slower (128 MB: 1 MB chunks 4.6 ms; eight threads,
// 512 KB chunks 6.1 ms), threads do not pay below (16 MB 0.77-1.0 ms with any
// number), and under 2 MB a plain copy into memory the program has used
// before is faster (a pass with 1 MB of labels 821 / 909 us, 96 arrays of 0.2
// MB 12.9 / 13.4 ms).  Making the slots takes 0.1 ms (1 MB), so the first copy
// is plain unless it is large; the large form's 16 MB take up to 5 ms to make,
// use first and give back, so they stay with the graph and not with each
// session (one-shot runs with a 32 MB result: plain 4.0 ms, slots made and
// freed by each session 4.6-5.2, the graph's 2.4; 16 MB 1.38 / 1.20 / 1.05, 64
// MB 8.7 / 5.5-6.6 / 6.1).
constexpr size_t kCopyDirect = 2 << 20;
constexpr size_t kCopyLarge = 16 << 20;
constexpr size_t kSmallChunk = 512 << 10;
constexpr size_t kLargeChunk = 2 << 20;

CopySlots::~CopySlots() {
    for (auto& e : done)
        if (e) (void)hipEventDestroy(e);
    if (slot[0]) (void)hipHostFree(slot[0]);
}

bool CopySlots::create(size_t bytes) {
    if (chunk) return true;
    hipError_t err = hipSuccess;
    if (!slot[0]) {
        void* p = nullptr;
        err = hipHostMalloc(&p, 2 * bytes, hipHostMallocDefault);
        if (err == hipSuccess) {
            slot[0] = static_cast<char*>(p);
            slot[1] = slot[0] + bytes;
        }
    }
    for (auto& e : done)
        if (err == hipSuccess && !e) err = hipEventCreateWithFlags(&e, hipEventDisableTiming);
    if (err != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    chunk = bytes;
    return true;
}

Staging::~Staging() {
    if (stream) (void)hipStreamDestroy(stream);
}

bool Staging::ready(size_t bytes) {
    if (!stream && hipStreamCreateWithFlags(&stream, hipStreamNonBlocking) != hipSuccess) {
        stream = nullptr;
        (void)hipGetLastError();
        return false;
    }
    if (bytes < kCopyLarge) return small.create(kSmallChunk);
    for (auto& w : large)
        if (!w.create(kLargeChunk)) return false;
    return true;
}

// Chunk i + 1 crosses the link while chunk i goes from its slot to its place.
static hipError_t copy_range(CopySlots& w, char* dst, const char* src, size_t bytes, hipStream_t s) {
    hipError_t e = hipSuccess;
    const size_t chunks = (bytes + w.chunk - 1) / w.chunk;
    auto issue = [&](size_t i) {
        const size_t at = i * w.chunk;
        e = hipMemcpyAsync(w.slot[i & 1], src + at, std::min(w.chunk, bytes - at), hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipEventRecord(w.done[i & 1], s);
    };
    if (chunks) issue(0);
    for (size_t i = 0; i < chunks && e == hipSuccess; ++i) {
        if (i + 1 < chunks) issue(i + 1);
        if (e == hipSuccess) e = hipEventSynchronize(w.done[i & 1]);
        const size_t at = i * w.chunk;
        if (e == hipSuccess) std::memcpy(dst + at, w.slot[i & 1], std::min(w.chunk, bytes - at));
    }
    // a slot's copy must not outlive a failed call
    if (e != hipSuccess) (void)hipStreamSynchronize(s);
    return e;
}

// A worker's share of a large copy.  (Threads are made by pthread_create,
// which reports what it cannot do; std::thread allocates and throws.)
struct CopyShare {
    CopySlots* slots;
    char* dst;
    const char* src;
    size_t bytes;
    hipStream_t s;
    int dev;
    hipError_t err;
};
static void* copy_share(void* arg) {
    CopyShare& c = *static_cast<CopyShare*>(arg);
    c.err = hipSetDevice(c.dev);
    if (c.err == hipSuccess) c.err = copy_range(*c.slots, c.dst, c.src, c.bytes, c.s);
    return nullptr;
}

// The copy through st's slots (its lock held), st.ready for it.
static hipError_t copy_staged(Staging& st, char* to, const char* from, size_t bytes) {
    if (bytes < kCopyLarge) return copy_range(st.small, to, from, bytes, st.stream);
    int dev = 0;
    const hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const size_t share = ((bytes + kLargeChunk - 1) / kLargeChunk + kCopyWorkers - 1) / kCopyWorkers * kLargeChunk;
    CopyShare part[kCopyWorkers];
    pthread_t helper[kCopyWorkers];
    bool runs[kCopyWorkers] = {};
    for (int i = 0; i < kCopyWorkers; ++i) {
        const size_t b = std::min(bytes, (size_t)i * share), end = std::min(bytes, b + share);
        part[i] = CopyShare{&st.large[i], to + b, from + b, end - b, st.stream, dev, hipSuccess};
        if (i) runs[i] = pthread_create(&helper[i], nullptr, copy_share, &part[i]) == 0;
    }
    // this thread takes the first share, and those for which no thread was to be had
    for (int i = 0; i < kCopyWorkers; ++i)
        if (!runs[i]) (void)copy_share(&part[i]);
    for (int i = 0; i < kCopyWorkers; ++i)
        if (runs[i]) (void)pthread_join(helper[i], nullptr);
    for (const CopyShare& p : part)
        if (p.err != hipSuccess) return p.err;
    return hipSuccess;
}

int copy_to_host(Staging& st, void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (bytes >= kCopyDirect) {
        GLP_HIP(hipStreamSynchronize(s));  // (the copies are not on s)
        std::lock_guard<std::mutex> lock(st.mu);
        const bool staged = (st.used || bytes >= kCopyLarge) && st.ready(bytes);
        st.used = true;
        if (staged) {
            const hipError_t e = copy_staged(st, static_cast<char*>(dst), static_cast<const char*>(src), bytes);
            return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "copying results: %s", hipGetErrorString(e));
        }
    }
    if (bytes == 0) return GLP_OK;
    GLP_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
    GLP_HIP(hipStreamSynchronize(s));
    return GLP_OK;
}

}  // namespace glp
