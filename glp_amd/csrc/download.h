// Copies of results to the caller's memory (download.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <cstddef>
#include <mutex>

namespace glp {

// Pinned double buffers of one worker.
struct CopySlots {
    char* slot[2] = {nullptr, nullptr};
    hipEvent_t done[2] = {nullptr, nullptr};
    size_t chunk = 0;
    bool create(size_t chunk);  // false: no memory or events to be had
    ~CopySlots();
};

constexpr int kCopyWorkers = 4;
// The pinned buffers and the stream of copies, made when copies repeat and
// kept: a graph's, for all sessions on it, as long as its device copy or one
// of them is there, or a server's (1 MB, and 16 MB once its copies are large).
struct Staging {
    std::mutex mu;  // held by the copy that uses them
    hipStream_t stream = nullptr;
    CopySlots small, large[kCopyWorkers];
    bool used = false;  // a copy that could have used them was made
    bool ready(size_t bytes);  // makes what a copy of `bytes` needs; false: not to be had
    ~Staging();
};

// Copies `bytes` from the device to pageable host memory after the work
// queued on s; returns when they are there.  Where the buffers cannot be had
// the copy is a plain one.
int copy_to_host(Staging& st, void* dst, const void* src, size_t bytes, hipStream_t s);

}  // namespace glp
