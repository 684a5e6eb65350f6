// pp_hostcopy.h -- solutions to pageable host arrays, by several host threads.
//
// The runtime copies to pageable memory through one thread (16 MB: 1.0 ms, 1.5 ms where the array's
// pages are new) though the link takes 0.3 ms.  Here the device writes chunks to a ring of pinned memory
// and four threads (the caller and three helpers, gone on return) empty it: 0.47 and 0.61 ms.
// Measured per 16 MB: one thread 0.75, chunks of 256 KB 0.74, of 512 KB 0.52, of 1 MB 0.47, of
// 2 MB 0.51 ms; the copy engine instead of a kernel 0.61 (10 us a chunk between its copies).  The
// other direction stays with the runtime, which is as fast there (0.47 against 0.53 ms).
//
// No counterpart in the reference, whose arrays live on the device (src/pencilDcmp.cpp).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace pp {

constexpr int kCopyThreads = 4;

// one object's ring of pinned memory: each thread moves every kCopyThreads-th chunk through
// slots of its own, so threads share nothing but the stream's order
struct HostRing {
    static constexpr int kSlots = 2;
    static constexpr size_t kChunk = (size_t)1 << 20;
    char *buf = nullptr;
    int device = -1;  // of its events
    hipEvent_t ev[kCopyThreads * kSlots] = {};
    std::mutex in_use;
};
void free_ring(HostRing &r);

// dst (host) <- src (device, 16-byte aligned) on `s`, finished and the stream drained on return.
// Copies under kRingMin (2 MB: 0.11 against 0.12 ms, 4 MB: 0.19 against 0.24), registered host memory, the
// per-thread stream (another one on each helper), a ring that another thread is using, a stream, source or
// ring of another device than the caller's current one, and whatever fails on the way are the runtime's.
constexpr size_t kRingMin = (size_t)4 << 20;
hipError_t copy_to_host(HostRing &r, double *dst, const double *src, size_t count, hipStream_t s);

// host memory to host memory by a thread per 512 KB, four at most
void copy_by_threads(void *dst, const void *src, size_t bytes);

}  // namespace pp
