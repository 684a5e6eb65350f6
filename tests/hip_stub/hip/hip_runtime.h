// The few names of the HIP runtime that pp_hostcopy.hip uses, on the host and with two devices: kernels
// and events of one device fail on a stream of another, as they do on a machine with several GPUs, where a
// plain copy goes through.  For tests/host_copy_check.cpp alone.
#pragma once
#include <atomic>
#include <cstddef>
#include <cstdlib>
#include <cstring>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorInvalidHandle = 400 };
struct StubStream {
    int device;
};
typedef StubStream *hipStream_t;
struct StubEvent {
    int device;
};
typedef StubEvent *hipEvent_t;
typedef int hipDevice_t;
struct dim3 {
    unsigned x, y, z;
    dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
struct double2 {
    double x, y;
};
enum { hipMemcpyDeviceToHost = 2, hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeDevice = 2 };
struct hipPointerAttribute_t {
    hipMemoryType type;
    int device;
};
#define __global__
#define __launch_bounds__(...)
#define hipStreamPerThread (reinterpret_cast<hipStream_t>(2))

inline thread_local int stub_device = 0;
inline thread_local dim3 blockIdx, threadIdx, gridDim;
inline std::atomic<int> stub_kernels{0}, stub_copies{0}, stub_fail_at{-1};
// the one device array of the test and its device
inline const char *stub_array = nullptr;
inline size_t stub_array_bytes = 0;
inline int stub_array_device = 0;

inline hipError_t hipGetDevice(int *d) { return *d = stub_device, hipSuccess; }
inline hipError_t hipSetDevice(int d) { return stub_device = d, hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) { return *d = s ? s->device : stub_device, hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return (*p = std::malloc(n)) ? hipSuccess : hipErrorInvalidValue; }
inline hipError_t hipHostFree(void *p) { return std::free(p), hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = new StubEvent{stub_device}, hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    return e->device == (s ? s->device : stub_device) ? hipSuccess : hipErrorInvalidHandle;
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    const char *c = (const char *)p;
    const bool dev = c >= stub_array && c < stub_array + stub_array_bytes;
    a->type = dev ? hipMemoryTypeDevice : hipMemoryTypeUnregistered;
    a->device = dev ? stub_array_device : 0;
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t)
{
    stub_copies++;
    std::memcpy(d, s, n);
    return hipSuccess;
}

// a launch's result is what hipGetLastError says next
inline thread_local hipError_t stub_launch = hipSuccess;
inline hipError_t hipGetLastError()
{
    const hipError_t e = stub_launch;
    stub_launch = hipSuccess;
    return e;
}
template <typename K, typename... A>
void hipLaunchKernelGGL(K kernel, dim3 grid, dim3 block, size_t, hipStream_t s, A... args)
{
    const int at = stub_kernels++;
    if ((s && s->device != stub_device) || at == stub_fail_at) {
        stub_launch = hipErrorInvalidHandle;
        return;
    }
    gridDim = grid;
    for (blockIdx.x = 0; blockIdx.x < grid.x; blockIdx.x++)
        for (threadIdx.x = 0; threadIdx.x < block.x; threadIdx.x++) kernel(args...);
}
