// pp_hostcopy.hip -- host copies by several threads (pp_hostcopy.h).
#include "pp_hostcopy.h"

#include <algorithm>
#include <cstring>
#include <thread>

namespace pp {

namespace {

// device -> mapped pinned memory; bound by the link (128 blocks write 55 GB/s)
__global__ void __launch_bounds__(256) k_to_host(double *__restrict__ out, const double *__restrict__ in, long n)
{
    const long n2 = n / 2;
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n2; i += gridDim.x * 256L)
        reinterpret_cast<double2 *>(out)[i] = reinterpret_cast<const double2 *>(in)[i];
    if (n % 2 && blockIdx.x == 0 && threadIdx.x == 0) out[n - 1] = in[n - 1];
}

bool ring_ready(HostRing &r, int device)
{
    if (r.buf) return r.device == device;
    const int n = kCopyThreads * HostRing::kSlots;
    if (hipHostMalloc((void **)&r.buf, n * HostRing::kChunk, hipHostMallocDefault) != hipSuccess) {
        r.buf = nullptr;
        (void)hipGetLastError();
        return false;
    }
    for (int i = 0; i < n; i++)
        if (hipEventCreateWithFlags(&r.ev[i], hipEventDisableTiming) != hipSuccess) {
            r.ev[i] = nullptr;
            (void)hipGetLastError();
            free_ring(r);
            return false;
        }
    r.device = device;
    return true;
}

// kernels and events of one device serve its own streams alone: the current device, if the stream and the
// source are its own too, else -1
int one_device(const double *src, hipStream_t s)
{
    int device = 0;
    hipDevice_t of_stream = 0;
    hipPointerAttribute_t a{};
    bool ok = hipGetDevice(&device) == hipSuccess && hipPointerGetAttributes(&a, src) == hipSuccess && a.device == device;
    if (ok && s) ok = hipStreamGetDevice(s, &of_stream) == hipSuccess && of_stream == device;
    if (!ok) (void)hipGetLastError();
    return ok ? device : -1;
}

// memory the device reaches by itself
bool registered(const void *p)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

// run(0) here and run(1) .. run(n - 1) on threads of their own (here too where there are none to be had)
template <typename F>
void on_threads(int n, const F &run)
{
    std::thread t[kCopyThreads];
    int started = 1;
    try {
        for (; started < n; started++) t[started] = std::thread([&run, w = started] { run(w); });
    } catch (...) {
    }
    run(0);
    for (int w = started; w < n; w++) run(w);
    for (int w = 1; w < started; w++) t[w].join();
}

// chunks w, w + kCopyThreads, ... of the copy
hipError_t empty_chunks(const HostRing &r, int w, double *dst, const double *src, size_t count, hipStream_t s)
{
    constexpr int W = kCopyThreads, S = HostRing::kSlots;
    constexpr size_t C = HostRing::kChunk / sizeof(double);
    const long chunks = (long)((count + C - 1) / C);
    const long mine = w < chunks ? (chunks - w + W - 1) / W : 0;
    auto at = [&](long k) { return (size_t)(w + k * W) * C; };
    auto len = [&](long k) { return std::min(C, count - at(k)); };
    auto slot = [&](long k) { return reinterpret_cast<double *>(r.buf) + (size_t)(w * S + k % S) * C; };
    auto fill = [&](long k) {
        hipLaunchKernelGGL(k_to_host, dim3(128), dim3(256), 0, s, slot(k), src + at(k), (long)len(k));
        const hipError_t e = hipGetLastError();
        return e != hipSuccess ? e : hipEventRecord(r.ev[w * S + k % S], s);
    };
    hipError_t e = hipSuccess;
    for (long k = 0; k < std::min<long>(S, mine) && e == hipSuccess; k++) e = fill(k);
    for (long k = 0; k < mine && e == hipSuccess; k++) {
        if ((e = hipEventSynchronize(r.ev[w * S + k % S])) != hipSuccess) break;
        std::memcpy(dst + at(k), slot(k), len(k) * sizeof(double));
        if (k + S < mine) e = fill(k + S);
    }
    return e;
}

}  // namespace

void free_ring(HostRing &r)
{
    for (hipEvent_t &e : r.ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (r.buf) (void)hipHostFree(r.buf);
    r.buf = nullptr;
}

hipError_t copy_to_host(HostRing &r, double *dst, const double *src, size_t count, hipStream_t s)
{
    const size_t bytes = count * sizeof(double);
    auto plain = [&] {
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipStreamSynchronize(s);
    };
    int device = -1;
    std::unique_lock<std::mutex> lk(r.in_use, std::try_to_lock);
    if (!lk.owns_lock() || bytes < kRingMin || s == hipStreamPerThread || registered(dst) ||
        (device = one_device(src, s)) < 0 || !ring_ready(r, device))
        return plain();
    hipError_t err[kCopyThreads];
    on_threads(kCopyThreads, [&](int w) {
        err[w] = hipSetDevice(device);
        if (err[w] == hipSuccess) err[w] = empty_chunks(r, w, dst, src, count, s);
    });
    // also after an error: nothing may be in flight in the ring when it is used again
    hipError_t e = hipStreamSynchronize(s);
    for (hipError_t w : err)
        if (w != hipSuccess) e = w;
    if (e == hipSuccess) return e;
    (void)hipGetLastError();
    return plain();
}

void copy_by_threads(void *dst, const void *src, size_t bytes)
{
    const int n = (int)std::clamp<size_t>(bytes >> 19, 1, kCopyThreads);
    const size_t part = (bytes / n + 4095) / 4096 * 4096;
    on_threads(n, [&](int w) {
        const size_t a = std::min(bytes, w * part), b = w == n - 1 ? bytes : std::min(bytes, a + part);
        if (b > a) std::memcpy((char *)dst + a, (const char *)src + a, b - a);
    });
}

}  // namespace pp
