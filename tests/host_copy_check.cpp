// pp_hostcopy.hip on the host, through hip_stub/hip/hip_runtime.h: what each call of copy_to_host returns and
// copies with the stream, the source, the ring and the caller on one device or on two, and when a launch
// fails on the way.  Prints a line for each case; returns the number of wrong ones.
#include <cstdio>
#include <vector>

#include "../pittpack_amd/csrc/pp_hostcopy.hip"

static int wrong = 0;

static void copy(const char *name, pp::HostRing &ring, std::vector<double> &src, int src_device, hipStream_t s, int current,
                 bool by_ring, int fail_at = -1)
{
    std::vector<double> dst(src.size(), -1.0);
    stub_array = (const char *)src.data();
    stub_array_bytes = src.size() * sizeof(double);
    stub_array_device = src_device;
    stub_kernels = stub_copies = 0;
    stub_fail_at = fail_at;
    stub_device = current;
    const hipError_t e = pp::copy_to_host(ring, dst.data(), src.data(), src.size(), s);
    const bool ring_used = stub_kernels > 0 && stub_copies == 0;
    const bool ok = e == hipSuccess && dst == src && ring_used == by_ring && stub_device == current;
    std::printf("%s: %s (error %d, %d kernels, %d plain copies)\n", name, ok ? "ok" : "WRONG", (int)e, stub_kernels.load(),
                stub_copies.load());
    wrong += !ok;
}

int main()
{
    StubStream s0{0}, s1{1};
    for (size_t n : {(size_t)1 << 19, ((size_t)1 << 19) + 1, ((size_t)9 << 17) + 12345}) {
        std::vector<double> src(n);
        for (size_t i = 0; i < n; i++) src[i] = (double)(i * 2654435761u % 1000003);
        pp::HostRing ring;
        copy("one device", ring, src, 0, &s0, 0, true);
        copy("null stream", ring, src, 0, nullptr, 0, true);
        copy("caller on another device", ring, src, 0, &s0, 1, false);
        copy("null stream, caller on another device", ring, src, 0, nullptr, 1, false);
        copy("stream of another device", ring, src, 0, &s1, 0, false);
        copy("ring of another device", ring, src, 1, &s1, 1, false);
        copy("a launch fails", ring, src, 0, &s0, 0, false, 3);
        copy("one device again", ring, src, 0, &s0, 0, true);
        pp::free_ring(ring);
        copy("all on the second device", ring, src, 1, &s1, 1, true);
        pp::free_ring(ring);
    }
    return wrong;
}
