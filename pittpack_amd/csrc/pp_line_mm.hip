// pp_line_mm.hip -- the matrices of the dense-product line transforms (pp_line_mm.h), written on
// the device from one octant of cosines: N / 2 x N / 2 values a half are 1 MB at N = 512, so only
// 2 (N + 1) doubles cross the bus.  Angles are reduced exactly in integers.
#include "pp_line_mm.h"

namespace pp {

// one direction's matrices [e, o] x [depth][row] of length N, zero where padded
__global__ void k_mm_table(double *out, const double *oct, int N, int fam, int fwd)
{
    const int D8 = mm_depth8(N, fam), R16 = mm_rows16(N, fam), H = mm_depth(N, fam), K = mm_rows(N, fam);
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 2L * D8 * R16) return;
    const int part = (int)(t / ((long)D8 * R16));
    const int rem = (int)(t - (long)part * D8 * R16);
    const int j = rem / R16, k = rem - j * R16;
    double v = 0.0;
    if (j < H && k < K) {
        if (fam == 0) {
            // cos(pi mode (2 n + 1) / (2 N)): forward sums over n into modes 2 k + part, inverse
            // over modes 2 j + part into n
            const int mode = 2 * (fwd ? k : j) + part, n = fwd ? j : k;
            if (mode < N) v = mm_cos8(oct, N, 2L * mode * (2 * n + 1));
        } else if (fam == 1) {
            // cos(pi (2 j + 1) (2 k + 1) / (4 N)), outputs k and K + k
            const int row = k + part * K;
            if (row < N) v = mm_cos8(oct, N, (2L * j + 1) * (2 * row + 1));
        } else {
            // cos / sin(2 pi j k / N)
            v = mm_cos8(oct, N, 8L * j * k + (part ? 6L * N : 0));
        }
    }
    out[t] = v;
}

hipError_t launch_mm_tables(double *out, const double *oct, int N, int kind, hipStream_t s)
{
    const int fam = mm_family(kind);
    const size_t n = mm_table_size(N, fam);
    for (int inv = 0; inv <= (fam == 0 ? 1 : 0); inv++) {
        hipLaunchKernelGGL(k_mm_table, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, out + inv * n, oct, N, fam, !inv);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace pp
