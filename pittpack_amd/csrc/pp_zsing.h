// pp_zsing.h -- the singular z column (eigenvalue sum exactly -2, so the interior rows are
// 1 -2 1) by one wave.
//
// The reference runs Thomas sweeps on it (thomasLowMemNoBCV1, src/triDiag.cpp:1629-1687, and
// shermanMorrisonThomasV1, 2112-2255 for periodic z): nz dependent divisions, 82 us of a 342 us
// 256^3 solve when one thread runs them.  Its second differences integrate instead: with
// d_j = x_j - x_{j-1}, row j says d_{j+1} - d_j = r_j, so d is a suffix sum of r and x a prefix sum
// of d, each a scan over 64 lanes of up to 16 rows (256^3 PPPPPP 342 -> 265 us).
#pragma once
#include <hip/hip_runtime.h>

namespace pp {

// rows j = 1 .. n-2: x_{j-1} - 2 x_j + x_{j+1} = r_j; last: x_{n-2} + bn x_{n-1} = r_{n-1}; x_0 given.
// r (LDS, n values, n >= 3) is overwritten with x.  One whole wave calls it.
__device__ __forceinline__ void singular_column(double *r, int n, double x0, double bn, int lane)
{
    const int C = (n + 63) / 64, j0 = lane * C, j1 = min(j0 + C, n - 1);  // rows j0 .. j1 - 1 (below n - 1)
    const double rl = r[n - 1];
    // S_j = r_j + ... + r_{n-2}
    double t = 0.0;
    for (int j = max(j0, 1); j < j1; j++) t += r[j];
    double run = t;  // sum over this lane's rows and all later ones
    for (int s = 1; s < 64; s <<= 1) {
        const double u = __shfl_down(run, s, 64);
        if (lane + s < 64) run += u;
    }
    const double tail = __shfl_down(run, 1, 64);
    run = lane < 63 ? tail : 0.0;  // the lanes after this one
    double sum = 0.0;
    for (int j = j1 - 1; j >= max(j0, 1); j--) {
        run += r[j];
        r[j] = run;
        sum += run;
    }
    double total = sum;
    for (int s = 32; s > 0; s >>= 1) total += __shfl_xor(total, s, 64);
    // d_j = D - S_j with D = d_{n-1} from the last row
    const double g = 1.0 + bn;
    const double D = (rl - g * (x0 - total)) / (g * (double)(n - 1) - 1.0);
    // x_j = x_0 + d_1 + ... + d_j
    const int e1 = min(j0 + C, n);
    t = 0.0;
    for (int j = max(j0, 1); j < e1; j++) t += j < n - 1 ? D - r[j] : D;
    double pre = t;
    for (int s = 1; s < 64; s <<= 1) {
        const double u = __shfl_up(pre, s, 64);
        if (lane >= s) pre += u;
    }
    pre = __shfl_up(pre, 1, 64);
    double x = x0 + (lane > 0 ? pre : 0.0);
    for (int j = max(j0, 1); j < e1; j++) {
        x += j < n - 1 ? D - r[j] : D;
        r[j] = x;
    }
    if (lane == 0) r[0] = x0;
}

// The periodic column as the reference solves it (row 0 replaced by x_0 + x_{n-1} = target): T y = r
// with row 0 alone (2 y_0 = target) and last row x_{n-2} - x_{n-1}, then Sherman-Morrison with
// T^-1 (-1, 0 .. 0, 1) = -1/2 - j.
__device__ __forceinline__ void singular_periodic_column(double *r, int n, double target, int lane)
{
    singular_column(r, n, 0.5 * target, -1.0, lane);
    __builtin_amdgcn_wave_barrier();
    const double fact = (r[0] - r[n - 1]) / (double)n;
    __builtin_amdgcn_wave_barrier();
    for (int j = lane; j < n; j += 64) r[j] += fact * (0.5 + (double)j);
}

}  // namespace pp
