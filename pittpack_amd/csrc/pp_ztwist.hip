// pp_ztwist.hip -- FP64 z solve of columns of up to 128 rows: Thomas from both ends of a column at once.
//
// Splitting a short column over 16 lanes (k_zsolve) is more arithmetic than its transfer: the PCR steps
// and the explicit end rows are some 170 instructions a row at 64 rows, where the sweeps themselves take
// fewer than 20.  Here two lanes of a wave, 32 apart, eliminate one column, one from row 0 downward and one
// from row n - 1 upward, up to the middle, where
//   x_T = dT + rT x_B,  x_B = dB + rB x_T   =>   x_T = (dT + rT dB) / (1 - rT rB)
// and both substitute back outward: Thomas' operations, half as long a chain, one exchange
// between lanes.  The pivots are kept as w = 1 - r, with s = eig + 2 <= 0:
//   t = w - s,  r = 1 / (1 + t),  w' = t r   (w = 0 at a Neumann end, 2 at a Dirichlet end)
// where nothing cancels, and 1 - rT rB = wT + wB - wT wB.  Nearly singular columns need no other
// sweeps, then: at 64 rows and |eig + 2| = 0.001 the error is 6e-16 of the column's largest value, where
// Thomas' sweeps lose 1e-14 and the PCR steps 4e-14 (0.5: 2.0, 2.2 and 3.2e-16; the pinned column
// 5e-16 like the PCR steps; 80-bit sweeps on random columns).  A wave takes the 32 columns of two tiles, row by row in 128-byte segments,
// the whole column in flight at once; no staging in LDS.
//
// Bound by memory on large grids, on small ones by the launch and by fetching the unrolled code (a chain of
// pivots half as long, two rows a step, was no faster).  z stage, us, before and now:
// 512x512x16 37.5 15.0, 512x512x64 104 44.6, 512x512x128 137 89.5 (96 at 5.6 TB/s), 1024x1024x32 214 82.0,
// 256x256x128 42.7 29.8, 128x128x64 12.7 8.2 (nearly singular columns included); 1000 solves of
// 24x20x18 in a batch 144 30.
//
// Replaces solveThmBatch (src/pencilDcmp.cpp:5062-5234, src/triDiag.cpp:1629-1822) like k_zsolve.
#include <utility>

#include "pp_launch.h"
#include "pp_zsolve.h"

namespace pp {

namespace {

// K = ceil(nz / 16): at most H = 8 K rows a lane, at least 8 K - 8.  Thomas factors stay in registers
// up to 32 rows, beyond in LDS (32 KB a wave at 64 rows)
template <int K, bool TILED>
__global__ void __launch_bounds__(64) k_ztwist(ZArgs a0)
{
    constexpr int H = 8 * K;
    constexpr bool CP_LDS = H > 32;
    ZArgs a = a0;
    const bool down = !a0.items && ztwist_by_column(a0.SX, a0.SY, a0.nz);
    int bx = down ? blockIdx.y : blockIdx.x, pair = down ? blockIdx.x : blockIdx.y;
    if (a0.items) {
        const ZItem it = a0.items[bx];
        const ZSolve sv = a0.solves[it.solve];
        a.data = reinterpret_cast<double *>(a0.data) + sv.offset;
        a.SX = sv.SX;
        a.SY = sv.SY;
        a.nz = sv.nz;
        a.zlo_dirichlet = sv.zlo_dirichlet;
        a.zhi_dirichlet = sv.zhi_dirichlet;
        a.Cx = sv.Cx;
        a.Cy = sv.Cy;
        a.lamx = sv.lamx;
        a.lamy = sv.lamy;
        bx = it.bx;
        pair = it.by;
    }
    const int n = a.nz, half = (n + 1) / 2;
    const int lane = threadIdx.x, c = lane & 15;
    const bool up = lane >= 32;  // from the last row
    // y lines 2 pair and 2 pair + 1 of tile column bx
    const bool second = lane & 16;
    const bool one = 2 * pair + 1 >= a.SY;
    const int sy = 2 * pair + (second && !one ? 1 : 0);
    int sx = bx * 16 + c;
    const bool store = sx < a.SX && !(second && one);
    if (sx >= a.SX) sx = a.SX - 1;

    // eigenvalue of this (kx, ky) column, src/pencilDcmp.cpp:4393-4417, without contraction
    const double eig = __dadd_rn(__dadd_rn(-2.0, __dmul_rn(a.lamx[sx], a.Cx)), __dmul_rn(a.lamy[sy], a.Cy));
    bool pin = fabs(eig + 2.) < 1.e-10;
    if (pin && a.zero_mode == 1 && (a.zlo_dirichlet || a.zhi_dirichlet)) pin = false;
    const double s = eig + 2.;

    // row j of this lane: j from its end
    const int rows = up ? n - half : half;
    double *data = reinterpret_cast<double *>(a.data);
    const int trows = a.tile_rows ? a.tile_rows : (n + 15) / 16 * 16;
    double *const tile = data + ((long)bx * a.SY + 2 * pair) * trows * 16;
    unsigned first = ((second && !one ? trows : 0) + (up ? n - 1 : 0)) * 16 + c, step = up ? -16 : 16;
    const long zs = (long)a.SX * a.SY;
    double *col = data + (long)sy * a.SX + sx + (up ? (n - 1) * zs : 0);
    const long cstep = up ? -zs : zs;
    auto at = [&](int j) -> double * {
        if constexpr (TILED) return tile + (first + (unsigned)j * step);
        else return col + j * cstep;
    };

    double d[H];
#pragma unroll
    for (int j = 0; j < H; j++) d[j] = *at(j < H - 8 ? j : min(j, rows - 1));  // past the middle: its last row again

    __shared__ double lds[CP_LDS ? 64 * H : 1];
    double rr[CP_LDS ? 1 : H];
    double w = (up ? a.zhi_dirichlet : a.zlo_dirichlet) ? 2.0 : 0.0, rprev, dprev;
    {
        // the pinned column's row 0 is x_0 = d_0
        const bool fixed = pin && !up;
        const double t = w - s, r = rcp_nr(1.0 + t);
        rprev = fixed ? 0.0 : r;
        w = fixed ? 1.0 : t * r;
        dprev = fixed ? d[0] : -d[0] * r;
        d[0] = dprev;
        if constexpr (CP_LDS) lds[lane] = rprev;
        else rr[0] = rprev;
    }
#pragma unroll
    for (int j = 1; j < H; j++) {
        const double t = w - s, r = rcp_nr(1.0 + t);
        const double dj = (dprev - d[j]) * r;
        const bool on = j < H - 8 || j < rows;
        w = on ? t * r : w;
        rprev = on ? r : rprev;
        dprev = on ? dj : dprev;
        d[j] = dprev;
        if constexpr (CP_LDS) {
            lds[64 * j + lane] = rprev;
            asm volatile("" : "+v"(d[j]));  // the update stays here, not in the backward sweep
        } else {
            rr[j] = rprev;
        }
    }
    // the middle (the rows' offsets are computed again for the stores, not held since the loads)
    asm volatile("" : "+v"(first), "+v"(col));
    const double wo = __shfl_xor(w, 32, 64), dO = __shfl_xor(dprev, 32, 64);
    double x = (dprev + rprev * dO) * rcp_nr(w + wo - w * wo);
#pragma unroll
    for (int j = H - 1; j >= 0; j--) {
        double rj;
        if constexpr (CP_LDS) rj = lds[64 * j + lane];
        else rj = rr[j];
        const double xj = d[j] + rj * x;
        if (j >= H - 9) x = j < rows - 1 ? xj : x;  // row rows - 1 is the middle's
        else x = xj;
        if (store && (j < H - 8 || j < rows)) *at(j) = x;
        if constexpr (CP_LDS) {
            if (j % 4 == 0) asm volatile("" : "+v"(x)::"memory");  // factors loaded a few rows ahead only
        }
    }
}

template <int K>
hipError_t launch_k(const ZArgs &a, hipStream_t s)
{
    dim3 grid((unsigned)((a.SX + 15) / 16), (unsigned)((a.SY + 1) / 2));
    if (a.items) grid = dim3((unsigned)a.nitems);
    if (!a.items && ztwist_by_column(a.SX, a.SY, a.nz)) std::swap(grid.x, grid.y);
    if (a.tiled) hipLaunchKernelGGL((k_ztwist<K, true>), grid, dim3(64), 0, s, a);
    else hipLaunchKernelGGL((k_ztwist<K, false>), grid, dim3(64), 0, s, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_ztwist(int nz, const ZArgs &a, hipStream_t s)
{
    if (nz < 4 || nz > 128 || a.pinned_zero || (a.tiled && a.tile_w != 16)) return hipErrorInvalidValue;
    switch ((nz + 15) / 16) {
    case 1: return launch_k<1>(a, s);
    case 2: return launch_k<2>(a, s);
    case 3: return launch_k<3>(a, s);
    case 4: return launch_k<4>(a, s);
    case 5: return launch_k<5>(a, s);
    case 6: return launch_k<6>(a, s);
    case 7: return launch_k<7>(a, s);
    default: return launch_k<8>(a, s);
    }
}

}  // namespace pp
