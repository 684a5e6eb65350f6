// pp_plane_mm.h -- both transforms of a small plane in one kernel, as dense products on the FP64
// matrix cores (pp_line_mm.h).
//
// A plane of at most 64 x 64 points fits a block's LDS, so the x and y transforms of a solve's
// forward half -- and of its inverse half -- need no trip through memory between them: three
// launches a solve instead of five and 48 bytes a point instead of 80.  A block's time is the
// latency of its phases one after the other (24 x 20: load and fold 1.2 us, x products 1.0, fold
// 0.6, y products and store 1.1, and 2 of launch): loads of the matrices before the data's, for
// both axes, took longer (the L1 passes 64 bytes a cycle: 2.2 us for 24 loads a wave).  Threads
// keep their folded position over the lines they stage: 560 and 480 vector instructions a wave
// where per-element positions took 708 and 806.
//
// Replaces, per plane, assignRhs / modifyRhsDirichlet (src/pencilDcmp.cpp:5591-5647, 4623-4835),
// the two SignalProc + FFT stages and the x <-> y plane transposes (2279-2515), rescale (3503-3531).
#pragma once
#include <hip/hip_runtime.h>

#include "pp_line_mm.h"

namespace pp {

// waves of a block: each has one job (16 outputs of 16 lines) an axis
constexpr int kPlaneWaves = 8;
inline int plane_jobs(int nx, int ny, int kx, int ky)
{
    const int jx = (ny + 15) / 16 * (mm_rows16(nx, mm_family(kx)) / 16);
    const int jy = (nx + 15) / 16 * (mm_rows16(ny, mm_family(ky)) / 16);
    return jx > jy ? jx : jy;
}
// (a single solve: at least four, to load the plane; a batch's other blocks do that)
inline int plane_waves(int nx, int ny, int kx, int ky)
{
    const int j = plane_jobs(nx, ny, kx, ky);
    return j < 4 ? 4 : j;
}

// Planes these kernels take (FP64 form), all members of a batch by the same rule as a single solve.
// Measured against the line kernels, a solve / a batch of hundreds of members (us):
//   DD, NN up to 32 points         20x20x16 14.4 : 22.9, 24x20x18 - / 185 : 198, 32x32x16 14.6 : 17.2 / 232 : 214
//   ND, DN up to 28 points         28x28x16 16.2 : 24.7, but 32x32x16 16.2 : 15.6, 32x16x100 - / 304 : 262
//   without a compiled plan        33x33x16 21.6 : 24.6, 63x63x63 26.8 : 29.4 / 366 : 596
//   not: periodic, compiled        32x32x16 22.9 : 27.1 / 388 : 290 then, the lines since 192 (17 outputs pad to 32)
//   not: compiled past 32          48x48x48 - / 525 : 481 then, the lines since 320; 64x64x64 - / 501 : 465
//   not: planes of < 96 points     8x8x32 20 : 22 / 358 : 238, but 10x12x16 - / 189 : 229
// A batch fills the chip, so there the products' padding counts; a single solve does not.
constexpr int kPlaneMax = 64;
inline bool plane_axis(int n, int kind)
{
    const int fam = mm_family(kind);
    return n <= kPlaneMax && (!line_compiled(n) || n <= (fam == 0 ? 32 : fam == 1 ? 28 : 0));
}
inline bool mm_plane(int nx, int ny, int kx, int ky)
{
    return plane_axis(nx, kx) && plane_axis(ny, ky) && nx * ny >= 96 && plane_jobs(nx, ny, kx, ky) <= kPlaneWaves;
}

// doubles of LDS for a plane: region A holds one axis' folded rows, region B the plane between the
// axes, then the x forward's per-line Dirichlet constants
__host__ __device__ inline int plane_cs(int nx)
{
    const int c16 = (nx + 15) / 16 * 16;
    return c16 % 32 == 0 ? c16 + 16 : c16;  // two depth rows of 16 columns on different banks
}
__host__ __device__ inline int plane_a(int nx, int ny, int famx, int famy)
{
    const int ax = (ny + 15) / 16 * 16 * mm_xstride(nx, famx);
    const int ay = mm_parts(famy) * mm_depth8(ny, famy) * plane_cs(nx);
    return ax > ay ? ax : ay;
}
__host__ __device__ inline int plane_sb(int nx) { return nx | 1; }
inline size_t plane_lds(int nx, int ny, int kx, int ky)
{
    return (size_t)(plane_a(nx, ny, mm_family(kx), mm_family(ky)) + ny * plane_sb(nx) + 3 * ny) * sizeof(double);
}

// batched: a member's kinds and matrices per axis
struct PlaneSolve {
    int kind[2];
    const double *mm[2], *mmi[2];
};

// forward: ax.in (right-hand side) -> ay.out (z tiles or field); inverse: ay.in -> ax.out.  ax and ay
// are the arguments the two line launches would take (mm / mmi set); batched: ax.items = {solve, z}
// over ax.solves and ps, lds the largest member's, waves (a power of two) no fewer than any has jobs
hipError_t launch_plane_mm(int fwd, int kx, int ky, const LineArgs &ax, const LineArgs &ay, size_t lds, hipStream_t s,
                           const PlaneSolve *ps = nullptr, int waves = 0);

}  // namespace pp
