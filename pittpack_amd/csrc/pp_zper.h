// pp_zper.h -- lengths and block shapes of the one-pass periodic z solve (pp_zperiodic.hip).
#pragma once
#include "pp_line.h"

namespace pp {

// The half lengths M = nz / 2: the line transforms' and, whole in one thread's registers, 5 and 7
// (columns of 10 and 14 points, us a whole solve, one pass : z-line transforms: 512x512x10 77.7 : 148,
// 512x512x14 83.7 : 139, 64x64x10 21.1 : 27.7; 200 members of 24x24x10 in a batch, whose z-line transforms are
// three launches of each member's own, 50.9 : 1687)
#define PP_ZPER_LENGTHS(X) X(5) X(7) PP_FFT_LENGTHS(X)

// Threads a column: the line transforms' FP64 shape along y.  Columns per block: 16 (128-byte FP64 rows) while the
// slices fit 80 KB, 8 for longer lines, as the y transforms on the field in place, and no fewer than fill a
// wave: a quarter or half of one per block (16 columns of one or two threads) was slower than full-length
// complex lines (z stage, us, with those / quarter or half waves / now: 512x512x16 24.5 38.7 16.6, 787x192x20
// 31.9 32.9 17.6, 20x240x16 6.9 9.4 6.6, 512x512x48 66 61 39, 512x512x80 138 130 71)
constexpr int zper_threads(int M) { return M == 5 || M == 7 ? 1 : line_wide(M, 1) ? line_threads_alt(M) : line_threads(M, 1); }
template <int M>
constexpr int zper_lines_m()
{
    constexpr int T = zper_threads(M), L = line_lines<double, M, 1, T>();
    return T >= 64 && L > 8 ? 8 : T < 4 ? 64 / T : L;
}

// LDS slots of a column: an odd number, so that the 16 columns of a wave's access start on different banks (z stage,
// us, with the line transforms' number / odd: 112 elements, whose 120 slots start on two, 512x512x224 582 323 and
// 20x240x224 32.9 22.4, where full-length lines took 584 and 25.2; 56 elements, 60 slots, 512x512x112 138 109)
template <int M>
constexpr int zper_slots() { return line_slots<M>() | 1; }

}  // namespace pp
