// pp_zperiodic.hip -- z solve for periodic z faces.
//
// The reference solves each (kx, ky) column's cyclic tridiagonal system (diagonal eig, unit
// off-diagonals, wrap-around corners) by Sherman-Morrison on top of two Thomas sweeps
// (shermanMorrisonThomas, src/triDiag.cpp:1961-2108).  That system is circulant, so here a
// block diagonalises it exactly instead: real FFT of the column along z, division of mode
// k by eig + 2 cos(2 pi k / nz), inverse FFT -- one read and one write of the column, with the
// Stockham passes of the line transforms (pp_fft.h) running on z-columns.
//
// The singular column (|eig + 2| < 1e-10: x and y in {P, N}, mode (0, 0)) follows the
// reference's own branch (shermanMorrisonThomasV1, src/triDiag.cpp:2112-2255: first row
// replaced by the average of the first and last right-hand sides, pinned Thomas sweeps and
// the Sherman-Morrison correction), in FP64 by k_smt_v1.  The mixed form
// solves that column from FP64 plane sums instead (k_mode00, pp_mixed.hip) and has it
// written as zeros here.
//
// Lengths without a plan (PP_ZPER_LENGTHS) take three passes instead of one: real z-line
// transforms of any length (the line kernels) around a division kernel (k_zper_divide).
//
// Storage is FP64 (FP64 form) or FP32 (the mixed form's work field); the arithmetic of the
// one-pass kernel and of the division is FP64 in both.  Batched launches take one block per
// item (solve, column block, y row) over the solves' descriptors.
#include <hip/hip_runtime.h>

#include "pp_fft.h"
#include "pp_launch.h"
#include "pp_line.h"
#include "pp_zper.h"
#include "pp_zsing.h"
#include "pp_zsolve.h"

namespace pp {

// ZPerArgs (pp_launch.h): data [nz][SY][SX] in place, nz = 2 M; tw = exp(-2 pi i e / M), e < M, and
// A = exp(-2 pi i k / nz), k <= M, interleaved; c2 = 2 cos(2 pi k / nz), k < nz.  S is the storage
// type: the FP64 form and the mixed form's FP32 work field both compute in FP64 (the transform and
// the division by the mode's eigenvalue), so near-singular columns need no separate treatment in
// either form.
//
// A real column is one complex line of half its length, z_m = x_2m + i x_2m+1, whose rows arrive and
// leave in the FFT's own register layout (no LDS scatter).  With Z its FFT, Zc = conj Z_{M-k},
// P = (Z_k + Zc) / 2, R = (Z_k - Zc) / 2, w = exp(-2 pi i k / nz) and s_k = 1 / (nz (eig + c2_k)),
// splitting Z into the column's spectrum, dividing and packing it again collapses to
//     Z'_k = (s_k + s_{M-k}) Z_k + i (s_k - s_{M-k}) (conj(w) P - w R),
// one mirrored LDS read between the two FFTs (256^3: 86 us with full-length complex lines -> 56 us).
// At least four waves per SIMD (128 registers) where a thread holds 8 elements
template <int M, int T, int LINES>
constexpr int zper_min_waves() { return M / T == 8 ? 4 : 2; }

template <typename S, int M, int T, int LINES>
__global__ void __launch_bounds__(T *LINES, (zper_min_waves<M, T, LINES>())) k_zper(ZPerArgs a)
{
    using R = double;
    constexpr int E = M / T;
    constexpr int LS = zper_slots<M>();
    extern __shared__ __align__(16) unsigned char smem_zp[];
    cpx<R> *lds = reinterpret_cast<cpx<R> *>(smem_zp);
    const int tid = threadIdx.x;
    const int l = tid % LINES, t = tid / LINES;
    cpx<R> *L = lds + l * LS;
    int bx = blockIdx.x, sy = blockIdx.y;
    S *data = reinterpret_cast<S *>(a.data);
    if (a.items) {
        // batched: this block's solve, its sizes and eigenvalue factors
        const ZItem it = a.items[blockIdx.x];
        const ZSolve sv = a.solves[it.solve];
        data += sv.offset;
        a.SX = sv.SX;
        a.SY = sv.SY;
        a.Cx = sv.Cx;
        a.Cy = sv.Cy;
        a.lamx = sv.lamx;
        a.lamy = sv.lamy;
        bx = it.bx;
        sy = it.by;
    }
    const int sx0 = bx * LINES + l;
    const bool valid = sx0 < a.SX;
    const int sx = valid ? sx0 : a.SX - 1;
    // row 2 (t + T m) + h of the lane's column: a block-uniform pointer per (m, h) and one 32-bit
    // byte offset per lane (2 T planes of at most 1024^2 doubles: below 2^31)
    const bool tiled = a.tile_rows > 0;
    const long stride = tiled ? 16 : (long)a.SX * a.SY;
    const int c0 = bx * LINES;
    S *const col0 = data + (tiled ? ((long)(c0 / 16) * a.SY + sy) * a.tile_rows * 16 + c0 % 16 : (long)sy * a.SX + c0);
    // (in place, columns past the grid read the last one; a tile's padding columns are its own)
    const unsigned lane_bytes = (unsigned)((2L * t * stride + (tiled ? l : sx - c0)) * (long)sizeof(S));
    auto at = [&](int m, int h) {
        return reinterpret_cast<S *>(reinterpret_cast<char *>(col0 + (2L * T * m + h) * stride) + lane_bytes);
    };

    cpx<R> v[E];
#pragma unroll
    for (int m = 0; m < E; m++) v[m] = {(R)*at(m, 0), (R)*at(m, 1)};
    FFTSeeds<R, M, T> fs;
    fs.load(t, a.tw);
    c64 w = ld64(a.A, t);
    const c64 wT = ld64(a.A, T);
    // eigenvalue of this (kx, ky) column, src/pencilDcmp.cpp:4393-4417, without contraction
    double eig = __dadd_rn(__dadd_rn(-2.0, __dmul_rn(a.lamx[sx], a.Cx)), __dmul_rn(a.lamy[sy], a.Cy));
    const bool singular = fabs(eig + 2.) < 1.e-10;

    line_fft<R, M, T, -1>(v, L, t, fs);
#pragma unroll
    for (int m = 0; m < E; m++) L[padc(t + T * m)] = v[m];
    __syncthreads();
    // (the factors of a mode are formed where they are used: hoisted above the FFT, which the
    // compiler does for all modes at once unless held back, they cost a wave per SIMD)
    int kt = t;
    asm volatile("" : "+v"(eig), "+v"(kt));
#pragma unroll
    for (int m = 0; m < E; m++) {
        const int k = kt + T * m;
        const cpx<R> Zk = v[m], Zc = c_conj(L[padc(k == 0 ? 0 : M - k)]);
        const cpx<R> wk = to_c<R>(w);
        w = m64(w, wT);
        const double c2 = a.c2[k];  // mode M - k has -c2
        const double s0 = singular ? 0.0 : rcp_nr((eig + c2) * (double)(2 * M));
        const double s1 = singular ? 0.0 : rcp_nr((eig - c2) * (double)(2 * M));
        const cpx<R> P = c_scale(c_add(Zk, Zc), 0.5), Q = c_scale(c_sub(Zk, Zc), 0.5);
        const cpx<R> q = c_scale(c_sub(c_mulc(P, wk), c_mul(Q, wk)), s0 - s1);
        v[m] = {(s0 + s1) * Zk.x - q.y, (s0 + s1) * Zk.y + q.x};
        if (m % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    line_fft<R, M, T, +1>(v, L, t, fs);
    // the singular column: zeros (pinned_zero, v is zero) or left for k_smt_v1
    if (valid && (!singular || a.pinned_zero)) {
#pragma unroll
        for (int m = 0; m < E; m++) {
            *at(m, 0) = (S)v[m].x;
            *at(m, 1) = (S)v[m].y;
        }
    }
}

// the reference's singular periodic branch on one column, FP64: by scans where the
// diagonal is exactly -2 (mode (0, 0) of periodic and Neumann axes); a diagonal only within 1e-10 of
// it (cells 1e5 times thinner in z) takes the reference's sweeps, whose factors carry it
__device__ void smt_v1_body(double *data, long stride, int nz, double diag)
{
    extern __shared__ double sv[];
    double *rh = sv, *rh1 = sv + nz, *tmp = sv + 2 * nz;
    for (int i = threadIdx.x; i < nz; i += blockDim.x) rh[i] = data[i * stride];
    __syncthreads();
    if (diag == -2.0 && nz >= 3) {
        if (threadIdx.x < 64) singular_periodic_column(rh, nz, (rh[0] + rh[nz - 1]) * 0.5, threadIdx.x);
    } else if (threadIdx.x == 0) {
        const int N = nz;
        const double alpha = 1.0, beta = 1.0;
        // shermanMorrisonThomasV1 with b = {1, diag, diag}
        const double b0 = 1.0;
        const double gamma = -b0;
        const double bb[3] = {b0 - gamma, diag, diag - alpha * beta / gamma};
        // thomasLowMemNoBCV1 (src/triDiag.cpp:1629-1687): row 0 decoupled
        auto sweep = [&](double *r) {
            double bet;
            r[0] = r[0] / (bet = bb[0]);
            int j = 1;
            tmp[j] = 0.0;
            bet = bb[1] - tmp[j];
            r[1] = (r[1] - r[j - 1]) / bet;
            for (j = 2; j < N - 1; j++) {
                tmp[j] = 1.0 / bet;
                bet = bb[1] - tmp[j];
                r[j] = (r[j] - r[j - 1]) / bet;
            }
            j = N - 1;
            tmp[j] = 1.0 / bet;
            bet = bb[2] - tmp[j];
            r[j] = (r[j] - r[j - 1]) / bet;
            for (j = N - 2; j >= 0; j--) r[j] -= tmp[j + 1] * r[j + 1];
        };
        rh[0] = (rh[0] + rh[N - 1]) * 0.5;
        sweep(rh);
        rh1[0] = gamma;
        rh1[N - 1] = alpha;
        for (int i = 1; i < N - 1; i++) rh1[i] = 0.0;
        sweep(rh1);
        const double part1 = (rh[0] + beta * rh[N - 1] / gamma);
        const double part2 = (1. + rh1[0] + beta * rh1[N - 1] / gamma);
        const double fact = part1 / part2;
        for (int i = 0; i < N; i++) rh[i] -= fact * rh1[i];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nz; i += blockDim.x) data[i * stride] = rh[i];
}

__global__ void k_smt_v1(double *data, SmtItem it) { smt_v1_body(data + it.offset, it.stride, it.nz, it.diag); }

// batched: block b solves the singular column of items[b]
__global__ void k_smt_v1_batch(double *data, const SmtItem *items)
{
    const SmtItem it = items[blockIdx.x];
    smt_v1_body(data + it.offset, it.stride, it.nz, it.diag);
}

// grid: column blocks x SY (one solve), or nitems blocks (batched, a.items set)
template <typename S, int M>
static hipError_t launch_zper_m(const ZPerArgs &a, int nitems, hipStream_t s)
{
    constexpr int T = zper_threads(M);
    constexpr int LINES = zper_lines_m<M>();
    const size_t lds = (size_t)LINES * zper_slots<M>() * sizeof(cpx<double>);
    auto kern = k_zper<S, M, T, LINES>;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const dim3 grid = a.items ? dim3((unsigned)nitems) : dim3((unsigned)((a.SX + LINES - 1) / LINES), (unsigned)a.SY);
    if (a.items && nitems == 0) return hipSuccess;
    hipLaunchKernelGGL(kern, grid, dim3(T * LINES), lds, s, a);
    return hipGetLastError();
}

bool zperiodic_supported(int nz) { return nz >= 8 && nz % 2 == 0 && zper_threads(nz / 2) > 0; }

int zper_lines(int nz)
{
    switch (zperiodic_supported(nz) ? nz / 2 : 0) {
#define PPM(m) \
    case m: return zper_lines_m<m>();
        PP_ZPER_LENGTHS(PPM)
#undef PPM
    default: return 0;
    }
}

// Periodic z of any other length: the field's z lines go through the real line transforms
// (R2HC forward, HC2R inverse, pp_line.h / pp_line_bs.h, launched by the host on the
// [nz][SY*SX] view) and this kernel divides half-complex entry p of column (sx, sy) by
// nz * (eig + 2 cos(2 pi p / nz)) -- modes k and nz - k share the factor, so the real and
// imaginary parts of a mode divide alike.  The singular column only takes 1 / nz, so the
// inverse transform restores its right-hand side for the reference's branch (k_smt_v1), or
// is zeroed (pinned_zero).
template <typename S>
__global__ void k_zper_divide(ZPerArgs a)
{
    const long plane = (long)a.SX * a.SY;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= plane * a.nz) return;
    const int p = (int)(i / plane);
    const long c = i - (long)p * plane;
    const int sy = (int)(c / a.SX), sx = (int)(c - (long)sy * a.SX);
    const double eig = __dadd_rn(__dadd_rn(-2.0, __dmul_rn(a.lamx[sx], a.Cx)), __dmul_rn(a.lamy[sy], a.Cy));
    const bool singular = fabs(eig + 2.) < 1.e-10;
    const double den = singular ? (double)a.nz : (eig + a.c2[p]) * (double)a.nz;
    S *data = reinterpret_cast<S *>(a.data);
    data[i] = (singular && a.pinned_zero) ? (S)0 : (S)((double)data[i] / den);
}

template <typename S>
static hipError_t launch_zper_divide_s(const ZPerArgs &a, hipStream_t s)
{
    const long n = (long)a.SX * a.SY * a.nz;
    hipLaunchKernelGGL(k_zper_divide<S>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_zper_divide(const ZPerArgs &a, hipStream_t s) { return launch_zper_divide_s<double>(a, s); }

hipError_t launch_zper_divide_f32(const ZPerArgs &a, hipStream_t s) { return launch_zper_divide_s<float>(a, s); }

template <typename S>
static hipError_t launch_zperiodic_s(const ZPerArgs &a, int nitems, hipStream_t s)
{
    switch (zperiodic_supported(a.nz) ? a.nz / 2 : 0) {
#define PPM(m) \
    case m: return launch_zper_m<S, m>(a, nitems, s);
        PP_ZPER_LENGTHS(PPM)
#undef PPM
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_zperiodic_f64(const ZPerArgs &a, hipStream_t s) { return launch_zperiodic_s<double>(a, 0, s); }

hipError_t launch_zperiodic_f32(const ZPerArgs &a, hipStream_t s) { return launch_zperiodic_s<float>(a, 0, s); }

hipError_t launch_zperiodic_f64_batch(const ZPerArgs &a, int nitems, hipStream_t s)
{
    return a.items ? launch_zperiodic_s<double>(a, nitems, s) : hipErrorInvalidValue;
}

hipError_t launch_zperiodic_f32_batch(const ZPerArgs &a, int nitems, hipStream_t s)
{
    return a.items ? launch_zperiodic_s<float>(a, nitems, s) : hipErrorInvalidValue;
}

hipError_t launch_smt_v1(double *data, const SmtItem &it, hipStream_t s)
{
    hipLaunchKernelGGL(k_smt_v1, dim3(1), dim3(256), 3 * (size_t)it.nz * sizeof(double), s, data, it);
    return hipGetLastError();
}

hipError_t launch_smt_v1_batch(double *data, const SmtItem *items, int nitems, int nz_max, hipStream_t s)
{
    if (nitems == 0) return hipSuccess;
    hipLaunchKernelGGL(k_smt_v1_batch, dim3((unsigned)nitems), dim3(256), 3 * (size_t)nz_max * sizeof(double), s, data,
                       items);
    return hipGetLastError();
}

}  // namespace pp
