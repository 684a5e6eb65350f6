// pp_line_mm.h -- line transforms as dense products on the FP64 matrix cores of gfx950, for
// line lengths the compiled Stockham plans of pp_line.h do not cover.
//
// The reference takes any length from FFTW / cuFFT plans (src/poissonCPU.cpp:56,87,162,211,
// src/poissonGPU.cpp:13,37) and SignalProc handles odd sizes (src/signalProc.cpp:34-44,161-195).
// Every line transform here is a real matrix, and all but the quarter-wave ones split in two of
// half the size by the symmetry of their basis functions about the middle of the line:
//
//   NN / DD forward  s_j = x_j + x_{N-1-j}, d_j = x_j - x_{N-1-j};   X_2m from s, X_2m+1 from d
//   NN / DD inverse  e_n from X_2m, o_n from X_2m+1;   x_n = e_n + o_n, x_{N-1-n} = e_n - o_n
//   PP forward       the same fold about j and N - j; real parts from s, imaginary from d
//   PP inverse       e_n from the real, o_n from the imaginary parts; x_n, x_{N-n} = e_n +- o_n
//   ND / DN          no such symmetry: the two halves of the outputs, each from the whole line
//
// so a line costs N / 2 multiply-adds per point (N quarter-wave), all of them on the matrix cores
// (v_mfma_f64_16x16x4: 68 TFLOP/s measured, about 45 on full-entropy data, whose power lowers the
// clock), where the chirp convolution (pp_line_bs.h) spends two complex FFTs of 2 to 4 N points
// on every real line.  The sum runs in two interleaved chains, which keeps its rounding below
// the convolution's (relative L2 against extended precision, N = 33 / 101 / 202 / 331 / 509:
// 1.2 / 1.9 / 2.5 / 3.0 / 3.8e-16 against 2.5 / 3.1 / 3.5 / 3.4 / 4.2e-16).  On 16M points, one
// transform: N = 101 70-100 -> 39 us, 202 195-300 -> 119-137 us, 331 260-436 -> 146-160 us; the
// memory traffic alone would take 47 us at 5.5 TB/s, the products 54 us (N = 202) or 84 us (331):
// loads and products of the two blocks a CU holds overlap only partly (skipping either one in a
// copy leaves the other's time), and a block that walks over tiles with the next tile's loads in
// flight measured the same.  DD is NN with alternating signs and reversed modes, DN is ND reversed with alternating
// signs (the identities of SignalProc::swap, src/signalProc.cpp:235-265).
//
// A block stages `tiles` units of 16 lines (x) or 16 columns of one plane (y), folded, in LDS
// (so the fused input scaling, the Dirichlet term and the line sums happen on the way in), then
// its waves take output row tiles of 16: two accumulator sets (e and o) per unit, PW units (one, or two,
// mm_plan) per wave, so that one matrix element loaded from L2 feeds PW products.  Results go
// from the accumulators straight to global memory: the data is the A operand for x (lanes of a
// result row are 16 consecutive outputs of one line) and the B operand for y (16 consecutive
// columns), so stores are whole 128-byte segments without an LDS round trip.  Even and odd
// steps of the sum accumulate separately, which halves the length of a rounding chain.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "pp_line.h"
#include "pp_line_bs.h"

namespace pp {

// symmetry family of a kind: 0 DCT/DST-II/III (NN, DD), 1 DCT/DST-IV (ND, DN), 2 real DFT (PP)
__host__ __device__ constexpr int mm_family(int kind) { return kind == KIND_PP ? 2 : (kind == KIND_NN || kind == KIND_DD) ? 0 : 1; }
// length of one half's sum (rows of staged data) and its number of outputs
__host__ __device__ constexpr int mm_depth(int N, int fam) { return fam == 2 ? N / 2 + 1 : fam == 0 ? (N + 1) / 2 : N; }
__host__ __device__ constexpr int mm_rows(int N, int fam) { return fam == 2 ? N / 2 + 1 : (N + 1) / 2; }
// padded to whole matrix-instruction steps (two of depth 4) and row tiles; padding is zero
__host__ __device__ constexpr int mm_depth8(int N, int fam) { return (mm_depth(N, fam) + 7) / 8 * 8; }
__host__ __device__ constexpr int mm_rows16(int N, int fam) { return (mm_rows(N, fam) + 15) / 16 * 16; }
// doubles of one direction's matrices: [e, o] x [depth][row] (row fastest)
inline size_t mm_table_size(int N, int fam) { return 2 * (size_t)mm_depth8(N, fam) * mm_rows16(N, fam); }
// staged halves: the quarter-wave kinds take both output halves from one copy of the line
__host__ __device__ constexpr int mm_parts(int fam) { return fam == 1 ? 1 : 2; }

// doubles of LDS per unit of 16 lines / columns.  y: [part][depth][16] (a 32-lane read of two
// depth rows covers all banks); x: [line][part x depth + 2] (stride = 2 mod 4, so that 16 lines
// by two depths fall on 32 different bank pairs)
__host__ __device__ constexpr int mm_xstride(int N, int fam) { return mm_parts(fam) * mm_depth8(N, fam) + 2; }
__host__ __device__ constexpr int mm_unit(int N, int fam, int axis)
{
    return 16 * (axis == 0 ? mm_xstride(N, fam) : mm_parts(fam) * mm_depth8(N, fam));
}
// x forward: per-line constants of the Dirichlet term after the staged lines
constexpr int mm_xextra = 3 * 16;

typedef double mm_d4 __attribute__((ext_vector_type(4)));

// output position and sign of mode / element k for the reversed kinds
template <int KIND, int FWD>
__device__ __forceinline__ int mm_out(int N, int k, double &v)
{
    if constexpr (KIND == KIND_DD) {
        if constexpr (FWD) return N - 1 - k;
        else v = (k & 1) ? -v : v;
    } else if constexpr (KIND == KIND_DN) {
        v = (k & 1) ? -v : v;
    }
    return k;
}

// The two inputs folded into row m: their positions (-1: none) and how they combine.
// part 0 gets s0 * a + s1 * b, part 1 gets t0 * a + t1 * b.
struct MmIn {
    int ja, jb;
    double s0, s1, t0, t1;
};

template <int KIND, int FWD>
__device__ __forceinline__ MmIn mm_in(int N, int m)
{
    MmIn r = {-1, -1, 0, 0, 0, 0};
    constexpr int FAM = mm_family(KIND);
    if (m >= mm_depth(N, FAM)) return r;
    if constexpr (FAM == 1) {
        r.ja = (KIND == KIND_DN) ? N - 1 - m : m;
        r.s0 = 1.0;
    } else if constexpr (FWD) {
        r.ja = m;
        if constexpr (FAM == 0) {
            // DD: DST-II through the DCT-II of (-1)^j x_j
            r.s0 = (KIND == KIND_DD && (m & 1)) ? -1.0 : 1.0;
            const int j2 = N - 1 - m;
            if (j2 != m) {
                r.jb = j2;
                r.s1 = (KIND == KIND_DD && (j2 & 1)) ? -1.0 : 1.0;
                r.t0 = r.s0;
                r.t1 = -r.s1;
            }
        } else {
            r.s0 = 1.0;
            if (m > 0 && 2 * m != N) {
                r.jb = N - m;
                r.s1 = 1.0;
                r.t0 = 1.0;
                r.t1 = -1.0;
            }
        }
    } else {
        if constexpr (FAM == 0) {
            // X_2m to part 0 (half of X_0), X_2m+1 to part 1; DD reads the modes reversed
            const int k0 = 2 * m, k1 = 2 * m + 1;
            r.ja = (KIND == KIND_DD) ? N - 1 - k0 : k0;
            r.s0 = m == 0 ? 0.5 : 1.0;
            if (k1 < N) {
                r.jb = (KIND == KIND_DD) ? N - 1 - k1 : k1;
                r.t1 = 1.0;
            }
        } else {
            r.ja = m;
            r.s0 = (m == 0 || 2 * m == N) ? 1.0 : 2.0;
            if (m > 0 && 2 * m != N) {
                r.jb = N - m;
                r.t1 = -2.0;
            }
        }
    }
    return r;
}

// Matrix products of one wave: PW units (`unit` doubles apart in LDS), row tile i of `mm`
// ([e, o] x [D8][R16]); `stride` is a line's in LDS for x, a depth row's for y.  The loop is software-pipelined by hand: matrix elements are loaded (as
// buffer loads: a scalar offset walks the matrix, no address arithmetic per load) two pairs of
// steps ahead, staged values one pair ahead, so that the wait for L2 (some 500 cycles) and LDS lies
// under the 64-cycle products of the pairs between.
template <int AX, int FAM, int PW>
__device__ __forceinline__ void mm_products(const double *mm, int D8, int R16, int i, const double *lds, int unit,
                                            int stride, int lane, mm_d4 (&e)[PW], mm_d4 (&o)[PW])
{
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    const int r = lane >> 4, c = lane & 15;
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(mm), 0, 2 * D8 * R16 * 8, 0x00027000);
    const int vo = (r * R16 + 16 * i + c) * 8, half = D8 * R16 * 8, cs = 4 * R16 * 8;
    auto coef = [&](int so) { return __builtin_bit_cast(double, (u2)__builtin_amdgcn_raw_buffer_load_b64(rs, vo, so, 0)); };
    const double *ld = lds + (AX == 0 ? c * stride + r : r * stride + c);
    const int DS = AX == 0 ? 4 : 4 * stride;                       // one step of depth 4
    const int po = FAM == 1 ? 0 : (AX == 0 ? D8 : D8 * stride);    // the second part
    mm_d4 acc[2][2][PW];
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int p = 0; p < PW; p++) acc[q][h][p] = mm_d4{0, 0, 0, 0};
    const int S = D8 / 8;  // pairs of steps
    // reads past the last pair of steps repeat it (in bounds)
    double cf[2][2][2];  // [pair parity][step][half]
    double dv[2][PW][2];  // [step][unit][part]
    auto load_coef = [&](int s, double (&v)[2][2]) {
        const int so = (s < S ? s : S - 1) * 2 * cs;
        v[0][0] = coef(so);
        v[0][1] = coef(so + half);
        v[1][0] = coef(so + cs);
        v[1][1] = coef(so + cs + half);
    };
    auto load_data = [&](int s, double (&v)[2][PW][2]) {
        const double *d = ld + (s < S ? s : S - 1) * 2 * DS;
#pragma unroll
        for (int p = 0; p < PW; p++)
#pragma unroll
            for (int q = 0; q < 2; q++) {
                v[q][p][0] = d[p * unit + q * DS];
                v[q][p][1] = FAM == 1 ? v[q][p][0] : d[p * unit + q * DS + po];
            }
    };
    load_coef(0, cf[0]);
    load_coef(1, cf[1]);
    load_data(0, dv);
    auto pair = [&](int s, double (&cc)[2][2]) {
        double nx[2][PW][2];
        load_data(s + 1, nx);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int p = 0; p < PW; p++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    if constexpr (AX == 0) acc[q][h][p] = __builtin_amdgcn_mfma_f64_16x16x4f64(dv[q][p][h], cc[q][h], acc[q][h][p], 0, 0, 0);
                    else acc[q][h][p] = __builtin_amdgcn_mfma_f64_16x16x4f64(cc[q][h], dv[q][p][h], acc[q][h][p], 0, 0, 0);
                }
        __builtin_amdgcn_sched_barrier(0);
        load_coef(s + 2, cc);
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int p = 0; p < PW; p++)
#pragma unroll
                for (int h = 0; h < 2; h++) dv[q][p][h] = nx[q][p][h];
    };
    int s = 0;
    for (; s + 1 < S; s += 2) {
        pair(s, cf[0]);
        pair(s + 1, cf[1]);
    }
    if (s < S) pair(s, cf[0]);
#pragma unroll
    for (int p = 0; p < PW; p++) {
        e[p] = acc[0][0][p] + acc[1][0][p];
        o[p] = acc[0][1][p] + acc[1][1][p];
    }
}

// the outputs that row m of the two halves gives: put(position, value)
template <int KIND, int FWD, typename PUT>
__device__ __forceinline__ void mm_emit(int N, int m, double e, double o, const PUT &put)
{
    constexpr int FAM = mm_family(KIND);
    if (m >= mm_rows(N, FAM)) return;
    if constexpr (FAM == 1) {
        const double f = FWD ? 2.0 : 1.0;
        const int k1 = mm_rows(N, 1) + m;
        double v = f * e, w = f * o;
        const int p0 = mm_out<KIND, FWD>(N, m, v), p1 = mm_out<KIND, FWD>(N, k1, w);
        put(p0, v);
        if (k1 < N) put(p1, w);
    } else if constexpr (FAM == 0 && FWD) {
        double v = 2.0 * e, w = 2.0 * o;
        const int p0 = mm_out<KIND, FWD>(N, 2 * m, v), p1 = mm_out<KIND, FWD>(N, 2 * m + 1, w);
        put(p0, v);
        if (2 * m + 1 < N) put(p1, w);
    } else if constexpr (FAM == 0) {
        double v = e + o, w = e - o;
        const int m2 = N - 1 - m;
        const int p0 = mm_out<KIND, FWD>(N, m, v), p1 = mm_out<KIND, FWD>(N, m2, w);
        put(p0, v);
        if (m2 != m) put(p1, w);
    } else if constexpr (FWD) {
        put(m, e);
        if (m > 0 && 2 * m != N) put(N - m, -o);
    } else {
        put(m, e + o);
        if (m > 0 && 2 * m != N) put(N - m, e - o);
    }
}

template <typename TIn, typename TOut, int AX, int FWD, int KIND, int PW>
__global__ void __launch_bounds__(1024) k_line_mm(LineArgs a0, int units)
{
    constexpr int FAM = mm_family(KIND);
    LineArgs a = a0;
    int bx = blockIdx.x, by = blockIdx.y;
    if (a0.items) {
        line_block<TIn, TOut, double, 16, AX>(a0, a, bx, by);
    } else if constexpr (AX == 1) {
        // neighbouring column blocks share lines of memory where nx is no multiple of 16: one XCD
        const int lin = xcd_logical(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
        bx = lin % gridDim.x;
        by = lin / gridDim.x;
    }
    const int N = a0.n;
    const int D8 = mm_depth8(N, FAM), R16 = mm_rows16(N, FAM);
    const int unit = mm_unit(N, FAM, AX), xs = mm_xstride(N, FAM);
    const int part = AX == 0 ? D8 : D8 * 16;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double *lds = reinterpret_cast<double *>(smem_raw);
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nw = blockDim.x >> 6;
    const TIn *in = reinterpret_cast<const TIn *>(a.in);
    TOut *out = reinterpret_cast<TOut *>(a.out);

    // y: the unit's columns and plane -- consecutive planes of one column block, or (one plane:
    // the z lines of a periodic solve) consecutive column blocks
    const bool flat = AX == 1 && a.nplanes == 1;
    auto unit_col = [&](int p) { return 16 * (flat ? bx * units + p : bx); };
    auto unit_z = [&](int p) { return flat ? 0 : by * units + p; };

    // ---- load, fold, stage ----
    if constexpr (AX == 0) {
        const long line0 = (long)bx * 16 * units;
        // per-line constants of the Dirichlet term
        double *dl = lds + units * unit;
        if constexpr (FWD) {
            if (a.dmask) {
                for (int l = tid; l < 16 * units; l += blockDim.x) {
                    const long line = line0 + l < a.nlines ? line0 + l : 0;
                    const DirLine d = dirichlet_line(a, (int)(line % a.ny), (int)(line / a.ny));
                    dl[3 * l] = d.cyz;
                    dl[3 * l + 1] = d.cx0;
                    dl[3 * l + 2] = d.cxn;
                }
                __syncthreads();
            }
        }
        // LW lanes per line (a power of two no wider than the folded line needs)
        const int LW = D8 <= 8 ? 8 : D8 <= 16 ? 16 : D8 <= 32 ? 32 : 64;
        const int sub = lane / LW, m1 = lane % LW, lpw = 64 / LW;
        constexpr int U = 4;
        for (int l0 = wv * lpw + sub; l0 < 16 * units; l0 += nw * lpw * U) {
            double sum[U] = {0, 0, 0, 0};
            for (int m = m1; m < D8; m += LW) {
                const MmIn f = mm_in<KIND, FWD>(N, m);
                double xa[U], xb[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int l = l0 + u * nw * lpw;
                    long line = line0 + (l < 16 * units ? l : 0);
                    if (line >= a.nlines) line = 0;
                    const TIn *src = in + line * N;
                    xa[u] = (double)src[f.ja < 0 ? 0 : f.ja];
                    xb[u] = (double)src[f.jb < 0 ? 0 : f.jb];
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int l = l0 + u * nw * lpw;
                    if (l >= 16 * units) continue;
                    double va = xa[u], vb = xb[u];
                    if constexpr (FWD) {
                        va = va * a.in_scale;  // rhs * c3 * c3 (src/pencilDcmp.cpp:5639)
                        va = va * a.in_scale;
                        vb = vb * a.in_scale;
                        vb = vb * a.in_scale;
                        if (a.dmask) {
                            const double cyz = dl[3 * l];
                            if (cyz != 0.0) {
                                if (f.ja >= 0) va -= gld(a.dtab, f.ja) * cyz;
                                if (f.jb >= 0) vb -= gld(a.dtab, f.jb) * cyz;
                            }
                            // elements 0 and N - 1
                            if (f.ja == 0) va -= dl[3 * l + 1];
                            if (f.jb == 0) vb -= dl[3 * l + 1];
                            if (f.ja == N - 1) va -= dl[3 * l + 2];
                            if (f.jb == N - 1) vb -= dl[3 * l + 2];
                        }
                        // the line's sum, of the values that are transformed
                        if (f.ja >= 0) sum[u] += va;
                        if (f.jb >= 0) sum[u] += vb;
                    }
                    double *row = lds + (l >> 4) * unit + (l & 15) * xs + m;
                    // (an absent input is not read into the sum: it may be anything, NaN too)
                    if (f.ja < 0) va = 0.0;
                    if (f.jb < 0) vb = 0.0;
                    row[0] = f.s0 * va + f.s1 * vb;
                    if constexpr (mm_parts(FAM) == 2) row[part] = f.t0 * va + f.t1 * vb;
                }
            }
            if constexpr (FWD) {
                if (a.line_sums) {
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        double s = sum[u];
                        for (int off = LW / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
                        const int l = l0 + u * nw * lpw;
                        if (m1 == 0 && l < 16 * units && line0 + l < a.nlines) a.line_sums[line0 + l] = s;
                    }
                }
            }
        }
    } else {
        const int c = tid & 15, q0 = tid >> 4, nq = blockDim.x >> 4;
        const bool tin = a.ztiled & ZT_IN;
        const int W = a.tile_w ? a.tile_w : 16;
        const long stride = tin ? (long)a.tnz * W : a.ncols;
        for (int p = 0; p < units; p++) {
            // columns and planes past the grid read the last one (in bounds) and are not stored
            int col = unit_col(p) + c, z = unit_z(p);
            if (z >= a.nplanes) z = a.nplanes - 1;
            long base;
            if (tin) {
                // tiles hold whole blocks of columns, padded
                const int tc = unit_col(p) < a.ncols ? col : 0;
                base = ((long)(tc / W) * N * a.tnz + z) * W + tc % W;
            } else {
                if (col >= a.ncols) col = a.ncols - 1;
                base = (long)z * N * a.ncols + col;
            }
            double *dst = lds + p * unit + c;
            constexpr int U = 4;
            for (int m0 = q0; m0 < D8; m0 += nq * U) {
                double xa[U], xb[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const MmIn f = mm_in<KIND, FWD>(N, m0 + u * nq);
                    xa[u] = (double)in[base + (long)(f.ja < 0 ? 0 : f.ja) * stride];
                    xb[u] = (double)in[base + (long)(f.jb < 0 ? 0 : f.jb) * stride];
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int m = m0 + u * nq;
                    if (m >= D8) continue;
                    const MmIn f = mm_in<KIND, FWD>(N, m);
                    const double va = f.ja < 0 ? 0.0 : xa[u], vb = f.jb < 0 ? 0.0 : xb[u];
                    dst[m * 16] = f.s0 * va + f.s1 * vb;
                    if constexpr (mm_parts(FAM) == 2) dst[part + m * 16] = f.t0 * va + f.t1 * vb;
                }
            }
        }
    }
    __syncthreads();

    // ---- products and stores: wave -> (group of PW units, row tile) ----
    const int KT = R16 / 16, groups = units / PW;
    const double *mm = FWD ? a0.mm : a0.mmi;
    for (int job = wv; job < groups * KT; job += nw) {
        const int g = job / KT, i = job - g * KT;
        mm_d4 e[PW], o[PW];
        const int p0 = g * PW;
        mm_products<AX, FAM, PW>(mm, D8, R16, i, lds + p0 * unit, unit, AX == 0 ? xs : 16, lane, e, o);
#pragma unroll
        for (int p = 0; p < PW; p++) {
            if constexpr (AX == 0) {
                // result row = line 4 r + lane / 16 of the unit, column = output lane % 16
                const int m = 16 * i + (lane & 15);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const long line = ((long)bx * units + p0 + p) * 16 + 4 * r + (lane >> 4);
                    if (line >= a.nlines) continue;
                    const long base = line * N;
                    double padd = 0.0;
                    if constexpr (!FWD) {
                        if (a.plane_add) padd = a.plane_add[line / a.ny];
                    }
                    mm_emit<KIND, FWD>(N, m, e[p][r], o[p][r], [&](int pos, double v) {
                        v = a.out_scale * v;
                        if constexpr (!FWD) {
                            if (a.plane_add) v += padd;
                            if (a.accumulate) v += (double)out[base + pos];
                            else if (a.acc0) v += (double)a.acc0[base + pos] + (a.acc1 ? (double)a.acc1[base + pos] : 0.0);
                        }
                        out[base + pos] = (TOut)v;
                    });
                }
            } else {
                // result row = output 4 r + lane / 16, column = the unit's column lane % 16
                const int col = unit_col(p0 + p) + (lane & 15), z = unit_z(p0 + p);
                if (col >= a.ncols || z >= a.nplanes) continue;
                long base, stride;
                if (a.ztiled & ZT_OUT) {
                    const int W = a.tile_w ? a.tile_w : 16;
                    base = ((long)(col / W) * N * a.tnz + z) * W + col % W;
                    stride = (long)a.tnz * W;
                } else {
                    base = (long)z * N * a.ncols + col;
                    stride = a.ncols;
                }
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    mm_emit<KIND, FWD>(N, 16 * i + 4 * r + (lane >> 4), e[p][r], o[p][r],
                                       [&](int pos, double v) { out[base + (long)pos * stride] = (TOut)v; });
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------------------
// matrices
// ---------------------------------------------------------------------------------------

// cos(2 pi q / (8 N)) from the octant table oct = {cos, sin}(2 pi q / (8 N)), q = 0 .. N
__device__ __forceinline__ double mm_cos8(const double *oct, int N, long q)
{
    int m = (int)(q % (8L * N));
    if (m > 4 * N) m = 8 * N - m;
    double sg = 1.0;
    if (m > 2 * N) {
        m = 4 * N - m;
        sg = -1.0;
    }
    return sg * (m <= N ? oct[2 * m] : oct[2 * (2 * N - m) + 1]);
}

// doubles of the octant table of length N, and of both directions' matrices (the real DFT's and
// the quarter-wave kinds' are their own transposes: one set serves both)
inline size_t mm_octant_size(int N) { return 2 * (size_t)(N + 1); }
inline size_t mm_tables_size(int N, int kind)
{
    const int fam = mm_family(kind);
    return (fam == 0 ? 2 : 1) * mm_table_size(N, fam);
}
inline size_t mm_inverse_offset(int N, int kind)
{
    return mm_family(kind) == 0 ? mm_table_size(N, 0) : 0;
}
// write both directions' matrices of (N, kind) to `out` (mm_tables_size doubles) from the device
// octant table (pp_line_mm.hip)
hipError_t launch_mm_tables(double *out, const double *oct, int N, int kind, hipStream_t s);

// ---------------------------------------------------------------------------------------
// launch
// ---------------------------------------------------------------------------------------

// The lines these kernels serve (given their matrices): those without a compiled plan, up to the
// length where N / 2 multiply-adds per point (N quarter-wave) cost more than the chirp convolution.
// Measured against it on 16M points, us per transform, dense / chirp:
//   x, folded kinds:   331: 153 / 264   509: 183 / 183   602: 280 / 293   650: 301 / 277
//   y, folded kinds:   331: 152 / 436   602: 268 / 517   750: 260 / 440  1000: 318 / 361
//   x, quarter-wave:   331: 227 / 262   402: 335 / 223
//   y, quarter-wave:   331: 227 / 437   509: 282 / 315   602: 514 / 513
// (x: 440 to 512 folded and 280 up quarter-wave are no faster, and the matrix cores' power slows the rest
// of a solve by 3 %).  A long line's products are a chain of loads from L2 whatever the number of lines,
// which the convolution's few passes beat while lines are few -- 1024 / 4096 lines, x then y (us):
//   101: 8.5 9.1, 7.8 9.1 / 9.0 11.6, 10.9 12.1    201: 12.0 13.8, 10.8 13.0 / 9.2 17.7, 12.0 21.4
//   401: 25 30, 22 25 / 14 34, 15 45               601: 45 50, 39 45 / 22 58, 27 87
//   x, quarter-wave (twice the products)  67: 9.7 10.2 / 9.0 11.1    27, 1280 lines: a solve 33.1 / 32.2
// Quarter-wave lines along x just short of 256 points have the chirp of 512 at its best: a whole solve, dense /
// chirp, 2112, 3072, 4096, 16384 and 65536 lines
//   138: 0.97 0.98 0.86 0.76 0.79    170: 1.02 1.05 0.94 0.88 0.93    201: 1.10 1.09 0.96 0.94 1.00
//   222: 1.12 1.13 1.01 0.96 1.03    243: 1.15 1.16 1.03 1.00 1.02    271: 1.00 1.02 0.90 0.74 0.78
// Columns fill units of 16, the convolution's blocks (8 columns from 129 points on, 4 from 257) less, and the
// units of long lines go over the CUs in rounds of 256: mm_stretch is how much longer the products take for both.
// y, a whole solve, dense / chirp, cols x planes:
//   folded        12x320  401: 0.86  509: 0.96  767: 1.00 1021: 1.43    40x128 1021: 1.18  767: 0.83
//                 4x960   201: 0.89  254: 0.92  331: 1.14  509: 1.52    8x512   613: 0.85  767: 1.03
//   quarter-wave  12x320  254: 0.87  331: 1.03  509: 1.44               40x128  331: 0.89  401: 1.07
//                 20x160  250: 1.10                                     20x200  254: 0.87
//                 4x960   130: 0.87  201: 1.15  331: 1.60               8x512   201: 1.00  254: 1.11
// and whole units, 256, 264, 384 and 512 of them (rounds 1.00, 1.94, 1.33 and 1.00 times as long as they are full):
//   y folded  767: 0.63 0.89 0.73 0.64    1021: 0.90 1.30 1.05 0.90    quarter-wave 331: 0.78 0.88 0.79 0.67
//   x folded  371: 0.88 1.07 0.93 0.80     613: 0.91 1.24 0.99 0.84    quarter-wave 509: 0.95 1.22 1.08 0.94 (y)
//   x quarter-wave  185: 0.96 1.10 1.02 0.90    213: 0.98 1.13 1.04 0.94    280: 0.92 1.03 0.89 0.77
// Lines of a few points fill little of a tile of 16 outputs, so many of them are the convolution's, one
// thread's each, and 2 points always.  A whole solve, dense / chirp, 4096, 16384, 65536 and 262144 lines:
//   x   2 points 1.04 1.06 1.04 1.12    5 0.99 1.02 1.01 1.02    13 0.91 0.95 0.91 0.80
//   y   2 points 1.02 1.01 1.03 1.55    5 0.98 0.97 1.02 1.30    13 0.98 0.95 1.03 1.21    17 0.99 0.92 0.89 0.93
constexpr int kMmMaxN = 1024;
inline double mm_stretch(int axis, int cols, long lines, int block)
{
    if (axis == 0) return (double)((lines + 4095) / 4096) * 4096 / lines;
    const long units = (long)((cols + 15) / 16) * (lines / cols);
    return (double)((units + 255) / 256) * 4096 / ((double)((cols + block - 1) / block * block) * (lines / cols));
}
inline bool mm_columns(int n, bool quarter, int cols, long lines)
{
    const int block = bs_block_lines<double>(n, 1);
    if (n <= 256) {
        // (rounds tell less: of shorter lines more than one block runs on a CU; few units leave either idle)
        const long dense = (cols + 15) / 16 * 16, chirp = (cols + block - 1) / block * block, units = dense / 16 * (lines / cols);
        const double rounds = units <= 256 ? 1.0 : (double)((units + 255) / 256 * 256) / units;
        return quarter ? n * dense * (0.4 + 0.6 * rounds) <= 410 * chirp : n * dense <= 1100 * chirp;
    }
    const double s = mm_stretch(1, cols, lines, block);
    if (quarter) return n <= 512 && n * std::sqrt((double)n) * s <= 11900;
    return n <= 512 ? n * s <= 1100 : (double)n * n * s <= 1.17e6;
}

// cols: y, the columns of a plane
inline bool mm_serves(int n, int kind, int axis, int cols, long lines)
{
    if (line_compiled(n) || n < 3) return false;
    if (n < (axis == 1 ? 16 : 8) && lines > (n == 3 ? 4096 : 16384)) return false;
    const bool quarter = mm_family(kind) == 1;
    const int any = axis == 1 ? (quarter ? 112 : 208) : quarter ? 0 : 112;  // up to here any number of lines
    if (n > any && lines < (axis == 0 && quarter && n > 150 ? 4096 : n <= 256 ? 2048 : 3072)) return false;
    if (axis == 1) return mm_columns(n, quarter, cols, lines);
    if (n <= (quarter ? 150 : 256)) return true;
    const double s = n * mm_stretch(0, 0, lines, 1);
    if (quarter) return n <= 232 ? s <= 255 : n > 256 && n <= 280 && s <= 500;
    return n <= 440 ? s <= 560 : n > 512 && n <= 620 && s <= 842;
}

// Shape of a launch over `nunits` units of 16 lines / columns.  One unit a wave: two halve the matrix traffic
// from L2, but half as many blocks end in emptier last rounds, and short lines are left with too few waves.  A
// whole solve, two / one a wave, over the convolution's time, 1056, 2046 and 4092 units (ND: quarter-wave):
//   x   19 0.96/0.91 0.94/0.89 0.88/0.84   185 ND 1.12/0.93 0.94/0.89 0.97/0.87   331 0.82/0.76 0.66/0.68 0.69/0.72
//   y   67 0.61/0.59 0.50/0.54 0.51/0.47   201 ND 0.82/0.72 0.76/0.69 0.70/0.66   439 0.72/0.63 0.65/0.60 0.55/0.56
// Two are faster at 4096 units and more of folded lines of 113 to 256 points (x 254 points 0.81/0.85, y 127 points
// at 16384 0.54/0.58, but 67 points 0.62/0.63, 300 points 0.69/0.62), and where their block has a CU of its own,
// with up to 16 waves, as long as its rounds over the CUs are as full (x 331 points, 1536 units 0.68/0.72).  More
// units per block while the block stays small (8 waves, 64 KB: two or more blocks per CU, so
// one block's loads overlap another's products) and three blocks per CU remain.
struct MmPlan {
    int pw, units, waves;
};
inline MmPlan mm_plan(int N, int kind, int axis, long nunits)
{
    const int fam = mm_family(kind), KT = mm_rows16(N, fam) / 16;
    const long ub = (long)(mm_unit(N, fam, axis) + (axis == 0 ? mm_xextra : 0)) * 8;
    MmPlan p;
    const bool whole = nunits >= 1024 && (nunits + 511) / 512 * 2 <= (nunits + 255) / 256;  // two cost no round more
    const bool pair = N > 256 ? 2 * ub > 80 * 1024 && 2 * ub <= 158 * 1024 && whole : N > 112 && nunits >= 4096;
    p.pw = fam != 1 && pair ? 2 : 1;
    int g = 1;
    while ((g + 1) * KT <= 8 && (g + 1) * p.pw * ub <= 64 * 1024 && nunits >= 768L * (g + 1) * p.pw) g++;
    p.units = g * p.pw;
    const int jobs = g * KT, most = p.units * ub > 80 * 1024 ? 16 : 8;
    const int rounds = (jobs + most - 1) / most;
    p.waves = (jobs + rounds - 1) / rounds;
    // short lines: enough threads to stage the units, more while units are few (256 units of quarter-wave x
    // lines of 19 points, a whole solve: 23.8 us with one wave a block, 21.8 with two, the convolution 22.8;
    // from 4096 units more threads are more waves than the loads need: y lines of 17 points 0.84 -> 0.90 of it)
    const int per = nunits <= 1024 ? 128 : 32;
    while (p.waves < 4 && p.waves * 64 < per * p.units) p.waves++;
    return p;
}

template <typename TIn, typename TOut, int AX, int FWD, int KIND, int PW>
hipError_t launch_line_mm_pw(const LineArgs &a, const MmPlan &p, dim3 grid, hipStream_t s)
{
    const int fam = mm_family(KIND);
    const size_t lds = (size_t)p.units * (mm_unit(a.n, fam, AX) + (AX == 0 ? mm_xextra : 0)) * sizeof(double);
    auto kern = k_line_mm<TIn, TOut, AX, FWD, KIND, PW>;
    // the limit is a property of the kernel on the current device; lengths share the kernel, so
    // it is set to the most any of them takes
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, grid, dim3(64 * p.waves), lds, s, a, p.units);
    return hipGetLastError();
}

template <typename TIn, typename TOut, int AX, int FWD, int KIND>
hipError_t launch_line_mm_cfg(const LineArgs &a, hipStream_t s)
{
    if (a.n < 2 || a.n > kMmMaxN || !a.mm || !a.mmi) return hipErrorInvalidValue;
    MmPlan p{a.mm_pw, a.mm_units, a.mm_waves};
    dim3 grid;
    if (a.items) {
        grid = dim3((unsigned)a.nlines);  // batched: nlines holds the item count
    } else {
        const long blocks = (a.nlines + 15) / 16;  // of lines, or of columns in one plane
        p = mm_plan(a.n, KIND, AX, AX == 0 ? blocks : blocks * a.nplanes);
        if (AX == 0 || a.nplanes == 1) grid = dim3((unsigned)((blocks + p.units - 1) / p.units));
        else grid = dim3((unsigned)blocks, (unsigned)((a.nplanes + p.units - 1) / p.units));
    }
    if (p.pw == 2) return launch_line_mm_pw<TIn, TOut, AX, FWD, KIND, 2>(a, p, grid, s);
    return launch_line_mm_pw<TIn, TOut, AX, FWD, KIND, 1>(a, p, grid, s);
}

// what serves a line: a compiled plan or the chirp convolution, or the dense products
enum class LineRoute { PLAN, DENSE };
inline LineRoute line_route(int n, int kind, int axis, int cols, long lines)
{
    return mm_serves(n, kind, axis, cols, lines) ? LineRoute::DENSE : LineRoute::PLAN;
}

// lines (x) or columns (y) per block of the launch that serves length N (dense x launches take
// whole multiples of it, mm_plan)
template <typename R>
inline int line_lines_any(int N, LineRoute route, int AX)
{
    if (route == LineRoute::DENSE) return 16;
    return line_compiled(N) ? line_block_lines<R>(N, AX) : bs_block_lines<R>(N, AX);
}

// every precision form, axis and direction of one kind (LineForm as in launch_line_kind)
template <int KIND>
hipError_t launch_line_mm_kind(int form, int AX, int FWD, const LineArgs &a, hipStream_t s)
{
    switch (form) {
    case FORM_F64:
        if (AX == 0) return FWD ? launch_line_mm_cfg<double, double, 0, 1, KIND>(a, s)
                                : launch_line_mm_cfg<double, double, 0, 0, KIND>(a, s);
        return FWD ? launch_line_mm_cfg<double, double, 1, 1, KIND>(a, s)
                   : launch_line_mm_cfg<double, double, 1, 0, KIND>(a, s);
    // FP32 storage, FP64 products
    case FORM_F32:
        if (AX == 0) return FWD ? launch_line_mm_cfg<float, float, 0, 1, KIND>(a, s)
                                : launch_line_mm_cfg<float, float, 0, 0, KIND>(a, s);
        return FWD ? launch_line_mm_cfg<float, float, 1, 1, KIND>(a, s)
                   : launch_line_mm_cfg<float, float, 1, 0, KIND>(a, s);
    case FORM_F64_TO_F32:
        if (AX == 0 && FWD) return launch_line_mm_cfg<double, float, 0, 1, KIND>(a, s);
        return hipErrorInvalidValue;
    case FORM_F32_TO_F64:
        if (AX == 0 && !FWD) return launch_line_mm_cfg<float, double, 0, 0, KIND>(a, s);
        return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
    }
}

}  // namespace pp
