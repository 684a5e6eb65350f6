// pp_plane_mm.hip -- the plane kernels of pp_plane_mm.h: one block per plane.
#include "pp_plane_mm.h"

namespace pp {

namespace {

// one block's plane and the LDS regions of pp_plane_mm.h
struct Plane {
    LineArgs ax, ay;
    int kx, ky, z;
    double *A, *B, *dl;
    int tid, nt, lane, wv, nw;
};

// x rows, folded, into A: from the right-hand side (forward, with the fused scaling and
// Dirichlet term) or from the plane in B (inverse).  A thread keeps its folded position m over the
// lines it takes
template <int KIND, int FWD>
__device__ __forceinline__ void stage_x(const Plane &p)
{
    constexpr int FAM = mm_family(KIND);
    const LineArgs &a = p.ax;
    const int N = a.nx, ny = a.ny, D8 = mm_depth8(N, FAM), xs = mm_xstride(N, FAM), sb = plane_sb(N);
    const unsigned inv = 0xffffffffu / (unsigned)D8 + 1u;
    const int step = (int)__umulhi((unsigned)p.nt, inv), l0 = (int)__umulhi((unsigned)p.tid, inv), m = p.tid - l0 * D8;
    if (l0 >= step) return;
    const MmIn f = mm_in<KIND, FWD>(N, m);
    const int ja = max(f.ja, 0), jb = max(f.jb, 0);
    const double *src = reinterpret_cast<const double *>(a.in) + (long)p.z * ny * N;
    constexpr int U = 4;
    for (int l = l0; l < ny; l += step * U) {
        double xa[U], xb[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int lu = min(l + u * step, ny - 1);
            const int row = FWD ? lu * N : lu * sb;
            xa[u] = FWD ? src[row + ja] : p.B[row + ja];
            xb[u] = FWD ? src[row + jb] : p.B[row + jb];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int lu = l + u * step;
            if (lu >= ny) break;
            double va = xa[u], vb = xb[u];
            if constexpr (FWD) {
                va = va * a.in_scale;  // rhs * c3 * c3 (src/pencilDcmp.cpp:5639)
                va = va * a.in_scale;
                vb = vb * a.in_scale;
                vb = vb * a.in_scale;
                if (a.dmask) {
                    const double cyz = p.dl[3 * lu];
                    if (cyz != 0.0) {
                        if (f.ja >= 0) va -= gld(a.dtab, f.ja) * cyz;
                        if (f.jb >= 0) vb -= gld(a.dtab, f.jb) * cyz;
                    }
                    // elements 0 and N - 1
                    if (f.ja == 0) va -= p.dl[3 * lu + 1];
                    if (f.jb == 0) vb -= p.dl[3 * lu + 1];
                    if (f.ja == N - 1) va -= p.dl[3 * lu + 2];
                    if (f.jb == N - 1) vb -= p.dl[3 * lu + 2];
                }
            }
            if (f.ja < 0) va = 0.0;
            if (f.jb < 0) vb = 0.0;
            double *row = p.A + lu * xs + m;
            row[0] = f.s0 * va + f.s1 * vb;
            if constexpr (mm_parts(FAM) == 2) row[D8] = f.t0 * va + f.t1 * vb;
        }
    }
}

// x products: to the plane in B (forward) or the solution (inverse)
template <int KIND, int FWD>
__device__ __forceinline__ void mult_x(const Plane &p)
{
    constexpr int FAM = mm_family(KIND);
    const LineArgs &a = p.ax;
    const int N = a.nx, ny = a.ny, D8 = mm_depth8(N, FAM), R16 = mm_rows16(N, FAM), xs = mm_xstride(N, FAM);
    const int KT = R16 / 16, jobs = (ny + 15) / 16 * KT, sb = plane_sb(N);
    const double *mm = FWD ? a.mm : a.mmi;
    double *out = reinterpret_cast<double *>(a.out) + (long)p.z * ny * N;
    for (int job = p.wv; job < jobs; job += p.nw) {
        const int u = job / KT, i = job - u * KT;
        mm_d4 e[1], o[1];
        mm_products<0, FAM, 1>(mm, D8, R16, i, p.A + u * 16 * xs, 0, xs, p.lane, e, o);
        // result row = line 4 r + lane / 16 of the unit, column = output lane % 16
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int l = 16 * u + 4 * r + (p.lane >> 4);
            if (l >= ny) continue;
            mm_emit<KIND, FWD>(N, 16 * i + (p.lane & 15), e[0][r], o[0][r], [&](int pos, double v) {
                if constexpr (FWD) p.B[l * sb + pos] = v;
                else out[l * N + pos] = a.out_scale * v;
            });
        }
    }
}

// y side of the plane: element (column 16 u + c, row 0), the next unit of 16 columns and the next row
struct YPlace {
    long base, unit, row;
};
__device__ __forceinline__ YPlace y_place(const LineArgs &a, int z, bool tiled, int c)
{
    if (tiled) return {(long)z * 16 + c, (long)a.ny * a.tnz * 16, (long)a.tnz * 16};
    return {(long)z * a.ny * a.nx + c, 16, a.nx};
}

// y rows, folded, into A: from the plane in B (forward) or the z solve's output (inverse)
template <int KIND, int FWD>
__device__ __forceinline__ void stage_y(const Plane &p)
{
    constexpr int FAM = mm_family(KIND);
    const LineArgs &a = p.ay;
    const int N = a.ny, nx = a.nx, D8 = mm_depth8(N, FAM), cs = plane_cs(nx), sb = plane_sb(nx);
    const int c = p.tid & 15;
    const YPlace y = y_place(a, p.z, a.ztiled & ZT_IN, c);
    const double *src = reinterpret_cast<const double *>(a.in) + y.base;
    constexpr int U = kPlaneMax / 16;
    for (int m = p.tid >> 4; m < D8; m += p.nt >> 4) {
        const MmIn f = mm_in<KIND, FWD>(N, m);
        const long ra = max(f.ja, 0) * (FWD ? (long)sb : y.row), rb = max(f.jb, 0) * (FWD ? (long)sb : y.row);
        double xa[U], xb[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            xa[u] = xb[u] = 0.0;
            if (16 * u + c >= nx) continue;
            if constexpr (FWD) {
                xa[u] = p.B[(int)ra + 16 * u + c];
                xb[u] = p.B[(int)rb + 16 * u + c];
            } else {
                xa[u] = src[u * y.unit + ra];
                xb[u] = src[u * y.unit + rb];
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (16 * u + c >= nx) continue;
            const double va = f.ja < 0 ? 0.0 : xa[u], vb = f.jb < 0 ? 0.0 : xb[u];
            double *row = p.A + m * cs + 16 * u + c;
            row[0] = f.s0 * va + f.s1 * vb;
            if constexpr (mm_parts(FAM) == 2) row[D8 * cs] = f.t0 * va + f.t1 * vb;
        }
    }
}

// y products: to the z solve's input (forward) or the plane in B (inverse)
template <int KIND, int FWD>
__device__ __forceinline__ void mult_y(const Plane &p)
{
    constexpr int FAM = mm_family(KIND);
    const LineArgs &a = p.ay;
    const int N = a.ny, nx = a.nx, D8 = mm_depth8(N, FAM), R16 = mm_rows16(N, FAM), cs = plane_cs(nx);
    const int KT = R16 / 16, jobs = (nx + 15) / 16 * KT, sb = plane_sb(nx);
    const double *mm = FWD ? a.mm : a.mmi;
    double *out = reinterpret_cast<double *>(a.out);
    for (int job = p.wv; job < jobs; job += p.nw) {
        const int u = job / KT, i = job - u * KT;
        mm_d4 e[1], o[1];
        mm_products<1, FAM, 1>(mm, D8, R16, i, p.A + u * 16, 0, cs, p.lane, e, o);
        // result row = output 4 r + lane / 16, column = the unit's column lane % 16
        const int col = 16 * u + (p.lane & 15);
        if (col >= nx) continue;
        const YPlace y = y_place(a, p.z, a.ztiled & ZT_OUT, p.lane & 15);
        double *dst = out + y.base + u * y.unit;
#pragma unroll
        for (int r = 0; r < 4; r++)
            mm_emit<KIND, FWD>(N, 16 * i + 4 * r + (p.lane >> 4), e[0][r], o[0][r], [&](int pos, double v) {
                if constexpr (FWD) dst[pos * y.row] = v;
                else p.B[pos * sb + col] = v;
            });
    }
}

#define PP_BY_KIND(kind, call)                     \
    switch (kind) {                                \
    case KIND_DD: call<KIND_DD, FWD>(p); break;    \
    case KIND_NN: call<KIND_NN, FWD>(p); break;    \
    case KIND_PP: call<KIND_PP, FWD>(p); break;    \
    case KIND_ND: call<KIND_ND, FWD>(p); break;    \
    default: call<KIND_DN, FWD>(p); break;         \
    }

template <int FWD>
__global__ void __launch_bounds__(64 * kPlaneWaves) k_plane_mm(LineArgs ax0, LineArgs ay0, int kx, int ky, const PlaneSolve *ps)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    Plane p;
    p.ax = ax0;
    p.ay = ay0;
    p.kx = kx;
    p.ky = ky;
    p.z = blockIdx.x;
    if (ax0.items) {
        int by;
        line_item<double, double, 0>(ax0, p.ax, blockIdx.x, p.z, by);
        line_item<double, double, 1>(ay0, p.ay, blockIdx.x, p.z, by);
        const PlaneSolve *sv = ps + ax0.items[blockIdx.x].solve;
        p.kx = sv->kind[0];
        p.ky = sv->kind[1];
        p.ax.mm = sv->mm[0];
        p.ax.mmi = sv->mmi[0];
        p.ay.mm = sv->mm[1];
        p.ay.mmi = sv->mmi[1];
    }
    p.tid = threadIdx.x;
    p.nt = blockDim.x;
    p.lane = p.tid & 63;
    p.wv = p.tid >> 6;
    p.nw = p.nt >> 6;
    const int nx = p.ax.nx, ny = p.ax.ny;
    p.A = reinterpret_cast<double *>(smem_raw);
    p.B = p.A + plane_a(nx, ny, mm_family(p.kx), mm_family(p.ky));
    p.dl = p.B + ny * plane_sb(nx);
    if constexpr (FWD) {
        if (p.ax.dmask) {
            for (int l = p.tid; l < ny; l += p.nt) {
                const DirLine d = dirichlet_line(p.ax, l, p.z);
                p.dl[3 * l] = d.cyz;
                p.dl[3 * l + 1] = d.cx0;
                p.dl[3 * l + 2] = d.cxn;
            }
            __syncthreads();
        }
        PP_BY_KIND(p.kx, stage_x)
        __syncthreads();
        PP_BY_KIND(p.kx, mult_x)
        __syncthreads();
        PP_BY_KIND(p.ky, stage_y)
        __syncthreads();
        PP_BY_KIND(p.ky, mult_y)
    } else {
        PP_BY_KIND(p.ky, stage_y)
        __syncthreads();
        PP_BY_KIND(p.ky, mult_y)
        __syncthreads();
        PP_BY_KIND(p.kx, stage_x)
        __syncthreads();
        PP_BY_KIND(p.kx, mult_x)
    }
}

}  // namespace

hipError_t launch_plane_mm(int fwd, int kx, int ky, const LineArgs &ax, const LineArgs &ay, size_t lds, hipStream_t s,
                           const PlaneSolve *ps, int waves)
{
    if (ax.items ? !ps : (!mm_plane(ax.nx, ax.ny, kx, ky) || !ax.mm || !ay.mm)) return hipErrorInvalidValue;
    if (lds > 160 * 1024 || (ay.ztiled && ay.tile_w != 16)) return hipErrorInvalidValue;
    auto kern = fwd ? k_plane_mm<1> : k_plane_mm<0>;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
    }
    const unsigned blocks = ax.items ? (unsigned)ax.nlines : (unsigned)ax.nz;  // batched: the item count
    const unsigned threads = 64u * (unsigned)(ax.items ? waves : plane_waves(ax.nx, ax.ny, kx, ky));
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(threads), lds, s, ax, ay, kx, ky, ps);
    return hipGetLastError();
}

}  // namespace pp
