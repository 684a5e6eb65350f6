// pp_noalloc.h -- where the tables of pp_solve_device_oop_noalloc lie in its fixed device array (host code).
//
// Small solves' tables and dense-product matrices take some 0.1 MB of the 2 MiB; matrices of long lines
// take 8 N^2 bytes.  An axis whose matrices do not fit beside the others' tables runs as the chirp
// convolution (45 thousand doubles at most); the largest go first, so the axes that lose their products are
// as few as can be: 101 x 509 x 97 keeps its x products (238 us a solve with both, 357 with neither, 306
// with those of x).
#pragma once
#include "pp_plane_mm.h"
#include "pp_setup.h"

namespace pp {

constexpr size_t kScratchDoubles = 256 * 1024;  // 2 MiB per GPU

// offsets (doubles)
struct NoallocTables {
    size_t tab[2][5] = {};  // tw, A, B, C, D per axis
    size_t ztab[5] = {};    // periodic z in three passes: real z-line tables
    size_t lamx = 0, lamy = 0, dtab = 0, ztw = 0, zA = 0, zc2 = 0;
    // dense-product lines (x, y, periodic z): where their matrices are written (0: none) and
    // their octant tables
    size_t mm[3] = {}, oct[3] = {};
    size_t used = 0;  // doubles copied from the host; the matrices lie behind
};

// lines of axis a (0 x, 1 y; 2 periodic z) that are dense products, or whose matrices the handle would have
inline bool noalloc_dense(const SolveSetup &g, int a)
{
    if (a == 2) return mm_serves(g.nz, KIND_PP, 1, g.nx * g.ny, (long)g.nx * g.ny);
    return mm_serves(a == 0 ? g.nx : g.ny, g.kind[a], a, g.nx, (long)(a == 0 ? g.ny : g.nx) * g.nz);
}
inline bool noalloc_matrices(const SolveSetup &g, int a, bool one_pass)
{
    if (a == 2) return g.zper && !one_pass && noalloc_dense(g, 2);
    return noalloc_dense(g, a) || mm_plane(g.nx, g.ny, g.kind[0], g.kind[1]);
}

// one_pass: periodic z of this length needs no z lines.  False where the tables exceed the array
inline bool noalloc_layout(const SolveSetup &g, bool one_pass, NoallocTables &r)
{
    const int n[3] = {g.nx, g.ny, g.nz}, kind[3] = {g.kind[0], g.kind[1], KIND_PP};
    bool mm[3];
    for (int a = 0; a < 3; a++) mm[a] = noalloc_matrices(g, a, one_pass);
    for (;;) {
        NoallocTables t;
        size_t o = 0;
        auto take = [&](size_t count) {
            const size_t at = o;
            o += (count + 31) / 32 * 32;  // 256-byte aligned sub-arrays
            return at;
        };
        auto lines = [&](int a, size_t *tab) {
            const AxisTableSizes z = axis_table_sizes(n[a]);
            for (int i = 0; i < 5; i++) tab[i] = take(z.n[i]);
        };
        for (int a = 0; a < 2; a++) {
            if (mm[a]) t.oct[a] = take(mm_octant_size(n[a]));
            if (!mm[a] || !noalloc_dense(g, a)) lines(a, t.tab[a]);
        }
        t.lamx = take((size_t)g.nx);
        t.lamy = take((size_t)g.ny);
        t.dtab = take(dirichlet_table_size(g));
        if (g.zper) {
            if (one_pass) {
                t.ztw = take((size_t)g.nz);
                t.zA = take((size_t)g.nz + 2);
            } else if (mm[2]) {
                t.oct[2] = take(mm_octant_size(g.nz));
            } else {
                lines(2, t.ztab);
            }
            t.zc2 = take((size_t)g.nz);
        }
        t.used = o;
        int largest = -1;
        for (int a = 0; a < 3; a++) {
            if (!mm[a]) continue;
            t.mm[a] = take(mm_tables_size(n[a], kind[a]));
            if (largest < 0 || mm_tables_size(n[a], kind[a]) > mm_tables_size(n[largest], kind[largest])) largest = a;
        }
        if (o <= kScratchDoubles) {
            r = t;
            return true;
        }
        if (largest < 0) return false;
        mm[largest] = false;
    }
}

}  // namespace pp
