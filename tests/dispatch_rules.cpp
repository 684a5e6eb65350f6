// The host rules that choose a transform's kernel, for tests/test_dispatch_rules.py: built for the host alone.
#include <type_traits>

#include "pp_noalloc.h"
#include "pp_resx.h"
#include "pp_zper.h"

using namespace pp;

// (a kind in the place of the route would look like dense products for all kinds but one)
static_assert(!std::is_invocable_v<decltype(line_lines_any<double>), int, int, int>);

extern "C" {

// 1 dense products, 0 a compiled plan or the chirp convolution
int rule_dense(int n, int kind, int axis, int cols, long lines) { return mm_serves(n, kind, axis, cols, lines); }
int rule_plane(int nx, int ny, int kx, int ky) { return mm_plane(nx, ny, kx, ky); }
// columns of an FP64 y block of the launch that serves the line
int rule_y_block(int n, int kind, int cols, long lines)
{
    return line_lines_any<double>(n, line_route(n, kind, 1, cols, lines), 1);
}
// lanes a line's staging takes in an x launch
int rule_stage_lanes(int n, int kind)
{
    const int d = mm_depth8(n, mm_family(kind));
    return d <= 8 ? 8 : d <= 16 ? 16 : d <= 32 ? 32 : 64;
}

// waves that a dense launch over `units` units of 16 lines / columns brings to the chip
long rule_dense_waves(int n, int kind, int axis, long units)
{
    const MmPlan p = mm_plan(n, kind, axis, units);
    return (units + p.units - 1) / p.units * p.waves;
}

// threads a block, and LDS slots a column, of the one-pass periodic z solve of nz rows (0: other lengths)
int rule_zper(int nz, int *slots)
{
    switch (nz / 2) {
#define PPM(m) case m: *slots = zper_slots<m>(); return zper_threads(m) * zper_lines_m<m>();
        PP_ZPER_LENGTHS(PPM)
#undef PPM
    default: return 0;
    }
}
// elements a thread holds of a line of n points in the fused correction step
int rule_resx_elements(int n) { return n / 2 / resx_threads(n / 2); }

// the layout of the no-allocation entry point: 0 where it does not fit, else a bit for each axis with its
// matrices; ends[i] of starts[i] .. ends[i]: its sub-arrays (*count of them), in doubles
int rule_noalloc(int nx, int ny, int nz, const char *bc, int one_pass, long *starts, long *ends, int *count, long *room)
{
    SolveSetup g;
    g.nx = nx;
    g.ny = ny;
    g.nz = nz;
    if (setup_boundary(g, bc)) return -1;
    NoallocTables t;
    *count = 0;
    *room = (long)kScratchDoubles;
    if (!noalloc_layout(g, one_pass != 0, t)) return 0;
    const int n[3] = {nx, ny, nz}, kind[3] = {g.kind[0], g.kind[1], KIND_PP};
    auto add = [&](size_t at, size_t len) {
        starts[*count] = (long)at;
        ends[(*count)++] = (long)(at + len);
    };
    int bits = 8;
    for (int a = 0; a < 3; a++) {
        const bool lines = a < 2 ? !(t.mm[a] && noalloc_dense(g, a)) : g.zper && !one_pass && !t.mm[a];
        const AxisTableSizes z = axis_table_sizes(n[a]);
        for (int i = 0; lines && i < 5; i++) add(a < 2 ? t.tab[a][i] : t.ztab[i], z.n[i]);
        if (!t.mm[a]) continue;
        bits |= 1 << a;
        add(t.oct[a], mm_octant_size(n[a]));
        add(t.mm[a], mm_tables_size(n[a], kind[a]));
    }
    add(t.lamx, nx);
    add(t.lamy, ny);
    add(t.dtab, dirichlet_table_size(g));
    if (g.zper) {
        add(t.zc2, nz);
        if (one_pass) {
            add(t.ztw, nz);
            add(t.zA, nz + 2);
        }
    }
    return bits;
}

}  // extern "C"
