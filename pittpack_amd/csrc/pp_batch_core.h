// pp_batch_core.h -- the engine of the batched form, shared by pp_batch (one batch, its own
// device memory) and pp_server (many batches in flight, memory from one pool).
//
// A batch is planned on the host (member offsets, per-member descriptors, per-launch block
// items), then bound to one contiguous device region, uploaded asynchronously and run on a
// stream.  Every stage is one launch per shape class: line length and transform kind for
// the x and y transforms, rows per lane for the z solve.
#pragma once
#include <hip/hip_runtime.h>

#include <array>
#include <map>
#include <set>
#include <vector>

#include "pp_launch.h"
#include "pp_line.h"
#include "pp_line_mm.h"
#include "pp_mixed.h"
#include "pp_plane_mm.h"
#include "pp_setup.h"
#include "pp_zsolve.h"

namespace pp {

struct AxisDev {
    double *tw = nullptr, *A = nullptr, *B = nullptr, *C = nullptr, *D = nullptr;
    const double *mm = nullptr, *mmi = nullptr;  // dense-product matrices
};

// FP64 tables per line length (and, dense products, symmetry family), resident on the device
// until destruction
class TableCache {
  public:
    ~TableCache();
    // tables of lines of length N (dense: as products of `kind`)
    int get(int N, int kind, bool dense, AxisDev &out);
    // dense-product matrices of (N, kind): where the caller has placed them, else allocated
    int get_mm(int N, int kind, const double *&mm, const double *&mmi);
    // ... in the caller's memory (mm_bytes, 256-byte aligned) until drop_mm; kinds of one family share them
    static size_t mm_bytes(int N, int kind);
    int place_mm(int N, int kind, char *at);
    void drop_mm(int N, int kind) { m_.erase({N, mm_family(kind)}); }

  private:
    struct Matrices {
        double *own = nullptr;  // its allocation (null: placed by the caller)
        const double *mm = nullptr, *mmi = nullptr;
    };
    int write_mm(int N, int kind, double *base, Matrices &e);
    std::map<int, AxisDev> t_;  // by length; -length: periodic z only
    std::map<std::pair<int, int>, Matrices> m_;  // {length, symmetry family}
};

// events recorded between the launches of one run (null ev: no timing)
struct Marks {
    hipEvent_t *ev = nullptr;
    int n = 0, max = 0;
};

// Streams beside a batch's own on which the classes of a stage run at the same time while a solve is
// captured: branches of its graph.  A class' launch fills the chip only in its middle, and 48 members
// of 16..96 points a side are some 70 launches of 6 to 65 us: 1.68 ms in series, 1.28 to 1.37 ms over four
// branches (mixed form 4.25 and 3.61; 200 members 4.1 and 3.6, 1000 members 19.6 and 19.5).  A stage's split
// and merge cost some 15 us, so batches under kMinPoints stay in series (4.7 million points: 0.21 in
// series, 0.26 over branches; 12.3 million: 0.51 and 0.43, 13.0 million: 0.41 and 0.40); launched one by one
// they cost more (4.7 million points: 0.37 ms), so there is no such split outside a graph.
struct BatchLanes {
    static constexpr long kMinPoints = 10000000;
    static constexpr int kSide = 3;  // with the batch's own, the process' four hardware queues
    hipStream_t side[kSide] = {};
    hipEvent_t fork = nullptr, join[kSide] = {};
    int create();  // PP code; nothing is left behind on failure
    void destroy();
    // work launched on `s` so far happens before the side streams' / the side streams' before `s`'
    hipError_t split(hipStream_t s);
    hipError_t merge(hipStream_t s);
};

// Matrices of lines of up to this many points count as tables (35 KB at most, some 2 MB if every length
// and family of them is met); longer ones take some 8 N^2 bytes (the real DFT's 4 N^2), 4.8 GB all
// together, which a server places in its pool (pp_server.hip)
constexpr int kMmResident = 64;

struct BatchMember {
    SolveSetup g;
    long offset = 0;  // element offset of the member's field in the rhs / solution / work arenas
    long lam_off[2] = {0, 0};
    long dtab_off = 0;
    bool pinned = false;  // mixed form: pinned (0,0) column solved in FP64 from plane sums
    long sums_off = 0, plane_off = 0, upart_off = 0;
    bool dense = true;   // may multiply with matrices of more than kMmResident points
    bool plane = false;  // FP64: both transforms of a plane in one launch (pp_plane_mm.h)
    long toff = 0;  // FP64: offset of the member's z tiles in the tile arena (-1: none)
};

class BatchCore {
  public:
    // options (set before plan)
    int precision = 0;  // 0 FP64, 1 FP32 + FP64 refinement
    int refine = 2;
    int zero_mode = 1;
    double tau = 0.05;
    double zthomas_tau = 1e-3;  // FP64: columns below it by the reference's Thomas sweeps (0: off)
    int force_var = -1;  // FP64 line classes: -1 tuned / default shapes, 0 default, 1 alternative
    int fuse_res = 1;    // mixed form: corrections fused into the x forward where a member's rows allow

    std::vector<BatchMember> mem;

    // validates and appends a member; *id = its index
    int add(int nx, int ny, int nz, const char *bc, const double *X, int *id);
    // host plan: offsets, descriptors, launch items; sets region_bytes
    int plan();
    // device pointers inside [base, base + region_bytes), table pointers from tc
    int bind(char *base, TableCache *tc);
    // asynchronous uploads of the planned tables (host copies stay alive in this object)
    int upload(hipStream_t s);
    // planned: the matrices of more than kMmResident points its lines multiply with, {length, kind} (one
    // kind of each family)
    std::set<std::pair<int, int>> matrices() const;
    // the solve of every member (right-hand sides kept, solutions in the solution arena)
    int run(hipStream_t s, Marks *mk);
    BatchLanes *lanes = nullptr;  // a captured run's stages, class by class over these (null: in series)
    // FP64: time each line class in both launch shapes on this batch (bound, uploaded) and
    // keep the faster per class and direction; the right-hand-side arena is overwritten
    int tune_lines(hipStream_t s);
    int alt_classes() const;

    long long points() const;
    size_t region_bytes = 0;
    bool planned = false, bound = false;

    // device pointers (valid after bind)
    double *d_rhs = nullptr, *d_sol = nullptr;
    double *d_tiles = nullptr;  // FP64: z tiles between the y transforms and the z solve
    float *d_w = nullptr;
    float *d_u0 = nullptr, *d_cacc = nullptr;  // mixed form: the solution's FP32 parts while refined
    long arena_elems = 0;
    int launches[3] = {0, 0, 0};

  private:
    struct HostClass {
        int key = 0, kind = 0, nitems = 0;
        bool dense = false;  // line classes: dense products (mm), not a plan or convolution
        MmPlan mm{};  // dense-product line classes: the launch shape
        std::vector<LineItem> li;
        std::vector<ZItem> zi;
        size_t off = 0;
        void *d_items = nullptr;
        // FP64 line classes: launch shape per direction (forward, inverse) and, for x, the
        // block items of the alternative shape (its lines per block differ)
        int var[2] = {0, 0};
        std::vector<LineItem> li_alt;
        size_t off_alt = 0;
        void *d_items_alt = nullptr;
        int th_first = 0, th_count = 0;  // FP64 z classes: their Thomas columns in zth_
        size_t lds = 0;      // plane classes: of their largest plane
        int lane = 0;        // stream of the class within its stage (0: the batch's own)
        bool fused = false;  // correction x classes: members whose residual runs in k_resx
    };
    // are the member's lines along axis a (0 x, 1 y; 2 periodic z without a plan) dense products?
    static bool dense(const BatchMember &m, int a);
    hipStream_t lane(hipStream_t s, int k) const { return forked_ && k > 0 ? lanes->side[k - 1] : s; }
    void plan_lanes(std::initializer_list<std::vector<HostClass> *> stage);
    int launch_class(hipStream_t s, const HostClass &c, int form, int axis, int fwd, const void *in, void *out,
                     int bflags, double *sums, const double *plane, int accumulate, int ztiled,
                     const float *acc0 = nullptr, const float *acc1 = nullptr);
    template <typename R>
    int plan_lines(int axis, std::vector<HostClass> &out);
    void plan_z();
    int plan_mixed();
    int run_line_stage(hipStream_t s, std::vector<HostClass> &cls, int form, int axis, int fwd, const void *in,
                       void *out, int bflags, double *sums, const double *plane, int accumulate, int ztiled = 0,
                       const float *acc0 = nullptr, const float *acc1 = nullptr);
    int run_z_stage(hipStream_t s, bool f32);
    template <typename F>
    int run_stage(hipStream_t s, size_t classes, const F &launches);
    size_t z_classes() const { return lz_.size() + lzp_.size() + zlong_.size() + zpl_.size(); }
    int run_z_columns(hipStream_t s);
    int run_planes(hipStream_t s, int fwd);
    int run_fp64(hipStream_t s, Marks *mk);
    int mixed_inner(hipStream_t s, Marks *mk);
    int run_mixed(hipStream_t s, Marks *mk);

    // host copies of everything uploaded
    std::vector<double> lam_, dtab_;
    std::vector<LineSolve> ls_;
    std::vector<ZSolve> zs_;
    std::vector<HostClass> lx_, ly_, lz_;
    std::vector<HostClass> lp_;  // FP64: plane launches, items {member, z}, by waves a block
    bool forked_ = false;        // inside run_stage, over the side streams
    std::vector<PlaneSolve> ps_;
    PlaneSolve *d_ps_ = nullptr;
    size_t o_ps_ = 0;
    // mixed form: the corrections' x forward, each x class split into the members whose
    // residual is computed inside it (k_resx: ny a multiple of its lines per block, as the
    // single-solve handle decides) and the rest (residual kernel, then the FP32 transform)
    std::vector<HostClass> lxc_;
    std::vector<char> mfused_;
    // periodic z: one-pass classes (key nz, a compiled complex plan; items {member, column
    // block, y row}), members of other lengths (real z-line transforms, one launch each), the
    // singular columns of FP64 members, and 2 cos(2 pi k / nz) per distinct periodic length
    std::vector<HostClass> lzp_;
    std::vector<int> zpl_;
    std::vector<SmtItem> smt_;
    std::vector<double> zc2_;
    std::map<int, long> zc2_off_;
    // FP64 members with 513..1024-row columns: the long-column kernel, one launch each
    std::vector<int> zlong_;
    // FP64: nearly singular columns of the PCR classes' members, solved by the reference's
    // Thomas sweeps in blocks of their z class' launch, and their factor tables
    std::vector<ZThomasItem> zth_;
    std::vector<double> zth_tab_;
    std::vector<int4> fix_;
    std::vector<HostClass> lfix_;  // 16-column tiles holding near-singular columns, per J
    std::vector<Mode00Item> m00_;
    std::vector<int> m00_mem_;  // member of each m00_ entry
    std::vector<ResArgs> res_;
    std::vector<int4> ritems_;   // residual tiles of odd-nx members (64 columns)
    std::vector<int4> rpitems_;  // residual tiles of even-nx members (two cells per lane, 128 columns)
    bool res_two_ = false;   // some odd-nx member's residual tiles need the second halo load
    bool resp_two_ = false;  // some even-nx member has ny = 1 (mod 4)
    int nz_max_ = 0;
    long nsums_ = 0, nplane_ = 0, nupart_ = 0, ntiles_ = 0;
    // region layout (byte offsets)
    size_t o_zth_ = 0, o_zth_tab_ = 0, o_u0_ = 0, o_cacc_ = 0, o_zc2_ = 0, o_smt_ = 0, o_rhs_ = 0, o_sol_ = 0, o_tiles_ = 0, o_w_ = 0, o_lam_ = 0, o_dtab_ = 0, o_ls_ = 0, o_zs_ = 0, o_sums_ = 0, o_plane_ = 0,
           o_upart_ = 0, o_fix_ = 0, o_m00_ = 0, o_res_ = 0, o_ritems_ = 0, o_rpitems_ = 0;
    std::map<std::array<int, 3>, AxisDev> tabs_;  // {length, kind, dense}; kind -1: periodic z
    // device pointers of the tables
    double *d_lam_ = nullptr, *d_dtab_ = nullptr, *d_sums_ = nullptr, *d_plane_ = nullptr, *d_upart_ = nullptr;
    LineSolve *d_ls_ = nullptr;
    ZSolve *d_zs_ = nullptr;
    int4 *d_fix_ = nullptr, *d_ritems_ = nullptr, *d_rpitems_ = nullptr;
    double *d_zc2_ = nullptr;
    ZThomasItem *d_zth_ = nullptr;
    double *d_zth_tab_ = nullptr;
    SmtItem *d_smt_ = nullptr;
    int smt_nz_max_ = 0;

    Mode00Item *d_m00_ = nullptr;
    ResArgs *d_res_ = nullptr;
};

}  // namespace pp
