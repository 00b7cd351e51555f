// Host-side engine of the MI355X SnuSolver path: device state of one matrix
// (struct snumat), the launch lists of its factorization and solves, and the
// executors that run a set of matrices (one, or a batch) with one launch per
// step across all of them.
#pragma once
#include <hip/hip_runtime.h>

#include <climits>
#include <string>
#include <type_traits>
#include <vector>

#include "snu_internal.h"
#include "snu_kernels.h"

#define HIPCHK(x)                                                          \
  do {                                                                     \
    hipError_t e_ = (x);                                                   \
    if (e_ != hipSuccess)                                                  \
      return snu::set_error(SNU_ERR_HIP, std::string("HIP error ") +       \
                                             hipGetErrorString(e_) + " at " #x); \
  } while (0)

namespace snu {

// One grouped launch.  key orders the launches of one matrix; launches of
// several matrices with equal (key, kind) are independent and are merged
// into one launch.
struct Launch {
  int kind;  // 0 diagonal blocks and their panels (tiles: panel workgroups); GEMM (64 tile) 1: C = AB, 2: C -= AB, 6: C = -AB;
             // GEMM (128 tile) 5: C -= AB, 10: C = AB, 11: C = -AB; 3: copy
             // C = A (GEMM descriptors, 64 x 64 tiles); GEMV 7: y = Ax, 8: y -= Ax
             // (one column), 17 / 18: the same on groups of 16 columns
  int p0, np, tiles;
  double flops;
  long long key;
  int wgs = 0;          // GEMV: workgroups (one column: of the split-K partial pass, 0: unsplit)
  long long part = 0;   // GEMV: partial-sum values of the launch (0: unsplit)
  int gstep = 1, groups = 1;  // 16 columns: groups per workgroup, most groups of a problem
};
inline bool is_gemm(int kind) {
  return kind == 1 || kind == 2 || kind == 5 || kind == 6 || kind == 10 || kind == 11;
}
// C = +-AB launches (products by triangular inverses) as opposed to C -= AB
inline bool is_assign_gemm(int kind) { return kind == 1 || kind == 6 || kind == 10 || kind == 11; }

// Launch list with its descriptors (device copies once uploaded).
template <typename T>
struct DensePlan {
  std::vector<DiagProbT<T>> dp;
  std::vector<GemmProbT<T>> gp;
  std::vector<GemmSegT<T>> gs;
  std::vector<Launch> launches;
  DiagProbT<T> *d_dp = nullptr;
  GemmProbT<T> *d_gp = nullptr;
  GemmSegT<T> *d_gs = nullptr;
};
template <typename T>
struct GemvPlan {
  std::vector<GemvProbT<T>> vp;
  std::vector<GemvSegT<T>> vs;
  std::vector<Launch> fwd, bwd;
  GemvProbT<T> *d_vp = nullptr;
  GemvSegT<T> *d_vs = nullptr;
  T *d_part = nullptr;            // split-K partial sums (launches run in turn)
  int *d_done = nullptr;          // their arrival counters (0 between launches)
  size_t cap_vp = 0, cap_vs = 0, cap_part = 0, cap_done = 0;  // device capacities (grow-only)
};

// Multifrontal leaf factorization of a launch set (one matrix, or a batch
// merged): per height of the leaves' front trees, the fronts the LDS kernel
// takes whole and the larger fronts' extend-add tiles; the larger fronts'
// blocked partial LU as a keyed launch list (key: height, step within it);
// the extend-add tiles of the separator blocks (after the last height).
struct FrontLevel {
  // small fronts from small0 on, by class: orders up to kFrontWave, up to
  // kFrontLo, above; the largest order of each
  int small0 = 0, nsmall[3] = {0, 0, 0}, max_f[3] = {0, 0, 0};
  int tile0 = 0, ntile = 0;
};
template <typename T>
struct FrontPlan {
  std::vector<FrontDev> small;
  std::vector<AddTile> tiles;  // by height, then the separator tiles
  std::vector<AddSrc> src;
  int sep0 = 0;             // first separator tile
  std::vector<FrontLevel> levels;
  DensePlan<T> dense;
  FrontDev *d_small = nullptr;
  AddTile *d_tiles = nullptr;
  AddSrc *d_src = nullptr;
};
// Values kept behind a front for its pivot blocks (kFrontInv; larger fronts).
inline long long front_inv_size(int f, int nk, int fmax) {
  return f > fmax ? (nk + 63) / 64 * (long long)kFrontInv : 0;
}
inline long long front_key(int height, int step, int kind) {
  return (long long)height * 100000000LL + step * 8LL + kind;
}
inline int front_key_height(long long key) { return (int)(key / 100000000LL); }

// Value-typed device state of one matrix (FP64, or FP32 refined in FP64).
template <typename T>
struct Values {
  T *arena = nullptr;  // the separators' dense blocks
  T *inv = nullptr;    // per separator: full L^-1 then U^-1 (s x s each)
  T *lu = nullptr;     // per separator: LU of its 64 x 64 diagonal blocks
  T *tmp = nullptr;    // products of a level's panels, then of its triangular inversion
  T *farena = nullptr; // leaf fronts (each f x f, a larger one's pivot blocks behind it)
  FrontPlan<T> fronts;
  DensePlan<T> fact;
  // standalone solves: right-hand sides, dense-solve vectors (separator rows
  // alone), the fronts' update rows; w1: update rows of one column (allocation-free solves)
  T *bp = nullptr, *ys = nullptr, *wbuf = nullptr, *w1 = nullptr;
  int plan_nrhs = -1;
  GemvPlan<T> sp;
  // allocation-free solves: the same plan over buffers in the library's
  // static per-device scratch (its device pointers point into the scratch
  // and are never freed)
  GemvPlan<T> sp_scratch;
  int scratch_nrhs = -1;
  bool scratch_own_w = true;
  int scratch_over = INT_MAX;  // columns known not to fit the scratch as groups
};

// Tables of a standalone solve, one copy to the device.
struct SolveTab {
  VecDev vec;
  PermDev perm;
  IrDev ir;  // (SNU_FP32)
};

// Host copies of the per-leaf work lists (kept for batching).
struct WorkLists {
  std::vector<TargetDev> targets;  // separator rows receiving leaf contributions
  std::vector<int> tsrc;           // their sources: update rows of root fronts
};

// Device copies of the work lists of a launch set (one matrix or a batch).
struct WorkDev {
  LeafDev *leaves = nullptr;
  int nleaves = 0;
  TargetDev *targets = nullptr;
  int *tsrc = nullptr, ntarget = 0;
};

// Second stream of a factorization: the next height's diagonal blocks while the
// Schur updates that they do not need run.  One per matrix or batch that has
// work for it (make_side), made right after the owner's first stream: streams
// made one after the other get different hardware queues (made at the first
// factorization, with several handles alive, it shared its owner's, and
// nothing overlapped).
struct SideStream {
  hipStream_t st = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
};
// What a launch of the dense plan does to it, before it runs (kSideJoin: the
// first stream waits for the second; kSideFork: the second waits for the
// first), and whether it runs on it.
enum { kSideJoin = 1, kSideFork = 2, kSideRun = 4 };
// A factorization's launch sequence captured once into a HIP graph and
// replayed (no memset nodes: buffers are cleared by kernels).
struct FactorGraph {
  hipGraphExec_t exec = nullptr;
};

}  // namespace snu

struct snumat {
  snu::Plan P;
  snu_opts_t opts;
  int prec = SNU_FP64;
  bool on_device = false;
  bool factored = false;
  bool staged = false;  // a factorize_stage ran on the current values
  bool scattered = false;  // and it was stage 0: the fronts hold no factors
  int device = -1;
  hipStream_t stream = nullptr;
  std::vector<void *> allocs;
  size_t dev_bytes = 0;
  long long arena_len = 0;
  double *d_aval = nullptr;  // A's values in the caller's CSR order (FP64)
  long long *d_adest = nullptr;  // A's separator entries: place in the arena,
  int *d_asrc = nullptr;         // index in A's values
  long long nsep_ent = 0;
  std::vector<long long> leaf_foff;  // first front value of each leaf (np + 1)
  int *d_arow = nullptr, *d_acol = nullptr;  // A's pattern (refinement residuals)
  int *d_order = nullptr;
  // leaves and work lists
  std::vector<snu::LeafDev> h_leaves;  // vec = 0
  snu::WorkLists wl;
  snu::WorkDev wd;
  int wrows = 0;       // update rows of the leaf fronts (solves)
  // dense tables
  std::vector<long long> inv_off, lu_off;
  std::vector<int> sep_rows;  // separator rows before each separator (at np: all)
  long long inv_total = 0, tmp_panels = 0, tmp_inversion = 0;
  snu::Values<double> v64;
  snu::Values<float> v32;
  // standalone solves
  double *d_bx = nullptr;  // staging for host-pointer solves,
  int stage_cap = 0;       // columns it holds
  size_t alloc_limit = ~size_t(0);  // larger device allocations fail (tests)
  unsigned long long *d_norms = nullptr;     // |A|inf (bits of a double)
  double *d_colnorms = nullptr;              // refinement column norms (norm_values)
  int *d_active = nullptr;
  snu::SolveTab *d_tab = nullptr;  // the tables of a standalone solve
  snu::PrepDev *d_prep = nullptr;
  double anorm = 0;
  int nrhs_cap = 0;
  int ir_steps = 0;
  double ir_berr = 0;
  // timing
  bool profile = false;
  bool use_graph = false;
  snu::FactorGraph graph;
  snu::SideStream side;
  std::vector<hipEvent_t> ev, pev;
  double t[16] = {0};
  // C -= AB launches by tile: 64 x 64 (time ms, launches, GFLOP), then 128 x 128
  double gsplit[6] = {0};
  // SNU_FP32: FP64 factorization of the same matrix on the same device, built
  // and factorized on the first solve whose refinement stalls above 1e-12,
  // refactorized after every new factorization of this handle
  snumat *fb64 = nullptr;
  bool fb64_current = false;
};

namespace snu {

template <typename T>
Values<T> &vals(snumat *h) {
  if constexpr (std::is_same<T, double>::value) return h->v64;
  else return h->v32;
}
template <typename T>
const Values<T> &vals(const snumat *h) {
  if constexpr (std::is_same<T, double>::value) return h->v64;
  else return h->v32;
}

int upload(snumat *h);
// The multifrontal plan of one uploaded matrix (value arrays allocated).
template <typename T>
int build_front_plan(snumat *h);
// Merge the front plans of several matrices into out's host tables (per
// height: their fronts side by side; dense launches merged by key).
template <typename T>
void merge_fronts(const std::vector<const FrontPlan<T> *> &in, FrontPlan<T> &out);
// GEMM tile (64 or 128) for a C block of M x N, by precision; autotune_tiles
// measures the table once per process (on the current device)
template <typename T>
void autotune_tiles();
int tile_for(int prec, int M, int N);
int tile_table(int prec, int *out3);
void free_device(snumat *h);
size_t estimate_device_bytes(const snumat *h);
int device_alloc(snumat *h, void **p, size_t bytes);
float ev_ms(hipEvent_t a, hipEvent_t b);

// Append problem C (M x N) -= / = sum_seg A_seg B_seg to a grouped GEMM
// launch with tb x tb tiles; returns 1 if a problem was added.
template <typename T>
int add_gemm(std::vector<GemmProbT<T>> &gp, std::vector<GemmSegT<T>> &gs, int &tiles,
             T *C, long long ldc, int M, int N, const std::vector<GemmSegT<T>> &segs,
             double &flops, int tb = 64);

// GEMV plan of one matrix's dense solves into the packed vectors bp / ys at
// this matrix's segment (VecDev form, nrhs columns); keys order fwd / bwd.
template <typename T>
void build_solve_plan(const snumat *h, T *bp, T *ys, int nrhs, GemvPlan<T> &out);
// Copy the plan's descriptors to the device on stream st, growing the
// device arrays only when they are too small (the host vectors must stay
// unchanged until st has passed the copy).
template <typename T>
int upload_gemv_plan(GemvPlan<T> &g, hipStream_t st = nullptr);
// The split-K layout of the plan's launches (no device work); returns the
// partial-sum values and the arrival counters its largest launch needs.
struct SplitNeed {
  size_t part = 0, done = 0;
};
template <typename T>
SplitNeed layout_gemv_plan(GemvPlan<T> &g);
template <typename T>
void free_gemv_plan(GemvPlan<T> &g);
template <typename T>
int upload_dense_plan(DensePlan<T> &d);
template <typename T>
void free_dense_plan(DensePlan<T> &d);

// Merge the launch lists of several matrices: launches with equal (key,
// kind) become one launch over the concatenated problems.
template <typename T>
void merge_dense(const std::vector<const DensePlan<T> *> &in, DensePlan<T> &out);
template <typename T>
void merge_gemv(const std::vector<const GemvPlan<T> *> &in, GemvPlan<T> &out);

// Executors over a launch set.
struct FactorSet {
  SideStream *side = nullptr;  // (null: one stream)
  int nmat;
  const PrepDev *prep = nullptr;  // scatter_only: its table, largest arena and entries
  long long max_len = 0, max_nnz = 0;
  const IrDev *ir;           // FP32 only: |A| norms into anorm_out
  unsigned long long *anorm_out;
  int max_n;
  const void *fronts;  // FrontPlan of the set's value type
  double eps;
  bool split = false;  // FP32: GEMM tiles through bf16 splits (SNU_GEMM_SPLIT)
  bool scatter_only = false;  // A's values into place, nothing factored
};
// graph (optional, not with profile): capture the launches on the first
// call, replay them afterwards; the phase events then all mark the end.
template <typename T>
int run_factor(const FactorSet &fs, const DensePlan<T> &plan, hipStream_t st,
               const std::vector<hipEvent_t> *ev, bool profile, std::vector<hipEvent_t> *pev,
               double *gemm_ms, FactorGraph *graph = nullptr);
void free_graph(FactorGraph &g);
// (no stream if no height of the plans, taken together, has work for it)
template <typename T>
int make_side(const std::vector<const DensePlan<T> *> &in, SideStream &s);
void free_side(SideStream &s);
// Per launch of the plan, the kSide* flags; at its end the first stream waits
// for the second once more.
template <typename T>
std::vector<int> side_schedule(const DensePlan<T> &plan);
// The dense plan of a handle (built for the structure alone if the handle is
// on no device).
template <typename T>
const DensePlan<T> &plan_of(snumat *h);
struct SolveSet {
  const PermDev *perm;
  const VecDev *vec;
  int nmat;
  long long max_elems;  // largest n x groups of a matrix
  int max_groups;
  bool one, many;       // matrices with one / several columns present
  const WorkDev *wd;
};
// Forward and backward sweep over the packed vectors.
template <typename T>
void run_sweep(const SolveSet &ss, T *bp, T *wbuf, const GemvPlan<T> &plan, hipStream_t st);
// b into the packed vectors, the sweep, x out of them.
template <typename T>
void run_solve(const SolveSet &ss, T *bp, T *wbuf, const GemvPlan<T> &plan, hipStream_t st);
struct RefineSet {
  SolveSet sweep;
  const IrDev *ir;
  int nmat, max_n;
  double *norms;  // norm_values(): column maxima of |b|, |r|, |x|, then workgroups' maxima
  int nslots;
  const std::vector<int> *slot_mat;   // matrix of each column slot
  const std::vector<double> *anorm;   // |A|inf per matrix
  int *d_active;                      // nmat flags
  int max_steps;
  double tol;
};
int run_refined(const RefineSet &rs, float *bp, float *wbuf, const GemvPlan<float> &plan,
                hipStream_t st, int *steps_out, std::vector<double> *berr_mat);

// Buffers of one standalone solve: the permuted right-hand sides and the
// leaf fronts' update rows (value type of the handle), the dense-solve launch
// plan with its device descriptors, and (SNU_FP32) the column norms of the
// refinement.
struct SolveBuffers {
  void *bp = nullptr, *wbuf = nullptr;
  const void *plan = nullptr;  // GemvPlan<T> of the handle's value type
  double *colnorms = nullptr;
};
// Solve with device pointers (caller's b / x, column-major) on the given
// buffers, on the handle's stream; returns when the work is done.  fallback:
// a refinement that stalls above 1e-12 is answered by the handle's FP64 twin
// (built on first need); otherwise SNU_ERR_NOT_CONVERGED is returned with x
// holding the last iterate.
int solve_core(snumat *h, const double *d_b, long long ldb, double *d_x, long long ldx, int nrhs,
               const SolveBuffers &B, bool fallback);
// x = A^-1 b with FP64 factors of an SNU_FP32 handle's matrix (its FP64
// twin: same plan, FP64 arena, the handle's current values; built and
// factorized on first need, refactorized after the handle's next
// factorization); returns when the work is done.
int fp64_fallback_solve(snumat *h, const double *d_b, long long ldb, double *d_x, long long ldx, int nrhs);

}  // namespace snu
