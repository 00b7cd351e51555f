// Device-side descriptors and kernel launchers of the MI355X SnuSolver path.
// Value-carrying kernels are templated on the value type T (double for the
// FP64 path, float for the FP32 factorization refined in FP64); launchers are
// instantiated for both in snu_kernels.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace snu {

// Solve work of the leaf fronts.  A unit is what one wave does between two
// barriers: a whole front (orders the LDS factor kernel takes), or of a larger
// front one 64-pivot block (forward or backward), one 64-row tile of its
// boundary rows (forward) or one 64-pivot block's product with a chunk of its
// boundary columns (backward).
enum SolveUnitKind { kFwdFront = 0, kFwdPivots, kFwdRows, kBwdFront, kBwdCols, kBwdPivots };
struct SolveUnit {
  const void *F, *inv;       // the front (column-major), a larger one's pivot blocks (kFrontInv)
  int ld, nk, nb;            // front order, pivots, boundary entries B
  int kpos;                  // solve position of the first pivot (pivots are consecutive)
  int wrow;                  // first row of the front's update vector
  int pull;                  // first entry of the front's rows in pull
  int bidx;                  // first entry of B in bidx
  int kind;
  int row0;                  // kFwdRows: first row of the tile
  int s, q, nq;              // pivot block; column chunk and chunks per block (kBwdCols, kBwdPivots)
};
// One leaf (one reference rank) of one matrix: device pointers into the
// owning matrix's arrays, so that leaves of several matrices can share a
// launch.
struct LeafDev {
  const SolveUnit *units;                // the leaf's solve units, by phase
  const int *fphase, *bphase;            // bounds of the forward / backward phases in units
  // per front row {s0, s1}: the children's update rows to add, in order (-1:
  // none; s1 <= -2: the list at pulllist[-2 - s1], its length first)
  const int *pull, *pulllist;
  const int *bidx;                       // solve positions of the fronts' B entries
  int nfphase, nbphase;
  int vec;                               // the matrix's slot in the launch's VecDev table
  int pad;
};
// Multifrontal leaf factorization.  A front is an f x f column-major matrix
// whose first nk rows / columns are its pivots; after its partial LU the
// trailing (f - nk) x (f - nk) block holds its update for the parent.
struct FrontChild {
  const void *U;     // the child's update block (its front at (nk, nk)), ld
  const int *rel;    // per entry of the child's B: index in this front (ascending)
  int ld, nb;        // the child's front order, |B| of the child
};
// One entry of A in a front or tile: position (from its first value), index in
// A's values.
struct AEntry {
  int pos, idx;
};
// A front factored whole in LDS.
struct FrontDev {
  void *F;                  // the front's values (f x f, column-major)
  const double *aval;       // A's values
  const AEntry *ent;        // its entries of A
  const FrontChild *child;  // children in ascending order (their updates are added in it)
  int f, nk, nent, nchild;
};
// Extend-add: one 64 x 64 tile of a target (a larger front, or a separator's
// dense block) and the pieces of update blocks that land in it, added in
// order.  pos: per entry of the update block's B, its index in the target;
// entries [rb, rb + rn) are the tile's rows at pos - r0, [cb, cb + cn) its
// columns at pos - c0.
struct AddSrc {
  const void *U;
  const int *pos;
  int ld, rb, rn, cb, cn, r0, c0, pad;
};
struct AddTile {
  void *C;
  const double *aval;
  const AEntry *ent;
  long long ldc;
  int nr, nc;               // rows, columns of the tile
  int s0, s1;               // its sources
  int nent;                 // entries of A added after them
  int pad;
};

// A matrix's right-hand sides in the packed solve vectors.  One column: n
// consecutive values at base.  Several: groups of 16 columns (the last one
// padded with zeros), each n x 16 with the columns of a row adjacent, so that
// a row is one cache line and an MFMA operand is one contiguous load.  Update
// vectors of the leaf fronts: wrows rows at wbase in the same form.
struct VecDev {
  long long base, wbase;
  int n, nrhs, wrows, pad;
};
constexpr int kColGroup = 16;
__host__ __device__ inline int vec_groups(int nrhs) {
  return nrhs <= 1 ? (nrhs > 0 ? 1 : 0) : (nrhs + kColGroup - 1) / kColGroup;
}
__host__ __device__ inline int vec_width(int nrhs) { return nrhs == 1 ? 1 : kColGroup; }
// Separator row receiving leaf contributions: the update rows [s0, s1) of
// tsrc, added in order; vec: its matrix.
struct TargetDev {
  int row, s0, s1, vec;
};
// Caller-side vectors of one matrix for the (un)permutation.
struct PermDev {
  const int *order;
  const double *b;
  double *x;
  long long ldb, ldx;
  int n, vec;
};
// Set-up of one matrix for the scatter alone: the separators' dense blocks are
// zeroed, then A's separator entries put into place.
struct PrepDev {
  void *arena;
  long long arena_len;
  const double *aval;
  const long long *adest;   // per separator entry: place in the arena
  const int *asrc;          // and index in A's values
  long long nnz;
};
// FP64 refinement of one matrix: A in its CSR order, column-major vectors.
struct IrDev {
  const int *rowptr, *colidx;
  const double *val;
  const int *order;  // solve position of each row
  const double *b;
  const double *x;
  long long ldb, ldx;
  int n, nrhs;
  int norm0;  // first slot of this matrix's columns in the norm arrays
  int vec;    // its slot in the VecDev table
};

template <typename T>
struct GemmSegT {
  const T *A, *B;
  long long lda, ldb;
  int K;
};
template <typename T>
struct GemmProbT {
  T *C;
  long long ldc;
  int M, N;
  int seg0, nseg;
  int tiles_n, tile0;
};
// One 64-column step of a blocked LU: the diagonal block D (nb x nb), whose
// factors go to LU (D itself keeps its values: several workgroups read it) and
// whose triangles' inverses to Linv / Uinv; and the panels beside it, in place:
// the m rows below D (D + nb) times U^-1, L^-1 times the m columns right of it
// (D + nb ld), 64 rows / columns per workgroup from tile0 on.
template <typename T>
struct DiagProbT {
  T *D;
  long long ld;
  int nb, m;
  T *Linv, *Uinv;  // nb x nb diagonal blocks of the full inverses
  long long ldi;
  T *LU;           // 64 x 64
  int tile0;
  T eps;           // pivots of magnitude below eps become +-eps (0: none)
};
// Its panel workgroups (one also for a block without panels).
inline int panel_tiles(int m) { return m > 0 ? 2 * ((m + 63) / 64) : 1; }
constexpr int kFrontInv = 3 * 4096;  // values per 64-pivot block of a larger front: L^-1, U^-1, LU
// y = / -= sum_seg A_seg (M x K) x_seg; tri: 0 dense, 1 lower triangular
// single segment (columns k <= row), 2 upper (k >= row).  One column
// (groups 0), or `groups` groups of 16 columns: x and y rows hold 16 adjacent
// values, consecutive groups are ldx / ldy values apart.
template <typename T>
struct GemvSegT {
  const T *A, *x;
  long long lda, ldx;
  int K;
};
template <typename T>
struct GemvProbT {
  T *y;
  long long ldy;
  int M, seg0, nseg, tri, tile0, groups;
  // split K: each segment in pieces of kGemvPiece (16 columns: kGemvPiece16)
  // columns of A, one workgroup per (64-row tile, piece) writing partial sums
  // at poff; wg0 numbers the problem's first workgroup in its launch
  int parts, wg0;
  long long poff;
};
constexpr int kGemvPiece = 128, kGemvPiece16 = 256;
using GemmSeg = GemmSegT<double>;
using GemmProb = GemmProbT<double>;
using DiagProb = DiagProbT<double>;
using GemvSeg = GemvSegT<double>;
using GemvProb = GemvProbT<double>;


template <typename T>
void launch_fill(T *p, long long n, hipStream_t st);
// zero arena, scatter A's values (one matrix per table entry)
template <typename T>
void launch_prepare(const PrepDev *tab, int nmat, long long max_len, long long max_nnz,
                    hipStream_t st);
// dst = src, bytes a multiple of 16
void launch_copy(const void *src, void *dst, long long bytes, hipStream_t st);
// mode 0: C -= sum A B; 1: C = A B; 2: C = -A B
// C = A (first segment) per problem, 64 x 64 tiles numbered as the GEMM's
template <typename T>
void launch_copy2d(const GemmProbT<T> *probs, int nprob, const GemmSegT<T> *segs, int total_tiles,
                   hipStream_t st);
template <typename T>
void launch_gemm(const GemmProbT<T> *probs, int nprob, const GemmSegT<T> *segs,
                 int total_tiles, int mode, hipStream_t st);
template <typename T>
void launch_gemm128(const GemmProbT<T> *probs, int nprob, const GemmSegT<T> *segs,
                    int total_tiles, int mode, hipStream_t st);
// FP32 128 x 128 tiles through three-piece bf16 splits on the bf16 MFMA
// (FP32-accurate; modes as launch_gemm128, same tile counts)
void launch_gemm128_split(const GemmProbT<float> *probs, int nprob, const GemmSegT<float> *segs,
                          int total_tiles, int mode, hipStream_t st);
// the same on 64 x 64 tiles (modes and tile counts of launch_gemm)
void launch_gemm_split(const GemmProbT<float> *probs, int nprob, const GemmSegT<float> *segs,
                       int total_tiles, int mode, hipStream_t st);
template <typename T>
void launch_gemm_variant(const GemmProbT<T> *probs, int nprob, const GemmSegT<T> *segs,
                         int total_tiles, int tile, int kb, int depth, hipStream_t st);
// mode 0: y -= A x; 1: y = A x
// Split-K GEMV: partial sums per (tile, piece) into part, added in fixed order
// by a tile's last workgroup.  done: an arrival counter per tile, 0 before the
// launch and after it.
template <typename T>
void launch_gemv_split(const GemvProbT<T> *probs, int nprob, const GemvSegT<T> *segs, int total_wgs, int mode,
                       T *part, int *done, hipStream_t st);
template <typename T>
void launch_gemv(const GemvProbT<T> *probs, int nprob, const GemvSegT<T> *segs,
                 int total_tiles, int mode, hipStream_t st);
// 16-column groups on MFMA; gstep groups per workgroup (1, 2 or 4); part
// non-null: split K, max_groups the most groups of a problem.
template <typename T>
void launch_gemv16(const GemvProbT<T> *probs, int nprob, const GemvSegT<T> *segs, int total_tiles,
                   int total_wgs, int gstep, int max_groups, int mode, T *part, hipStream_t st);
// Diagonal blocks and their panels (tiles: panel workgroups of all problems).
template <typename T>
void launch_diag_lu(const DiagProbT<T> *probs, int nprob, int tiles, hipStream_t st);
// Right-hand sides into / solutions out of the packed vectors; max_elems: the
// largest n x groups of the matrices.  Out: add: x += instead of x =, for the
// matrices whose active flag is set (null: all).
template <typename T>
void launch_permute_in(const PermDev *pd, int nmat, const VecDev *vd, T *bp,
                       long long max_elems, hipStream_t st);
template <typename T>
void launch_permute_out(const PermDev *pd, int nmat, const VecDev *vd, const T *bp,
                        long long max_elems, bool add, const int *active, hipStream_t st);
// Separator rows += the root fronts' update rows.
template <typename T>
void launch_assemble_rhs(const TargetDev *targets, int ntarget, const int *tsrc, const VecDev *vd,
                         const T *wbuf, T *bp, int max_groups, bool one, bool many, hipStream_t st);
// Forward / backward solve with the leaf fronts.  one / many: whether matrices
// with one / several columns are in the launch set.
template <typename T>
void launch_leaf_sweep(const LeafDev *leaves, int nleaves, const VecDev *vd, T *bp, T *wbuf,
                       int max_groups, bool one, bool many, bool bwd, hipStream_t st);

// ---- multifrontal leaf factorization ----
// Fronts held whole in LDS (f <= max_f): assembly from A's entries and the
// children's updates, partial LU with the pivot clamp, the whole front (factors
// and update block) to global memory.
template <typename T>
void launch_front_small(const FrontDev *fr, int nfront, int max_f, double eps, hipStream_t st);
// The same, one wave per front, for orders up to kFrontWave.
constexpr int kFrontWave = 48;
template <typename T>
void launch_front_wave(const FrontDev *fr, int nfront, int max_f, double eps, hipStream_t st);
// Largest front order the LDS kernel takes for this value type.
template <typename T>
int front_small_max();
// Extend-add of update blocks into target tiles (larger fronts before their
// partial LU on the dense kernels; separator blocks), one workgroup per tile.
template <typename T>
void launch_extend_add(const AddTile *tiles, int ntile, const AddSrc *src, hipStream_t st);

// ---- FP64 iterative refinement (one matrix per table entry) ----
// r = b - A x into the packed vectors and max |b|, |r|, |x| per column into
// the three areas of norms (nslots each; the workgroups' maxima after them)
constexpr int kResidualBlocks = 2048;
int residual_blocks(int nmat, int max_n);
inline size_t norm_values(int nmat, int max_n, int nslots) {
  return 3 * (size_t)nslots * (1 + residual_blocks(nmat, max_n));
}
template <typename T>
void launch_residual(const IrDev *tab, const VecDev *vd, int nmat, int max_n, T *bp, double *norms, int nslots,
                     hipStream_t st);
void launch_rowabs_max(const IrDev *tab, int nmat, int max_n, unsigned long long *out,
                       hipStream_t st);
}  // namespace snu
