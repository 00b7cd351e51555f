// Kernels of the solves (gfx950, wave64): permutation into the packed
// vectors, forward and backward sweeps over the leaf fronts, separator
// right-hand sides, and the grouped products of the dense solves.
//
// One column runs on vector instructions (a wave's lanes are 64 rows, the
// values of x are read lane by lane); several columns run 16 at a time on
// MFMA.  Both read a factor entry once per 16 columns and are bound by that
// traffic and by the chain of front heights, not by arithmetic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "snu_device.h"
#include "snu_kernels.h"

namespace snu {

// ---------------------------------------------------------------------------
// permutation
// ---------------------------------------------------------------------------
// One matrix per blockIdx.y, one row of one column group per thread.
template <typename T>
__global__ void k_permute_in(const PermDev *__restrict__ pd, const VecDev *__restrict__ vd, T *bp) {
  const PermDev P = pd[blockIdx.y];
  const VecDev V = vd[P.vec];
  const long long tot = (long long)P.n * vec_groups(V.nrhs);
  T *x = bp + V.base;
  const auto order = gptr(P.order);
  const auto rhs = gptr(P.b);
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < tot;
       i += (long long)gridDim.x * blockDim.x) {
    if (V.nrhs == 1) {
      x[order[i]] = (T)rhs[i];
      continue;
    }
    const int g = (int)(i / P.n), r = (int)(i % P.n);
    T *d = x + ((long long)g * P.n + order[r]) * kColGroup;
    const auto b = rhs + r + (long long)g * kColGroup * P.ldb;
    T v[kColGroup];
#pragma unroll
    for (int c = 0; c < kColGroup; c++)
      v[c] = g * kColGroup + c < V.nrhs ? (T)b[c * P.ldb] : T(0);
#pragma unroll
    for (int c = 0; c < kColGroup; c++) d[c] = v[c];
  }
}
template <typename T, bool ADD>
__global__ void k_permute_out(const PermDev *__restrict__ pd, const VecDev *__restrict__ vd, const T *bp,
                              const int *__restrict__ active) {
  const long long first = (long long)blockIdx.x * blockDim.x + threadIdx.x, step = (long long)gridDim.x * blockDim.x;
  if (ADD && active && !active[blockIdx.y]) return;
  const PermDev P = pd[blockIdx.y];
  const VecDev V = vd[P.vec];
  const long long tot = (long long)P.n * vec_groups(V.nrhs);
  const T *x = bp + V.base;
  const auto order = gptr(P.order);
  const auto sol = gptr(P.x);
  for (long long i = first; i < tot; i += step) {
    if (V.nrhs == 1) {
      const double v = (double)x[order[i]];
      sol[i] = ADD ? sol[i] + v : v;
      continue;
    }
    const int g = (int)(i / P.n), r = (int)(i % P.n);
    const T *s = x + ((long long)g * P.n + order[r]) * kColGroup;
    const auto d = sol + r + (long long)g * kColGroup * P.ldx;
    const int nc = V.nrhs - g * kColGroup;
    T v[kColGroup];
    double o[kColGroup];
#pragma unroll
    for (int c = 0; c < kColGroup; c++) {
      v[c] = s[c];
      o[c] = ADD && c < nc ? d[c * P.ldx] : 0.0;
    }
#pragma unroll
    for (int c = 0; c < kColGroup; c++)
      if (c < nc) d[c * P.ldx] = ADD ? o[c] + (double)v[c] : (double)v[c];
  }
}
static unsigned perm_blocks(long long max_elems) {
  long long b = (max_elems + 255) / 256;
  return (unsigned)std::max(1LL, std::min(b, 2048LL));
}
template <typename T>
void launch_permute_in(const PermDev *pd, int nmat, const VecDev *vd, T *bp, long long max_elems,
                       hipStream_t st) {
  if (nmat <= 0 || max_elems <= 0) return;
  hipLaunchKernelGGL(k_permute_in<T>, dim3(perm_blocks(max_elems), nmat), dim3(256), 0, st, pd, vd, bp);
}
template <typename T>
void launch_permute_out(const PermDev *pd, int nmat, const VecDev *vd, const T *bp, long long max_elems, bool add,
                        const int *active, hipStream_t st) {
  if (nmat <= 0 || max_elems <= 0) return;
  const dim3 g(perm_blocks(max_elems), nmat);
  if (add)
    hipLaunchKernelGGL((k_permute_out<T, true>), g, dim3(256), 0, st, pd, vd, bp, active);
  else
    hipLaunchKernelGGL((k_permute_out<T, false>), g, dim3(256), 0, st, pd, vd, bp, active);
}

// ---------------------------------------------------------------------------
// leaf fronts
// ---------------------------------------------------------------------------
// Forward, per front: w = (b of its pivots, 0) + the children's updates; y =
// L11^-1 w_K replaces b, and w_B - L21 y is the front's update for its
// parent (root fronts: for the separators, k_assemble_rhs).  Backward: x_K =
// U11^-1 (y_K - U12 x_B).  Both by substitution with divisions by the pivots.
// (The inverses of triangles of 16 and 64 pivots in its place are shorter
// chains, but their error grows with the triangle's condition number: one front
// of a chain with diagonal 2, -3 below and -0.3 above, FP64, has backward error
// 1.4e-12 at order 48 and 6e-3 at order 65 with them, 2e-16 by substitution.)
// A row's products are summed and then taken from it, so that rounding goes
// with their sum (errors of x against the exact solution 3.8e-16 to 4.6e-16 on
// 2D and 3D grids; 4.7e-16 to 5.8e-16 taking them from the row one by one).
// A front's rows read their children's update rows through lists in a fixed
// order, so no two units write one place and results do not depend on
// scheduling.
// One workgroup per leaf and column group walks the leaf's front tree height
// by height; between two barriers its waves take the units of a phase in turn.
// That keeps the whole sweep in one launch (the tree is 3 to 12 heights of at
// most a few hundred units) and a unit is sized so that a wave has 16 or more
// loads in flight.  Bound by the latency of the units' loads and substitutions
// down the chain of heights; forward / backward: 64^3 7-point FP64, one column
// 214 / 250 us (row by row over the leaf's CSR factors, hundreds of level sets:
// 554 / 828; with the inverses 202 / 242); 48^3 27-point FP64, 16 columns 499 /
// 428 us (2916 / 4719; 493 / 381); 1000^2 5-point FP32, 64 columns 1.42 / 1.23
// ms (3.8 / 4.8; 1.54 / 1.15).
// 1024 threads per leaf for one column (261 / 292 us with 512 and the
// inverses); the 16-column fragments need over 200 registers, so 512.
template <int NC>
constexpr int leaf_threads() {
  return NC == 1 ? 1024 : 512;
}

// descriptors through the scalar cache (they are written by the host only)
typedef __attribute__((address_space(4))) const int ccint;
__device__ __forceinline__ ccint *cptr(const int *p) { return (ccint *)p; }
typedef int int16_v __attribute__((ext_vector_type(16)));
__device__ __forceinline__ SolveUnit load_unit(const SolveUnit *p) {
  static_assert(sizeof(SolveUnit) == sizeof(int16_v), "one 64-byte load");
  return __builtin_bit_cast(SolveUnit, *(__attribute__((address_space(4))) const int16_v *)p);
}

// l16: a fragment's column of the lane, lk: its row group (rows 4 lk .. 4 lk + 3,
// one per register), ar: the row of A that the lane loads as the first operand.
// For FP64 the product's register r of group lk is row 4 r + lk of the
// instruction; loading A's rows in that order (ar) makes it row 4 lk + r of the
// block as for FP32, so that four consecutive rows are in one lane, where
// substitution needs them.
struct SweepCtx {
  int lane, l16, lk, ar;
};
template <typename T>
__device__ __forceinline__ constexpr int lane_of_row(int row) {
  return std::is_same<T, double>::value ? 4 * (row & 3) + (row >> 2) : row;
}
__device__ __forceinline__ int sweep_row(int r, int lk) { return 4 * lk + r; }
// LU of the unit's 64-pivot block of a larger front (64 x 64)
template <typename T>
__device__ __forceinline__ const T *pivot_block(const SolveUnit &U) {
  return (const T *)U.inv + (long long)U.s * kFrontInv + 2 * 4096;
}

// ---- one column ----
typedef int int2_v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) const int2_v gcint2;
// the sources of front row r
__device__ __forceinline__ int2_v pull_entry(const LeafDev &L, const SolveUnit &U, int r) {
  return ((gcint2 *)L.pull)[U.pull + r];
}
// their sum (NC values per row, col of them)
template <typename T, int NC>
__device__ __forceinline__ T pull_sum(const LeafDev &L, const T *W, int2_v e, int col) {
  T s = e[0] >= 0 ? W[(long long)e[0] * NC + col] : T(0);
  s += e[1] >= 0 ? W[(long long)e[1] * NC + col] : T(0);
  if (__any(e[1] < -1)) {
    if (e[1] < -1) {
      const auto l = gptr(L.pulllist) - 2 - e[1];
      const int n = l[0];
      for (int i = 1; i <= n; i++) s += W[(long long)l[i] * NC + col];
    }
  }
  return s;
}
// sum_k a[k ld] v(k) over k < K, 16 columns in flight (a: this lane's row)
template <typename T, class V>
__device__ __forceinline__ T dot_cols(const T *a, long long ld, int K, int lane, V v) {
  const auto p = gptr(a);
  T s0 = T(0), s1 = T(0), s2 = T(0), s3 = T(0);
  for (int kc = 0; kc < K; kc += 64) {
    const int kn = min(64, K - kc);
    const T x = lane < kn ? v(kc + lane) : T(0);
    for (int k = 0; k < kn; k += 16) {
      T c[16];
#pragma unroll
      for (int j = 0; j < 16; j++) c[j] = p[(long long)(kc + min(k + j, kn - 1)) * ld];
#pragma unroll
      for (int j = 0; j < 16; j += 4) {
        s0 += c[j] * rld(x, k + j);
        s1 += c[j + 1] * rld(x, k + j + 1);
        s2 += c[j + 2] * rld(x, k + j + 2);
        s3 += c[j + 3] * rld(x, k + j + 3);
      }
    }
  }
  return (s0 + s1) + (s2 + s3);
}
// w -= L y for the `rows` rows of a lower trapezoid (unit diagonal, n columns;
// y: w's first n rows on the way), RPL rows per lane.  A row's products are
// summed and taken from it at once: rounding relative to their sum, not to the
// row at every step.  (Rows that are done go on summing, which nothing reads.)
template <typename T, int RPL>
__device__ __forceinline__ void solve_lower1(const T *A, int ld, int rows, int n, T (&w)[RPL], int lane) {
  const auto F = gptr(A);
  T s[RPL], y[RPL];
#pragma unroll
  for (int i = 0; i < RPL; i++) s[i] = y[i] = T(0);
  for (int k0 = 0; k0 < n; k0 += 16) {
    T c[RPL][16];
#pragma unroll
    for (int i = 0; i < RPL; i++)
#pragma unroll
      for (int j = 0; j < 16; j++) c[i][j] = F[min(lane + 64 * i, rows - 1) + min(k0 + j, n - 1) * ld];
#pragma unroll
    for (int j = 0; j < 16; j++) {
      const int k = k0 + j;
      T yk;
      auto take = [&](int i) __attribute__((always_inline)) {
        const T d = w[i] - s[i];
        y[i] = lane + 64 * i == k ? d : y[i];
        yk = rld(d, k & 63);
      };
      if (RPL == 1 || k < 64) take(0);
      else take(RPL - 1);
      if (k >= n) yk = T(0);  // (no branch: the loads of later steps would move behind it)
#pragma unroll
      for (int i = 0; i < RPL; i++) s[i] += c[i][j] * yk;
    }
  }
#pragma unroll
  for (int i = 0; i < RPL; i++) w[i] = lane + 64 * i < n ? y[i] : w[i] - s[i];
}
// an upper triangle's pivots
template <typename T, int RPL>
__device__ __forceinline__ void pivots1(const T *A, int ld, int n, Pivot<T> (&by)[RPL], int lane) {
#pragma unroll
  for (int i = 0; i < RPL; i++) {
    const int r = lane + 64 * i;
    by[i] = Pivot<T>(r < n ? gptr(A)[(long long)r * (ld + 1)] : T(1));
  }
}
// t = U^-1 (t - s), n rows
template <typename T, int RPL>
__device__ __forceinline__ void solve_upper1(const T *A, int ld, int n, const Pivot<T> (&by)[RPL], T (&t)[RPL],
                                             T (&s)[RPL], int lane) {
  const auto F = gptr(A);
  T v[RPL];
#pragma unroll
  for (int i = 0; i < RPL; i++) v[i] = by[i].scaled(t[i]);
  for (int k0 = n - 1; k0 >= 0; k0 -= 16) {
    T c[RPL][16];
#pragma unroll
    for (int i = 0; i < RPL; i++)
#pragma unroll
      for (int j = 0; j < 16; j++) c[i][j] = F[min(lane + 64 * i, n - 1) + max(k0 - j, 0) * ld];
#pragma unroll
    for (int j = 0; j < 16; j++) {
      const int k = k0 - j;
      T xk;
      auto take = [&](int i) __attribute__((always_inline)) {
        const T q = by[i].solve(v[i], s[i]);
        t[i] = lane + 64 * i == k ? q : t[i];
        xk = rld(q, k & 63);
      };
      if (RPL == 1 || k < 64) take(0);
      else take(RPL - 1);
      if (k < 0) xk = T(0);
#pragma unroll
      for (int i = 0; i < RPL; i++) s[i] += c[i][j] * xk;
    }
  }
}
// RPL rows per lane (front order <= 64 RPL)
template <typename T, int RPL>
__device__ __forceinline__ void fwd_front1(const LeafDev &L, const SolveUnit &U, T *x, T *W, int lane) {
  const int f = U.ld, nk = U.nk;
  T w[RPL];
#pragma unroll
  for (int i = 0; i < RPL; i++) {
    const int r = lane + 64 * i;
    w[i] = r < nk ? x[U.kpos + r] : T(0);
    w[i] += pull_sum<T, 1>(L, W, r < f ? pull_entry(L, U, r) : int2_v{-1, -1}, 0);
  }
  solve_lower1<T, RPL>((const T *)U.F, f, f, nk, w, lane);
#pragma unroll
  for (int i = 0; i < RPL; i++) {
    const int r = lane + 64 * i;
    if (r < nk) x[U.kpos + r] = w[i];
    else if (r < f) W[U.wrow + r - nk] = w[i];
  }
}
template <typename T, int RPL>
__device__ __forceinline__ void bwd_front1(const LeafDev &L, const SolveUnit &U, T *x, int lane) {
  const auto F = gptr((const T *)U.F);
  const int f = U.ld, nk = U.nk, nb = U.nb;
  T xb[RPL], t[RPL], s[RPL];
  Pivot<T> by[RPL];
  pivots1<T, RPL>((const T *)U.F, f, nk, by, lane);
#pragma unroll
  for (int i = 0; i < RPL; i++) {
    const int r = lane + 64 * i;
    xb[i] = r < nb ? x[gptr(L.bidx)[U.bidx + r]] : T(0);
    t[i] = r < nk ? x[U.kpos + r] : T(0);
    s[i] = T(0);
  }
  // U12 x_B: 64 / gw columns per load when the pivots leave lanes free
  const int gw = nk > 32 ? 64 : nk > 16 ? 32 : nk > 8 ? 16 : 8;
  const int ng = 64 / gw, sub = lane / gw, row = lane & (gw - 1);
  for (int j0 = 0; j0 < nb; j0 += 8 * ng) {
    T c[RPL][8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int j = min(j0 + q * ng + sub, nb - 1);
#pragma unroll
      for (int i = 0; i < RPL; i++) c[i][q] = F[min(row + 64 * i, nk - 1) + (nk + j) * f];
    }
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int j = j0 + q * ng + sub;
      T xj = __shfl(xb[0], j & 63, 64);
      if (RPL > 1) {
        const T x1 = __shfl(xb[RPL - 1], j & 63, 64);
        xj = j < 64 ? xj : x1;
      }
      if (j >= nb) xj = T(0);
#pragma unroll
      for (int i = 0; i < RPL; i++) s[i] += c[i][q] * xj;
    }
  }
#pragma unroll
  for (int i = 0; i < RPL; i++) {
    for (int o = gw; o < 64; o <<= 1) s[i] += __shfl_xor(s[i], o, 64);
  }
  solve_upper1<T, RPL>((const T *)U.F, f, nk, by, t, s, lane);
#pragma unroll
  for (int i = 0; i < RPL; i++)
    if (lane + 64 * i < nk) x[U.kpos + lane + 64 * i] = t[i];
}
template <typename T, bool BWD>
__device__ __forceinline__ void unit1(const LeafDev &L, const SolveUnit &U, T *x, T *W, int lane) {
  constexpr int RPL = sizeof(T) == 8 ? 1 : 2;
  const T *F = (const T *)U.F, *lu = pivot_block<T>(U);
  const int f = U.ld, nk = U.nk, r0 = 64 * U.s, nbk = min(64, nk - r0), r = r0 + min(lane, nbk - 1);
  if constexpr (!BWD) switch (U.kind) {
    case kFwdFront:  // (most FP32 fronts need one row per lane too: a batch of 96 4.09 -> 3.92 ms)
      if (RPL == 1 || f <= 64) fwd_front1<T, 1>(L, U, x, W, lane);
      else fwd_front1<T, RPL>(L, U, x, W, lane);
      break;
    case kFwdPivots: {
      T w = lane < nbk ? x[U.kpos + r] : T(0);
      w += pull_sum<T, 1>(L, W, lane < nbk ? pull_entry(L, U, r) : int2_v{-1, -1}, 0);
      if (r0) {
        const T p = dot_cols(F + r, f, r0, lane, [&](int k) { return x[U.kpos + k]; });
        if (lane < nbk) w -= p;
      }
      T y[1] = {w};
      solve_lower1<T, 1>(lu, 64, nbk, nbk, y, lane);
      if (lane < nbk) x[U.kpos + r] = y[0];
      break;
    }
    case kFwdRows: {
      const int b = U.row0 + lane, bc = min(b, U.nb - 1);
      const T w = pull_sum<T, 1>(L, W, pull_entry(L, U, nk + bc), 0);
      const T p = dot_cols(F + nk + bc, f, nk, lane, [&](int k) { return x[U.kpos + k]; });
      if (b < U.nb) W[U.wrow + b] = w - p;
      break;
    }
  }
  else switch (U.kind) {
    case kBwdFront:
      if (RPL == 1 || f <= 64) bwd_front1<T, 1>(L, U, x, lane);
      else bwd_front1<T, RPL>(L, U, x, lane);
      break;
    case kBwdCols: {
      const int cw = 64 * ((nk + 63) / 64), j0 = U.q * cw, j1 = min(U.nb, j0 + cw);
      const auto bi = gptr(L.bidx) + U.bidx + j0;
      const T p = dot_cols(F + r + (long long)(nk + j0) * f, f, j1 - j0, lane, [&](int k) { return x[bi[k]]; });
      W[U.wrow + (U.s * U.nq + U.q) * 64 + lane] = p;
      break;
    }
    case kBwdPivots: {
      Pivot<T> by[1];
      pivots1<T, 1>(lu, 64, nbk, by, lane);
      T y[1] = {lane < nbk ? x[U.kpos + r] : T(0)}, s[1] = {T(0)};
      for (int q = 0; q < U.nq; q++) s[0] += W[U.wrow + (U.s * U.nq + q) * 64 + lane];
      if (r0 + 64 < nk)
        s[0] += dot_cols(F + r + (long long)(r0 + 64) * f, f, nk - r0 - 64, lane,
                         [&](int k) { return x[U.kpos + r0 + 64 + k]; });
      solve_upper1<T, 1>(lu, 64, nbk, by, y, s, lane);
      if (lane < nbk) x[U.kpos + r] = y[0];
      break;
    }
  }
}

// ---- 16 columns ----
// rows [row0, row0 + 16) of a vector group, those from nvalid on zero
template <typename T>
__device__ __forceinline__ Frag<T> load_frag(const T *X, int row0, int nvalid, const SweepCtx &c) {
  Frag<T> v;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int row = row0 + sweep_row(r, c.lk);
    v[r] = row < nvalid ? X[(long long)row * kColGroup + c.l16] : T(0);
  }
  return v;
}
template <typename T>
__device__ __forceinline__ void store_frag(T *X, int row0, int nvalid, const Frag<T> &v, const SweepCtx &c) {
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int row = row0 + sweep_row(r, c.lk);
    if (row < nvalid) X[(long long)row * kColGroup + c.l16] = v[r];
  }
}
// the children's updates of front rows [row0, row0 + 16), zero from rend on
template <typename T>
__device__ __forceinline__ Frag<T> pull_frag(const LeafDev &L, const SolveUnit &U, const T *W, int row0, int rend,
                                             const SweepCtx &c) {
  int2_v e[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int row = row0 + sweep_row(r, c.lk);
    e[r] = row < rend ? pull_entry(L, U, row) : int2_v{-1, -1};
  }
  Frag<T> v;
  bool more = false;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    v[r] = e[r][0] >= 0 ? W[(long long)e[r][0] * kColGroup + c.l16] : T(0);
    v[r] += e[r][1] >= 0 ? W[(long long)e[r][1] * kColGroup + c.l16] : T(0);
    more |= e[r][1] < -1;
  }
  if (__any(more)) {
#pragma unroll
    for (int r = 0; r < 4; r++)
      if (e[r][1] < -1) {
        const auto l = gptr(L.pulllist) - 2 - e[r][1];
        const int n = l[0];
        for (int i = 1; i <= n; i++) v[r] += W[(long long)l[i] * kColGroup + c.l16];
      }
  }
  return v;
}
template <typename T>
__device__ __forceinline__ void mask_frag(Frag<T> &v, int row0, int nvalid, const SweepCtx &c) {
#pragma unroll
  for (int r = 0; r < 4; r++)
    if (row0 + sweep_row(r, c.lk) >= nvalid) v[r] = T(0);
}
// acc += A[16 rows][columns k0 .. k0 + 15] b; a: this lane's row, columns
// clamped to kmax (their b rows are zero)
template <typename T>
__device__ __forceinline__ void frag_mm(Frag<T> &acc, const T *a, int ld, int k0, int kmax, const Frag<T> &b,
                                        const SweepCtx &c) {
  const auto p = gptr(a);
  T v[4];
#pragma unroll
  for (int r = 0; r < 4; r++) v[r] = p[(long long)min(k0 + sweep_row(r, c.lk), kmax) * ld];
#pragma unroll
  for (int r = 0; r < 4; r++) acc = mfma4(v[r], b[r], acc);
}
// A 16 x 16 block of a triangle (unit lower, or upper), n of its rows and
// columns used: entry (ar, 4 g + lk) of its strict part in a[g].
template <typename T, bool UPPER>
struct Tri16 {
  T a[4];
  Pivot<T> by;  // (UPPER) row ar's pivot
  __device__ __forceinline__ void load(const T *F, int ld, int n, const SweepCtx &c) {
    const auto p = gptr(F) + min(c.ar, n - 1);
#pragma unroll
    for (int g = 0; g < 4; g++) a[g] = p[(long long)min(4 * g + c.lk, n - 1) * ld];
    if constexpr (UPPER) by = Pivot<T>(c.ar < n ? p[(long long)min(c.ar, n - 1) * ld] : T(1));
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const int k = 4 * g + c.lk;
      if (!(UPPER ? k > c.ar && k < n : k < c.ar && c.ar < n)) a[g] = T(0);
    }
  }
  // w - acc solved with it (both zero beyond n).  Four rows at a time: the lanes
  // that hold them (the others compute along) solve them with the block's
  // entries and pivots read lane by lane, then one product adds their share to
  // the rows left.  (The four steps as a loop: half the code, but a block's loads
  // are then waited for at its head: 1000^2, 64 columns 10.5 -> 12.5 ms per solve.)
  template <int g>
  __device__ __forceinline__ void rows(const Frag<T> &w, Frag<T> &acc, Frag<T> &y, const SweepCtx &c) const {
    T p[4], s[4];
#pragma unroll
    for (int i = 0; i < 4; i++) p[i] = acc[i];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int j = UPPER ? 3 - q : q;
      if constexpr (UPPER) {
        const Pivot<T> d = by.of_lane(lane_of_row<T>(4 * g + j));
        s[j] = d.solve(d.scaled(w[j]), p[j]);
      } else {
        s[j] = w[j] - p[j];
      }
#pragma unroll
      for (int i = UPPER ? 0 : j + 1; i < (UPPER ? j : 4); i++)
        p[i] += rld(a[g], lane_of_row<T>(4 * g + i) + 16 * j) * s[j];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) y[i] = c.lk == g ? s[i] : y[i];
    if (g != (UPPER ? 0 : 3))
      acc = mfma4((UPPER ? c.ar < 4 * g : c.ar >= 4 * g + 4) ? a[g] : T(0), spread_group<g>(s), acc);
  }
  __device__ __forceinline__ Frag<T> solve(const Frag<T> &w, Frag<T> acc, const SweepCtx &c) const {
    Frag<T> y = w;
    if constexpr (UPPER) rows<3>(w, acc, y, c), rows<2>(w, acc, y, c), rows<1>(w, acc, y, c), rows<0>(w, acc, y, c);
    else rows<0>(w, acc, y, c), rows<1>(w, acc, y, c), rows<2>(w, acc, y, c), rows<3>(w, acc, y, c);
    return y;
  }
};
// Whole front with at most 16 KB pivots and 16 BB boundary entries; EXACT: no
// block is empty, so the code is straight-line and all its loads are in flight
// before the first product (a branch per block would expose each block's
// latency in turn).
template <typename T, int KB, int BB, bool EXACT>
__device__ __forceinline__ void fwd_front16(const LeafDev &L, const SolveUnit &U, T *x, T *W, const SweepCtx &c) {
  const T *F = (const T *)U.F;
  const int f = U.ld, nk = U.nk, nb = U.nb;
  T *xk = x + (long long)U.kpos * kColGroup, *wb = W + (long long)U.wrow * kColGroup;
  // (the stores to x last: the loads are not moved over them)
  Tri16<T, false> t[KB];
  if constexpr (EXACT) {
#pragma unroll
    for (int b = 0; b < KB; b++) t[b].load(F + 16 * b * (f + 1), f, min(16, nk - 16 * b), c);
  }
  Frag<T> y[KB];
#pragma unroll
  for (int b = 0; b < KB; b++) {
    y[b] = frag_zero<T>();
    if (EXACT || 16 * b < nk) {
      if constexpr (!EXACT) t[b].load(F + 16 * b * (f + 1), f, min(16, nk - 16 * b), c);
      Frag<T> acc = frag_zero<T>();
#pragma unroll
      for (int a = 0; a < b; a++) frag_mm(acc, F + min(16 * b + c.ar, nk - 1), f, 16 * a, nk - 1, y[a], c);
      Frag<T> w = load_frag(xk, 16 * b, nk, c) + pull_frag(L, U, W, 16 * b, nk, c);
      mask_frag(acc, 16 * b, nk, c);
      y[b] = t[b].solve(w, acc, c);
    }
  }
#pragma unroll
  for (int b = 0; b < BB; b++)
    if (EXACT || 16 * b < nb) {
      Frag<T> acc = frag_zero<T>();
#pragma unroll
      for (int a = 0; a < KB; a++)
        if (EXACT || 16 * a < nk) frag_mm(acc, F + min(nk + 16 * b + c.ar, f - 1), f, 16 * a, nk - 1, y[a], c);
      store_frag(wb, 16 * b, nb, pull_frag(L, U, W, nk + 16 * b, f, c) - acc, c);
    }
#pragma unroll
  for (int b = 0; b < KB; b++)
    if (EXACT || 16 * b < nk) store_frag(xk, 16 * b, nk, y[b], c);
}
// rows of x at the positions idx[row0 ..], zero from n on
template <typename T>
__device__ __forceinline__ Frag<T> gather_frag(const T *x, const int *idx, int row0, int n, const SweepCtx &c) {
  const auto p = gptr(idx);
  int at[4];
#pragma unroll
  for (int r = 0; r < 4; r++) at[r] = p[min(row0 + sweep_row(r, c.lk), n - 1)];
  Frag<T> v;
#pragma unroll
  for (int r = 0; r < 4; r++)
    v[r] = row0 + sweep_row(r, c.lk) < n ? x[(long long)at[r] * kColGroup + c.l16] : T(0);
  return v;
}
template <typename T, int KB, int BB, bool EXACT>
__device__ __forceinline__ void bwd_front16(const LeafDev &L, const SolveUnit &U, T *x, const SweepCtx &c) {
  const T *F = (const T *)U.F;
  const int f = U.ld, nk = U.nk, nb = U.nb;
  T *xk = x + (long long)U.kpos * kColGroup;
  Tri16<T, true> tri[KB];
  if constexpr (EXACT) {
#pragma unroll
    for (int b = 0; b < KB; b++) tri[b].load(F + 16 * b * (f + 1), f, min(16, nk - 16 * b), c);
  }
  Frag<T> t[KB];
#pragma unroll
  for (int b = 0; b < KB; b++) t[b] = frag_zero<T>();
#pragma unroll
  for (int a = 0; a < BB; a++)
    if (EXACT || 16 * a < nb) {
      const Frag<T> xb = gather_frag(x, L.bidx + U.bidx, 16 * a, nb, c);
#pragma unroll
      for (int b = 0; b < KB; b++)
        if (EXACT || 16 * b < nk)
          frag_mm(t[b], F + min(16 * b + c.ar, nk - 1) + (long long)nk * f, f, 16 * a, nb - 1, xb, c);
    }
#pragma unroll
  for (int b = KB - 1; b >= 0; b--)
    if (EXACT || 16 * b < nk) {
      if constexpr (!EXACT) tri[b].load(F + 16 * b * (f + 1), f, min(16, nk - 16 * b), c);
      Frag<T> acc = t[b];
#pragma unroll
      for (int a = b + 1; a < KB; a++)
        if (EXACT || 16 * a < nk) frag_mm(acc, F + min(16 * b + c.ar, nk - 1), f, 16 * a, nk - 1, t[a], c);
      const Frag<T> w = load_frag(xk, 16 * b, nk, c);
      mask_frag(acc, 16 * b, nk, c);
      t[b] = tri[b].solve(w, acc, c);
    }
#pragma unroll
  for (int b = 0; b < KB; b++)
    if (EXACT || 16 * b < nk) store_frag(xk, 16 * b, nk, t[b], c);
}
// the straight-line form for the block counts of most fronts
template <typename T, bool BWD>
__device__ __forceinline__ void front16(const LeafDev &L, const SolveUnit &U, T *x, T *W, const SweepCtx &c) {
  constexpr int MB = sizeof(T) == 8 ? 4 : 6;
  const int kb = (U.nk + 15) >> 4, bb = (U.nb + 15) >> 4;
#define SNU_FRONT16(K, B, E)                                 \
  do {                                                       \
    if constexpr (BWD) bwd_front16<T, K, B, E>(L, U, x, c);  \
    else fwd_front16<T, K, B, E>(L, U, x, W, c);             \
  } while (0)
  if (kb == 1 && bb == 1) SNU_FRONT16(1, 1, true);
  else if (kb == 1 && bb == 2) SNU_FRONT16(1, 2, true);
  else if (kb == 1 && bb == 3) SNU_FRONT16(1, 3, true);
  else if (kb == 2 && bb == 1) SNU_FRONT16(2, 1, true);
  else if (kb == 2 && bb == 2) SNU_FRONT16(2, 2, true);
  else SNU_FRONT16(MB, MB, false);
#undef SNU_FRONT16
}
// acc[4] += A[64 rows][K columns] X: a: the tile's first entry, rows clamped
// to rmax; vec(k) the fragment of X rows k .. k + 15
template <typename T, class V>
__device__ __forceinline__ void tile_mm(Frag<T> (&acc)[4], const T *a, int ld, int rmax, int K, const SweepCtx &c,
                                        V vec) {
  const auto p = gptr(a);
  int row[4];
#pragma unroll
  for (int b = 0; b < 4; b++) row[b] = min(16 * b + c.ar, rmax);
  Frag<T> x;
  T v[4][4];
  auto load = [&](int k0, Frag<T> &xn, T (&vn)[4][4]) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const auto pc = p + (long long)min(k0 + sweep_row(r, c.lk), K - 1) * ld;
#pragma unroll
      for (int b = 0; b < 4; b++) vn[b][r] = pc[row[b]];
    }
    xn = vec(k0);
  };
  auto mul = [&](const Frag<T> &xn, const T (&vn)[4][4]) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int b = 0; b < 4; b++) acc[b] = mfma4(vn[b][r], xn[r], acc[b]);
  };
  // the next 16 columns are loaded while these are multiplied
  load(0, x, v);
  for (int k0 = 16; k0 < K; k0 += 16) {
    Frag<T> xn;
    T vn[4][4];
    load(k0, xn, vn);
    mul(x, v);
    x = xn;
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int r = 0; r < 4; r++) v[b][r] = vn[b][r];
  }
  mul(x, v);
}
// the same with a 64-pivot block (64 x 64, nbk of its rows and columns used)
template <typename T, bool UPPER>
__device__ __forceinline__ void tri64(Frag<T> (&y)[4], const T *lu, int nbk, const Frag<T> (&w)[4],
                                      const Frag<T> (&sum)[4], const SweepCtx &c) {
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int b = UPPER ? 3 - q : q;
    y[b] = frag_zero<T>();
    if (16 * b >= nbk) continue;
    Frag<T> acc = sum[b];
#pragma unroll
    for (int a = UPPER ? b + 1 : 0; a < (UPPER ? 4 : b); a++)
      if (16 * a < nbk) frag_mm(acc, lu + min(16 * b + c.ar, nbk - 1), 64, 16 * a, nbk - 1, y[a], c);
    Tri16<T, UPPER> t;
    t.load(lu + 16 * b * 65, 64, min(16, nbk - 16 * b), c);
    mask_frag(acc, 16 * b, nbk, c);
    y[b] = t.solve(w[b], acc, c);
  }
}
template <typename T, bool BWD>
__device__ __forceinline__ void unit16(const LeafDev &L, const SolveUnit &U, T *x, T *W, const SweepCtx &c) {
  const T *F = (const T *)U.F, *lu = pivot_block<T>(U);
  const int f = U.ld, nk = U.nk, r0 = 64 * U.s, nbk = min(64, nk - r0);
  T *xk = x + (long long)U.kpos * kColGroup, *wf = W + (long long)U.wrow * kColGroup;
  Frag<T> acc[4];
#pragma unroll
  for (int b = 0; b < 4; b++) acc[b] = frag_zero<T>();
  if constexpr (!BWD) switch (U.kind) {
    case kFwdPivots: {
      if (r0) tile_mm(acc, F + r0, f, nbk - 1, r0, c, [&](int k) { return load_frag(xk, k, r0, c); });
      Frag<T> w[4], y[4];
#pragma unroll
      for (int b = 0; b < 4; b++) {
        w[b] = load_frag(xk, r0 + 16 * b, r0 + nbk, c) + pull_frag(L, U, W, r0 + 16 * b, r0 + nbk, c);
      }
      tri64<T, false>(y, lu, nbk, w, acc, c);
#pragma unroll
      for (int b = 0; b < 4; b++) store_frag(xk, r0 + 16 * b, r0 + nbk, y[b], c);
      break;
    }
    case kFwdRows: {
      tile_mm(acc, F + nk + U.row0, f, U.nb - 1 - U.row0, nk, c, [&](int k) { return load_frag(xk, k, nk, c); });
#pragma unroll
      for (int b = 0; b < 4; b++)
        store_frag(wf, U.row0 + 16 * b, U.nb, pull_frag(L, U, W, nk + U.row0 + 16 * b, f, c) - acc[b], c);
      break;
    }
  }
  else switch (U.kind) {
    case kBwdCols: {
      const int cw = 64 * ((nk + 63) / 64), j0 = U.q * cw, jn = min(U.nb, j0 + cw) - j0;
      const int *bi = L.bidx + U.bidx + j0;
      tile_mm(acc, F + r0 + (long long)(nk + j0) * f, f, nbk - 1, jn, c,
              [&](int k) { return gather_frag(x, bi, k, jn, c); });
#pragma unroll
      for (int b = 0; b < 4; b++) store_frag(wf + (U.s * U.nq + U.q) * 64 * kColGroup, 16 * b, 64, acc[b], c);
      break;
    }
    case kBwdPivots: {
      if (r0 + 64 < nk)
        tile_mm(acc, F + r0 + (long long)(r0 + 64) * f, f, nbk - 1, nk - r0 - 64, c,
                [&](int k) { return load_frag(xk + (r0 + 64) * kColGroup, k, nk - r0 - 64, c); });
      for (int q = 0; q < U.nq; q++)
#pragma unroll
        for (int b = 0; b < 4; b++)
          acc[b] += load_frag(wf + (U.s * U.nq + q) * 64 * kColGroup, 16 * b, 64, c);
      Frag<T> w[4], y[4];
#pragma unroll
      for (int b = 0; b < 4; b++) w[b] = load_frag(xk, r0 + 16 * b, r0 + nbk, c);
      tri64<T, true>(y, lu, nbk, w, acc, c);
#pragma unroll
      for (int b = 0; b < 4; b++) store_frag(xk, r0 + 16 * b, r0 + nbk, y[b], c);
      break;
    }
  }
}

template <typename T, int NC, bool BWD>
__global__ __launch_bounds__(leaf_threads<NC>()) void k_leaf_sweep(const LeafDev *__restrict__ leaves,
                                                             const VecDev *__restrict__ vd, T *bp, T *wbuf) {
  const LeafDev L = leaves[blockIdx.x];
  const VecDev V = vd[L.vec];
  const int g = blockIdx.y;
  if (vec_width(V.nrhs) != NC || g >= vec_groups(V.nrhs)) return;
  T *x = bp + V.base + (long long)g * V.n * NC, *W = wbuf + V.wbase + (long long)g * V.wrows * NC;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const SweepCtx c{lane, lane & 15, lane >> 4, lane_of_row<T>(lane & 15)};
  const auto ph = cptr(BWD ? L.bphase : L.fphase);
  const int np = BWD ? L.nbphase : L.nfphase;
  int u0 = ph[0];
  for (int p = 0; p < np; p++) {
    const int u1 = ph[p + 1];
    for (int u = u0 + wave; u < u1; u += leaf_threads<NC>() / 64) {
      const SolveUnit U = load_unit(L.units + u);
      if constexpr (NC == 1) unit1<T, BWD>(L, U, x, W, lane);
      else if (U.kind == (BWD ? kBwdFront : kFwdFront)) front16<T, BWD>(L, U, x, W, c);
      else unit16<T, BWD>(L, U, x, W, c);
    }
    u0 = u1;
    __syncthreads();
  }
}
template <typename T>
void launch_leaf_sweep(const LeafDev *leaves, int nleaves, const VecDev *vd, T *bp, T *wbuf, int max_groups,
                       bool one, bool many, bool bwd, hipStream_t st) {
  if (nleaves <= 0) return;
  if (one) {
    const dim3 b(leaf_threads<1>());
    if (bwd) hipLaunchKernelGGL((k_leaf_sweep<T, 1, true>), dim3(nleaves), b, 0, st, leaves, vd, bp, wbuf);
    else hipLaunchKernelGGL((k_leaf_sweep<T, 1, false>), dim3(nleaves), b, 0, st, leaves, vd, bp, wbuf);
  }
  if (many) {
    const dim3 g(nleaves, max_groups), b(leaf_threads<kColGroup>());
    if (bwd) hipLaunchKernelGGL((k_leaf_sweep<T, kColGroup, true>), g, b, 0, st, leaves, vd, bp, wbuf);
    else hipLaunchKernelGGL((k_leaf_sweep<T, kColGroup, false>), g, b, 0, st, leaves, vd, bp, wbuf);
  }
}

// Separator rows receiving leaf contributions: + the root fronts' update rows
// (ascending leaf, then front), one thread per target row, column group and
// column.
template <typename T, int NC>
__global__ __launch_bounds__(256) void k_assemble_rhs(const TargetDev *__restrict__ targets, int ntarget,
                                                      const int *__restrict__ tsrc,
                                                      const VecDev *__restrict__ vd, const T *wbuf, T *bp) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) / NC;
  if (i >= ntarget) return;
  const int c = threadIdx.x % NC, g = blockIdx.y;
  const TargetDev t = targets[i];
  const VecDev V = vd[t.vec];
  if (vec_width(V.nrhs) != NC || g >= vec_groups(V.nrhs)) return;
  const T *W = wbuf + V.wbase + (long long)g * V.wrows * NC + c;
  T *b = bp + V.base + ((long long)g * V.n + t.row) * NC + c;
  T acc = *b;
  for (int s = t.s0; s < t.s1; s++) acc += W[(long long)tsrc[s] * NC];
  *b = acc;
}
template <typename T>
void launch_assemble_rhs(const TargetDev *targets, int ntarget, const int *tsrc, const VecDev *vd, const T *wbuf,
                         T *bp, int max_groups, bool one, bool many, hipStream_t st) {
  if (ntarget <= 0) return;
  if (one)
    hipLaunchKernelGGL((k_assemble_rhs<T, 1>), dim3((ntarget + 255) / 256), dim3(256), 0, st, targets, ntarget,
                       tsrc, vd, wbuf, bp);
  if (many)
    hipLaunchKernelGGL((k_assemble_rhs<T, kColGroup>), dim3((unsigned)(((long long)ntarget * kColGroup + 255) / 256), max_groups),
                       dim3(256), 0, st, targets, ntarget, tsrc, vd, wbuf, bp);
}

// ---------------------------------------------------------------------------
// dense: grouped GEMV (the dense solves), one column
// ---------------------------------------------------------------------------
// One workgroup per 64 rows of a problem; lane = row, the 4 waves take
// interleaved columns and are combined in LDS (fixed order: deterministic).
// A is read once, coalesced down its columns; x through scalar loads.  kb, ke:
// the column range of a segment the workgroup sums.
template <typename T, class Range>
__device__ __forceinline__ T gemv_rows(const GemvProbT<T> &P, const GemvSegT<T> *__restrict__ segs, int mc, int w,
                                       Range range) {
  T acc = T(0);
  for (int sg = 0; sg < P.nseg; sg++) {
    const GemvSegT<T> S = segs[P.seg0 + sg];
    int kb, ke;
    range(S.K, kb, ke);
    auto A = gptr(S.A) + mc;
    auto X = gptr(S.x);
    int k = kb + w;
    // NF columns of A in flight per wave (the loads are independent of the
    // accumulation), added in groups of four: 8 in FP64, 16 in FP32 (the
    // same bytes in flight)
    constexpr int NF = sizeof(T) == 4 ? 16 : 8;
    for (; k + 4 * (NF - 1) < ke; k += 4 * NF) {
      T a[NF];
#pragma unroll
      for (int j = 0; j < NF; j++) a[j] = A[(long long)(k + 4 * j) * S.lda];
      auto xc = X + k;
#pragma unroll
      for (int j = 0; j < NF; j += 4)
        acc += a[j] * xc[4 * j] + a[j + 1] * xc[4 * j + 4] + a[j + 2] * xc[4 * j + 8] + a[j + 3] * xc[4 * j + 12];
    }
    for (; k + 12 < ke; k += 16) {
      T a0 = A[(long long)k * S.lda], a1 = A[(long long)(k + 4) * S.lda];
      T a2 = A[(long long)(k + 8) * S.lda], a3 = A[(long long)(k + 12) * S.lda];
      acc += a0 * X[k] + a1 * X[k + 4] + a2 * X[k + 8] + a3 * X[k + 12];
    }
    for (; k < ke; k += 4) acc += A[(long long)k * S.lda] * X[k];
  }
  return acc;
}
template <typename T, int MODE>
__global__ __launch_bounds__(256) void k_gemv(const GemvProbT<T> *__restrict__ probs, int nprob,
                                              const GemvSegT<T> *__restrict__ segs) {
  __shared__ T red[4][64];
  const int tile = blockIdx.x;
  int lo = 0, hi = nprob - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (probs[mid].tile0 <= tile) lo = mid;
    else hi = mid - 1;
  }
  const GemvProbT<T> P = probs[lo];
  const int m0 = (tile - P.tile0) * 64;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = m0 + lane;
  red[w][lane] = gemv_rows(P, segs, min(m, P.M - 1), w, [&](int K, int &kb, int &ke) {
    kb = P.tri == 2 ? m0 : 0;
    ke = P.tri == 1 ? min(K, m0 + 64) : K;
  });
  __syncthreads();
  if (w == 0 && m < P.M) {
    const T v = red[0][lane] + red[1][lane] + red[2][lane] + red[3][lane];
    auto y = gptr(P.y) + m;
    if (MODE == 1) *y = v;
    else *y = *y - v;
  }
}
// Partial sums that another workgroup of the launch adds: written through to,
// and read from, where the whole device sees them (the XCDs' L2 caches are not
// coherent).  Release and acquire fences would do the same for plain accesses,
// but write back and invalidate a whole L2 per workgroup (64^3, one column:
// 1.83 ms per solve).
template <typename T>
__device__ __forceinline__ void put_part(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T get_part(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void parts_written() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// Whether the calling wave's workgroup is the last of `parts` to arrive at
// *done (left at 0 again for the next launch): what the others had written by
// parts_written() before arriving can then be read.
__device__ __forceinline__ bool last_to_arrive(int *done, int parts, int lane) {
  int at = 0;
  if (lane == 0) at = __hip_atomic_fetch_add(done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const bool last = __builtin_amdgcn_readfirstlane(at) == parts - 1;
  if (last && lane == 0) __hip_atomic_store(done, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("" ::: "memory");
  return last;
}
// Split-K GEMV: workgroup (problem, tile lt, piece) sums A[rows of lt][k] x[k]
// over k in [piece * kGemvPiece, (piece + 1) * kGemvPiece) of every segment
// (within the triangle for tri problems), in the order of the unsplit kernel,
// and stores the 64 partial sums; the tile's last workgroup to arrive adds the
// pieces in ascending order.  The decomposition depends on the problem alone,
// so a problem gives the same bits in any launch.  64^3: 1.05 ms per solve, 1.12
// with a second launch per product to add the pieces.  (The products of 16
// columns keep theirs: there the last workgroup's sum takes as long, and with
// several groups longer: six packed matrices 4.70 ms against 4.63.)
template <typename T, int MODE>
__global__ __launch_bounds__(256) void k_gemv_split(const GemvProbT<T> *__restrict__ probs, int nprob,
                                                    const GemvSegT<T> *__restrict__ segs, T *part, int *done) {
  __shared__ T red[4][64];
  const int b = blockIdx.x;
  int lo = 0, hi = nprob - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (probs[mid].wg0 <= b) lo = mid;
    else hi = mid - 1;
  }
  const GemvProbT<T> P = probs[lo];
  const int local = b - P.wg0, lt = local / P.parts, pc = local % P.parts;
  const int m0 = lt * 64;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  red[w][lane] = gemv_rows(P, segs, min(m0 + lane, P.M - 1), w, [&](int K, int &kb, int &ke) {
    kb = max(P.tri == 2 ? m0 : 0, pc * kGemvPiece);
    ke = min(P.tri == 1 ? min(K, m0 + 64) : K, (pc + 1) * kGemvPiece);
  });
  __syncthreads();
  if (w != 0) return;
  T v = red[0][lane] + red[1][lane] + red[2][lane] + red[3][lane];
  if (P.parts > 1) {
    T *in = part + P.poff + (long long)lt * P.parts * 64 + lane;
    put_part(in + pc * 64, v);
    parts_written();
    if (!last_to_arrive(done + P.tile0 + lt, P.parts, lane)) return;
    v = get_part(in);
    int q = 1;
    for (; q + 3 < P.parts; q += 4) {
      const T a = get_part(in + q * 64), b1 = get_part(in + q * 64 + 64), c = get_part(in + q * 64 + 128),
              d = get_part(in + q * 64 + 192);
      v = v + a + b1 + c + d;
    }
    for (; q < P.parts; q++) v += get_part(in + q * 64);
  }
  if (m0 + lane < P.M) {
    auto y = gptr(P.y) + m0 + lane;
    if (MODE == 1) *y = v;
    else *y = *y - v;
  }
}
template <typename T>
void launch_gemv_split(const GemvProbT<T> *probs, int nprob, const GemvSegT<T> *segs, int total_wgs, int mode,
                       T *part, int *done, hipStream_t st) {
  if (total_wgs <= 0 || nprob <= 0) return;
  if (mode == 1)
    hipLaunchKernelGGL((k_gemv_split<T, 1>), dim3(total_wgs), dim3(256), 0, st, probs, nprob, segs, part, done);
  else
    hipLaunchKernelGGL((k_gemv_split<T, 0>), dim3(total_wgs), dim3(256), 0, st, probs, nprob, segs, part, done);
}
template <typename T>
void launch_gemv(const GemvProbT<T> *probs, int nprob, const GemvSegT<T> *segs, int total_tiles, int mode,
                 hipStream_t st) {
  if (total_tiles <= 0 || nprob <= 0) return;
  if (mode == 1)
    hipLaunchKernelGGL((k_gemv<T, 1>), dim3(total_tiles), dim3(256), 0, st, probs, nprob, segs);
  else
    hipLaunchKernelGGL((k_gemv<T, 0>), dim3(total_tiles), dim3(256), 0, st, probs, nprob, segs);
}

// ---------------------------------------------------------------------------
// dense: grouped products with 16-column groups
// ---------------------------------------------------------------------------
// Workgroup (problem, 64-row tile, K piece, GS column groups): the 4 waves
// take K blocks of 16 in turn (64 x 16 GS accumulators each, A straight from
// memory in operand layout, x one contiguous load per step) and are combined
// in LDS in fixed order.  A is read once for GS groups.  MODE 1: y = sum,
// 0: y -= sum, 2: partial sums (pieces of kGemvPiece16, added by
// k_gemv16_sum in ascending order); the decomposition depends on the problem
// alone.
template <typename T, int MODE, int GS>
__global__ __launch_bounds__(256) void k_gemv16(const GemvProbT<T> *__restrict__ probs, int nprob,
                                                const GemvSegT<T> *__restrict__ segs, T *__restrict__ part) {
  __shared__ T red[4][64][kColGroup];
  const int bid = blockIdx.x;
  int lo = 0, hi = nprob - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (probs[mid].wg0 <= bid) lo = mid;
    else hi = mid - 1;
  }
  const GemvProbT<T> P = probs[lo];
  const int gsteps = (P.groups + GS - 1) / GS;
  const int local = bid - P.wg0, g0 = (local % gsteps) * GS, pc = local / gsteps % P.parts,
            lt = local / (gsteps * P.parts);
  const int m0 = lt * 64, ng = min(GS, P.groups - g0);
  const int lane = threadIdx.x & 63, l16 = lane & 15, lk = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Frag<T> acc[GS][4];
#pragma unroll
  for (int g = 0; g < GS; g++)
#pragma unroll
    for (int b = 0; b < 4; b++) acc[g][b] = frag_zero<T>();
  int row[4];
#pragma unroll
  for (int b = 0; b < 4; b++) row[b] = min(m0 + 16 * b + l16, P.M - 1);
  for (int sg = 0; sg < P.nseg; sg++) {
    const GemvSegT<T> S = segs[P.seg0 + sg];
    int kb = P.tri == 2 ? m0 : 0, ke = P.tri == 1 ? min(S.K, m0 + 64) : S.K;
    if (MODE == 2) kb = max(kb, pc * kGemvPiece16), ke = min(ke, (pc + 1) * kGemvPiece16);
    const auto A = gptr(S.A);
    const auto X = gptr(S.x) + (long long)g0 * S.ldx + l16;
    for (int k0 = kb + 16 * w; k0 < ke; k0 += 64) {
      T a[4][4], x[GS][4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int k = k0 + frag_row<T>(r, lk), kc = min(k, ke - 1);
        const auto pc_ = A + (long long)kc * S.lda;
#pragma unroll
        for (int b = 0; b < 4; b++) a[b][r] = pc_[row[b]];
#pragma unroll
        for (int g = 0; g < GS; g++) {
          const T v = X[(g < ng ? g : 0) * S.ldx + (long long)kc * kColGroup];
          x[g][r] = k < ke ? v : T(0);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int g = 0; g < GS; g++)
#pragma unroll
          for (int b = 0; b < 4; b++) acc[g][b] = mfma4(a[b][r], x[g][r], acc[g][b]);
    }
  }
#pragma unroll
  for (int g = 0; g < GS; g++) {
    if (g >= ng) break;
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int r = 0; r < 4; r++) red[w][16 * b + frag_row<T>(r, lk)][l16] = acc[g][b][r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = 16 * w + 4 * r + lk;
      const T v = red[0][m][l16] + red[1][m][l16] + red[2][m][l16] + red[3][m][l16];
      if (MODE == 2) {
        part[P.poff + ((long long)(lt * P.parts + pc) * P.groups + g0 + g) * (64 * kColGroup) + m * kColGroup + l16] = v;
      } else if (m0 + m < P.M) {
        auto y = gptr(P.y) + (long long)(g0 + g) * P.ldy + (long long)(m0 + m) * kColGroup + l16;
        if (MODE == 1) *y = v;
        else *y = *y - v;
      }
    }
  }
}
template <typename T, int MODE>
__global__ __launch_bounds__(256) void k_gemv16_sum(const GemvProbT<T> *__restrict__ probs, int nprob,
                                                    const T *__restrict__ part) {
  const int tile = blockIdx.x, g = blockIdx.y;
  int lo = 0, hi = nprob - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (probs[mid].tile0 <= tile) lo = mid;
    else hi = mid - 1;
  }
  const GemvProbT<T> P = probs[lo];
  if (g >= P.groups) return;
  const int lt = tile - P.tile0;
  const T *in = part + P.poff + ((long long)lt * P.parts * P.groups + g) * (64 * kColGroup);
#pragma unroll
  for (int e = threadIdx.x; e < 64 * kColGroup; e += 256) {
    const int m = lt * 64 + e / kColGroup;
    if (m >= P.M) break;
    T v = in[e];
    for (int pc = 1; pc < P.parts; pc++) v += in[(long long)pc * P.groups * (64 * kColGroup) + e];
    auto y = gptr(P.y) + (long long)g * P.ldy + (long long)m * kColGroup + e % kColGroup;
    if (MODE == 1) *y = v;
    else *y = *y - v;
  }
}
template <typename T, int GS>
static void launch_gemv16_gs(const GemvProbT<T> *probs, int nprob, const GemvSegT<T> *segs, int total_wgs, int mode,
                             T *part, hipStream_t st) {
  const dim3 g(total_wgs), b(256);
  if (part) hipLaunchKernelGGL((k_gemv16<T, 2, GS>), g, b, 0, st, probs, nprob, segs, part);
  else if (mode == 1) hipLaunchKernelGGL((k_gemv16<T, 1, GS>), g, b, 0, st, probs, nprob, segs, part);
  else hipLaunchKernelGGL((k_gemv16<T, 0, GS>), g, b, 0, st, probs, nprob, segs, part);
}
template <typename T>
void launch_gemv16(const GemvProbT<T> *probs, int nprob, const GemvSegT<T> *segs, int total_tiles, int total_wgs,
                   int gstep, int max_groups, int mode, T *part, hipStream_t st) {
  if (total_tiles <= 0 || nprob <= 0) return;
  if (gstep == 4) launch_gemv16_gs<T, 4>(probs, nprob, segs, total_wgs, mode, part, st);
  else if (gstep == 2) launch_gemv16_gs<T, 2>(probs, nprob, segs, total_wgs, mode, part, st);
  else launch_gemv16_gs<T, 1>(probs, nprob, segs, total_wgs, mode, part, st);
  if (!part) return;
  const dim3 g(total_tiles, max_groups), b(256);
  if (mode == 1) hipLaunchKernelGGL((k_gemv16_sum<T, 1>), g, b, 0, st, probs, nprob, part);
  else hipLaunchKernelGGL((k_gemv16_sum<T, 0>), g, b, 0, st, probs, nprob, part);
}

#define SNU_SOLVE_INST(T)                                                                            \
  template void launch_permute_in<T>(const PermDev *, int, const VecDev *, T *, long long, hipStream_t); \
  template void launch_permute_out<T>(const PermDev *, int, const VecDev *, const T *, long long,   \
                                      bool, const int *, hipStream_t);                              \
  template void launch_assemble_rhs<T>(const TargetDev *, int, const int *, const VecDev *, const T *, T *, int, \
                                       bool, bool, hipStream_t);                                    \
  template void launch_leaf_sweep<T>(const LeafDev *, int, const VecDev *, T *, T *, int, bool, bool, bool, \
                                     hipStream_t);                                                  \
  template void launch_gemv_split<T>(const GemvProbT<T> *, int, const GemvSegT<T> *, int, int, T *, int *, \
                                     hipStream_t);                                                  \
  template void launch_gemv<T>(const GemvProbT<T> *, int, const GemvSegT<T> *, int, int, hipStream_t); \
  template void launch_gemv16<T>(const GemvProbT<T> *, int, const GemvSegT<T> *, int, int, int, int, int, T *, \
                                 hipStream_t);
SNU_SOLVE_INST(double)
SNU_SOLVE_INST(float)
#undef SNU_SOLVE_INST

}  // namespace snu
