// Kernels of the multifrontal leaf factorization (gfx950, wave64).
//
// A leaf's no-pivot LU (the reference's core_numfact_v2 and core_GEMM,
// src/kernel_sparse.cu:740-781,953-971) runs as dense partial factorizations
// of frontal matrices, level by level of the leaves' front trees, every leaf
// of every matrix of a launch set sharing each launch:
//   small fronts (the whole front fits the LDS): k_front_wave does everything
//     in one wave per front, k_front_small in one workgroup;
//   larger fronts live in global memory: k_extend_add builds them, then the
//     blocked partial LU on the dense kernels (k_diag_panel, or k_diag_lu and
//     k_panel, with the pivot clamp; the update on the MFMA k_gemm);
//   k_extend_add then adds the root fronts' updates into the separator blocks
//     (the reference's boundary Schur assembly).
// The factors stay in the fronts, where the solves read them.
// Every position receives its contributions in a fixed order, so results do
// not depend on scheduling.
#include <hip/hip_runtime.h>

#include <utility>

#include "snu_device.h"
#include "snu_kernels.h"

namespace snu {

extern __shared__ __align__(16) char front_lds[];

// One workgroup per front, the whole front in LDS (f^2 values).
template <typename T>
__global__ __launch_bounds__(256) void k_front_small(const FrontDev *__restrict__ fr, T eps) {
  T *F = (T *)front_lds;
  const FrontDev D = fr[blockIdx.x];
  const int f = D.f, nk = D.nk, n2 = f * f, tid = threadIdx.x, nt = blockDim.x;
  for (int i = tid; i < n2; i += nt) F[i] = T(0);
  __syncthreads();
  for (int q = tid; q < D.nent; q += nt) {
    const AEntry e = D.ent[q];
    F[e.pos] = (T)D.aval[e.idx];
  }
  __syncthreads();
  // children's updates, one child after another (fixed summation order)
  // (lane = row within 64-row groups, wave = column modulo the waves)
  const int lane = tid & 63, wv = tid >> 6, nw = nt >> 6;
  for (int c = 0; c < D.nchild; c++) {
    const FrontChild C = D.child[c];
    const auto U = gptr((const T *)C.U);
    const auto rel = gptr(C.rel);
    const int nb = C.nb;
    for (int b = wv; b < nb; b += nw) {
      const int cb = rel[b] * f;
      for (int a = lane; a < nb; a += 64) F[rel[a] + cb] += U[a + (long long)b * C.ld];
    }
    __syncthreads();
  }
  // partial LU of the nk pivots (right-looking; each entry receives its
  // updates in ascending pivot order, as in the reference's elimination)
  for (int p = 0; p < nk; p++) {
    T d = F[p + p * f];
    if (d < eps && d > -eps) d = d < T(0) ? -eps : eps;
    const int m = f - p - 1;
    T *col = F + p * f + p + 1;
    for (int i = tid; i < m; i += nt) col[i] = col[i] / d;
    if (tid == 0) F[p + p * f] = d;
    __syncthreads();
    for (int c = p + 1 + wv; c < f; c += nw) {
      const T u = F[p + c * f];
      T *dst = F + c * f + p + 1;
      for (int r = lane; r < m; r += 64) dst[r] -= col[r] * u;
    }
    __syncthreads();
  }
  // the whole front to global memory: the solves read its factors, its
  // parent the update block
  const auto G = gptr((T *)D.F);
  for (int i = tid; i < n2; i += nt) G[i] = F[i];
}

// One wave per front of order <= kFrontWave: assembled in LDS (f^2 values), then
// lane = row with the columns in registers; the pivot row by v_readlane, so no
// barrier anywhere.  A front's columns come in chunks of 8 (those past f are
// skipped), its arithmetic is k_front_small's, operation for operation.
// Bound by instruction issue (three per column and pivot) and, where a launch
// fills the device, by the fronts written; k_front_small's two barriers per
// pivot left its waves waiting: 8190 fronts of order 31 with 15 pivots 123 -> 65
// us FP64, 32,898 of order 28 with 10 pivots 430 -> 252, 16 fronts 24 -> 13.
// Orders above 48 would take more than 128 registers.
constexpr int kFrontCol = 8;
// (the pivot row's entries are read with every lane active: its own lane takes
// no part in the update, and what the register holds there inside the branch is
// the register allocator's affair)
template <typename T, int P, int C>
__device__ __forceinline__ void wave_update(T (&a)[kFrontWave], T q, int f, int lane) {
  if constexpr (C < kFrontWave) {
    if (C < f) {
      T u[kFrontCol];
#pragma unroll
      for (int c = 0; c < kFrontCol; c++)
        if (C + c > P) u[c] = rld(a[C + c], P);
      if (lane > P) {
#pragma unroll
        for (int c = 0; c < kFrontCol; c++)
          if (C + c > P) a[C + c] -= q * u[c];
      }
      wave_update<T, P, C + kFrontCol>(a, q, f, lane);
    }
  }
}
template <typename T, int P>
__device__ __forceinline__ void wave_step(T (&a)[kFrontWave], int f, int nk, int lane, T eps) {
  if (P >= nk) return;
  T d = rld(a[P], P);
  if (d < eps && d > -eps) d = d < T(0) ? -eps : eps;
  const T q = a[P] / d;
  a[P] = lane > P ? q : lane == P ? d : a[P];
  wave_update<T, P, (P + 1) / kFrontCol * kFrontCol>(a, q, f, lane);
}
template <typename T, int... P>
__device__ __forceinline__ void wave_steps(std::integer_sequence<int, P...>, T (&a)[kFrontWave], int f, int nk,
                                           int lane, T eps) {
  (wave_step<T, P>(a, f, nk, lane, eps), ...);
}
template <typename T>
__global__ __launch_bounds__(64) void k_front_wave(const FrontDev *__restrict__ fr, T eps) {
  T *F = (T *)front_lds;
  const FrontDev D = fr[blockIdx.x];
  const int f = D.f, n2 = f * f, lane = threadIdx.x;
  for (int i = lane; i < n2; i += 64) F[i] = T(0);
  __syncthreads();  // (one wave: orders its LDS accesses)
  for (int q = lane; q < D.nent; q += 64) {
    const AEntry e = D.ent[q];
    F[e.pos] = (T)gptr(D.aval)[e.idx];
  }
  __syncthreads();
  // children's updates, one child after another (fixed summation order); lane
  // = row, 8 columns' loads in flight
  for (int c = 0; c < D.nchild; c++) {
    const FrontChild C = D.child[c];
    if (C.nb == 0) continue;
    const auto U = gptr((const T *)C.U) + min(lane, C.nb - 1);
    const auto rel = gptr(C.rel);
    const int row = rel[min(lane, C.nb - 1)];
    for (int b = 0; b < C.nb; b += 8) {
      T u[8];
      int col[8];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int bj = min(b + j, C.nb - 1);
        col[j] = rel[bj] * f;
        u[j] = U[(long long)bj * C.ld];
      }
#pragma unroll
      for (int j = 0; j < 8; j++)
        if (lane < C.nb && b + j < C.nb) F[row + col[j]] += u[j];
    }
    __syncthreads();
  }
  T a[kFrontWave];
#pragma unroll
  for (int c = 0; c < kFrontWave; c++) a[c] = c < f ? F[min(lane, f - 1) + c * f] : T(0);
  wave_steps<T>(std::make_integer_sequence<int, kFrontWave>{}, a, f, D.nk, lane, eps);
  const auto G = gptr((T *)D.F) + lane;
  if (lane < f) {
#pragma unroll
    for (int c = 0; c < kFrontWave; c++)
      if (c < f) G[c * f] = a[c];
  }
}

// Largest front factored whole in LDS (order): above it a front goes
// through HBM and the dense kernels.  Measured 64 / 80 / 96 / 128 (FP64) on
// the 64^3, 96^3 and batch workloads: smaller LDS fronts keep more
// workgroups per CU, and the larger ones are faster on MFMA.
template <typename T>
int front_small_max() {
  return sizeof(T) == 8 ? 64 : 96;
}

template <typename T>
void launch_front_small(const FrontDev *fr, int nfront, int max_f, double eps, hipStream_t st) {
  if (nfront <= 0) return;
  const size_t lds = (size_t)max_f * max_f * sizeof(T);
  (void)hipFuncSetAttribute((const void *)k_front_small<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds);
  hipLaunchKernelGGL(k_front_small<T>, dim3(nfront), dim3(256), lds, st, fr, (T)eps);
}

// One 64 x 64 tile of a target per workgroup, wave w its columns 16 w ..
// 16 w + 15, lane = row, summed in registers and written once: every source
// that lands in the tile (the host lists them, in order) is read through the
// maps tile row -> its row, tile column -> its column, which each wave builds
// in LDS from the source's ascending positions; A's entries are added last.
// Every stored tile is one, so nothing is cleared before (clearing the
// separator blocks, 2.0 GB, and reading them back took 0.5 ms of a 64^3
// factorization).  Bound by the update blocks read and the target written;
// 64^3 7-point FP64, all heights and the separator blocks together 1.6 ms.
// (Fronts zeroed, filled from CSR factor slots and added to child by child in
// memory took 3.5 ms, boundary Schur blocks gathered and then added 2.1 ms, the
// factors' write-back into CSR slots 1.5 ms.)
template <typename T>
__global__ __launch_bounds__(256) void k_extend_add(const AddTile *__restrict__ tiles,
                                                    const AddSrc *__restrict__ src) {
  __shared__ int rmap[4][64], cmap[4][64];
  const AddTile t = tiles[blockIdx.x];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c0 = 16 * wave;
  const auto C = gptr((T *)t.C) + min(lane, t.nr - 1);
  T v[16];
#pragma unroll
  for (int j = 0; j < 16; j++) v[j] = T(0);
  for (int s = t.s0; s < t.s1; s++) {
    const AddSrc S = src[s];
    const auto pos = gptr(S.pos);
    // (the fences keep the compiler from carrying a lane's own value over
    // another lane's store; the wave's LDS accesses run in order)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    rmap[wave][lane] = -1;
    cmap[wave][lane] = -1;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < S.rn) rmap[wave][pos[S.rb + lane] - S.r0] = S.rb + lane;
    if (lane < S.cn) cmap[wave][pos[S.cb + lane] - S.c0] = S.cb + lane;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int rr = rmap[wave][lane], cc = cmap[wave][lane];
    if (!__any(lane >= c0 && lane < c0 + 16 && cc >= 0)) continue;
    const auto U = gptr((const T *)S.U) + max(rr, 0);
    T u[16];
    int col[16];  // (read with every lane active)
#pragma unroll
    for (int j = 0; j < 16; j++) col[j] = rl(cc, c0 + j);
#pragma unroll
    for (int j = 0; j < 16; j++) u[j] = U[(long long)max(col[j], S.cb) * S.ld];
#pragma unroll
    for (int j = 0; j < 16; j++)
      if (rr >= 0 && col[j] >= 0) v[j] += u[j];
  }
  if (lane < t.nr) {
#pragma unroll
    for (int j = 0; j < 16; j++)
      if (c0 + j < t.nc) C[(c0 + j) * t.ldc] = v[j];
  }
  if (t.nent == 0) return;  // uniform
  __syncthreads();
  const auto base = gptr((T *)t.C);
  for (int q = threadIdx.x; q < t.nent; q += 256) {
    const AEntry e = t.ent[q];
    base[e.pos] += (T)gptr(t.aval)[e.idx];
  }
}
template <typename T>
void launch_front_wave(const FrontDev *fr, int nfront, int max_f, double eps, hipStream_t st) {
  if (nfront <= 0) return;
  const size_t lds = (size_t)max_f * max_f * sizeof(T);
  hipLaunchKernelGGL(k_front_wave<T>, dim3(nfront), dim3(64), lds, st, fr, (T)eps);
}
template <typename T>
void launch_extend_add(const AddTile *tiles, int ntile, const AddSrc *src, hipStream_t st) {
  if (ntile <= 0) return;
  hipLaunchKernelGGL(k_extend_add<T>, dim3(ntile), dim3(256), 0, st, tiles, src);
}

#define SNU_FRONT_INST(T)                                                                      \
  template int front_small_max<T>();                                                           \
  template void launch_front_small<T>(const FrontDev *, int, int, double, hipStream_t);        \
  template void launch_front_wave<T>(const FrontDev *, int, int, double, hipStream_t);         \
  template void launch_extend_add<T>(const AddTile *, int, const AddSrc *, hipStream_t);
SNU_FRONT_INST(double)
SNU_FRONT_INST(float)
#undef SNU_FRONT_INST

}  // namespace snu
