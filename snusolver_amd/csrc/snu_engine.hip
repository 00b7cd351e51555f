// Host-side engine: device layout of one matrix, launch lists of its dense
// factorization and dense solves, merging of the lists of several matrices,
// and the executors of the factor and solve sweeps.
//
// Phase map (reference -> here):
//   core_run (kernel_sparse.cu:1011-1037)        -> the leaf fronts, then
//        k_extend_add into the separator blocks
//   dense level loop (SnuMat_factorize.cu:258-284) -> per level: blocked
//        getrf/trsm (k_diag_panel), then grouped k_gemm for the Schur updates
//        of the level (K-concatenated over siblings: replaces reduction_gpu,
//        SnuMat_factorize.cu:78-124)
//   forward solve (core_trsm/core_update_b, trsm_Lxb/gemm on b; fused into
//        the factorization in the reference) and backward solve
//        (SnuMat_factorize.cu:286-345)     -> run_sweep
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <unordered_map>

#include "snu_engine.h"

namespace snu {

int device_alloc(snumat *h, void **p, size_t bytes) {
  *p = nullptr;
  if (bytes == 0) bytes = 1;
  const hipError_t e = bytes > h->alloc_limit ? hipErrorOutOfMemory : hipMalloc(p, bytes);
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();  // (reported here; the next launch's check must not see it)
    return set_error(SNU_ERR_OOM, "hipMalloc of " + std::to_string(bytes) + " bytes failed (" +
                                      hipGetErrorString(e) + ")");
  }
  h->allocs.push_back(*p);
  h->dev_bytes += bytes;
  return SNU_OK;
}

namespace {
template <class T>
int dalloc(snumat *h, T **p, size_t count) {
  return device_alloc(h, (void **)p, std::max<size_t>(1, count) * sizeof(T));
}
template <class T>
int dupload(snumat *h, T **p, const std::vector<T> &v) {
  int rc = dalloc(h, p, v.size());
  if (rc) return rc;
  if (!v.empty()) HIPCHK(hipMemcpy(*p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return SNU_OK;
}
}  // namespace

template <typename T>
int upload_list(T **p, const std::vector<T> &v) {
  *p = nullptr;
  HIPCHK(hipMalloc((void **)p, std::max<size_t>(1, v.size()) * sizeof(T)));
  if (!v.empty()) HIPCHK(hipMemcpy(*p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return SNU_OK;
}

float ev_ms(hipEvent_t a, hipEvent_t b) {
  float ms = 0;
  (void)hipEventElapsedTime(&ms, a, b);
  return ms;
}

// ---------------------------------------------------------------------------
// dense plan (structure only; pointers into the matrix's value arrays)
// ---------------------------------------------------------------------------
template <typename T>
int add_gemm(std::vector<GemmProbT<T>> &gp, std::vector<GemmSegT<T>> &gs, int &tiles,
             T *C, long long ldc, int M, int N, const std::vector<GemmSegT<T>> &segs,
             double &flops, int tb) {
  if (M <= 0 || N <= 0) return 0;
  GemmProbT<T> p;
  p.C = C;
  p.ldc = ldc;
  p.M = M;
  p.N = N;
  p.seg0 = (int)gs.size();
  p.nseg = 0;
  for (const GemmSegT<T> &s : segs)
    if (s.K > 0) {
      gs.push_back(s);
      p.nseg++;
      flops += 2.0 * M * N * s.K;
    }
  if (p.nseg == 0) return 0;
  p.tiles_n = (N + tb - 1) / tb;
  p.tile0 = tiles;
  tiles += ((M + tb - 1) / tb) * p.tiles_n;
  gp.push_back(p);
  return 1;
}
template int add_gemm<double>(std::vector<GemmProbT<double>> &, std::vector<GemmSegT<double>> &,
                              int &, double *, long long, int, int,
                              const std::vector<GemmSegT<double>> &, double &, int);
template int add_gemm<float>(std::vector<GemmProbT<float>> &, std::vector<GemmSegT<float>> &,
                             int &, float *, long long, int, int,
                             const std::vector<GemmSegT<float>> &, double &, int);

// ---------------------------------------------------------------------------
// tile-shape autotuner: per precision and size bucket of min(M, N), the
// faster of the 64 x 64 and 128 x 128 C -= AB kernels on a launch of many
// problems of the bucket's probe size (enough tiles to fill the device, as
// in the Schur-update launches), measured once per process on
// device-resident operands (both tiles compute every element with the same
// instruction sequence, so the choice never changes results)
// ---------------------------------------------------------------------------
namespace {
std::mutex g_tune_mu;
bool g_tuned[2] = {false, false};
int g_tile[2][3] = {{128, 128, 128}, {128, 128, 128}};
const int kBucketEdge[3] = {128, 512, 2048};
const int kBucketProbe[3] = {128, 1024, 4096};

template <typename T>
double time_gemm(int n, int count, int K, int tile, int reps) {
  T *dA = nullptr, *dB = nullptr, *dC = nullptr;
  GemmProbT<T> *dgp = nullptr;
  GemmSegT<T> *dgs = nullptr;
  double ms_out = -1;
  if (hipMalloc((void **)&dA, sizeof(T) * (size_t)n * K) == hipSuccess &&
      hipMalloc((void **)&dB, sizeof(T) * (size_t)K * n) == hipSuccess &&
      hipMalloc((void **)&dC, sizeof(T) * (size_t)n * n * count) == hipSuccess) {
    launch_fill(dA, (long long)n * K, nullptr);
    launch_fill(dB, (long long)K * n, nullptr);
    launch_fill(dC, (long long)n * n * count, nullptr);
    std::vector<GemmProbT<T>> gp;
    std::vector<GemmSegT<T>> gs;
    int tiles = 0;
    double fl = 0;
    for (int c = 0; c < count; c++)
      add_gemm<T>(gp, gs, tiles, dC + (size_t)n * n * c, n, n, n, {GemmSegT<T>{dA, dB, n, K, K}}, fl, tile);
    if (upload_list(&dgp, gp) == SNU_OK && upload_list(&dgs, gs) == SNU_OK) {
      auto run = [&]() {
        if (tile == 128) launch_gemm128<T>(dgp, count, dgs, tiles, 0, nullptr);
        else launch_gemm<T>(dgp, count, dgs, tiles, 0, nullptr);
      };
      hipEvent_t e0, e1;
      if (hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess) {
        run();
        (void)hipEventRecord(e0, nullptr);
        for (int r = 0; r < reps; r++) run();
        (void)hipEventRecord(e1, nullptr);
        if (hipEventSynchronize(e1) == hipSuccess) ms_out = ev_ms(e0, e1) / reps;
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
      }
    }
  }
  (void)hipDeviceSynchronize();
  if (dA) (void)hipFree(dA);
  if (dB) (void)hipFree(dB);
  if (dC) (void)hipFree(dC);
  if (dgp) (void)hipFree(dgp);
  if (dgs) (void)hipFree(dgs);
  return ms_out;
}
}  // namespace

template <typename T>
void autotune_tiles() {
  const int pi = std::is_same<T, float>::value ? 1 : 0;
  std::lock_guard<std::mutex> lk(g_tune_mu);
  if (g_tuned[pi]) return;
  for (int b = 0; b < 3; b++) {
    const int n = kBucketProbe[b], count = (4096 / n) * (4096 / n);
    const double t64 = time_gemm<T>(n, count, 1024, 64, 3), t128 = time_gemm<T>(n, count, 1024, 128, 3);
    if (t64 > 0 && t128 > 0) g_tile[pi][b] = t128 < t64 ? 128 : 64;
  }
  g_tuned[pi] = true;
}
template void autotune_tiles<double>();
template void autotune_tiles<float>();

int tile_for(int prec, int M, int N) {
  const int m = std::min(M, N);
  if (m < kBucketEdge[0]) return 64;
  const int b = m < kBucketEdge[1] ? 0 : m < kBucketEdge[2] ? 1 : 2;
  return g_tile[prec == SNU_FP32 ? 1 : 0][b];
}
int tile_table(int prec, int *out3) {
  for (int b = 0; b < 3; b++) out3[b] = g_tile[prec == SNU_FP32 ? 1 : 0][b];
  return g_tuned[prec == SNU_FP32 ? 1 : 0] ? 1 : 0;
}

namespace {

// A grouped C -= sum A B launch, split by tile size: problems whose size
// bucket the autotuner gave to the 128 x 128 kernel take it when the launch
// holds at least kMin128Tiles of those tiles (16 per CU: on smaller launches
// the 64 x 64 tiles, four times as many and more workgroups per CU, balance
// better: 64^3 factor 37.2 -> 35.1 ms, 96^3 FP64 440 -> 433 ms against a
// threshold of 512, measured); the rest take 64 x 64 tiles (launch kind 5
// and kind 2).
constexpr int kMin128Tiles = 4096;
// FP32 factorizations whose 128 x 128 tiles run as bf16 splits
// (SNU_GEMM_SPLIT: about twice the rate of the FP32 64 x 64 tile) take the
// large tile for every problem with min(M, N) >= 128, from kMin128Split
// tiles per launch.
constexpr int kMin128Split = 512;
struct TileRule {
  int prec = SNU_FP64;
  bool split = false;
  int pick(int M, int N) const {
    if (split) return std::min(M, N) >= 128 ? 128 : 64;
    return tile_for(prec, M, N);
  }
  long long min128() const { return split ? kMin128Split : kMin128Tiles; }
};
template <typename T>
TileRule tile_rule(const snumat *h) {
  TileRule r;
  r.prec = std::is_same<T, float>::value ? SNU_FP32 : SNU_FP64;
  r.split = r.prec == SNU_FP32 && h->opts.fp32_gemm == SNU_GEMM_SPLIT;
  return r;
}
template <typename T>
struct GemmBatch {
  struct Pend {
    T *C;
    long long ldc;
    int M, N;
    std::vector<GemmSegT<T>> segs;
  };
  std::vector<Pend> pend;
  TileRule rule;
  void add(T *C, long long ldc, int M, int N, const std::vector<GemmSegT<T>> &segs) {
    if (M > 0 && N > 0) pend.push_back(Pend{C, ldc, M, N, segs});
  }
  void flush(std::vector<GemmProbT<T>> &gp, std::vector<GemmSegT<T>> &gs, std::vector<Launch> &out,
             long long key) {
    long long big = 0;
    for (const Pend &q : pend)
      if (rule.pick(q.M, q.N) == 128) big += (long long)((q.M + 127) / 128) * ((q.N + 127) / 128);
    const bool use128 = big >= rule.min128();
    std::vector<GemmProbT<T>> p[2];
    int tiles[2] = {0, 0};
    double flops[2] = {0, 0};
    for (const Pend &q : pend) {
      const int t = use128 && rule.pick(q.M, q.N) == 128 ? 1 : 0;
      add_gemm(p[t], gs, tiles[t], q.C, q.ldc, q.M, q.N, q.segs, flops[t], t ? 128 : 64);
    }
    pend.clear();
    for (int t = 0; t < 2; t++) {
      if (p[t].empty()) continue;
      Launch L{t ? 5 : 2, (int)gp.size(), (int)p[t].size(), tiles[t], flops[t], key};
      gp.insert(gp.end(), p[t].begin(), p[t].end());
      out.push_back(L);
    }
  }
};

// A grouped GEMV launch (the dense solves).
template <typename T>
struct GemvBatch {
  std::vector<GemvProbT<T>> p;
  int tiles = 0;
  double bytes = 0;
  void add(std::vector<GemvSegT<T>> &vs, T *y, long long ldy, int M, int tri, int groups,
           const std::vector<GemvSegT<T>> &segs) {
    if (M <= 0) return;
    GemvProbT<T> q;
    q.y = y;
    q.ldy = ldy;
    q.M = M;
    q.tri = tri;
    q.groups = groups;
    q.seg0 = (int)vs.size();
    q.nseg = 0;
    for (const GemvSegT<T> &g : segs)
      if (g.K > 0) {
        vs.push_back(g);
        q.nseg++;
        bytes += (double)sizeof(T) * M * g.K * (tri ? 0.5 : 1.0);
      }
    if (!q.nseg) return;
    q.tile0 = tiles;
    tiles += (M + 63) / 64;
    p.push_back(q);
  }
  void flush(int kind, std::vector<GemvProbT<T>> &vp, std::vector<Launch> &out, long long key) {
    if (p.empty()) return;
    out.push_back(Launch{kind, (int)vp.size(), (int)p.size(), tiles, bytes, key});
    vp.insert(vp.end(), p.begin(), p.end());
    p.clear();
    tiles = 0;
    bytes = 0;
  }
};

// Maximal runs [r0, r1) of 64-aligned tiles of [0, len) that hold a
// structural nonzero according to any(x0, x1) (half-open, relative).
template <class F>
std::vector<std::pair<int, int>> nz_runs(int len, F any) {
  std::vector<std::pair<int, int>> out;
  for (int t0 = 0; t0 < len; t0 += 64) {
    int t1 = std::min(len, t0 + 64);
    if (!any(t0, t1)) continue;
    if (!out.empty() && out.back().second == t0) out.back().second = t1;
    else out.push_back({t0, t1});
  }
  return out;
}

// Outer panel width of the blocked LU of the separators' diagonal blocks.
constexpr int kPanel = 512;

// Small fronts by order, a launch per height each: one wave per front, one
// workgroup per front up to kFrontLo, and above it.
constexpr int kFrontLo = 64;
inline int front_class(int f) { return f <= kFrontWave ? 0 : f <= kFrontLo ? 1 : 2; }

// Launch keys: tree height (1 = parents of the leaves) major, then the step
// inside the level.  Matrices of different depths align at equal height.
constexpr long long kHeight = 100000000LL, kPanels = 60000000LL, kNextD = 90000000LL;
inline long long fkey(int height, long long step) { return height * kHeight + step; }

// Host-built launch descriptors of the dense factorization of one matrix.
// Per tree level, bottom-up:
//   for each 64-column step k of the diagonal blocks D: LU of the diagonal
//   block and the inverses of its triangles (written into the separator's full
//   L^-1 / U^-1), L21 <- L21 U11^-1 and U12 <- L11^-1 U12 inside D by the
//   block inverses, trailing update of D (GEMM);
//   then the full inverses L^-1, U^-1 of every separator of the level by
//   recursive doubling (two grouped GEMMs per doubling step);
//   then the panels in one pass each, Lp <- Lp U^-1 and Up <- L^-1 Up (GEMM
//   into scratch over the structurally nonzero rows / columns, K limited by
//   the triangle; copied back for the solves): the panels are read and written
//   once instead of once per 64-column step;
//   then the Schur updates of the ancestors, K-concatenated over the level's
//   separators below each of them: one grouped GEMM for the diagonal blocks of
//   the next level (step kNextD), which that level starts from, and one for
//   all others (kNextD + 1).
template <typename T>
void build_dense_plan(snumat *h) {
  using GemmSeg = GemmSegT<T>;
  using DiagProb = DiagProbT<T>;
  const Plan &P = h->P;
  const TileRule rule = tile_rule<T>(h);
  Values<T> &VV = vals<T>(h);
  T *dense = VV.arena;
  auto R = [&](int p) { return dense + P.offR[p]; };
  auto Lp = [&](int p) { return dense + P.offL[p]; };
  auto Li = [&](int p) { return VV.inv + h->inv_off[p]; };
  auto Ui = [&](int p) { return VV.inv + h->inv_off[p] + (long long)P.block_size[p] * P.block_size[p]; };
  DensePlan<T> &F = VV.fact;
  auto &h_dp = F.dp;
  auto &h_gp = F.gp;
  auto &h_gs = F.gs;
  auto &out = F.launches;
  h_dp.clear();
  h_gp.clear();
  h_gs.clear();
  out.clear();
  std::vector<T *> outL(P.np), outU(P.np);  // the products of a level's panels
  for (int l = P.max_level - 1; l >= 0; l--) {
    const int height = P.max_level - l;
    int lo = 1 << l, hi = std::min((2 << l) - 1, P.np - 1);
    int smax = 0;
    for (int i = lo; i <= hi; i++) smax = std::max(smax, P.block_size[i]);
    for (int k = 0; k < smax; k += 64) {
      const long long ks = (long long)(k / 64) * 8;
      Launch d{0, (int)h_dp.size(), 0, 0, 0, fkey(height, ks + 0)};
      for (int i = lo; i <= hi; i++) {
        int s = P.block_size[i];
        if (s <= k) continue;
        int nb = std::min(64, s - k);
        DiagProb dp{};  // eps = 0: separator pivots are not clamped
        dp.D = R(i) + k + (long long)k * s;
        dp.ld = s;
        dp.nb = nb;
        dp.Linv = Li(i) + k + (long long)k * s;
        dp.Uinv = Ui(i) + k + (long long)k * s;
        dp.ldi = s;
        dp.LU = VV.lu + h->lu_off[i] + (long long)(k / 64) * 4096;
        // L21 <- L21 U11^-1 (rows of D below the block) and U12 <- L11^-1 U12
        // (row block of D right of it)
        dp.m = s - k - nb;
        dp.tile0 = d.tiles;
        d.tiles += panel_tiles(dp.m);
        d.flops += 4.0 * dp.m * nb * nb;
        h_dp.push_back(dp);
        d.np++;
      }
      if (d.np) out.push_back(d);
      // trailing update of D, outer-blocked by kPanel columns: inside a
      // panel [K0, K1) a step updates only the L-shaped rest of the panel
      // (its columns below the step, its rows right of the panel); the last
      // step of the panel applies the panel's K1 - K0 rank-64 updates to the
      // trailing block D[K1:, K1:] as one product with K = K1 - K0 (a K = 64
      // update reads and writes the whole trailing block per step)
      GemmBatch<T> tu;
      tu.rule = rule;
      const int K0 = k - k % kPanel;
      for (int i = lo; i <= hi; i++) {
        const int s = P.block_size[i];
        if (s <= k) continue;
        const int nb = std::min(64, s - k), k2 = k + nb, K1 = std::min(s, K0 + kPanel);
        auto D = [&](int r, int c) { return R(i) + r + (long long)c * s; };
        if (k2 < K1) {
          tu.add(D(k2, k2), s, s - k2, K1 - k2, {GemmSeg{D(k2, k), D(k, k2), s, s, nb}});
          tu.add(D(k2, K1), s, K1 - k2, s - K1, {GemmSeg{D(k2, k), D(k, K1), s, s, nb}});
        } else {
          tu.add(D(K1, K1), s, s - K1, s - K1, {GemmSeg{D(K1, K0), D(K0, K1), s, s, K1 - K0}});
        }
      }
      tu.flush(h_gp, h_gs, out, fkey(height, ks + 3));
    }
    // full triangular inverses by recursive doubling:
    //   U: X[r0:, c0:] = -X[r0:, r0:] (U[r0:, c0:] X[c0:, c0:])
    //   L: X[c0:, r0:] = -X[c0:, c0:] (L[c0:, r0:] X[r0:, r0:])
    int step = 0;
    for (int hh = 64; hh < smax; hh *= 2, step++) {
      const long long base = 50000000LL + step * 4;
      Launch t1{1, (int)h_gp.size(), 0, 0, 0, fkey(height, base)};
      Launch t2{6, 0, 0, 0, 0, fkey(height, base + 1)};
      std::vector<GemmProbT<T>> fin;
      long long toff = 0;
      // per W-wide strip of each product, K limited to the triangle of the
      // triangular factor it meets (the rest of that factor is zero)
      long long big = 0;
      for (int i = lo; i <= hi; i++) {
        const int s = P.block_size[i];
        for (int r0 = 0; r0 + hh < s; r0 += 2 * hh) {
          const int hb = std::min(hh, s - r0 - hh);
          if (rule.pick(hh, hb) == 128) big += 2LL * ((hh + 127) / 128) * ((hb + 127) / 128);
        }
      }
      const int W = big >= rule.min128() ? 128 : 64;
      t1.kind = W == 128 ? 10 : 1;
      t2.kind = W == 128 ? 11 : 6;
      for (int i = lo; i <= hi; i++) {
        int s = P.block_size[i];
        for (int r0 = 0; r0 + hh < s; r0 += 2 * hh) {
          int c0 = r0 + hh, hb = std::min(hh, s - c0);
          T *TU = VV.tmp + h->tmp_panels + toff;
          toff += (long long)hh * hb;
          T *TL = VV.tmp + h->tmp_panels + toff;
          toff += (long long)hb * hh;
          // TU = U12 X22, X22 upper triangular: columns [n0, n0 + W) need
          // its rows [0, n0 + W)
          for (int n0 = 0; n0 < hb; n0 += W) {
            const int nt = std::min(W, hb - n0);
            t1.np += add_gemm(h_gp, h_gs, t1.tiles, TU + (long long)n0 * hh, hh, hh, nt,
                              {GemmSeg{R(i) + r0 + (long long)c0 * s, Ui(i) + c0 + (long long)(c0 + n0) * s,
                                       s, s, n0 + nt}},
                              t1.flops, W);
          }
          // TL = L21 X11, X11 lower triangular: columns [n0, n0 + W) need
          // its rows [n0, hh)
          for (int n0 = 0; n0 < hh; n0 += W) {
            const int nt = std::min(W, hh - n0);
            t1.np += add_gemm(h_gp, h_gs, t1.tiles, TL + (long long)n0 * hb, hb, hb, nt,
                              {GemmSeg{R(i) + c0 + (long long)(r0 + n0) * s,
                                       Li(i) + (r0 + n0) + (long long)(r0 + n0) * s, s, s, hh - n0}},
                              t1.flops, W);
          }
          // Ui[r0:, c0:] = -X11 TU, X11 upper triangular: rows [m0, m0 + W)
          // need its columns [m0, hh)
          for (int m0 = 0; m0 < hh; m0 += W) {
            const int mt = std::min(W, hh - m0);
            t2.np += add_gemm(fin, h_gs, t2.tiles, Ui(i) + r0 + m0 + (long long)c0 * s, s, mt, hb,
                              {GemmSeg{Ui(i) + (r0 + m0) + (long long)(r0 + m0) * s, TU + m0, s, hh, hh - m0}},
                              t2.flops, W);
          }
          // Li[c0:, r0:] = -X22 TL, X22 lower triangular: rows [m0, m0 + W)
          // need its columns [0, m0 + W)
          for (int m0 = 0; m0 < hb; m0 += W) {
            const int mt = std::min(W, hb - m0);
            t2.np += add_gemm(fin, h_gs, t2.tiles, Li(i) + c0 + m0 + (long long)r0 * s, s, mt, hh,
                              {GemmSeg{Li(i) + c0 + m0 + (long long)c0 * s, TL, s, hb, m0 + mt}},
                              t2.flops, W);
          }
        }
      }
      if (t1.np) out.push_back(t1);
      if (t2.np) {
        t2.p0 = (int)h_gp.size();
        h_gp.insert(h_gp.end(), fin.begin(), fin.end());
        out.push_back(t2);
      }
    }
    // panels: Lp <- Lp U^-1 per W-column strip of the result (U^-1 is upper
    // triangular: strip [n0, n0 + W) needs rows [0, n0 + W) of it), Up <-
    // L^-1 Up per W-row strip (rows [0, m0 + W) of Up), over the stored
    // (tile-compressed) rows / columns, into scratch; then copied back.
    // W = 128 (128 x 128 tiles) when the autotuner prefers that tile for the
    // level's panels and they hold enough such tiles to fill the device
    {
      long long big = 0;
      for (int i = lo; i <= hi; i++) {
        const int s = P.block_size[i], nl = P.nL[i], nu = P.nU[i];
        if (nl && rule.pick(nl, s) == 128) big += (long long)((nl + 127) / 128) * ((s + 127) / 128);
        if (nu && rule.pick(s, nu) == 128) big += (long long)((s + 127) / 128) * ((nu + 127) / 128);
      }
      const int W = big >= rule.min128() ? 128 : 64;
      Launch pm{W == 128 ? 10 : 1, (int)h_gp.size(), 0, 0, 0, fkey(height, kPanels)};
      std::vector<GemmProbT<T>> cp;
      Launch cl{3, 0, 0, 0, 0, fkey(height, kPanels + 1)};
      double cfl = 0;
      long long toff = 0;
      for (int i = lo; i <= hi; i++) {
        const int s = P.block_size[i], m = P.nL[i], nc = P.nU[i];
        if (m && s) {
          T *dst = outL[i] = VV.tmp + toff;
          toff += (long long)m * s;
          T *src = Lp(i);
          for (int n0 = 0; n0 < s; n0 += W) {
            const int nt = std::min(W, s - n0), kk = n0 + nt;
            pm.np += add_gemm(h_gp, h_gs, pm.tiles, dst + (long long)n0 * m, m, m, nt,
                              {GemmSeg{src, Ui(i) + (long long)n0 * s, m, s, kk}}, pm.flops, W);
          }
          cl.np += add_gemm(cp, h_gs, cl.tiles, src, m, m, s, {GemmSeg{dst, dst, m, m, 1}}, cfl);
        }
        if (nc && s) {
          T *dst = outU[i] = VV.tmp + toff;
          toff += (long long)s * nc;
          T *src = R(i) + (long long)s * s;
          for (int m0 = 0; m0 < s; m0 += W) {
            const int mt = std::min(W, s - m0), kk = m0 + mt;
            pm.np += add_gemm(h_gp, h_gs, pm.tiles, dst + m0, s, mt, nc,
                              {GemmSeg{Li(i) + m0, src, s, s, kk}}, pm.flops, W);
          }
          cl.np += add_gemm(cp, h_gs, cl.tiles, src, s, s, nc, {GemmSeg{dst, dst, s, s, 1}}, cfl);
        }
      }
      if (pm.np) out.push_back(pm);
      if (cl.np) {
        cl.p0 = (int)h_gp.size();
        h_gp.insert(h_gp.end(), cp.begin(), cp.end());
        out.push_back(cl);
      }
    }
    // Schur updates of every ancestor, K-concatenated over the level's
    // separators below it (the next level's diagonal blocks first).  Emitted per
    // target tile (64 rows / columns aligned to the first index of the block
    // they belong to, the tiles of the compressed storage), with only the
    // contributors that store both the L-panel rows and the U-panel columns
    // of that tile (the other products are exactly zero).
    GemmBatch<T> sc, sn;
    sc.rule = sn.rule = rule;
    for (int p = 1; p < lo; p++) {
      int lp = 31 - __builtin_clz(p);
      int first = p << (l - lp), last = ((p + 1) << (l - lp)) - 1;
      const int sp = P.block_size[p];
      // the tiles of p itself, then the stored tiles of p's ancestors (in
      // ancestor-space order; x: index in p's ancestor space), as
      // {position in the target, width, x}; x = -1 - t for p's own tile t
      std::vector<std::array<int, 3>> own, anL, anU;
      for (int t = 0; t < sp; t += 64) own.push_back({t, std::min(64, sp - t), -1 - t});
      for (int q = p / 2; q; q /= 2) {
        const int o = P.anc_off(p, q), sq = P.block_size[q];
        for (int t = 0; t < sq; t += 64) {
          const int w = std::min(64, sq - t);
          if (P.lmap[p][o + t] >= 0) anL.push_back({P.lmap[p][o + t], w, o + t});
          if (P.umap[p][o + t] >= 0) anU.push_back({sp + P.umap[p][o + t], w, o + t});
        }
      }
      for (int pass = 0; pass < 3; pass++) {  // 0: D_p (not a parent's: R_p = [D_p | Up_p]), 1: Up_p, 2: Lp_p
        const bool parent = lp == l - 1;
        std::vector<std::array<int, 3>> rows = pass == 2 ? anL : own, cols = pass == 1 ? anU : own;
        if (pass == 0 && !parent) cols.insert(cols.end(), anU.begin(), anU.end());
        if (pass == 1 && !parent) continue;
        const int tm = (int)rows.size(), tn = (int)cols.size();
        if (!tm || !tn) continue;
        T *Cb = pass == 2 ? Lp(p) : R(p);
        const int ldc = pass == 2 ? P.nL[p] : sp;
        // index of a tile in contributor i's ancestor space
        auto ix = [&](int i, const std::array<int, 3> &t) {
          return P.anc_off(i, p) + (t[2] < 0 ? -1 - t[2] : sp + t[2]);
        };
        // contributor set of every target tile
        std::vector<std::vector<int>> who((size_t)tm * tn);
        for (int a = 0; a < tm; a++)
          for (int b = 0; b < tn; b++)
            for (int i = first; i <= last; i++)
              if (P.lmap[i][ix(i, rows[a])] >= 0 && P.umap[i][ix(i, cols[b])] >= 0)
                who[(size_t)a * tn + b].push_back(i);
        auto segs_of = [&](const std::vector<int> &w, int a, int b) {
          std::vector<GemmSeg> segs;
          for (int i : w) {
            const int si = P.block_size[i];
            segs.push_back(GemmSeg{outL[i] + P.lmap[i][ix(i, rows[a])],
                                   outU[i] + (long long)P.umap[i][ix(i, cols[b])] * si, P.nL[i], si, si});
          }
          return segs;
        };
        auto emit = [&](int a, int b, int ta, int tb) {
          const std::vector<int> &w = who[(size_t)a * tn + b];
          int mt = 0, nt = 0;
          for (int x = 0; x < ta; x++) mt += rows[a + x][1];
          for (int y = 0; y < tb; y++) nt += cols[b + y][1];
          (parent && pass == 0 ? sn : sc).add(Cb + rows[a][0] + (long long)cols[b][0] * ldc, ldc, mt, nt, segs_of(w, a, b));
        };
        auto nonempty = [&](int a, int b) { return a < tm && b < tn && !who[(size_t)a * tn + b].empty(); };
        // tiles a, a + 1 (rows) are consecutive in every contributor's L
        // panel, b, b + 1 (columns) in its U panel
        auto merge_ok = [&](int a, int b) {
          for (int i : who[(size_t)a * tn + b])
            if (P.lmap[i][ix(i, rows[a + 1])] != P.lmap[i][ix(i, rows[a])] + rows[a][1] ||
                P.umap[i][ix(i, cols[b + 1])] != P.umap[i][ix(i, cols[b])] + cols[b][1])
              return false;
          return true;
        };
        // one problem per target tile with its contributor set, or per 2 x 2
        // tiles when the four share one set and are contiguous in every
        // contributor's panels (the tile kernel is then chosen per size
        // bucket), emitted in strips of 8 tile rows, two tile columns at a
        // time: consecutive tiles (which one XCD runs together) share A rows
        // (same tile row and contributor) and B columns (same tile column),
        // so their operands meet in that XCD's L2
        constexpr int kStrip = 8;
        for (int a0 = 0; a0 < tm; a0 += kStrip)
          for (int b = 0; b < tn; b += 2)
            for (int a = a0; a < std::min(tm, a0 + kStrip); a += 2) {
              const std::vector<int> &w = who[(size_t)a * tn + b];
              if (nonempty(a, b) && nonempty(a + 1, b) && nonempty(a, b + 1) && nonempty(a + 1, b + 1) &&
                  who[(size_t)(a + 1) * tn + b] == w && who[(size_t)a * tn + b + 1] == w &&
                  who[(size_t)(a + 1) * tn + b + 1] == w && merge_ok(a, b)) {
                emit(a, b, 2, 2);
                continue;
              }
              for (int q = 0; q < 4; q++) {
                const int x = a + (q & 1), y = b + (q >> 1);
                if (nonempty(x, y)) emit(x, y, 1, 1);
              }
            }
      }
    }
    sn.flush(h_gp, h_gs, out, fkey(height, kNextD));
    sc.flush(h_gp, h_gs, out, fkey(height, kNextD + 1));
  }
}

// Scratch of a level's panel products (they stay until the level's Schur
// updates have read them) and of the products of the triangular inversion,
// which run beside those: the most of any level, of any doubling step.
struct TmpSize {
  long long panels = 0, inversion = 0;
};
TmpSize tmp_size(const Plan &P) {
  TmpSize best;
  for (int l = P.max_level - 1; l >= 0; l--) {
    int lo = 1 << l, hi = std::min((2 << l) - 1, P.np - 1);
    int smax = 0;
    for (int i = lo; i <= hi; i++) smax = std::max(smax, P.block_size[i]);
    long long panels = 0;
    for (int i = lo; i <= hi; i++) panels += (long long)(P.nL[i] + P.nU[i]) * P.block_size[i];
    best.panels = std::max(best.panels, panels);
    for (int hh = 64; hh < smax; hh *= 2) {
      long long t = 0;
      for (int i = lo; i <= hi; i++) {
        int s = P.block_size[i];
        for (int r0 = 0; r0 + hh < s; r0 += 2 * hh) t += 2LL * hh * std::min(hh, s - r0 - hh);
      }
      best.inversion = std::max(best.inversion, t);
    }
  }
  return best;
}

}  // namespace

// Dense solves of one matrix, per level (y in ys, x overwriting b in bp):
//   forward (bottom-up):  y_i = L_i^-1 b_i;   b_p -= sum_i Lp_i[rows p] y_i
//   backward (top-down):  y_i -= Up_i x_anc;  x_i = U_i^-1 y_i
// Keys: forward launches ascend in height, backward ones descend, all
// backward after all forward.
template <typename T>
void build_solve_plan(const snumat *h, T *bp, T *ys, int nrhs, GemvPlan<T> &S) {
  using GemvSeg = GemvSegT<T>;
  const Values<T> &VV = vals<T>(h);
  const Plan &P = h->P;
  T *dense = VV.arena;
  // one column: groups 0, kinds 7 / 8; several: groups of 16, kinds 17 / 18
  const int w = vec_width(nrhs), groups = nrhs == 1 ? 0 : vec_groups(nrhs);
  const int kset = w == 1 ? 7 : 17, ksub = w == 1 ? 8 : 18;
  const long long n = (long long)P.n * w, ny = (long long)h->sep_rows[P.np] * w;  // values per column (group)
  auto R = [&](int p) { return dense + P.offR[p]; };
  auto Lp = [&](int p) { return dense + P.offL[p]; };
  auto Li = [&](int p) { return VV.inv + h->inv_off[p]; };
  auto Ui = [&](int p) { return VV.inv + h->inv_off[p] + (long long)P.block_size[p] * P.block_size[p]; };
  auto bseg = [&](int p) { return bp + (long long)P.block_start[p] * w; };
  auto yseg = [&](int p) { return ys + (long long)h->sep_rows[p] * w; };
  S.vp.clear();
  S.vs.clear();
  S.fwd.clear();
  S.bwd.clear();
  GemvBatch<T> g;
  for (int l = P.max_level - 1; l >= 0; l--) {
    const int height = P.max_level - l;
    int lo = 1 << l, hi = std::min((2 << l) - 1, P.np - 1);
    for (int i = lo; i <= hi; i++) {
      int s = P.block_size[i];
      g.add(S.vs, yseg(i), ny, s, 1, groups, {GemvSeg{Li(i), bseg(i), s, n, s}});
    }
    g.flush(kset, S.vp, S.fwd, height * 4LL + 0);
    for (int p = 1; p < lo; p++) {
      int lp = 31 - __builtin_clz(p);
      int first = p << (l - lp), last = ((p + 1) << (l - lp)) - 1;
      int sp = P.block_size[p];
      for (int m0 = 0; m0 < sp; m0 += 64) {
        int mt = std::min(64, sp - m0);
        std::vector<GemvSeg> segs;
        for (int i = first; i <= last; i++) {
          const int r = P.lmap[i][P.anc_off(i, p) + m0];  // the tile's stored rows (or -1)
          if (r < 0) continue;
          segs.push_back(GemvSeg{Lp(i) + r, yseg(i), P.nL[i], ny, P.block_size[i]});
        }
        g.add(S.vs, bseg(p) + m0 * w, n, mt, 0, groups, segs);
      }
    }
    g.flush(ksub, S.vp, S.fwd, height * 4LL + 1);
  }
  for (int l = 0; l < P.max_level; l++) {
    const int height = P.max_level - l;
    const long long bkey = 1000000000LL - height * 4LL;
    int lo = 1 << l, hi = std::min((2 << l) - 1, P.np - 1);
    for (int i = lo; i <= hi; i++) {
      int s = P.block_size[i];
      std::vector<GemvSeg> segs;
      for (int a = i / 2; a >= 1; a /= 2) {
        int off = P.anc_off(i, a);
        // stored column tiles of a, merged into runs (consecutive stored
        // tiles of one ancestor are consecutive columns of the panel)
        for (auto cr : nz_runs(P.block_size[a], [&](int x0, int x1) { return P.umap[i][off + x0] >= 0; }))
          segs.push_back(GemvSeg{R(i) + (long long)(s + P.umap[i][off + cr.first]) * s, bseg(a) + cr.first * w, s, n,
                                 cr.second - cr.first});
      }
      g.add(S.vs, yseg(i), ny, s, 0, groups, segs);
    }
    g.flush(ksub, S.vp, S.bwd, bkey + 0);
    for (int i = lo; i <= hi; i++) {
      int s = P.block_size[i];
      g.add(S.vs, bseg(i), n, s, 2, groups, {GemvSeg{Ui(i), yseg(i), s, ny, s}});
    }
    g.flush(kset, S.vp, S.bwd, bkey + 1);
  }
}

// Split-K layout: pieces per problem from its longest segment (the problem
// alone decides), workgroup and partial-sum offsets per launch; a launch
// whose problems are all single-piece runs unsplit.  Returns the partial-sum
// values and counters the largest launch needs (launches run in turn and share
// them).
template <typename T>
SplitNeed layout_gemv_plan(GemvPlan<T> &g) {
  SplitNeed need;
  for (std::vector<Launch> *ls : {&g.fwd, &g.bwd})
    for (Launch &L : *ls) {
      const bool one = L.kind == 7 || L.kind == 8;
      const int piece = one ? kGemvPiece : kGemvPiece16;
      int wgs = 0, split = 0, mg = 1;
      long long off = 0;
      for (int q = 0; q < L.np; q++) mg = std::max(mg, g.vp[L.p0 + q].groups);
      L.groups = mg;
      L.gstep = mg > 2 ? 4 : mg;
      for (int q = 0; q < L.np; q++) {
        GemvProbT<T> &p = g.vp[L.p0 + q];
        int kmax = 1;
        for (int j = 0; j < p.nseg; j++) kmax = std::max(kmax, g.vs[p.seg0 + j].K);
        p.parts = (kmax + piece - 1) / piece;
        split |= p.parts > 1;
      }
      for (int q = 0; q < L.np; q++) {
        GemvProbT<T> &p = g.vp[L.p0 + q];
        if (!split) p.parts = 1;
        p.wg0 = wgs;
        p.poff = off;
        const int tiles = (p.M + 63) / 64;
        wgs += tiles * p.parts * (one ? 1 : (p.groups + L.gstep - 1) / L.gstep);
        off += (long long)tiles * p.parts * 64 * (one ? 1 : p.groups * kColGroup);
      }
      L.wgs = one && !split ? 0 : wgs;
      L.part = split ? off : 0;
      need.part = std::max(need.part, (size_t)L.part);
      if (split && one) need.done = std::max(need.done, (size_t)L.tiles);
    }
  return need;
}

template <typename T>
int upload_gemv_plan(GemvPlan<T> &g, hipStream_t st) {
  auto grow = [](auto **p, size_t &cap, size_t need) -> int {
    if (need <= cap && *p) return SNU_OK;
    if (*p) HIPCHK(hipFree(*p));
    *p = nullptr;
    cap = 0;
    const size_t c = std::max<size_t>(need + need / 2, 64);
    if (hipMalloc((void **)p, c * sizeof(**p)) != hipSuccess) {
      *p = nullptr;
      (void)hipGetLastError();
      return set_error(SNU_ERR_OOM, "hipMalloc of " + std::to_string(c * sizeof(**p)) + " bytes for a solve failed");
    }
    cap = c;
    return SNU_OK;
  };
  const SplitNeed need = layout_gemv_plan(g);
  const bool fresh = need.done && (!g.d_done || need.done > g.cap_done);
  int rc;
  if ((rc = grow(&g.d_vp, g.cap_vp, g.vp.size())) || (rc = grow(&g.d_vs, g.cap_vs, g.vs.size())) ||
      (need.part && (rc = grow(&g.d_part, g.cap_part, need.part))) ||
      (need.done && (rc = grow(&g.d_done, g.cap_done, need.done))))
    return rc;
  if (fresh) launch_fill((float *)g.d_done, (long long)g.cap_done, st);
  if (!g.vp.empty())
    HIPCHK(hipMemcpyAsync(g.d_vp, g.vp.data(), g.vp.size() * sizeof(g.vp[0]), hipMemcpyHostToDevice, st));
  if (!g.vs.empty())
    HIPCHK(hipMemcpyAsync(g.d_vs, g.vs.data(), g.vs.size() * sizeof(g.vs[0]), hipMemcpyHostToDevice, st));
  return SNU_OK;
}
template <typename T>
void free_gemv_plan(GemvPlan<T> &g) {
  if (g.d_vp) (void)hipFree(g.d_vp);
  if (g.d_vs) (void)hipFree(g.d_vs);
  if (g.d_part) (void)hipFree(g.d_part);
  if (g.d_done) (void)hipFree(g.d_done);
  g = GemvPlan<T>();
}
template <typename T>
int upload_dense_plan(DensePlan<T> &d) {
  int rc;
  if ((rc = upload_list(&d.d_dp, d.dp)) || (rc = upload_list(&d.d_gp, d.gp)) ||
      (rc = upload_list(&d.d_gs, d.gs)))
    return rc;
  return SNU_OK;
}
template <typename T>
void free_dense_plan(DensePlan<T> &d) {
  if (d.d_dp) (void)hipFree(d.d_dp);
  if (d.d_gp) (void)hipFree(d.d_gp);
  if (d.d_gs) (void)hipFree(d.d_gs);
  d = DensePlan<T>();
}
// ---------------------------------------------------------------------------
// merging the launch lists of several matrices
// ---------------------------------------------------------------------------
namespace {
struct Ref {
  long long key;
  int kind, src, idx;
};
template <class GetLaunches>
std::vector<std::vector<Ref>> group_launches(int nsrc, GetLaunches get, bool descending = false) {
  std::vector<Ref> all;
  for (int s = 0; s < nsrc; s++) {
    const std::vector<Launch> &L = get(s);
    for (int i = 0; i < (int)L.size(); i++) all.push_back(Ref{L[i].key, L[i].kind, s, i});
  }
  std::stable_sort(all.begin(), all.end(), [&](const Ref &a, const Ref &b) {
    if (a.key != b.key) return descending ? a.key > b.key : a.key < b.key;
    return a.kind < b.kind;
  });
  std::vector<std::vector<Ref>> groups;
  for (size_t i = 0; i < all.size(); i++) {
    if (i == 0 || all[i].key != all[i - 1].key || all[i].kind != all[i - 1].kind) groups.emplace_back();
    groups.back().push_back(all[i]);
  }
  return groups;
}
}  // namespace

template <typename T>
void merge_dense(const std::vector<const DensePlan<T> *> &in, DensePlan<T> &out) {
  out.dp.clear();
  out.gp.clear();
  out.gs.clear();
  out.launches.clear();
  auto groups = group_launches((int)in.size(), [&](int s) -> const std::vector<Launch> & {
    return in[s]->launches;
  });
  for (auto &g : groups) {
    Launch M{g[0].kind, 0, 0, 0, 0, g[0].key};
    if (M.kind == 0) {
      M.p0 = (int)out.dp.size();
      for (const Ref &r : g) {
        const DensePlan<T> &D = *in[r.src];
        const Launch &L = D.launches[r.idx];
        for (int q = 0; q < L.np; q++) {
          out.dp.push_back(D.dp[L.p0 + q]);
          out.dp.back().tile0 += M.tiles;
        }
        M.np += L.np;
        M.tiles += L.tiles;
        M.flops += L.flops;
      }
    } else {
      M.p0 = (int)out.gp.size();
      for (const Ref &r : g) {
        const DensePlan<T> &D = *in[r.src];
        const Launch &L = D.launches[r.idx];
        for (int q = 0; q < L.np; q++) {
          GemmProbT<T> p = D.gp[L.p0 + q];
          int s0 = (int)out.gs.size();
          out.gs.insert(out.gs.end(), D.gs.begin() + p.seg0, D.gs.begin() + p.seg0 + p.nseg);
          p.seg0 = s0;
          p.tile0 += M.tiles;
          out.gp.push_back(p);
        }
        M.np += L.np;
        M.tiles += L.tiles;
        M.flops += L.flops;
      }
    }
    out.launches.push_back(M);
  }
}

template <typename T>
void merge_gemv(const std::vector<const GemvPlan<T> *> &in, GemvPlan<T> &out) {
  out.vp.clear();
  out.vs.clear();
  out.fwd.clear();
  out.bwd.clear();
  for (int dir = 0; dir < 2; dir++) {
    auto groups = group_launches((int)in.size(), [&](int s) -> const std::vector<Launch> & {
      return dir == 0 ? in[s]->fwd : in[s]->bwd;
    });
    for (auto &g : groups) {
      Launch M{g[0].kind, (int)out.vp.size(), 0, 0, 0, g[0].key};
      for (const Ref &r : g) {
        const GemvPlan<T> &D = *in[r.src];
        const Launch &L = (dir == 0 ? D.fwd : D.bwd)[r.idx];
        for (int q = 0; q < L.np; q++) {
          GemvProbT<T> p = D.vp[L.p0 + q];
          int s0 = (int)out.vs.size();
          out.vs.insert(out.vs.end(), D.vs.begin() + p.seg0, D.vs.begin() + p.seg0 + p.nseg);
          p.seg0 = s0;
          p.tile0 += M.tiles;
          out.vp.push_back(p);
        }
        M.np += L.np;
        M.tiles += L.tiles;
        M.flops += L.flops;
      }
      (dir == 0 ? out.fwd : out.bwd).push_back(M);
    }
  }
}

// ---------------------------------------------------------------------------
// device layout of one matrix
// ---------------------------------------------------------------------------
namespace {
template <typename T>
int alloc_values(snumat *h) {
  Values<T> &VV = vals<T>(h);
  int rc;
  if ((rc = dalloc(h, &VV.arena, (size_t)h->arena_len)) || (rc = dalloc(h, &VV.inv, (size_t)h->inv_total)) ||
      (rc = dalloc(h, &VV.tmp, (size_t)std::max(1LL, h->tmp_panels + h->tmp_inversion))) ||
      (rc = dalloc(h, &VV.lu, (size_t)std::max(1LL, h->lu_off[h->P.np]))))
    return rc;
  // the inverses' other triangles stay zero: factorizations write within the
  // 64 x 64 diagonal blocks and their own triangle alone
  launch_fill(VV.inv, h->inv_total, nullptr);
  HIPCHK(hipStreamSynchronize(nullptr));
  build_dense_plan<T>(h);
  return upload_dense_plan(VV.fact);
}
}  // namespace

// Multifrontal plan of one matrix's leaves (value arrays allocated): the front
// value arena, the fronts' entries of A, extend-add positions and child
// tables, per-height front tables and extend-add tiles, the larger fronts'
// blocked partial LU (per 64-column step: diagonal block LU with the pivot
// clamp, both triangular solves by the block inverses, the trailing update of
// the whole remaining front) and the extend-add tiles of the separator blocks.
template <typename T>
int build_front_plan(snumat *h) {
  using GemmSeg = GemmSegT<T>;
  Values<T> &VV = vals<T>(h);
  const Plan &P = h->P;
  const int np = P.np, fmax = front_small_max<T>();
  const T eps = (T)h->opts.eps;
  FrontPlan<T> &FP = VV.fronts;
  free_dense_plan(FP.dense);
  FP = FrontPlan<T>();
  int rc;
  // front value offsets; per B entry its index in the target: the parent
  // front, or (root fronts) the separator block it belongs to
  std::vector<int> rel;
  std::vector<size_t> o_rel(np);
  std::vector<std::vector<long long>> foff(np);
  h->leaf_foff.assign(np + 1, 0);
  long long ftotal = 0;
  int levels = 0;
  for (int r = 0; r < np; r++) {
    const LeafPlan &L = P.leaves[r];
    const int nf = (int)L.ff.size();
    o_rel[r] = rel.size();
    rel.insert(rel.end(), L.frel.begin(), L.frel.end());
    foff[r].resize(nf);
    for (int f = 0; f < nf; f++) {
      foff[r][f] = ftotal;
      ftotal += (long long)L.ff[f] * L.ff[f] + front_inv_size(L.ff[f], L.fnk[f], fmax);
      if (L.fpar[f] >= 0) continue;
      int k = 1;
      for (int q = L.fidx_ptr[f]; q < L.fidx_ptr[f + 1]; q++) {
        while (L.fidx[q] >= L.cstart[k + 1]) k++;
        rel[o_rel[r] + q] = L.fidx[q] - L.cstart[k];
      }
    }
    h->leaf_foff[r + 1] = ftotal;
    if (nf) levels = std::max(levels, L.fheight_max + 1);
  }
  int *d_rel = nullptr;
  if ((rc = dupload(h, &d_rel, rel)) || (rc = dalloc(h, &VV.farena, (size_t)std::max(1LL, ftotal)))) return rc;
  T *fa = VV.farena;
  // A's entries by front (small fronts: column-major position; larger ones:
  // by tile, position from the tile's first value); the rest go to the
  // separators
  std::vector<std::vector<int>> ent0(np);      // per front: first entry (nf + 1)
  std::vector<std::vector<int>> tile_ent(np);  // per leaf, larger fronts in turn: entries per tile
  std::vector<AEntry> ent;
  {
    auto leaf_of = [&](int q) {  // leaf of A's entry q, -1: a separator entry
      if (P.a_dest[q] >= P.leaf_total) return -1;
      return (int)(std::upper_bound(P.leaf_off.begin(), P.leaf_off.end(), P.a_dest[q]) - P.leaf_off.begin()) - 1;
    };
    std::vector<int> leaf(P.nnz);
    for (int r = 0; r < np; r++) ent0[r].assign(P.leaves[r].ff.size() + 1, 0);
    for (int q = 0; q < P.nnz; q++) {
      const int r = leaf[q] = leaf_of(q);
      if (r >= 0) ent0[r][P.leaves[r].afront[P.perm_map[q] - P.leaves[r].coo_off] + 1]++;
    }
    int total = 0;
    for (int r = 0; r < np; r++)
      for (int &e : ent0[r]) e = total += e;
    ent.resize(total);
    std::vector<std::vector<int>> at = ent0;
    for (int q = 0; q < P.nnz; q++) {
      const int r = leaf[q];
      if (r < 0) continue;
      const LeafPlan &L = P.leaves[r];
      const int k = P.perm_map[q] - L.coo_off;
      ent[at[r][L.afront[k]]++] = AEntry{L.apos[k], q};
    }
    // larger fronts: by tile
    std::vector<std::pair<int, AEntry>> tmp;
    for (int r = 0; r < np; r++) {
      const LeafPlan &L = P.leaves[r];
      for (int f = 0; f < (int)L.ff.size(); f++) {
        const int ff = L.ff[f], nt = (ff + 63) / 64;
        if (ff <= fmax) continue;
        const size_t tbase = tile_ent[r].size();
        tile_ent[r].resize(tbase + (size_t)nt * nt, 0);
        tmp.clear();
        for (int e = ent0[r][f]; e < ent0[r][f + 1]; e++) {
          const int row = ent[e].pos % ff, col = ent[e].pos / ff, t = (col / 64) * nt + row / 64;
          tile_ent[r][tbase + t]++;
          tmp.push_back({t, AEntry{row % 64 + (col % 64) * ff, ent[e].idx}});
        }
        std::sort(tmp.begin(), tmp.end(), [](const std::pair<int, AEntry> &x, const std::pair<int, AEntry> &y) {
          return x.first != y.first ? x.first < y.first : x.second.pos < y.second.pos;
        });
        for (size_t e = 0; e < tmp.size(); e++) ent[ent0[r][f] + e] = tmp[e].second;
      }
    }
  }
  AEntry *d_ent = nullptr;
  if ((rc = dupload(h, &d_ent, ent))) return rc;
  // children (of the fronts factored in LDS)
  std::vector<FrontChild> ch;
  std::vector<std::vector<int>> ch0(np);
  for (int r = 0; r < np; r++) {
    const LeafPlan &L = P.leaves[r];
    const int nf = (int)L.ff.size();
    ch0[r].resize(nf);
    for (int f = 0; f < nf; f++) {
      ch0[r][f] = (int)ch.size();
      if (L.ff[f] > fmax) continue;
      for (int q = L.fchild_ptr[f]; q < L.fchild_ptr[f + 1]; q++) {
        const int c = L.fchild[q], fc = L.ff[c], nkc = L.fnk[c];
        ch.push_back(FrontChild{fa + foff[r][c] + nkc + (long long)nkc * fc,
                                d_rel + o_rel[r] + L.fidx_ptr[c], fc, fc - nkc});
      }
    }
  }
  FrontChild *d_ch = nullptr;
  if ((rc = dupload(h, &d_ch, ch))) return rc;
  // fronts by height
  std::vector<std::vector<FrontDev>> sm(levels);
  struct Large { T *F, *inv; int f, nk, leaf, front, tile_ent; };
  std::vector<std::vector<Large>> lg(levels);
  for (int r = 0; r < np; r++) {
    const LeafPlan &L = P.leaves[r];
    int te = 0;
    for (int f = 0; f < (int)L.ff.size(); f++) {
      const int ff = L.ff[f];
      T *F = fa + foff[r][f], *inv = F + (long long)ff * ff;
      if (ff > fmax) {
        lg[L.fheight[f]].push_back(Large{F, inv, ff, L.fnk[f], r, f, te});
        te += ((ff + 63) / 64) * ((ff + 63) / 64);
        continue;
      }
      FrontDev D;
      D.F = F;
      D.aval = h->d_aval;
      D.ent = d_ent + ent0[r][f];
      D.child = d_ch + ch0[r][f];
      D.f = ff;
      D.nk = L.fnk[f];
      D.nent = ent0[r][f + 1] - ent0[r][f];
      D.nchild = L.fchild_ptr[f + 1] - L.fchild_ptr[f];
      sm[L.fheight[f]].push_back(D);
    }
  }
  FP.levels.assign(levels, FrontLevel());
  DensePlan<T> &DP = FP.dense;
  for (int hh = 0; hh < levels; hh++) {
    FrontLevel &lv = FP.levels[hh];
    lv.small0 = (int)FP.small.size();
    // by class: more workgroups of smaller fronts share a CU's LDS
    std::stable_sort(sm[hh].begin(), sm[hh].end(),
                     [](const FrontDev &x, const FrontDev &y) { return front_class(x.f) < front_class(y.f); });
    for (const FrontDev &D : sm[hh]) {
      const int k = front_class(D.f);
      lv.nsmall[k]++;
      lv.max_f[k] = std::max(lv.max_f[k], D.f);
    }
    FP.small.insert(FP.small.end(), sm[hh].begin(), sm[hh].end());
    // extend-add tiles of the larger fronts, column by column: each child's
    // entries per 64-index chunk of the front, every pair of chunks a source
    lv.tile0 = (int)FP.tiles.size();
    int kmax = 0;
    std::vector<int> bound;  // per child: first entry of each chunk (nt + 1)
    for (const Large &D : lg[hh]) {
      const LeafPlan &L = P.leaves[D.leaf];
      const int f = D.f, nt = (f + 63) / 64, nc = L.fchild_ptr[D.front + 1] - L.fchild_ptr[D.front];
      bound.resize((size_t)nc * (nt + 1));
      for (int k = 0; k < nc; k++) {
        const int c = L.fchild[L.fchild_ptr[D.front] + k];
        const int *rc0 = L.frel.data() + L.fidx_ptr[c], nb = L.fidx_ptr[c + 1] - L.fidx_ptr[c];
        int q = 0;
        for (int t = 0; t <= nt; t++) {
          while (q < nb && rc0[q] < 64 * t) q++;
          bound[(size_t)k * (nt + 1) + t] = q;
        }
      }
      int e = ent0[D.leaf][D.front];
      for (int ct = 0; ct < nt; ct++)
        for (int rt = 0; rt < nt; rt++) {
          AddTile t;
          t.C = D.F + 64 * rt + (long long)64 * ct * f;
          t.aval = h->d_aval;
          t.ent = d_ent + e;
          t.nent = tile_ent[D.leaf][D.tile_ent + ct * nt + rt];
          e += t.nent;
          t.ldc = f;
          t.nr = std::min(64, f - 64 * rt);
          t.nc = std::min(64, f - 64 * ct);
          t.s0 = (int)FP.src.size();
          for (int k = 0; k < nc; k++) {
            const int *bk = bound.data() + (size_t)k * (nt + 1);
            if (bk[rt] == bk[rt + 1] || bk[ct] == bk[ct + 1]) continue;
            const int c = L.fchild[L.fchild_ptr[D.front] + k], fc = L.ff[c], nkc = L.fnk[c];
            FP.src.push_back(AddSrc{fa + foff[D.leaf][c] + nkc + (long long)nkc * fc,
                                    d_rel + o_rel[D.leaf] + L.fidx_ptr[c], fc, bk[rt], bk[rt + 1] - bk[rt], bk[ct],
                                    bk[ct + 1] - bk[ct], 64 * rt, 64 * ct, 0});
          }
          t.s1 = (int)FP.src.size();
          FP.tiles.push_back(t);
        }
      kmax = std::max(kmax, D.nk);
    }
    lv.ntile = (int)FP.tiles.size() - lv.tile0;
    // blocked partial LU of this height's larger fronts, grouped per step
    for (int k = 0; k < kmax; k += 64) {
      const int step = k / 64;
      Launch d{0, (int)DP.dp.size(), 0, 0, 0, front_key(hh, step, 0)};
      GemmBatch<T> tu;
      tu.rule = tile_rule<T>(h);
      for (const Large &D : lg[hh]) {
        if (D.nk <= k) continue;
        const int f = D.f, nb = std::min(64, D.nk - k), m = f - k - nb;
        T *F = D.F;
        T *Li = D.inv + (long long)step * kFrontInv, *Ui = Li + 4096;
        DiagProbT<T> dp{};
        dp.D = F + k + (long long)k * f;
        dp.ld = f;
        dp.nb = nb;
        dp.Linv = Li;
        dp.Uinv = Ui;
        dp.ldi = 64;
        dp.LU = Ui + 4096;
        dp.eps = eps;
        // L21 <- L21 U11^-1 (rows below), U12 <- L11^-1 U12 (columns right)
        dp.m = m;
        dp.tile0 = d.tiles;
        d.tiles += panel_tiles(m);
        d.flops += 4.0 * m * nb * nb;
        DP.dp.push_back(dp);
        d.np++;
        T *X1 = F + (k + nb) + (long long)k * f, *X = F + k + (long long)(k + nb) * f;
        // trailing update of the remaining front, outer-blocked by kPanel
        // pivots as for the separators (the last step of a panel applies
        // its rank-64 updates to F[K1:, K1:] at once)
        const int k2 = k + nb, K0 = k - k % kPanel, K1 = std::min(D.nk, K0 + kPanel);
        auto at = [&](int r, int c) { return F + r + (long long)c * f; };
        if (k2 < K1) {
          tu.add(at(k2, k2), f, f - k2, K1 - k2, {GemmSeg{X1, X, f, f, nb}});
          tu.add(at(k2, K1), f, K1 - k2, f - K1, {GemmSeg{X1, at(k, K1), f, f, nb}});
        } else {
          tu.add(at(K1, K1), f, f - K1, f - K1, {GemmSeg{at(K1, K0), at(K0, K1), f, f, K1 - K0}});
        }
      }
      if (d.np) DP.launches.push_back(d);
      tu.flush(DP.gp, DP.gs, DP.launches, front_key(hh, step, 3));
    }
  }
  if ((rc = upload_dense_plan(DP))) return rc;
  // extend-add tiles of the separator blocks, all that are stored: the root
  // fronts' update blocks, per pair of 64-index tiles of the blocks their B
  // entries belong to (pairs whose panel tile is not stored are structurally
  // zero), and A's entries; every tile is written, so the blocks are not
  // cleared before.  A piece without rows stands for a tile itself.
  FP.sep0 = (int)FP.tiles.size();
  struct Piece { long long key; T *C; long long ldc; int nr, nc; AddSrc s; };
  std::vector<Piece> pieces;
  struct Group { int blk, t, b0, b1; };
  std::vector<Group> gr;
  std::vector<long long> tbase(P.num_block + 2, 0);  // tiles of the blocks before each block
  for (int b = 1; b <= P.num_block; b++) tbase[b + 1] = tbase[b] + (P.block_size[b] + 63) / 64;
  auto key_of = [&](int p, int t, int q, int u) { return (tbase[p] + t) * tbase[P.num_block + 1] + tbase[q] + u; };
  for (int p = 1; p < np; p++) {
    const int sp = P.block_size[p], tp = (sp + 63) / 64;
    auto add = [&](long long key, long long off, long long ldc, int nr, int nc) {
      pieces.push_back(Piece{key, VV.arena + off, ldc, nr, nc, AddSrc{}});
    };
    for (int t = 0; t < tp; t++)
      for (int u = 0; u < tp; u++)
        add(key_of(p, t, p, u), P.offR[p] + 64 * t + (long long)64 * u * sp, sp, std::min(64, sp - 64 * t), std::min(64, sp - 64 * u));
    for (int q = p / 2; q; q /= 2) {
      const int o = P.anc_off(p, q), sq = P.block_size[q];
      for (int u = 0; 64 * u < sq; u++) {
        const int cu = P.umap[p][o + 64 * u], rl = P.lmap[p][o + 64 * u], w = std::min(64, sq - 64 * u);
        for (int t = 0; t < tp; t++) {
          const int ht = std::min(64, sp - 64 * t);
          if (cu >= 0) add(key_of(p, t, q, u), P.offR[p] + 64 * t + (long long)(sp + cu) * sp, sp, ht, w);
          if (rl >= 0) add(key_of(q, u, p, t), P.offL[p] + rl + (long long)64 * t * P.nL[p], P.nL[p], w, ht);
        }
      }
    }
  }
  for (int r = 0; r < np; r++) {
    const LeafPlan &L = P.leaves[r];
    for (int f = 0; f < (int)L.ff.size(); f++) {
      if (L.fpar[f] >= 0) continue;
      const int fc = L.ff[f], nkc = L.fnk[f], i0 = L.fidx_ptr[f], nb = L.fidx_ptr[f + 1] - i0;
      const T *U = fa + foff[r][f] + nkc + (long long)nkc * fc;
      gr.clear();
      int k = 1;
      for (int q = 0; q < nb; q++) {
        while (L.fidx[i0 + q] >= L.cstart[k + 1]) k++;
        const int t = (L.fidx[i0 + q] - L.cstart[k]) / 64;
        if (gr.empty() || gr.back().blk != L.path[k] || gr.back().t != t) gr.push_back(Group{L.path[k], t, q, q});
        gr.back().b1 = q + 1;
      }
      for (const Group &a : gr)
        for (const Group &c : gr) {
          const int p = a.blk, q = c.blk, sp = P.block_size[p], sq = P.block_size[q];
          T *C;
          long long ldc;
          if (p == q) {
            C = VV.arena + P.offR[p] + 64 * a.t + (long long)64 * c.t * sp;
            ldc = sp;
          } else if (p > q) {  // row block deeper: its U panel
            const int u = P.umap[p][P.anc_off(p, q) + 64 * c.t];
            if (u < 0) continue;
            C = VV.arena + P.offR[p] + 64 * a.t + (long long)(sp + u) * sp;
            ldc = sp;
          } else {
            const int l = P.lmap[q][P.anc_off(q, p) + 64 * a.t];
            if (l < 0) continue;
            C = VV.arena + P.offL[q] + l + (long long)64 * c.t * P.nL[q];
            ldc = P.nL[q];
          }
          pieces.push_back(Piece{key_of(p, a.t, q, c.t), C, ldc,
                                 std::min(64, sp - 64 * a.t), std::min(64, sq - 64 * c.t),
                                 AddSrc{U, d_rel + o_rel[r] + i0, fc, a.b0, a.b1 - a.b0, c.b0, c.b1 - c.b0,
                                        64 * a.t, 64 * c.t, 0}});
        }
    }
  }
  std::vector<int> po(pieces.size());
  for (size_t q = 0; q < po.size(); q++) po[q] = (int)q;
  std::sort(po.begin(), po.end(), [&](int a, int b) {
    return pieces[a].key != pieces[b].key ? pieces[a].key < pieces[b].key : a < b;  // leaves in ascending order
  });
  for (size_t q = 0; q < po.size(); q++) {
    const Piece &x = pieces[po[q]];
    if (q == 0 || x.key != pieces[po[q - 1]].key) {
      AddTile t;
      t.C = x.C;
      t.aval = nullptr;
      t.ent = nullptr;
      t.ldc = x.ldc;
      t.nr = x.nr;
      t.nc = x.nc;
      t.s0 = t.s1 = (int)FP.src.size();
      t.nent = 0;
      FP.tiles.push_back(t);
    }
    if (x.s.rn == 0) continue;
    FP.src.push_back(x.s);
    FP.tiles.back().s1 = (int)FP.src.size();
  }
  // A's separator entries by tile
  std::vector<std::pair<int, AEntry>> sent_of;  // tile from sep0 on, entry
  {
    std::unordered_map<long long, int> tile_at;  // by its first value's place in the arena
    for (size_t q = FP.sep0; q < FP.tiles.size(); q++) tile_at[(T *)FP.tiles[q].C - VV.arena] = (int)q - FP.sep0;
    // first stored column (row) of every tile of each separator's panels
    std::vector<std::vector<int>> cu(np), rl(np);
    for (int p = 1; p < np; p++)
      for (int q = p / 2; q; q /= 2)
        for (int u = 0, o = P.anc_off(p, q); u < P.block_size[q]; u += 64) {
          if (P.umap[p][o + u] >= 0) cu[p].push_back(P.umap[p][o + u]);
          if (P.lmap[p][o + u] >= 0) rl[p].push_back(P.lmap[p][o + u]);
        }
    auto start = [](const std::vector<int> &v, int x) { return *(std::upper_bound(v.begin(), v.end(), x) - 1); };
    for (int q = 0; q < P.nnz; q++) {
      if (P.a_dest[q] < P.leaf_total) continue;
      const long long x = P.a_dest[q] - P.leaf_total;
      const int p = (int)(std::upper_bound(P.offR.begin() + 1, P.offR.begin() + np, x) - P.offR.begin()) - 1;
      const bool R = x < P.offL[p];
      const long long ld = R ? P.block_size[p] : P.nL[p], y = x - (R ? P.offR[p] : P.offL[p]), sp = P.block_size[p];
      const int row = (int)(y % ld), col = (int)(y / ld);
      const int r0 = R ? row / 64 * 64 : start(rl[p], row);
      const int c0 = !R || col < sp ? col / 64 * 64 : (int)sp + start(cu[p], col - (int)sp);
      sent_of.push_back({tile_at.at((R ? P.offR[p] : P.offL[p]) + r0 + c0 * ld),
                         AEntry{(int)(row - r0 + (col - c0) * ld), q}});
    }
    std::sort(sent_of.begin(), sent_of.end(), [](const std::pair<int, AEntry> &x, const std::pair<int, AEntry> &y) {
      return x.first != y.first ? x.first < y.first : x.second.pos < y.second.pos;
    });
  }
  std::vector<AEntry> sent;
  for (const auto &e : sent_of) sent.push_back(e.second);
  AEntry *d_sent = nullptr;
  if ((rc = dupload(h, &d_sent, sent))) return rc;
  for (size_t e = 0; e < sent_of.size(); e++) {
    AddTile &t = FP.tiles[FP.sep0 + sent_of[e].first];
    if (t.nent++ == 0) t.ent = d_sent + e, t.aval = h->d_aval;
  }
  if ((rc = dupload(h, &FP.d_small, FP.small)) ||
      (rc = dupload(h, &FP.d_tiles, FP.tiles)) || (rc = dupload(h, &FP.d_src, FP.src)))
    return rc;
  return SNU_OK;
}

template <typename T>
void merge_fronts(const std::vector<const FrontPlan<T> *> &in, FrontPlan<T> &out) {
  out.small.clear();
  out.tiles.clear();
  out.src.clear();
  std::vector<int> sbase;
  size_t levels = 0;
  for (const FrontPlan<T> *p : in) {
    sbase.push_back((int)out.src.size());
    out.src.insert(out.src.end(), p->src.begin(), p->src.end());
    levels = std::max(levels, p->levels.size());
  }
  auto add_tiles = [&](size_t pi, int first, int count) {
    for (int q = first; q < first + count; q++) {
      AddTile t = in[pi]->tiles[q];
      t.s0 += sbase[pi];
      t.s1 += sbase[pi];
      out.tiles.push_back(t);
    }
  };
  out.levels.assign(levels, FrontLevel());
  for (size_t hh = 0; hh < levels; hh++) {
    FrontLevel &lv = out.levels[hh];
    lv.small0 = (int)out.small.size();
    lv.tile0 = (int)out.tiles.size();
    for (int k = 0; k < 3; k++)  // every matrix's fronts of a class side by side
      for (const FrontPlan<T> *p : in) {
        if (hh >= p->levels.size()) continue;
        const FrontLevel &pl = p->levels[hh];
        int first = pl.small0;
        for (int j = 0; j < k; j++) first += pl.nsmall[j];
        out.small.insert(out.small.end(), p->small.begin() + first, p->small.begin() + first + pl.nsmall[k]);
        lv.nsmall[k] += pl.nsmall[k];
        lv.max_f[k] = std::max(lv.max_f[k], pl.max_f[k]);
      }
    for (size_t pi = 0; pi < in.size(); pi++)
      if (hh < in[pi]->levels.size()) add_tiles(pi, in[pi]->levels[hh].tile0, in[pi]->levels[hh].ntile);
    lv.ntile = (int)out.tiles.size() - lv.tile0;
  }
  out.sep0 = (int)out.tiles.size();
  for (size_t pi = 0; pi < in.size(); pi++) add_tiles(pi, in[pi]->sep0, (int)in[pi]->tiles.size() - in[pi]->sep0);
  std::vector<const DensePlan<T> *> dp;
  for (const FrontPlan<T> *p : in) dp.push_back(&p->dense);
  merge_dense(dp, out.dense);
}
// Places of the fronts' update rows of one leaf (size: rows per front) and the
// rows taken in all.  Rows live from their front's height to its parent's, where
// they are read (root fronts: to the end); the backward sweep uses a front's
// rows within its height.  Rows that are done with are given to fronts of later
// heights, first fit: 35 to 45% fewer rows than side by side on 2D and 3D grids.
static long long place_rows(const LeafPlan &L, const std::vector<long long> &size, std::vector<long long> &at) {
  const int nf = (int)L.ff.size();
  std::vector<std::vector<int>> begin(nf ? L.fheight_max + 1 : 0), done(begin.size());
  for (int f = 0; f < nf; f++) {
    begin[L.fheight[f]].push_back(f);
    if (L.fpar[f] >= 0) done[L.fheight[L.fpar[f]]].push_back(f);
  }
  at.assign(nf, 0);
  std::map<long long, long long> open;  // free rows below top: first, count (no two adjacent)
  long long top = 0;
  for (size_t h = 0; h < begin.size(); h++) {
    for (int f : begin[h]) {
      if (!size[f]) continue;
      auto it = open.begin();
      while (it != open.end() && it->second < size[f]) ++it;
      if (it == open.end()) {
        at[f] = top;
        top += size[f];
        continue;
      }
      at[f] = it->first;
      const long long left = it->second - size[f];
      open.erase(it);
      if (left) open[at[f] + size[f]] = left;
    }
    for (int f : done[h]) {
      if (!size[f]) continue;
      auto it = open.emplace(at[f], size[f]).first;
      auto next = std::next(it);
      if (next != open.end() && it->first + it->second == next->first) it->second += next->second, open.erase(next);
      if (it != open.begin()) {
        auto prev = std::prev(it);
        if (prev->first + prev->second == it->first) prev->second += it->second, open.erase(it);
      }
    }
  }
  return top;
}
// The leaf solves of one matrix: solve positions (leaf rows in front order, so
// a front's pivots are consecutive), update rows, the children's
// update rows each front row adds, the units of every phase (per height,
// forward upwards: whole fronts and first pivot blocks, further pivot blocks
// one phase each, boundary row tiles; backward downwards: boundary column
// chunks and whole fronts, then the pivot blocks last to first) and the
// separator rows' sources.
template <typename T>
static int build_leaf_solve(snumat *h) {
  Values<T> &VV = vals<T>(h);
  const Plan &P = h->P;
  const int np = P.np, fmax = front_small_max<T>();
  std::vector<int> pos(P.n), pull, plist, bidx, phase;
  std::vector<std::pair<int, int>> more;
  for (int i = 0; i < P.n; i++) pos[i] = i;
  std::vector<SolveUnit> units;
  struct Src { int R, row; };
  std::vector<Src> src;
  std::vector<std::array<size_t, 2>> o_phase(np);
  long long ftotal = 0, wrows = 0;
  for (int r = 0; r < np; r++) {
    const LeafPlan &L = P.leaves[r];
    LeafDev &D = h->h_leaves[r];
    const int nf = (int)L.ff.size(), g0 = P.block_start[L.leaf], ls = L.leaf_size;
    for (int q = 0; q < ls; q++) pos[g0 + L.fk[q]] = g0 + q;
    // global solve position of a core index
    auto gpos = [&](int x) {
      if (x < ls) return pos[g0 + x];
      int k = 1;
      while (x >= L.cstart[k + 1]) k++;
      return P.block_start[L.path[k]] + x - L.cstart[k];
    };
    std::vector<SolveUnit> base(nf);
    std::vector<std::vector<int>> byh(nf ? L.fheight_max + 1 : 0);
    // update rows, which the backward sweep's partial products share
    std::vector<long long> size(nf), at;
    auto chunks = [&](int f) {
      const int w = 64 * ((L.fnk[f] + 63) / 64);
      return L.ff[f] > fmax ? (L.ff[f] - L.fnk[f] + w - 1) / w : 0;
    };
    for (int f = 0; f < nf; f++)
      size[f] = std::max<long long>(L.ff[f] - L.fnk[f], 64LL * ((L.fnk[f] + 63) / 64) * chunks(f));
    const long long row0 = wrows;
    wrows += place_rows(L, size, at);
    for (int f = 0; f < nf; f++) {
      SolveUnit &U = base[f];
      std::memset(&U, 0, sizeof(U));
      U.ld = L.ff[f];
      U.nk = L.fnk[f];
      U.nb = U.ld - U.nk;
      U.F = VV.farena + ftotal;
      U.inv = VV.farena + ftotal + (long long)U.ld * U.ld;
      ftotal += (long long)U.ld * U.ld + front_inv_size(U.ld, U.nk, fmax);
      U.kpos = g0 + L.fkp[f];
      U.wrow = (int)(row0 + at[f]);
      U.nq = chunks(f);
      U.bidx = (int)bidx.size();
      for (int q = L.fidx_ptr[f]; q < L.fidx_ptr[f + 1]; q++) bidx.push_back(gpos(L.fidx[q]));
      U.pull = (int)(pull.size() / 2);
      pull.resize(pull.size() + 2 * (size_t)U.ld, -1);
      int *pf = pull.data() + 2 * (size_t)U.pull;
      more.clear();
      for (int k = L.fchild_ptr[f]; k < L.fchild_ptr[f + 1]; k++) {
        const int c = L.fchild[k];
        for (int q = L.fidx_ptr[c]; q < L.fidx_ptr[c + 1]; q++) {
          const int row = base[c].wrow + q - L.fidx_ptr[c], i = L.frel[q];
          if (pf[2 * i] < 0) pf[2 * i] = row;
          else if (pf[2 * i + 1] == -1) pf[2 * i + 1] = row;
          else more.push_back({i, row});
        }
      }
      // rows with three or more sources: a list from the second on
      std::stable_sort(more.begin(), more.end(),
                       [](const std::pair<int, int> &a, const std::pair<int, int> &b) { return a.first < b.first; });
      for (size_t q = 0; q < more.size();) {
        const int i = more[q].first;
        const size_t at = plist.size();
        plist.push_back(0);
        plist.push_back(pf[2 * i + 1]);
        for (; q < more.size() && more[q].first == i; q++) plist.push_back(more[q].second);
        plist[at] = (int)(plist.size() - at - 1);
        pf[2 * i + 1] = -2 - (int)at;
      }
      if (L.fpar[f] < 0)
        for (int q = L.fidx_ptr[f]; q < L.fidx_ptr[f + 1]; q++)
          if (L.fsrow[q] >= 0) src.push_back({gpos(L.fidx[q]), U.wrow + q - L.fidx_ptr[f]});
      byh[L.fheight[f]].push_back(f);
    }
    if (wrows > 2000000000LL || bidx.size() > 2000000000u || pull.size() > 2000000000u ||
        plist.size() > 2000000000u)
      return set_error(SNU_ERR_BAD_INPUT, "leaf fronts too large for 32-bit solve indices");
    auto emit = [&](int f, int kind, int row0, int sblk, int q) {
      SolveUnit U = base[f];
      U.kind = kind;
      U.row0 = row0;
      U.s = sblk;
      U.q = q;
      units.push_back(U);
    };
    auto close = [&] {  // ends a phase unless it is empty
      if ((size_t)phase.back() != units.size()) phase.push_back((int)units.size());
    };
    auto large = [&](int f) { return base[f].ld > fmax; };
    auto blocks = [&](int f) { return (base[f].nk + 63) / 64; };
    o_phase[r][0] = phase.size();
    phase.push_back((int)units.size());
    for (auto &fr : byh) {
      int smax = 0;
      for (int f : fr)
        if (large(f)) emit(f, kFwdPivots, 0, 0, 0), smax = std::max(smax, blocks(f));
      for (int f : fr)
        if (!large(f)) emit(f, kFwdFront, 0, 0, 0);
      close();
      for (int k = 1; k < smax; k++) {
        for (int f : fr)
          if (large(f) && blocks(f) > k) emit(f, kFwdPivots, 0, k, 0);
        close();
      }
      for (int f : fr)
        if (large(f))
          for (int t = 0; t < base[f].nb; t += 64) emit(f, kFwdRows, t, 0, 0);
      close();
    }
    D.nfphase = (int)(phase.size() - o_phase[r][0]) - 1;
    o_phase[r][1] = phase.size();
    phase.push_back((int)units.size());
    for (size_t hh = byh.size(); hh-- > 0;) {
      const std::vector<int> &fr = byh[hh];
      int smax = 0;
      for (int f : fr)
        if (large(f)) {
          smax = std::max(smax, blocks(f));
          for (int k = 0; k < blocks(f); k++)
            for (int q = 0; q < base[f].nq; q++) emit(f, kBwdCols, 0, k, q);
        }
      for (int f : fr)
        if (!large(f)) emit(f, kBwdFront, 0, 0, 0);
      close();
      for (int k = smax - 1; k >= 0; k--) {
        for (int f : fr)
          if (large(f) && blocks(f) > k) emit(f, kBwdPivots, 0, k, 0);
        close();
      }
    }
    D.nbphase = (int)(phase.size() - o_phase[r][1]) - 1;
  }
  h->wrows = (int)std::max(1LL, wrows);
  // separator rows and their sources, ascending row, then leaf and front
  std::stable_sort(src.begin(), src.end(), [](const Src &a, const Src &b) { return a.R < b.R; });
  WorkLists &W = h->wl;
  W.targets.clear();
  W.tsrc.clear();
  for (size_t q = 0; q < src.size(); q++) {
    if (q == 0 || src[q].R != src[q - 1].R) W.targets.push_back(TargetDev{src[q].R, (int)q, (int)q, 0});
    W.targets.back().s1 = (int)q + 1;
    W.tsrc.push_back(src[q].row);
  }
  // solve order of the caller's rows
  std::vector<int> order(P.n);
  for (int i = 0; i < P.n; i++) order[i] = pos[P.order[i]];
  int rc;
  SolveUnit *d_units = nullptr;
  int *d_phase = nullptr, *d_pull = nullptr, *d_plist = nullptr, *d_bidx = nullptr;
  if ((rc = dupload(h, &d_units, units)) || (rc = dupload(h, &d_phase, phase)) ||
      (rc = dupload(h, &d_pull, pull)) || (rc = dupload(h, &d_plist, plist)) ||
      (rc = dupload(h, &d_bidx, bidx)) || (rc = dupload(h, &h->d_order, order)) ||
      (rc = dupload(h, &h->wd.targets, W.targets)) || (rc = dupload(h, &h->wd.tsrc, W.tsrc)) ||
      (rc = dalloc(h, &VV.w1, (size_t)h->wrows)))
    return rc;
  h->wd.ntarget = (int)W.targets.size();
  for (int r = 0; r < np; r++) {
    LeafDev &D = h->h_leaves[r];
    D.units = d_units;
    D.fphase = d_phase + o_phase[r][0];
    D.bphase = d_phase + o_phase[r][1];
    D.pull = d_pull;
    D.pulllist = d_plist;
    D.bidx = d_bidx;
  }
  return SNU_OK;
}

template void merge_fronts<double>(const std::vector<const FrontPlan<double> *> &, FrontPlan<double> &);
template void merge_fronts<float>(const std::vector<const FrontPlan<float> *> &, FrontPlan<float> &);
template int build_front_plan<double>(snumat *);
template int build_front_plan<float>(snumat *);

// Offsets of the separators' blocks, inverses and scratch (structure only).
static void layout_dense(snumat *h) {
  const Plan &P = h->P;
  const int np = P.np;
  h->inv_off.assign(P.num_block + 1, 0);
  h->lu_off.assign(np + 1, 0);
  h->sep_rows.assign(np + 1, 0);
  for (int p = 1; p < np; p++) h->sep_rows[p + 1] = h->sep_rows[p] + P.block_size[p];
  for (int p = 1; p < np; p++) h->lu_off[p + 1] = h->lu_off[p] + (P.block_size[p] + 63) / 64 * 4096LL;
  long long inv_total = 0;
  for (int p = 1; p < np; p++) {
    h->inv_off[p] = inv_total;
    inv_total += 2LL * P.block_size[p] * P.block_size[p];
  }
  h->inv_total = inv_total;
  const TmpSize tmp = tmp_size(P);
  h->tmp_panels = tmp.panels;
  h->tmp_inversion = tmp.inversion;
  h->arena_len = P.dense_total;
}

int upload(snumat *h) {
  Plan &P = h->P;
  int rc;
  HIPCHK(hipSetDevice(h->device));
  if (h->prec == SNU_FP32) autotune_tiles<float>();
  else autotune_tiles<double>();
  const int np = P.np;
  h->h_leaves.assign(np, LeafDev());
  h->wl = WorkLists();
  layout_dense(h);
  // ---- structure uploads ----
  std::vector<long long> adest;
  std::vector<int> asrc;
  for (int q = 0; q < P.nnz; q++)
    if (P.a_dest[q] >= P.leaf_total) adest.push_back(P.a_dest[q] - P.leaf_total), asrc.push_back(q);
  h->nsep_ent = (long long)asrc.size();
  if ((rc = dalloc(h, &h->d_aval, (size_t)P.nnz)) || (rc = dupload(h, &h->d_adest, adest)) ||
      (rc = dupload(h, &h->d_asrc, asrc)))
    return rc;
  WorkDev &wd = h->wd;
  wd.nleaves = np;
  if ((rc = dalloc(h, &h->d_tab, 1)) ||
      (rc = dalloc(h, &h->d_prep, 1)) ||
      (rc = dalloc(h, &h->d_active, 1)) || (rc = dalloc(h, &h->d_norms, 1)))
    return rc;
  if (h->prec == SNU_FP32) {
    if ((rc = dupload(h, &h->d_arow, P.a_rowptr)) || (rc = dupload(h, &h->d_acol, P.a_colidx)))
      return rc;
    rc = alloc_values<float>(h);
    if (!rc) rc = build_front_plan<float>(h);
    if (!rc) rc = build_leaf_solve<float>(h);
  } else {
    rc = alloc_values<double>(h);
    if (!rc) rc = build_front_plan<double>(h);
    if (!rc) rc = build_leaf_solve<double>(h);
  }
  if (rc) return rc;
  if ((rc = dupload(h, &wd.leaves, h->h_leaves))) return rc;
  PrepDev pd;
  pd.arena = h->prec == SNU_FP32 ? (void *)h->v32.arena : (void *)h->v64.arena;
  pd.arena_len = h->arena_len;
  pd.aval = h->d_aval;
  pd.adest = h->d_adest;
  pd.asrc = h->d_asrc;
  pd.nnz = h->nsep_ent;
  HIPCHK(hipMemcpy(h->d_prep, &pd, sizeof(pd), hipMemcpyHostToDevice));
  return SNU_OK;
}

// Device bytes that upload() and a one-column solve take for this plan (the
// launch descriptor lists excluded).
size_t estimate_device_bytes(const snumat *h) {
  const Plan &P = h->P;
  const double vs = h->prec == SNU_FP32 ? 4.0 : 8.0;
  double idx = 0, inv = 0, fronts = 0;
  const int fmax = h->prec == SNU_FP32 ? front_small_max<float>() : front_small_max<double>();
  for (const LeafPlan &L : P.leaves) {
    // fronts: values with larger ones' pivot blocks; solve units,
    // children's update rows, positions of the B entries; extend-add tiles
    // and their sources
    fronts += (double)L.fentries;
    for (size_t f = 0; f < L.ff.size(); f++) {
      fronts += (double)front_inv_size(L.ff[f], L.fnk[f], fmax);
      const double nt = (L.ff[f] + 63) / 64;
      idx += L.ff[f] > fmax ? 14.0 * nt * nt + 12.0 * nt * nt : 18.0;
    }
    idx += 34.0 * L.ff.size() + 5.0 * L.fidx.size() + 3.0 * L.leaf_size;
  }
  for (int p = 1; p < P.np; p++)
    inv += 2.0 * P.block_size[p] * P.block_size[p] + (P.block_size[p] + 63) / 64 * 4096.0;
  const TmpSize tmp = tmp_size(P);
  double bytes = vs * ((double)P.dense_total + fronts + inv + (double)(tmp.panels + tmp.inversion));
  bytes += 24.0 * P.nnz + 4.0 * (idx + P.n) + 48.0 * P.num_block + 56.0 / 2048 * (double)P.dense_total;
  if (h->prec == SNU_FP32) bytes += 4.0 * (P.n + 1 + P.nnz);
  bytes += 2 * vs * P.n + 16.0 * P.n;
  return (size_t)bytes;
}

void free_graph(FactorGraph &g) {
  if (g.exec) (void)hipGraphExecDestroy(g.exec);
  g.exec = nullptr;
}

void free_side(SideStream &s) {
  if (s.fork) (void)hipEventDestroy(s.fork);
  if (s.join) (void)hipEventDestroy(s.join);
  if (s.st) (void)hipStreamDestroy(s.st);
  s = SideStream();
}
void free_device(snumat *h) {
  free_graph(h->graph);
  free_side(h->side);
  free_gemv_plan(h->v64.sp);
  free_gemv_plan(h->v32.sp);
  free_dense_plan(h->v64.fact);
  free_dense_plan(h->v32.fact);
  free_dense_plan(h->v64.fronts.dense);
  free_dense_plan(h->v32.fronts.dense);
  for (void *p : h->allocs) (void)hipFree(p);
  h->allocs.clear();
  for (hipEvent_t e : h->ev) (void)hipEventDestroy(e);
  h->ev.clear();
  for (hipEvent_t e : h->pev) (void)hipEventDestroy(e);
  h->pev.clear();
  if (h->stream) (void)hipStreamDestroy(h->stream);
  h->stream = nullptr;
}

// ---------------------------------------------------------------------------
// executors
// ---------------------------------------------------------------------------
namespace {
// SNU_GEMM_SPLIT factorizations run their 64 x 64 GEMM tiles as bf16 splits
// too
constexpr bool kSplit64 = true;
template <typename T>
void run_launch(const Launch &L, const GemmProbT<T> *gp, const GemmSegT<T> *gs,
                const DiagProbT<T> *dp, const GemvProbT<T> *vp, const GemvSegT<T> *vs,
                T *part, int *done, hipStream_t st, bool split = false) {
  if constexpr (std::is_same<T, float>::value) {
    if (split && (L.kind == 5 || L.kind == 10 || L.kind == 11)) {
      launch_gemm128_split(gp + L.p0, L.np, gs, L.tiles, L.kind == 5 ? 0 : L.kind == 10 ? 1 : 2, st);
      return;
    }
    if (split && kSplit64 && (L.kind == 1 || L.kind == 2 || L.kind == 6)) {
      launch_gemm_split(gp + L.p0, L.np, gs, L.tiles, L.kind == 2 ? 0 : L.kind == 1 ? 1 : 2, st);
      return;
    }
  }
  switch (L.kind) {
    case 0: launch_diag_lu(dp + L.p0, L.np, L.tiles, st); break;
    case 1: launch_gemm(gp + L.p0, L.np, gs, L.tiles, 1, st); break;
    case 2: launch_gemm(gp + L.p0, L.np, gs, L.tiles, 0, st); break;
    case 3: launch_copy2d(gp + L.p0, L.np, gs, L.tiles, st); break;
    case 5: launch_gemm128(gp + L.p0, L.np, gs, L.tiles, 0, st); break;
    case 10: launch_gemm128(gp + L.p0, L.np, gs, L.tiles, 1, st); break;
    case 11: launch_gemm128(gp + L.p0, L.np, gs, L.tiles, 2, st); break;
    case 6: launch_gemm(gp + L.p0, L.np, gs, L.tiles, 2, st); break;
    case 7:
    case 8:
      if (L.wgs > 0) launch_gemv_split(vp + L.p0, L.np, vs, L.wgs, L.kind == 7 ? 1 : 0, part, done, st);
      else launch_gemv(vp + L.p0, L.np, vs, L.tiles, L.kind == 7 ? 1 : 0, st);
      break;
    case 17:
    case 18:
      launch_gemv16(vp + L.p0, L.np, vs, L.tiles, L.wgs, L.gstep, L.groups, L.kind == 17 ? 1 : 0,
                    L.part ? part : nullptr, st);
      break;
  }
}
}  // namespace

// Whether the launches from i on, the Schur updates of a height that its
// parents' diagonal blocks do not need, are work enough to run those beside.  A
// chain of diagonal blocks leaves most CUs idle (a step: 22 us, at most 256
// workgroups), so its time goes where the updates take longer: 64^3 FP64 26.2
// -> 24.9 ms, 56^3 27-point FP32 15.2 -> 13.8, 45x37x29 4.37 -> 4.29.  Below
// about 20 us of updates a fork and its join cost what they give (a batch of 96
// 2D matrices: 3.55 ms from 1 GFLOP on, 3.60 from 0.2).
constexpr double kBesideFlops = 1e9;
inline bool beside(double flops) { return flops >= kBesideFlops; }
template <typename T>
bool beside(const DensePlan<T> &plan, size_t i) {
  const long long key = plan.launches[i].key;
  if (key % kHeight != kNextD + 1) return false;
  double flops = 0;
  for (; i < plan.launches.size() && plan.launches[i].key == key; i++) flops += plan.launches[i].flops;
  return beside(flops);
}
// The same for the height of launch i, one of its earlier launches.
template <typename T>
bool beside_later(const DensePlan<T> &plan, size_t i) {
  const long long height = plan.launches[i].key / kHeight;
  for (; i < plan.launches.size() && plan.launches[i].key / kHeight == height; i++)
    if (plan.launches[i].key % kHeight == kNextD + 1) return beside(plan, i);
  return false;
}
// The second stream's part in a factorization, launch by launch.  It takes the
// copy of a height's panels to where the solves read them, beside the height's
// Schur updates, and the diagonal blocks of the height above and their
// inverses, from the updates of those blocks (step kNextD) on, beside the
// height's other Schur updates.  Everything above those blocks waits for both
// streams: that height's panels, and, where it has none (separators that are
// empty or coupled to nothing above), the next launch of a greater height,
// whose blocks the updates running beside may write.
template <typename T>
std::vector<int> side_schedule(const DensePlan<T> &plan) {
  std::vector<int> out(plan.launches.size(), 0);
  long long fork = -1;  // height of the last fork not joined yet
  for (size_t i = 0; i < plan.launches.size(); i++) {
    const Launch &L = plan.launches[i];
    const long long height = L.key / kHeight, step = L.key % kHeight;
    const bool next = fork >= 0 && height == fork + 1 && step < kPanels;
    if (fork >= 0 && height > fork && !next) {
      out[i] |= kSideJoin;
      fork = -1;
    }
    if (next) out[i] |= kSideRun;
    else if (L.kind == 3 && beside_later(plan, i)) out[i] |= kSideFork | kSideRun;
    else if (fork < 0 && beside(plan, i)) {
      out[i] |= kSideFork;
      fork = height;
    }
  }
  return out;
}
template std::vector<int> side_schedule<double>(const DensePlan<double> &);
template std::vector<int> side_schedule<float>(const DensePlan<float> &);
template <typename T>
const DensePlan<T> &plan_of(snumat *h) {
  if (!h->on_device) {  // (pointers from null: the launches alone are meant)
    layout_dense(h);
    build_dense_plan<T>(h);
  }
  return vals<T>(h).fact;
}
template const DensePlan<double> &plan_of<double>(snumat *);
template const DensePlan<float> &plan_of<float>(snumat *);
template <typename T>
int make_side(const std::vector<const DensePlan<T> *> &in, SideStream &s) {
  std::map<long long, double> flops;
  for (const DensePlan<T> *p : in)
    for (const Launch &L : p->launches)
      if (L.key % kHeight == kNextD + 1) flops[L.key] += L.flops;
  if (std::none_of(flops.begin(), flops.end(), [](const auto &f) { return beside(f.second); })) return SNU_OK;
  hipError_t e = hipStreamCreateWithFlags(&s.st, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&s.fork, hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&s.join, hipEventDisableTiming);
  if (e == hipSuccess) return SNU_OK;
  free_side(s);
  return set_error(SNU_ERR_HIP, std::string("second stream: ") + hipGetErrorString(e));
}
// ev (optional): 6 events marking prepare / leaf fronts / leaf Schur /
// assembly / dense; pev (optional, with profile): a begin/end pair per GEMM
// launch (the leaf fronts' launches, then the dense ones), their times summed
// into gemm_ms[0] (dense C -= AB), gemm_ms[1] (dense C = +-AB), gemm_ms[2]
// (the dense C -= AB launches on 128 x 128 tiles, part of gemm_ms[0]) and
// gemm_ms[3] / gemm_ms[4] (the fronts' C -= AB launches on 64 x 64 / 128 x
// 128 tiles).
// The launches of one factorization on st (no host synchronisation).
template <typename T>
int enqueue_factor(const FactorSet &fs, const DensePlan<T> &plan, hipStream_t st,
                   const std::vector<hipEvent_t> *ev, bool profile, std::vector<hipEvent_t> *pev) {
  if (ev) HIPCHK(hipEventRecord((*ev)[0], st));
  if (fs.scatter_only) launch_prepare<T>(fs.prep, fs.nmat, fs.max_len, fs.max_nnz, st);
  if (fs.ir) launch_rowabs_max(fs.ir, fs.nmat, fs.max_n, fs.anorm_out, st);
  if (ev) HIPCHK(hipEventRecord((*ev)[1], st));
  if (fs.scatter_only) {
    if (ev)
      for (int q = 2; q <= 5; q++) HIPCHK(hipEventRecord((*ev)[q], st));
    HIPCHK(hipGetLastError());
    return SNU_OK;
  }
  // leaf fronts, height by height: whole fronts in LDS; larger fronts
  // assembled and factored by the dense launches of their height
  const FrontPlan<T> &fp = *(const FrontPlan<T> *)fs.fronts;
  int ngemm = 0;
  for (const Launch &L : fp.dense.launches) ngemm += is_gemm(L.kind);
  for (const Launch &L : plan.launches) ngemm += is_gemm(L.kind);
  const bool prof = profile && pev;
  if (prof && (int)pev->size() < 2 * ngemm) {
    for (hipEvent_t e : *pev) (void)hipEventDestroy(e);
    pev->assign(2 * ngemm, nullptr);
    for (auto &e : *pev) HIPCHK(hipEventCreate(&e));
  }
  int g = 0;
  auto run_timed = [&](const Launch &L, const DensePlan<T> &dp, hipStream_t on) -> int {
    const bool gm = prof && is_gemm(L.kind);
    if (gm) HIPCHK(hipEventRecord((*pev)[2 * g], st));
    run_launch<T>(L, dp.d_gp, dp.d_gs, dp.d_dp, nullptr, nullptr, nullptr, nullptr, on, fs.split);
    if (gm) HIPCHK(hipEventRecord((*pev)[2 * g++ + 1], st));
    return SNU_OK;
  };
  size_t li = 0;
  const size_t nl = fp.dense.launches.size();
  for (int hh = 0; hh < (int)fp.levels.size(); hh++) {
    const FrontLevel &lv = fp.levels[hh];
    const FrontDev *fr = fp.d_small + lv.small0;
    for (int k = 0; k < 3; fr += lv.nsmall[k++])
      (k == 0 ? launch_front_wave<T> : launch_front_small<T>)(fr, lv.nsmall[k], lv.max_f[k], fs.eps, st);
    launch_extend_add<T>(fp.d_tiles + lv.tile0, lv.ntile, fp.d_src, st);
    for (; li < nl && front_key_height(fp.dense.launches[li].key) == hh; li++) {
      int rc = run_timed(fp.dense.launches[li], fp.dense, st);
      if (rc) return rc;
    }
  }
  HIPCHK(hipGetLastError());
  if (ev) {
    HIPCHK(hipEventRecord((*ev)[2], st));
    HIPCHK(hipEventRecord((*ev)[3], st));
  }
  launch_extend_add<T>(fp.d_tiles + fp.sep0, (int)fp.tiles.size() - fp.sep0, fp.d_src, st);
  HIPCHK(hipGetLastError());
  if (ev) HIPCHK(hipEventRecord((*ev)[4], st));
  // (one stream when profiled: launches are timed one by one)
  SideStream *side = !prof && fs.side && fs.side->st ? fs.side : nullptr;
  const std::vector<int> how = side ? side_schedule(plan) : std::vector<int>(plan.launches.size(), 0);
  auto fork = [&]() -> int {
    HIPCHK(hipEventRecord(side->fork, st));
    HIPCHK(hipStreamWaitEvent(side->st, side->fork, 0));
    return SNU_OK;
  };
  auto join = [&]() -> int {
    HIPCHK(hipEventRecord(side->join, side->st));
    HIPCHK(hipStreamWaitEvent(st, side->join, 0));
    return SNU_OK;
  };
  int rc;
  bool pending = false;
  for (size_t i = 0; i < plan.launches.size(); i++) {
    if ((how[i] & kSideJoin) && (rc = join())) return rc;
    if ((how[i] & kSideFork) && (rc = fork())) return rc;
    pending = (pending && !(how[i] & kSideJoin)) || (how[i] & kSideFork);
    if ((rc = run_timed(plan.launches[i], plan, how[i] & kSideRun ? side->st : st))) return rc;
  }
  if (pending && (rc = join())) return rc;
  HIPCHK(hipGetLastError());
  if (ev) HIPCHK(hipEventRecord((*ev)[5], st));
  return SNU_OK;
}

template <typename T>
int run_factor(const FactorSet &fs, const DensePlan<T> &plan, hipStream_t st,
               const std::vector<hipEvent_t> *ev, bool profile, std::vector<hipEvent_t> *pev,
               double *gemm_ms, FactorGraph *graph) {
  int rc;
  if (graph && !profile) {
    // replay the captured launch sequence (captured on first use)
    if (!graph->exec) {
      hipGraph_t g = nullptr;
      HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
      rc = enqueue_factor<T>(fs, plan, st, nullptr, false, nullptr);
      hipError_t e = hipStreamEndCapture(st, &g);
      if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
      }
      if (e != hipSuccess) return set_error(SNU_ERR_HIP, std::string("graph capture: ") + hipGetErrorString(e));
      e = hipGraphInstantiate(&graph->exec, g, nullptr, nullptr, 0);
      (void)hipGraphDestroy(g);
      if (e != hipSuccess) {
        graph->exec = nullptr;
        return set_error(SNU_ERR_HIP, std::string("graph instantiate: ") + hipGetErrorString(e));
      }
    }
    if (ev) HIPCHK(hipEventRecord((*ev)[0], st));
    HIPCHK(hipGraphLaunch(graph->exec, st));
    if (ev) {
      for (int q = 1; q <= 5; q++) HIPCHK(hipEventRecord((*ev)[q], st));
    }
  } else if ((rc = enqueue_factor<T>(fs, plan, st, ev, profile, pev))) {
    return rc;
  }
  HIPCHK(hipStreamSynchronize(st));
  if (profile && pev && gemm_ms) {
    HIPCHK(hipStreamSynchronize(st));
    for (int q = 0; q < 5; q++) gemm_ms[q] = 0;
    int g = 0;
    const FrontPlan<T> &fp = *(const FrontPlan<T> *)fs.fronts;
    for (const Launch &L : fp.dense.launches) {
      if (!is_gemm(L.kind)) continue;
      const double ms = ev_ms((*pev)[2 * g], (*pev)[2 * g + 1]);
      if (L.kind == 2) gemm_ms[3] += ms;
      if (L.kind == 5) gemm_ms[4] += ms;
      g++;
    }
    for (const Launch &L : plan.launches) {
      if (!is_gemm(L.kind)) continue;
      const double ms = ev_ms((*pev)[2 * g], (*pev)[2 * g + 1]);
      gemm_ms[is_assign_gemm(L.kind) ? 1 : 0] += ms;
      if (L.kind == 5) gemm_ms[2] += ms;
      g++;
    }
  }
  return SNU_OK;
}

template <typename T>
void run_sweep(const SolveSet &ss, T *bp, T *wbuf, const GemvPlan<T> &plan, hipStream_t st) {
  const WorkDev &wd = *ss.wd;
  launch_leaf_sweep(wd.leaves, wd.nleaves, ss.vec, bp, wbuf, ss.max_groups, ss.one, ss.many, false, st);
  launch_assemble_rhs(wd.targets, wd.ntarget, wd.tsrc, ss.vec, wbuf, bp, ss.max_groups, ss.one, ss.many, st);
  for (const Launch &L : plan.fwd)
    run_launch<T>(L, nullptr, nullptr, nullptr, plan.d_vp, plan.d_vs, plan.d_part, plan.d_done, st);
  for (const Launch &L : plan.bwd)
    run_launch<T>(L, nullptr, nullptr, nullptr, plan.d_vp, plan.d_vs, plan.d_part, plan.d_done, st);
  launch_leaf_sweep(wd.leaves, wd.nleaves, ss.vec, bp, wbuf, ss.max_groups, ss.one, ss.many, true, st);
}
template <typename T>
void run_solve(const SolveSet &ss, T *bp, T *wbuf, const GemvPlan<T> &plan, hipStream_t st) {
  launch_permute_in(ss.perm, ss.nmat, ss.vec, bp, ss.max_elems, st);
  run_sweep<T>(ss, bp, wbuf, plan, st);
  launch_permute_out(ss.perm, ss.nmat, ss.vec, bp, ss.max_elems, false, nullptr, st);
}

// FP32 factors, FP64 refinement over a set of matrices: x = sweep(b), then
// x += sweep(b - A x) for the matrices whose backward error is above tol and
// still at least halving per step, at most max_steps corrections each.
int run_refined(const RefineSet &rs, float *bp, float *wbuf, const GemvPlan<float> &plan,
                hipStream_t st, int *steps_out, std::vector<double> *berr_mat) {
  const int nm = rs.nmat, ns = rs.nslots;
  const SolveSet &ss = rs.sweep;
  std::vector<double> u(3 * (size_t)ns);  // |b|, |r|, |x| per column
  const double *bn = u.data(), *rn = bn + ns, *xn = rn + ns;
  launch_permute_in(ss.perm, ss.nmat, ss.vec, bp, ss.max_elems, st);
  run_sweep<float>(ss, bp, wbuf, plan, st);
  launch_permute_out(ss.perm, ss.nmat, ss.vec, bp, ss.max_elems, false, nullptr, st);
  std::vector<double> prev(nm, INFINITY), berr(nm, INFINITY);
  std::vector<int> active(nm, 0), steps(nm, 0);
  int max_steps_taken = 0;
  for (;;) {
    launch_residual(rs.ir, ss.vec, nm, rs.max_n, bp, rs.norms, ns, st);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(u.data(), rs.norms, sizeof(double) * u.size(), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    std::fill(berr.begin(), berr.end(), 0.0);
    for (int i = 0; i < ns; i++) {
      const int m = (*rs.slot_mat)[i];
      const double den = (*rs.anorm)[m] * xn[i] + bn[i];
      double e = den > 0 ? rn[i] / den : (rn[i] > 0 ? INFINITY : 0.0);
      if (!(e == e)) e = INFINITY;
      if (!std::isfinite(bn[i])) e = 0.0;  // no solution to refine: x as the sweep left it
      berr[m] = std::max(berr[m], e);
    }
    int nact = 0;
    for (int m = 0; m < nm; m++) {
      active[m] = berr[m] > rs.tol && steps[m] < rs.max_steps && berr[m] < 0.5 * prev[m];
      nact += active[m];
    }
    if (!nact) break;
    for (int m = 0; m < nm; m++)
      if (active[m]) prev[m] = berr[m], steps[m]++, max_steps_taken = std::max(max_steps_taken, steps[m]);
    if (nact < nm)
      HIPCHK(hipMemcpyAsync(rs.d_active, active.data(), sizeof(int) * nm, hipMemcpyHostToDevice, st));
    run_sweep<float>(ss, bp, wbuf, plan, st);
    launch_permute_out(ss.perm, ss.nmat, ss.vec, bp, ss.max_elems, true, nact < nm ? rs.d_active : nullptr, st);
    HIPCHK(hipGetLastError());
  }
  if (steps_out) *steps_out = max_steps_taken;
  if (berr_mat) *berr_mat = berr;
  double worst = 0;
  for (double e : berr) worst = std::max(worst, e);
  if (!(worst <= 1e-12))
    return set_error(SNU_ERR_NOT_CONVERGED, "FP32 refinement stalled at backward error " +
                                                std::to_string(worst) + " after " +
                                                std::to_string(max_steps_taken) + " steps");
  return SNU_OK;
}

#define SNU_ENGINE_INST(T)                                                                    \
  template void build_solve_plan<T>(const snumat *, T *, T *, int, GemvPlan<T> &);            \
  template int upload_gemv_plan<T>(GemvPlan<T> &, hipStream_t);                               \
  template SplitNeed layout_gemv_plan<T>(GemvPlan<T> &);                                      \
  template void free_gemv_plan<T>(GemvPlan<T> &);                                             \
  template int upload_dense_plan<T>(DensePlan<T> &);                                          \
  template void free_dense_plan<T>(DensePlan<T> &);                                           \
  template void merge_dense<T>(const std::vector<const DensePlan<T> *> &, DensePlan<T> &);    \
  template void merge_gemv<T>(const std::vector<const GemvPlan<T> *> &, GemvPlan<T> &);       \
  template int make_side<T>(const std::vector<const DensePlan<T> *> &, SideStream &);           \
  template int run_factor<T>(const FactorSet &, const DensePlan<T> &, hipStream_t,            \
                             const std::vector<hipEvent_t> *, bool, std::vector<hipEvent_t> *, \
                             double *, FactorGraph *);                                        \
  template void run_solve<T>(const SolveSet &, T *, T *, const GemvPlan<T> &, hipStream_t);
SNU_ENGINE_INST(double)
SNU_ENGINE_INST(float)
#undef SNU_ENGINE_INST

}  // namespace snu
