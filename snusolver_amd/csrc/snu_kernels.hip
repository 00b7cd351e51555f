// HIP kernels for gfx950 (MI355X): blocked no-pivot dense LU on MFMA, FP64
// refinement and the factor set-up.
//
// Wave size 64 throughout.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "snu_device.h"
#include "snu_kernels.h"

#include <utility>

namespace snu {

// ---------------------------------------------------------------------------
// elementwise
// ---------------------------------------------------------------------------
template <typename T>
__global__ void k_fill(T *p, long long n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  long long stride = (long long)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = T(0);
}
template <typename T>
void launch_fill(T *p, long long n, hipStream_t st) {
  if (n <= 0) return;
  long long blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(k_fill<T>, dim3((unsigned)blocks), dim3(256), 0, st, p, n);
}


// ---------------------------------------------------------------------------
// dense: grouped GEMM on MFMA (FP64 v_mfma_f64_16x16x4f64, FP32
// v_mfma_f32_16x16x4f32)
// ---------------------------------------------------------------------------
// Operands are swapped (first operand <- B tile, second <- A tile): the
// product is D = B^T A^T, so the 16 lanes of a row group hold 16 consecutive
// rows of one column of C (coalesced epilogue).  Lane layouts (checked by
// lane-layout probes and the GEMM parity tests): A[i][k] in lane i + 16k,
// B[k][j] in lane j + 16k; FP64 D[i][j] in lane j + 16 (i mod 4), register
// i / 4; FP32 D[i][j] in lane j + 16 (i / 4), register i mod 4.
//
// Workgroup tile (32 BMB) x (32 BNB), 4 waves in 2 x 2, each (16 BMB) x
// (16 BNB); K chunk 16; double-buffered LDS fed from a register prefetch that
// stays in flight across the MFMA block (one barrier per chunk).
// MODE 0: C -= sum_seg A_seg B_seg (K concatenated over the segments).
// MODE 1 / 2: C = A B / C = -A B (one segment); C may alias A (N <= tile
// width) or B (M <= tile height): a workgroup reads its whole A row panel /
// B column panel before its epilogue writes.
// Workgroup ids are remapped so that each XCD (ids go round-robin over the 8
// XCDs) works on runs of consecutive tiles, which share operand panels in
// that XCD's L2.
// Chunks of kXcdChunk consecutive tiles go to the XCDs in turn (XCD x runs
// chunks x, x + 8, x + 16, ...): neighbouring tiles still share an L2, and
// tiles of unequal K (problems of one launch differ) spread evenly over the
// XCDs instead of one XCD receiving a whole run of long tiles.  The last
// partial round of 8 chunks keeps the identity order.
constexpr int kXcdChunk = 16;
__device__ __forceinline__ int xcd_remap(int bid, int nb) {
  const int full = nb / (8 * kXcdChunk) * (8 * kXcdChunk);
  if (bid >= full) return bid;
  const int x = bid & 7, i = bid >> 3;
  return ((i / kXcdChunk) * 8 + x) * kXcdChunk + (i % kXcdChunk);
}
// DEPTH: chunks of A and B in flight in registers ahead of the chunk being
// multiplied (1: the next chunk's loads overlap one MFMA block; 2: loads are
// issued two chunks ahead, alternating two register stages).
template <typename T, int MODE, int BMB, int BNB, int KB, int DEPTH = 1>
__global__ __launch_bounds__(256) void k_gemm(const GemmProbT<T> *__restrict__ probs,
                                              int nprob,
                                              const GemmSegT<T> *__restrict__ segs) {
  constexpr bool F64 = std::is_same<T, double>::value;
  constexpr int BM = 32 * BMB, BN = 32 * BNB;
  constexpr int NA = BM * KB / 256, NB = BN * KB / 256;
  // LDS tiles k-contiguous per row of A / column of B.  A lane reads GR
  // consecutive k of its row per access: FP32 128 x 128 tile 4 (16 bytes),
  // FP32 64 x 64 2, FP64 64 x 64 2 (16 bytes), FP64 128 x 128 1 (more
  // operands in registers would cost the second wave per SIMD).  Rows are
  // padded by GR elements: the row stride is then an odd multiple of the
  // access width modulo 32 banks, so the accesses of consecutive rows that
  // the LDS serves together (8 of 16 bytes, 16 of 8) hit disjoint banks.
  constexpr int GR = F64 ? (BMB * BNB >= 16 ? 1 : 2) : (BMB * BNB >= 16 ? 4 : 2);
  constexpr int KP = KB + GR;
  __shared__ __align__(16) T As[2][BM][KP];
  __shared__ __align__(16) T Bs[2][BN][KP];
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  int lo = 0, hi = nprob - 1;
  if (nprob == (int)gridDim.x) lo = hi = tile;  // one tile per problem
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (probs[mid].tile0 <= tile) lo = mid;
    else hi = mid - 1;
  }
  const GemmProbT<T> P = probs[lo];
  // grouped order: consecutive tile ids walk down a strip of GM tile rows
  // before moving right, so the tiles in flight on one XCD share both their
  // A and their B panels in its L2
  constexpr int GM = 8;
  const int lt = tile - P.tile0;
  const int tiles_m = (P.M + BM - 1) / BM;
  const int grp = lt / (GM * P.tiles_n), first = grp * GM;
  const int gsz = min(GM, tiles_m - first), li = lt - grp * GM * P.tiles_n;
  const int m0 = (first + li % gsz) * BM, n0 = (li / gsz) * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 16 * BMB, wn = (wave >> 1) * 16 * BNB;
  const int l16 = lane & 15, lk = lane >> 4;
  // one 16x16x4 product per 16 x 16 block, 4 output registers
  f4 accf[BMB][BNB];
  d4 accd[BMB][BNB];
#pragma unroll
  for (int a = 0; a < BMB; a++)
#pragma unroll
    for (int b = 0; b < BNB; b++) {
      accf[a][b] = f4{0.f, 0.f, 0.f, 0.f};
      accd[a][b] = d4{0.0, 0.0, 0.0, 0.0};
    }
  T ra[NA], rb[NB], ra2[NA], rb2[NB];
  // Loads are unconditional and unmasked with addresses clamped into the
  // operands, so they stay in flight across the MFMA block: a clamped row of
  // A (column of B) only feeds a row (column) of the tile that is never
  // stored; the K tail is zeroed in LDS after the store.  Element i of a
  // thread's A chunk is row m0 + tid % BM, column kk0 + NA (tid / BM) + i
  // (NA consecutive k: one vector store into LDS); of its B chunk row
  // kk0 + tid % KB, column n0 + tid / KB + i (256 / KB): on full chunks (no
  // K tail) and full tiles (no N edge), the uniform case, the addresses are
  // one base plus multiples of one stride.
  static_assert(256 % BM == 0 && 256 % KB == 0, "thread-to-element map");
  constexpr int BSTEP = 256 / KB;
  const int am = tid % BM, ak = tid / BM, bk = tid % KB, bn = tid / KB;
  auto load_into = [&](int sgi, int kk0, T (&xa)[NA], T (&xb)[NB]) {
    const GemmSegT<T> S = segs[P.seg0 + sgi];
    const auto pa = gptr(S.A) + min(m0 + am, P.M - 1);
    if (kk0 + KB <= S.K) {
      const auto p = pa + (long long)(kk0 + ak * NA) * S.lda;
#pragma unroll
      for (int i = 0; i < NA; i++) xa[i] = p[i * S.lda];
    } else {
#pragma unroll
      for (int i = 0; i < NA; i++) xa[i] = pa[(long long)min(kk0 + ak * NA + i, S.K - 1) * S.lda];
    }
    const auto pb = gptr(S.B) + min(kk0 + bk, S.K - 1);
    if (n0 + BN <= P.N) {
      const auto p = pb + (long long)(n0 + bn) * S.ldb;
      const long long st = (long long)BSTEP * S.ldb;
#pragma unroll
      for (int i = 0; i < NB; i++) xb[i] = p[i * st];
    } else {
#pragma unroll
      for (int i = 0; i < NB; i++) xb[i] = pb[(long long)min(n0 + bn + i * BSTEP, P.N - 1) * S.ldb];
    }
  };
  auto load = [&](int sgi, int kk0) { load_into(sgi, kk0, ra, rb); };
  // vectors of GR consecutive k
  typedef T vec_t __attribute__((ext_vector_type(GR)));
  static_assert(NA % GR == 0 && (KB / 4) % GR == 0, "vector LDS accesses");
  auto store_from = [&](int buf, int kvalid, const T (&xa)[NA], const T (&xb)[NB]) {
#pragma unroll
    for (int v = 0; v < NA / GR; v++) {
      vec_t w;
#pragma unroll
      for (int j = 0; j < GR; j++) w[j] = xa[v * GR + j];
      *(vec_t *)&As[buf][am][ak * NA + v * GR] = w;
    }
#pragma unroll
    for (int i = 0; i < NB; i++) Bs[buf][bn + i * BSTEP][bk] = xb[i];
    if (kvalid < KB && bk >= kvalid) {  // last chunk of a segment whose K % KB != 0
#pragma unroll
      for (int i = 0; i < NB; i++) Bs[buf][bn + i * BSTEP][bk] = T(0);
    }
  };
  auto store = [&](int buf, int kvalid) { store_from(buf, kvalid, ra, rb); };
  auto advance = [&](int &sgi, int &kk0) {
    kk0 += KB;
    while (sgi < P.nseg && kk0 >= segs[P.seg0 + sgi].K) {
      sgi++;
      kk0 = 0;
    }
  };
  // One K chunk from LDS buffer buf.  The chunk's k indices are permuted
  // between the MFMA steps (A and B alike, so the sum is the same): at step
  // kq, lanes 16 k' .. 16 k' + 15 hold k = (KB / 4) k' + kq, so a lane's
  // operands for GR consecutive steps are GR consecutive values of its row
  // of A (column of B): one LDS read per row block per GR steps.
  constexpr int KQ = KB / 4;
  auto compute = [&](int buf) {
#pragma unroll
    for (int g0 = 0; g0 < KQ; g0 += GR) {
      vec_t bv[BNB], av[BMB];
#pragma unroll
      for (int b = 0; b < BNB; b++) bv[b] = *(const vec_t *)&Bs[buf][wn + b * 16 + l16][KQ * lk + g0];
#pragma unroll
      for (int a = 0; a < BMB; a++) av[a] = *(const vec_t *)&As[buf][wm + a * 16 + l16][KQ * lk + g0];
#pragma unroll
      for (int j = 0; j < GR; j++) {
        if constexpr (F64) {
#pragma unroll
          for (int a = 0; a < BMB; a++)
#pragma unroll
            for (int b = 0; b < BNB; b++)
              accd[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[b][j], av[a][j], accd[a][b], 0, 0, 0);
        } else {
#pragma unroll
          for (int a = 0; a < BMB; a++)
#pragma unroll
            for (int b = 0; b < BNB; b++)
              accf[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[b][j], av[a][j], accf[a][b], 0, 0, 0);
        }
      }
    }
  };
  // element (a, b, r) of this lane's accumulators: its place in C and value
  auto elem = [&](int a, int b, int r, int &m, int &n, T &v) __attribute__((always_inline)) {
    if constexpr (F64) {
      // D = B^T A^T: register r of lane l holds C[l % 16][4 r + l / 16]
      m = m0 + wm + a * 16 + l16;
      n = n0 + wn + b * 16 + 4 * r + lk;
      v = accd[a][b][r];
    } else {
      // D = B^T A^T: register r of lane l holds C[l % 16][4 (l / 16) + r]
      m = m0 + wm + a * 16 + l16;
      n = n0 + wn + b * 16 + 4 * lk + r;
      v = accf[a][b][r];
    }
  };
  // C -= AB: after the K loop the C values of a group of block rows are all
  // loaded before any is stored, so they are in flight together (one round
  // trip per group, not one per element; groups of 2 block rows keep the
  // registers of the large tile in bounds)
  constexpr int AG = BMB > 2 ? 2 : BMB;
  T cold[BMB][BNB][4];
  auto load_c = [&](int a0) __attribute__((always_inline)) {
    if constexpr (MODE == 0) {
#pragma unroll
      for (int a = a0; a < a0 + AG; a++)
#pragma unroll
        for (int b = 0; b < BNB; b++)
#pragma unroll
          for (int r = 0; r < 4; r++) {
            int m, n;
            T v;
            elem(a, b, r, m, n, v);
            cold[a][b][r] = (m < P.M && n < P.N) ? gptr(P.C)[m + (long long)n * P.ldc] : T(0);
          }
    }
  };
  int sg = 0, k0 = 0;
  if (P.nseg == 0) return;
  if constexpr (DEPTH == 1) {
    load(sg, k0);
    store(0, segs[P.seg0].K - k0);
    __syncthreads();
    int buf = 0;
    for (;;) {
      int nsg = sg, nk0 = k0;
      advance(nsg, nk0);
      const bool more = nsg < P.nseg;
      if (more) load(nsg, nk0);
      compute(buf);
      if (!more) break;
      store(buf ^ 1, segs[P.seg0 + nsg].K - nk0);
      __syncthreads();
      buf ^= 1;
      sg = nsg;
      k0 = nk0;
    }
  } else {
    // chunk c is multiplied from LDS while chunk c+1 sits in one register
    // stage (stored after the MFMA block) and chunk c+2 is in flight into
    // the other; the stages alternate, so no register copies wait on loads
    load(sg, k0);
    store(0, segs[P.seg0].K - k0);
    __syncthreads();
    int s1 = sg, k1 = k0;
    advance(s1, k1);
    int s2 = s1, k2 = k1;
    if (s1 < P.nseg) {
      load_into(s1, k1, ra, rb);
      advance(s2, k2);
      if (s2 < P.nseg) load_into(s2, k2, ra2, rb2);
    }
    int buf = 0;
    for (;;) {
      // stage a holds (s1, k1), stage b holds (s2, k2)
      compute(buf);
      if (s1 >= P.nseg) break;
      store_from(buf ^ 1, segs[P.seg0 + s1].K - k1, ra, rb);
      __syncthreads();
      buf ^= 1;
      int s3 = s2, k3 = k2;
      if (s3 < P.nseg) {
        advance(s3, k3);
        if (s3 < P.nseg) load_into(s3, k3, ra, rb);
      }
      compute(buf);
      if (s2 >= P.nseg) break;
      store_from(buf ^ 1, segs[P.seg0 + s2].K - k2, ra2, rb2);
      __syncthreads();
      buf ^= 1;
      s1 = s3;
      k1 = k3;
      s2 = s3;
      k2 = k3;
      if (s2 < P.nseg) {
        advance(s2, k2);
        if (s2 < P.nseg) load_into(s2, k2, ra2, rb2);
      }
    }
  }
#pragma unroll
  for (int a0 = 0; a0 < BMB; a0 += AG) {
    load_c(a0);
#pragma unroll
    for (int a = a0; a < a0 + AG; a++)
#pragma unroll
      for (int b = 0; b < BNB; b++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          int m, n;
          T v;
          elem(a, b, r, m, n, v);
          if (m < P.M && n < P.N) {
            auto c = gptr(P.C) + m + (long long)n * P.ldc;
            if (MODE == 1) *c = v;
            else if (MODE == 2) *c = -v;
            else *c = cold[a][b][r] - v;
          }
        }
  }
}
// ---------------------------------------------------------------------------
// FP32 grouped GEMM on the bf16 MFMA (v_mfma_f32_16x16x32_bf16; the
// SNU_GEMM_SPLIT form of the FP32 factorization's GEMM launches)
// ---------------------------------------------------------------------------
// Every FP32 operand x is split into three bf16 pieces with x = h + m + l
// exactly: h = bf16(x), m = bf16(x - h), l = bf16(x - h - m), each rounded
// to nearest even.  x - h and x - h - m are exact in FP32, |m| <= 2^-8 |x|
// and |l| <= 2^-16 |x|, and x - h - m has at most 8 significant bits, so l
// is exact as well.  C accumulates in FP32 the six products of pieces of
// weight >= 2^-16, hh + hm + mh + hl + mm + lh (each bf16 product is exact
// in FP32); the three left out (ml, lm, ll) total at most about
// 2^-23 |a| |b|, two units of FP32's own rounding of one product.  Per
// 16 x 16 x 32 block that is six bf16 MFMAs (16 cycles each) in place of
// eight 16x16x4 f32 MFMAs (32 cycles each).
// Workgroup tile (32 BMB) x (32 BNB) (128 x 128 or 64 x 64), 4 waves in
// 2 x 2; K chunk 32 (one bf16 MFMA deep).  LDS holds one chunk, pieces per
// row of A and per column of B as [h 0..31 | m 0..31 | l 0..31 | pad 8] bf16
// (52 dwords: the 16-byte reads of 8 consecutive rows fall on disjoint
// banks); the next chunk is in flight in registers during the MFMA block,
// and several workgroups share a CU (2 of the large tile, 4 of the small),
// so one splits and stores while another multiplies.
// Tiles, problems, modes, aliasing and the XCD order are those of k_gemm
// with the same tile size (the same tile counts).
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float fl2_t __attribute__((ext_vector_type(2)));
constexpr int kSplitRow = 104;  // bf16 per LDS row: 3 pieces x 32 + 8
// pieces of two FP32 values as packed bf16 pairs (element 0 in the low half)
__device__ __forceinline__ void split_pair(float x0, float x1, unsigned &h, unsigned &m, unsigned &l) {
  const fl2_t x = fl2_t{x0, x1};
  const bf16x2_t hb = __builtin_convertvector(x, bf16x2_t);
  const fl2_t r = x - __builtin_convertvector(hb, fl2_t);
  const bf16x2_t mb = __builtin_convertvector(r, bf16x2_t);
  const fl2_t r2 = r - __builtin_convertvector(mb, fl2_t);
  const bf16x2_t lb = __builtin_convertvector(r2, bf16x2_t);
  h = __builtin_bit_cast(unsigned, hb);
  m = __builtin_bit_cast(unsigned, mb);
  l = __builtin_bit_cast(unsigned, lb);
}
template <int MODE, int BMB, int BNB>
__global__ __launch_bounds__(256, BMB * BNB >= 16 ? 2 : 4) void k_gemm_split(
    const GemmProbT<float> *__restrict__ probs, int nprob, const GemmSegT<float> *__restrict__ segs) {
  constexpr int BM = 32 * BMB, BN = 32 * BNB, KB = 32;
  constexpr int NA = BM / 8, NBC = BN / 16;  // A: NA consecutive k per thread; B: NBC columns
  constexpr int RW = kSplitRow / 2;          // dwords per LDS row
  __shared__ __align__(16) unsigned As[BM * RW];
  __shared__ __align__(16) unsigned Bs[BN * RW];
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  int lo = 0, hi = nprob - 1;
  if (nprob == (int)gridDim.x) lo = hi = tile;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (probs[mid].tile0 <= tile) lo = mid;
    else hi = mid - 1;
  }
  const GemmProbT<float> P = probs[lo];
  constexpr int GM = 8;
  const int lt = tile - P.tile0;
  const int tiles_m = (P.M + BM - 1) / BM;
  const int grp = lt / (GM * P.tiles_n), first = grp * GM;
  const int gsz = min(GM, tiles_m - first), li = lt - grp * GM * P.tiles_n;
  const int m0 = (first + li % gsz) * BM, n0 = (li / gsz) * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 16 * BMB, wn = (wave >> 1) * 16 * BNB;
  const int l16 = lane & 15, lk = lane >> 4;
  f4 acc[BMB][BNB];
#pragma unroll
  for (int a = 0; a < BMB; a++)
#pragma unroll
    for (int b = 0; b < BNB; b++) acc[a][b] = f4{0.f, 0.f, 0.f, 0.f};
  // A chunk: row m0 + am, k = NA ak + 0..NA-1 (coalesced over rows); B
  // chunk: columns n0 + bc + 16 i (i < NBC), k = 2 bp, 2 bp + 1 (a lane
  // pair's two loads cover 8 bytes, 16 lanes one 128-byte column segment).
  // Addresses are clamped into the operands as in k_gemm; the K tail of B is
  // zeroed before the split.
  static_assert(NA % 8 == 0 && 256 % BM == 0, "thread-to-element map");
  const int am = tid % BM, ak = tid / BM, bp = tid & 15, bc = tid >> 4;
  float xa[NA], xb[2 * NBC];
  auto load = [&](int sgi, int kk0) {
    const GemmSegT<float> S = segs[P.seg0 + sgi];
    const auto pa = gptr(S.A) + min(m0 + am, P.M - 1);
    if (kk0 + KB <= S.K) {
      const auto p = pa + (long long)(kk0 + NA * ak) * S.lda;
#pragma unroll
      for (int i = 0; i < NA; i++) xa[i] = p[i * S.lda];
    } else {
#pragma unroll
      for (int i = 0; i < NA; i++) xa[i] = pa[(long long)min(kk0 + NA * ak + i, S.K - 1) * S.lda];
    }
    const auto pb = gptr(S.B);
    if (kk0 + KB <= S.K && n0 + BN <= P.N) {
      const auto p = pb + kk0 + 2 * bp + (long long)(n0 + bc) * S.ldb;
      const long long st = 16 * S.ldb;
#pragma unroll
      for (int i = 0; i < NBC; i++) {
        xb[2 * i] = p[i * st];
        xb[2 * i + 1] = p[i * st + 1];
      }
    } else {
      const int k0c = min(kk0 + 2 * bp, S.K - 1), k1c = min(kk0 + 2 * bp + 1, S.K - 1);
#pragma unroll
      for (int i = 0; i < NBC; i++) {
        const auto p = pb + (long long)min(n0 + bc + 16 * i, P.N - 1) * S.ldb;
        xb[2 * i] = p[k0c];
        xb[2 * i + 1] = p[k1c];
      }
    }
  };
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  auto store = [&](int kvalid) {
    unsigned h[NA / 2], m[NA / 2], l[NA / 2];
#pragma unroll
    for (int j = 0; j < NA / 2; j++) split_pair(xa[2 * j], xa[2 * j + 1], h[j], m[j], l[j]);
    unsigned *ra = As + am * RW + (NA / 2) * ak;
#pragma unroll
    for (int v = 0; v < NA / 8; v++) {
      *(u4 *)(ra + 4 * v) = u4{h[4 * v], h[4 * v + 1], h[4 * v + 2], h[4 * v + 3]};
      *(u4 *)(ra + 16 + 4 * v) = u4{m[4 * v], m[4 * v + 1], m[4 * v + 2], m[4 * v + 3]};
      *(u4 *)(ra + 32 + 4 * v) = u4{l[4 * v], l[4 * v + 1], l[4 * v + 2], l[4 * v + 3]};
    }
    const bool z0 = 2 * bp >= kvalid, z1 = 2 * bp + 1 >= kvalid;
#pragma unroll
    for (int i = 0; i < NBC; i++) {
      unsigned hb, mb, lb;
      split_pair(z0 ? 0.f : xb[2 * i], z1 ? 0.f : xb[2 * i + 1], hb, mb, lb);
      unsigned *rb = Bs + (bc + 16 * i) * RW + bp;
      rb[0] = hb;
      rb[16] = mb;
      rb[32] = lb;
    }
  };
  auto advance = [&](int &sgi, int &kk0) {
    kk0 += KB;
    while (sgi < P.nseg && kk0 >= segs[P.seg0 + sgi].K) {
      sgi++;
      kk0 = 0;
    }
  };
  // lane l16 + 16 lk supplies row (column) l16 of its block with k slots
  // 8 lk .. 8 lk + 7 of every piece, for both operands alike
  auto compute = [&]() {
    bf16x8_t av[BMB][3];
#pragma unroll
    for (int a = 0; a < BMB; a++)
#pragma unroll
      for (int p = 0; p < 3; p++)
        av[a][p] = __builtin_bit_cast(bf16x8_t, *(const u4 *)(As + (wm + a * 16 + l16) * RW + 16 * p + 4 * lk));
#pragma unroll
    for (int b = 0; b < BNB; b++) {
      bf16x8_t bv[3];
#pragma unroll
      for (int p = 0; p < 3; p++)
        bv[p] = __builtin_bit_cast(bf16x8_t, *(const u4 *)(Bs + (wn + b * 16 + l16) * RW + 16 * p + 4 * lk));
#pragma unroll
      for (int a = 0; a < BMB; a++) {
        // small terms first: l h, m m, h l, m h, h m, h h
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv[2], av[a][0], acc[a][b], 0, 0, 0);
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv[1], av[a][1], acc[a][b], 0, 0, 0);
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv[0], av[a][2], acc[a][b], 0, 0, 0);
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv[1], av[a][0], acc[a][b], 0, 0, 0);
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv[0], av[a][1], acc[a][b], 0, 0, 0);
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv[0], av[a][0], acc[a][b], 0, 0, 0);
      }
    }
  };
  if (P.nseg == 0) return;
  int sg = 0, k0 = 0;
  load(sg, k0);
  store(segs[P.seg0].K - k0);
  __syncthreads();
  for (;;) {
    int nsg = sg, nk0 = k0;
    advance(nsg, nk0);
    const bool more = nsg < P.nseg;
    if (more) load(nsg, nk0);
    compute();
    if (!more) break;
    __syncthreads();
    store(segs[P.seg0 + nsg].K - nk0);
    __syncthreads();
    sg = nsg;
    k0 = nk0;
  }
  // D = B^T A^T: register r of lane l holds C[l % 16][4 (l / 16) + r]
  constexpr int AG = BMB > 2 ? 2 : BMB;
#pragma unroll
  for (int a0 = 0; a0 < BMB; a0 += AG) {
    float cold[AG][BNB][4];
    if constexpr (MODE == 0) {
#pragma unroll
      for (int a = 0; a < AG; a++)
#pragma unroll
        for (int b = 0; b < BNB; b++)
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const int m = m0 + wm + (a0 + a) * 16 + l16, n = n0 + wn + b * 16 + 4 * lk + r;
            cold[a][b][r] = (m < P.M && n < P.N) ? gptr(P.C)[m + (long long)n * P.ldc] : 0.f;
          }
    }
#pragma unroll
    for (int a = 0; a < AG; a++)
#pragma unroll
      for (int b = 0; b < BNB; b++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int m = m0 + wm + (a0 + a) * 16 + l16, n = n0 + wn + b * 16 + 4 * lk + r;
          if (m < P.M && n < P.N) {
            auto c = gptr(P.C) + m + (long long)n * P.ldc;
            const float v = acc[a0 + a][b][r];
            if (MODE == 1) *c = v;
            else if (MODE == 2) *c = -v;
            else *c = cold[a][b][r] - v;
          }
        }
  }
}
void launch_gemm128_split(const GemmProbT<float> *probs, int nprob, const GemmSegT<float> *segs,
                          int total_tiles, int mode, hipStream_t st) {
  if (total_tiles <= 0 || nprob <= 0) return;
  if (mode == 1)
    hipLaunchKernelGGL((k_gemm_split<1, 4, 4>), dim3(total_tiles), dim3(256), 0, st, probs, nprob, segs);
  else if (mode == 2)
    hipLaunchKernelGGL((k_gemm_split<2, 4, 4>), dim3(total_tiles), dim3(256), 0, st, probs, nprob, segs);
  else
    hipLaunchKernelGGL((k_gemm_split<0, 4, 4>), dim3(total_tiles), dim3(256), 0, st, probs, nprob, segs);
}
void launch_gemm_split(const GemmProbT<float> *probs, int nprob, const GemmSegT<float> *segs,
                       int total_tiles, int mode, hipStream_t st) {
  if (total_tiles <= 0 || nprob <= 0) return;
  if (mode == 1)
    hipLaunchKernelGGL((k_gemm_split<1, 2, 2>), dim3(total_tiles), dim3(256), 0, st, probs, nprob, segs);
  else if (mode == 2)
    hipLaunchKernelGGL((k_gemm_split<2, 2, 2>), dim3(total_tiles), dim3(256), 0, st, probs, nprob, segs);
  else
    hipLaunchKernelGGL((k_gemm_split<0, 2, 2>), dim3(total_tiles), dim3(256), 0, st, probs, nprob, segs);
}

// Grouped 2-D copy over GEMM descriptors: C (ldc) = A of the problem's first
// segment (lda), one workgroup per 64 x 64 tile, rows contiguous per wave.
template <typename T>
__global__ __launch_bounds__(256) void k_copy2d(const GemmProbT<T> *__restrict__ probs, int nprob,
                                                const GemmSegT<T> *__restrict__ segs) {
  const int tile = blockIdx.x;
  int lo = 0, hi = nprob - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (probs[mid].tile0 <= tile) lo = mid;
    else hi = mid - 1;
  }
  const GemmProbT<T> P = probs[lo];
  const GemmSegT<T> S = segs[P.seg0];
  const int lt = tile - P.tile0;
  const int m0 = (lt / P.tiles_n) * 64, n0 = (lt % P.tiles_n) * 64;
  const int r = threadIdx.x & 63;
  if (m0 + r >= P.M) return;
  const T *src = S.A + (m0 + r) + (long long)n0 * S.lda;
  T *dst = P.C + (m0 + r) + (long long)n0 * P.ldc;
  const int nc = min(64, P.N - n0);
  for (int c = threadIdx.x >> 6; c < nc; c += 4) dst[(long long)c * P.ldc] = src[(long long)c * S.lda];
}
template <typename T>
void launch_copy2d(const GemmProbT<T> *probs, int nprob, const GemmSegT<T> *segs, int total_tiles,
                   hipStream_t st) {
  if (total_tiles <= 0 || nprob <= 0) return;
  hipLaunchKernelGGL(k_copy2d<T>, dim3(total_tiles), dim3(256), 0, st, probs, nprob, segs);
}
// K chunk of the production launches: 32 in FP32 (the 128 x 128 tile
// 110 -> 122 TF/s at 4096^3, the 64 x 64 tile even with 16), 16 in FP64
// (32 costs the FP64 tiles their second workgroup per CU)
template <typename T>
constexpr int gemm_kb() {
  return sizeof(T) == 4 ? 32 : 16;
}
template <typename T>
void launch_gemm(const GemmProbT<T> *probs, int nprob, const GemmSegT<T> *segs,
                 int total_tiles, int mode, hipStream_t st) {
  if (total_tiles <= 0 || nprob <= 0) return;
  // loads one chunk ahead (two ahead measured slower in both precisions
  // once the accumulators stay in VGPRs)
  constexpr int KB = gemm_kb<T>();
  if (mode == 1)
    hipLaunchKernelGGL((k_gemm<T, 1, 2, 2, KB, 1>), dim3(total_tiles), dim3(256), 0, st, probs, nprob,
                       segs);
  else if (mode == 2)
    hipLaunchKernelGGL((k_gemm<T, 2, 2, 2, KB, 1>), dim3(total_tiles), dim3(256), 0, st, probs, nprob,
                       segs);
  else
    hipLaunchKernelGGL((k_gemm<T, 0, 2, 2, KB, 1>), dim3(total_tiles), dim3(256), 0, st, probs, nprob,
                       segs);
}
// 128 x 128 tiles, mode 0 (C -= AB), 1 (C = AB) or 2 (C = -AB); loads one
// chunk ahead (with accumulators in VGPRs the large tile is fastest that way
// in both precisions)
template <typename T>
void launch_gemm128(const GemmProbT<T> *probs, int nprob, const GemmSegT<T> *segs,
                    int total_tiles, int mode, hipStream_t st) {
  if (total_tiles <= 0 || nprob <= 0) return;
  constexpr int KB = gemm_kb<T>();
  if (mode == 1)
    hipLaunchKernelGGL((k_gemm<T, 1, 4, 4, KB, 1>), dim3(total_tiles), dim3(256), 0, st, probs, nprob,
                       segs);
  else if (mode == 2)
    hipLaunchKernelGGL((k_gemm<T, 2, 4, 4, KB, 1>), dim3(total_tiles), dim3(256), 0, st, probs, nprob,
                       segs);
  else
    hipLaunchKernelGGL((k_gemm<T, 0, 4, 4, KB, 1>), dim3(total_tiles), dim3(256), 0, st, probs, nprob,
                       segs);
}
// C -= AB variants for tuning: tile 64 or 128, K chunk 16 or 32, register
// prefetch depth 1 or 2 (the tile count is that of the tile size)
template <typename T>
void launch_gemm_variant(const GemmProbT<T> *probs, int nprob, const GemmSegT<T> *segs,
                         int total_tiles, int tile, int kb, int depth, hipStream_t st) {
  if (total_tiles <= 0 || nprob <= 0) return;
  const dim3 g(total_tiles), b(256);
  if (tile == 128) {
    if (depth == 2) hipLaunchKernelGGL((k_gemm<T, 0, 4, 4, 16, 2>), g, b, 0, st, probs, nprob, segs);
    else if (kb == 32) hipLaunchKernelGGL((k_gemm<T, 0, 4, 4, 32, 1>), g, b, 0, st, probs, nprob, segs);
    else hipLaunchKernelGGL((k_gemm<T, 0, 4, 4, 16, 1>), g, b, 0, st, probs, nprob, segs);
  } else {
    if (depth == 2) hipLaunchKernelGGL((k_gemm<T, 0, 2, 2, 16, 2>), g, b, 0, st, probs, nprob, segs);
    else if (kb == 32) hipLaunchKernelGGL((k_gemm<T, 0, 2, 2, 32, 1>), g, b, 0, st, probs, nprob, segs);
    else hipLaunchKernelGGL((k_gemm<T, 0, 2, 2, 16, 1>), g, b, 0, st, probs, nprob, segs);
  }
}

// ---------------------------------------------------------------------------
// dense: diagonal block LU (no pivoting, as cusolverDnDgetrf with a null
// ipiv / LAPACKE_mkl_dgetrfnp) and the inverses of its triangular factors.
// ---------------------------------------------------------------------------
// One workgroup of 4 waves per block (padded to 64 x 64 with a unit diagonal),
// in LDS, blocked by 16 columns.  Per block column kb:
//   (1) two waves, each factoring the 16 x 16 diagonal block for itself in
//       registers (every group of 16 lanes holds it, row per lane, and takes a
//       pivot row by DPP broadcast: no barrier, no scalar registers), carry it
//       over to what needs the inverse of its factors:
//         lane = row: U11^-1 for the rows below the block (L21) and, of
//         Y = U^-1, the rows above it; the block's own rows start from the
//         identity and become Y's diagonal block;
//         lane = column: L11^-1 for the columns right of the block (U12) and,
//         of X = L^-1, those left of it; the block's own become X's;
//   (2) all waves: the rank-16 updates A22 -= L21 U12, X -= L21 X_kb,
//       Y -= Y_kb U12 on MFMA tiles.
// X and Y replace the factors in place: L21 and U12 are read by (2) of their
// own block column alone, which leaves X's and Y's blocks there (all tiles are
// computed before any is written).  [column][row]; odd leading dimension:
// accesses along rows are conflict-free too.  42 KB FP64: three blocks share a
// CU (84 KB and 8 waves, with X and Y beside the factors, kept it to one).
// Bound by the pivot chain of (1): of one block's 45,000 cycles (18.6 us,
// FP64) 19,000 are its 64 dependent broadcast, division and update steps,
// 14,000 the tiles of (2), 7,000 reading the block and storing the results.
// Broadcast inside the FMA (DPP), one reciprocal for the two quotients of a
// step and tiles loaded together brought a step's launch with panels from 26.1
// to 22.4 us FP64 and from 21.4 to 18.6 us FP32.
template <typename T>
struct DiagLds {
  T A[64][65], Xd[4][16][17];
};
// d[c] -= md u, v[c] -= mv u, u: lane J's d[c], for N columns from C on.
// (s_nop: a DPP source must not have been written by the two instructions
// before; the compiler's own hazard check does not see into the block.)
#define SNU_RANK1(type, op)                                                                                        \
  template <int J, int C, int N>                                                                                  \
  __device__ __forceinline__ void rank1_block(type(&d)[16], type(&v)[16], type md, type mv) {                     \
    static_assert(N == 1 || N == 2 || N == 4, "columns");                                                         \
    if constexpr (N == 4)                                                                                         \
      asm volatile("s_nop 1\n\t" op " %4, %0, -%9 row_newbcast:%10\n\t" op " %0, %0, -%8 row_newbcast:%10\n\t"     \
                   op " %5, %1, -%9 row_newbcast:%10\n\t" op " %1, %1, -%8 row_newbcast:%10\n\t"                   \
                   op " %6, %2, -%9 row_newbcast:%10\n\t" op " %2, %2, -%8 row_newbcast:%10\n\t"                   \
                   op " %7, %3, -%9 row_newbcast:%10\n\t" op " %3, %3, -%8 row_newbcast:%10"                       \
                   : "+v"(d[C]), "+v"(d[C + 1]), "+v"(d[C + 2]), "+v"(d[C + 3]), "+v"(v[C]), "+v"(v[C + 1]),       \
                     "+v"(v[C + 2]), "+v"(v[C + 3])                                                               \
                   : "v"(md), "v"(mv), "n"(J));                                                                   \
    else if constexpr (N == 2)                                                                                    \
      asm volatile("s_nop 1\n\t" op " %2, %0, -%5 row_newbcast:%6\n\t" op " %0, %0, -%4 row_newbcast:%6\n\t"       \
                   op " %3, %1, -%5 row_newbcast:%6\n\t" op " %1, %1, -%4 row_newbcast:%6"                         \
                   : "+v"(d[C]), "+v"(d[C + 1]), "+v"(v[C]), "+v"(v[C + 1])                                       \
                   : "v"(md), "v"(mv), "n"(J));                                                                   \
    else                                                                                                          \
      asm volatile("s_nop 1\n\t" op " %1, %0, -%3 row_newbcast:%4\n\t" op " %0, %0, -%2 row_newbcast:%4\n\ts_nop 1" \
                   : "+v"(d[C]), "+v"(v[C])                                                                       \
                   : "v"(md), "v"(mv), "n"(J));                                                                   \
  }
SNU_RANK1(double, "v_fmac_f64_dpp")
SNU_RANK1(float, "v_fmac_f32_dpp")
#undef SNU_RANK1
template <typename T, int J, int C>
__device__ __forceinline__ void rank1(T (&d)[16], T (&v)[16], T md, T mv) {
  // (two columns at least in a step's first block: the next step broadcasts
  // its first column)
  if constexpr (C < 16) {
    constexpr int N = 16 - C >= 4 ? 4 : 16 - C >= 2 ? 2 : 1;
    rank1_block<J, C, N>(d, v, md, mv);
    rank1<T, J, C + N>(d, v, md, mv);
  }
}
// Column J of the diagonal block d (entry l16 of its columns per lane; becomes
// its LU factors) and of what a wave carries along in v.  keep: v[J] stays as
// it is instead of being divided by the pivot.  One code path for both waves:
// fetching variants of the unrolled steps cost more than the arithmetic.
// d[J] / pivot and v[J] / pivot are rounded as by two divisions (Divisor), with
// one reciprocal.
template <typename T, int J>
__device__ __forceinline__ void diag_step(T (&d)[16], T (&v)[16], int l16, bool keep, T eps) {
  // pivots of magnitude below eps become +-eps (the leaf pivots' rule; eps = 0
  // leaves them)
  T piv = bcast16<J>(d[J]);
  const T cl = piv < T(0) ? -eps : eps;
  piv = fabs(piv) < eps ? cl : piv;
  const Divisor<T> by(piv);
  const T a = by.quotient(d[J]), b = by.quotient(v[J]);
  const T md = l16 > J ? a : T(0);
  d[J] = l16 > J ? a : l16 == J ? piv : d[J];
  v[J] = keep ? v[J] : b;
  asm volatile("" : "+v"(d[J]), "+v"(v[J]));  // (not left, with its inputs, for the end)
  rank1<T, J, J + 1>(d, v, md, b);
}
template <typename T, int... J>
__device__ __forceinline__ void diag_block(std::integer_sequence<int, J...>, T (&d)[16], T (&v)[16], int l16,
                                           bool keep, T eps) {
  (diag_step<T, J>(d, v, l16, keep, eps), ...);
}
// store: this workgroup writes the block's factors to LU.
template <typename T>
__device__ __forceinline__ void factor_block(DiagLds<T> &S, const DiagProbT<T> &P, int lane, int wave, bool store) {
  const int nb = P.nb;
  {
    const auto D = gptr((const T *)P.D);
    T v[16];
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int c = wave + 4 * q;
      v[q] = D[min(lane, nb - 1) + (long long)min(c, nb - 1) * P.ld];
    }
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int c = wave + 4 * q;
      S.A[c][lane] = lane < nb && c < nb ? v[q] : (lane == c ? T(1) : T(0));
    }
  }
  __syncthreads();
  const auto LU = gptr(P.LU);
#pragma unroll 1
  for (int kb = 0; kb < 4; kb++) {
    asm volatile("" : "+v"(lane));  // (addresses and masks by lane are not kept from one pass to the next)
    const int k0 = 16 * kb, l16 = lane & 15, lk = lane >> 4;
    if (wave < 2) {
      // wave 0: lane = row.  Wave 1: lane = column, all transposed (the scaled
      // pivot row then plays the part of the multipliers).
      const bool tr = wave == 1, own = lk == kb;
      const T *ds = &S.A[0][0] + (tr ? (k0 + l16) * 65 + k0 : k0 * 65 + k0 + l16);
      T *vs = &S.A[0][0] + (tr ? lane * 65 + k0 : k0 * 65 + lane);
      T d[16], v[16];
      if (tr) {
#pragma unroll
        for (int j = 0; j < 16; j++) d[j] = ds[j], v[j] = vs[j];
      } else {
#pragma unroll
        for (int j = 0; j < 16; j++) d[j] = ds[j * 65], v[j] = vs[j * 65];
      }
#pragma unroll
      for (int j = 0; j < 16; j++) v[j] = own ? (j == l16 ? T(1) : T(0)) : v[j];
      diag_block<T>(std::make_integer_sequence<int, 16>{}, d, v, l16, tr, P.eps);
      // (the diagonal block is read by both before wave 0 writes it)
      __syncthreads();
      if (tr) {
        if (own) vs = &S.Xd[kb][l16][0];
#pragma unroll
        for (int j = 0; j < 16; j++) vs[j] = v[j];
      } else {
#pragma unroll
        for (int j = 0; j < 16; j++) vs[j * 65] = v[j];
        if (store && lane < 16) {
#pragma unroll
          for (int j = 0; j < 16; j++) LU[k0 * 65 + lane + j * 64] = d[j];
        }
      }
    } else {
      __syncthreads();
    }
    __syncthreads();
    // tile (i, j) (16 x 16 blocks) -= (i, kb) (kb, j) for i > kb (column
    // j = wave), then for i <= kb, j > kb; X's and Y's first contribution
    // (j == kb, i == kb) replaces L21 and U12.  A wave's tiles are loaded
    // together, those past the last one as copies of it.
    if (kb == 3) break;
    // (i, j) of tile t: the digits of 4 i + j in base 16
    const int nt = kb == 0 ? 15 : kb == 1 ? 12 : 7;
    const unsigned long long list = kb == 0 ? 0x3321FEDCBA987654ull : kb == 1 ? 0x77777632FEDCBA98ull : 0xBBBBBBBBBB73FEDCull;
    Frag<T> acc[4];
    T av[4][4], bv[4][4];
    int at[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int ij = (int)(list >> (4 * (wave + 4 * q))) & 15, i = ij >> 2, j = ij & 3;
      at[q] = 16 * j * 65 + 16 * i;
      const T *a = &S.A[k0][16 * i], *b = j == kb ? &S.Xd[kb][0][0] : &S.A[16 * j][k0], *c = &S.A[0][0] + at[q];
      const int ldb = j == kb ? 17 : 65;
      const bool first = i == kb || j == kb;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int k = frag_row<T>(r, lk);
        const T x = c[l16 * 65 + k];
        acc[q][r] = first ? T(0) : x;
        av[q][r] = a[k * 65 + l16];
        bv[q][r] = b[l16 * ldb + k];
      }
    }
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int q = 0; q < 4; q++) acc[q] = mfma4(-av[q][r], bv[q][r], acc[q]);
    if (store) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int ij = (int)(list >> (4 * (wave + 4 * q))) & 15, i = ij >> 2, j = ij & 3;
        if (i != kb && j != kb) continue;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int k = k0 + frag_row<T>(r, lk);
          LU[i == kb ? k + (16 * j + l16) * 64 : 16 * i + l16 + k * 64] = i == kb ? bv[q][r] : av[q][r];
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (wave + 4 * q < nt) {
#pragma unroll
        for (int r = 0; r < 4; r++) (&S.A[0][0])[at[q] + l16 * 65 + frag_row<T>(r, lk)] = acc[q][r];
      }
    __syncthreads();
  }
}
// The inverses (lower: L^-1, upper: U^-1) into their places.
template <typename T>
__device__ __forceinline__ void store_block(const DiagLds<T> &S, const DiagProbT<T> &P, int lane, int wave, bool lower,
                                            bool upper) {
  const int rb = lane >> 4, l16 = lane & 15;
#pragma unroll
  for (int q = 0; q < 16; q++) {
    const int c = wave + 4 * q, cb = q >> 2;
    const T a = S.A[c][lane], xd = S.Xd[cb][c & 15][l16];
    if (lane < P.nb && c < P.nb) {
      if (lower) gptr(P.Linv)[lane + c * P.ldi] = rb > cb ? a : rb == cb ? xd : T(0);
      if (upper) gptr(P.Uinv)[lane + c * P.ldi] = rb <= cb ? a : T(0);
    }
  }
}
// Panel tile q of a problem: rows 64 q .. below the block times U^-1, or (from
// the middle on) L^-1 times the columns right of it.  A wave takes 16 rows
// (columns) of the tile; its operand from the panel is loaded in MFMA layout
// before the block is factored.
template <typename T>
struct PanelTile {
  bool rows;     // below the block (else right of it)
  int at, left;  // this lane's row / column of the panel, entries of it left from the tile's block
  T v[16];
};
template <typename T>
__device__ __forceinline__ void load_panel(PanelTile<T> &t, const DiagProbT<T> &P, int q, int lane, int wave) {
  const int mt = (P.m + 63) >> 6, l16 = lane & 15, lk = lane >> 4;
  t.rows = q < mt;
  const int base = 64 * (t.rows ? q : q - mt) + 16 * wave;
  t.at = base;
  t.left = P.m - base;
  if (P.m == 0) return;  // a block without panels
  const int i = min(base + l16, P.m - 1);
  const auto src = gptr((const T *)P.D) + (t.rows ? P.nb + i : (P.nb + (long long)i) * P.ld);
#pragma unroll
  for (int j = 0; j < 16; j++) {
    const int k = 16 * (j >> 2) + frag_row<T>(j & 3, lk);
    t.v[j] = src[min(k, P.nb - 1) * (t.rows ? P.ld : 1LL)];
  }
#pragma unroll
  for (int j = 0; j < 16; j++)
    if (16 * (j >> 2) + frag_row<T>(j & 3, lk) >= P.nb) t.v[j] = T(0);
}
// inv(kb, o, k): entry (16 kb + k, 16 o + l16) of U^-1 (rows), or (16 o + l16,
// 16 kb + k) of L^-1.  The operand order leaves consecutive rows of C in
// consecutive lanes.
template <typename T, class Inv>
__device__ __forceinline__ void panel_product(const DiagProbT<T> &P, const PanelTile<T> &t, int lane, Inv inv) {
  const int l16 = lane & 15, lk = lane >> 4;
  if (t.left <= 0) return;
  const auto C = gptr(P.D + (t.rows ? P.nb + t.at : (P.nb + (long long)t.at) * P.ld));
  Frag<T> acc[4];
#pragma unroll
  for (int o = 0; o < 4; o++) acc[o] = frag_zero<T>();
#pragma unroll
  for (int kb = 0; kb < 4; kb++) {
    T w[4][4];  // (the inverse is triangular: blocks o >= kb)
#pragma unroll
    for (int o = kb; o < 4; o++)
#pragma unroll
      for (int r = 0; r < 4; r++) w[o][r] = inv(kb, o, frag_row<T>(r, lk));
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int o = kb; o < 4; o++)
        acc[o] = t.rows ? mfma4(w[o][r], t.v[4 * kb + r], acc[o]) : mfma4(t.v[4 * kb + r], w[o][r], acc[o]);
  }
#pragma unroll
  for (int o = 0; o < 4; o++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int a = frag_row<T>(r, lk);
      if (t.rows) {  // row at + l16, column 16 o + a
        if (l16 < t.left && 16 * o + a < P.nb) C[l16 + (16 * o + a) * P.ld] = acc[o][r];
      } else {  // row 16 o + l16, column at + a
        if (a < t.left && 16 * o + l16 < P.nb) C[16 * o + l16 + a * P.ld] = acc[o][r];
      }
    }
}
template <typename T>
__device__ __forceinline__ int find_tile(const DiagProbT<T> *__restrict__ probs, int nprob, int tile) {
  int lo = 0, hi = nprob - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (probs[mid].tile0 <= tile) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}
// One block per workgroup.
template <typename T>
__global__ __launch_bounds__(256, 3) void k_diag_lu(const DiagProbT<T> *__restrict__ probs) {
  __shared__ DiagLds<T> S;
  __builtin_amdgcn_s_setprio(3);  // (before waves of Schur updates on the same CU: 14.0 -> 13.8 ms, 56^3 FP32)
  const DiagProbT<T> P = probs[blockIdx.x];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  factor_block(S, P, lane, wave, true);
  store_block(S, P, lane, wave, true, true);
}
// One panel tile per workgroup, which factors the block for itself first (the
// problem's first ones store it).
template <typename T>
__global__ __launch_bounds__(256, 3) void k_diag_panel(const DiagProbT<T> *__restrict__ probs, int nprob) {
  __shared__ DiagLds<T> S;
  __builtin_amdgcn_s_setprio(3);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const DiagProbT<T> P = probs[find_tile(probs, nprob, blockIdx.x)];
  const int q = blockIdx.x - P.tile0, l16 = lane & 15;
  PanelTile<T> t = {};
  load_panel(t, P, q, lane, wave);
  factor_block(S, P, lane, wave, q == 0);
  // every wave holds its part of the tile before any overwrites it
#pragma unroll
  for (int j = 0; j < 16; j++) asm volatile("" : "+v"(t.v[j]));
  __syncthreads();
  if (t.rows)
    panel_product(P, t, lane, [&](int kb, int o, int k) { return S.A[16 * o + l16][16 * kb + k]; });
  else
    panel_product(P, t, lane, [&](int kb, int o, int k) { return kb == o ? S.Xd[o][k][l16] : S.A[16 * kb + k][16 * o + l16]; });
  // (L^-1 by the first, U^-1 by the second if there are panels)
  if (q <= (P.m > 0)) store_block(S, P, lane, wave, q == 0, q == 1 || P.m == 0);
}
// One panel tile per workgroup, by the stored inverse.
template <typename T>
__global__ __launch_bounds__(256) void k_panel(const DiagProbT<T> *__restrict__ probs, int nprob) {
  __shared__ T W[64][65];  // the inverse that the tile takes, [column][row]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const DiagProbT<T> P = probs[find_tile(probs, nprob, blockIdx.x)];
  if (P.m == 0) return;
  const int l16 = lane & 15;
  PanelTile<T> t = {};
  load_panel(t, P, blockIdx.x - P.tile0, lane, wave);
  const auto inv = gptr((const T *)(t.rows ? P.Uinv : P.Linv));
  T w[16];
#pragma unroll
  for (int q = 0; q < 16; q++) w[q] = inv[min(lane, P.nb - 1) + min(wave + 4 * q, P.nb - 1) * P.ldi];
#pragma unroll
  for (int q = 0; q < 16; q++) {
    const int c = wave + 4 * q;
    W[c][lane] = lane < P.nb && c < P.nb ? w[q] : (lane == c ? T(1) : T(0));
  }
#pragma unroll
  for (int j = 0; j < 16; j++) asm volatile("" : "+v"(t.v[j]));
  __syncthreads();
  if (t.rows)
    panel_product(P, t, lane, [&](int kb, int o, int k) { return W[16 * o + l16][16 * kb + k]; });
  else
    panel_product(P, t, lane, [&](int kb, int o, int k) { return W[16 * kb + k][16 * o + l16]; });
}
// A step's blocks and panels as one launch, every panel workgroup factoring
// its block for itself, while the launch has at most one workgroup per CU (256).
// The chain of a factorization's upper levels is a sequence of such steps: 22
// us FP64 and 18.5 us FP32 each, against 19 / 16 for the blocks and 8 to 10
// more for a launch of the panels.  With more panel tiles the blocks are
// factored once each first.  The product is the same code on the same values
// either way.
template <typename T>
void launch_diag_lu(const DiagProbT<T> *probs, int nprob, int tiles, hipStream_t st) {
  if (nprob <= 0) return;
  constexpr int kFused = 256;
  if (tiles > 0 && tiles <= kFused) {
    hipLaunchKernelGGL(k_diag_panel<T>, dim3(tiles), dim3(256), 0, st, probs, nprob);
    return;
  }
  hipLaunchKernelGGL(k_diag_lu<T>, dim3(nprob), dim3(256), 0, st, probs);
  if (tiles > 0) hipLaunchKernelGGL(k_panel<T>, dim3(tiles), dim3(256), 0, st, probs, nprob);
}

// ---------------------------------------------------------------------------
// FP64 iterative refinement around the FP32 factors (original CSR order)
// ---------------------------------------------------------------------------
// One matrix per blockIdx.y throughout; FP64 arithmetic.
static unsigned ir_blocks(long long rows_x_lanes) {
  long long b = (rows_x_lanes + 255) / 256;
  return (unsigned)std::max(1LL, std::min(b, 1024LL));
}
__device__ __forceinline__ double block_max(double v, double *red) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
  if (lane == 0) red[w] = v;
  __syncthreads();
  v = red[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); i++) v = fmax(v, red[i]);
  return v;
}
// Maximum of |v| that takes a NaN for an infinity (fmax alone would leave it
// out, and a solution of NaNs pass for an exact one): the largest high word
// tells, which is cheaper per value than a comparison in FP64.
struct NormMax {
  double m = 0.0;
  unsigned hi = 0;
  __device__ __forceinline__ void add(double v) {
    m = fmax(m, fabs(v));
    hi = max(hi, (unsigned)__double2hiint(v) & 0x7fffffffu);
  }
  __device__ __forceinline__ double value() const { return hi < 0x7ff00000u ? m : HUGE_VAL; }
};
// r = b - A x, rounded to T straight into the packed vectors (the next
// sweep's right-hand sides, so no FP64 residual goes through memory), and the
// column maxima of |b|, |r| and |x| in the same pass: each workgroup stores its
// own, k_norm_max combines them (atomic maxima from all workgroups queue up on
// a few cache lines: six packed matrices 230 -> 184 us).  One column: 8 lanes
// per row.  Several: a lane is a row, 8 columns at a time, so every load covers
// 512 contiguous bytes of one column and A's entries are read once per 8
// columns (16 rows x 4 columns per load: 1.18 ms against 0.84 for 1000^2
// 5-point with 64 columns; 0.69 now).  As separate passes, column by column, the same
// work took 2.58 ms for the residual and 2 x 0.39 ms for the norms; the
// vectors alone (1.3 GB) take 0.25 ms.
template <typename T>
__global__ __launch_bounds__(256) void k_residual(const IrDev *__restrict__ tab, const VecDev *__restrict__ vd,
                                                  T *__restrict__ bp, double *__restrict__ part, int nslots) {
  __shared__ double red[3][4][kColGroup];
  const IrDev M = tab[blockIdx.y];
  const VecDev V = vd[M.vec];
  const int nblk = gridDim.x;
  T *out = bp + V.base;
  const auto rowptr = gptr(M.rowptr), colidx = gptr(M.colidx), order = gptr(M.order);
  const auto val = gptr(M.val), x = gptr(M.x), rhs = gptr(M.b);
  const int sub = threadIdx.x & 7, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long long first = ((long long)blockIdx.x * 256 + threadIdx.x) >> 3, step = ((long long)gridDim.x * 256) >> 3;
  if (M.nrhs == 1) {
    NormMax nb, nr;
    double mx = 0.0;
    for (long long row = first; row < M.n; row += step) {
      const int p0 = rowptr[row], p1 = rowptr[row + 1];
      double s = 0.0;
      for (int p = p0 + sub; p < p1; p += 8) s += val[p] * x[colidx[p]];
      s += __shfl_xor(s, 1, 8);
      s += __shfl_xor(s, 2, 8);
      s += __shfl_xor(s, 4, 8);
      if (sub == 0) {
        const double b = rhs[row], r = b - s;
        out[order[row]] = (T)r;
        nb.add(b);
        nr.add(r);
        mx = fmax(mx, fabs(x[row]));
      }
    }
    double *rd = &red[0][0][0];
    const double mb = block_max(nb.value(), rd), mr = block_max(nr.value(), rd);
    mx = block_max(mx, rd);
    if (threadIdx.x == 0) {
      part[(long long)M.norm0 * nblk + blockIdx.x] = mb;
      part[((long long)nslots + M.norm0) * nblk + blockIdx.x] = mr;
      part[(2LL * nslots + M.norm0) * nblk + blockIdx.x] = mx;
    }
    return;
  }
  // consecutive rows per workgroup, and consecutive workgroups of one XCD (ids
  // go round-robin over the 8) on consecutive rows: neighbouring rows share
  // their x entries in that XCD's L2
  constexpr int NC = 8;
  const int nw = gridDim.x & ~7, wg = (int)blockIdx.x < nw ? (blockIdx.x & 7) * (nw >> 3) + (blockIdx.x >> 3) : blockIdx.x;
  const int chunk = (M.n + gridDim.x - 1) / gridDim.x;
  const int row_end = min((long long)M.n, (long long)(wg + 1) * chunk);
  for (int c0 = 0; c0 < M.nrhs; c0 += NC) {
    T *oc = out + (long long)(c0 / kColGroup) * V.n * kColGroup + c0 % kColGroup;
    NormMax nb[NC], nr[NC];
    double m[3][NC];
#pragma unroll
    for (int c = 0; c < NC; c++) m[2][c] = 0.0;
    for (int row = wg * chunk + threadIdx.x; row < row_end; row += 256) {
      const int p0 = rowptr[row], p1 = rowptr[row + 1];
      T *o = oc + (long long)order[row] * kColGroup;
      double b[NC], xr[NC], s[NC];
#pragma unroll
      for (int c = 0; c < NC; c++) {
        const long long cc = min(c0 + c, M.nrhs - 1);
        b[c] = rhs[row + cc * M.ldb];
        xr[c] = x[row + cc * M.ldx];
        s[c] = 0.0;
      }
      for (int p = p0; p < p1; p++) {
        const double v = val[p];
        const auto xi = x + colidx[p];
#pragma unroll
        for (int c = 0; c < NC; c++) s[c] += v * xi[min(c0 + c, M.nrhs - 1) * M.ldx];
      }
#pragma unroll
      for (int c = 0; c < NC; c++) {
        const double r = b[c] - s[c];
        o[c] = c0 + c < M.nrhs ? (T)r : T(0);
        nb[c].add(b[c]);
        nr[c].add(r);
        m[2][c] = fmax(m[2][c], fabs(xr[c]));
      }
    }
#pragma unroll
    for (int c = 0; c < NC; c++) m[0][c] = nb[c].value(), m[1][c] = nr[c].value();
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
      for (int c = 0; c < NC; c++) {
        for (int o = 1; o < 64; o <<= 1) m[q][c] = fmax(m[q][c], __shfl_xor(m[q][c], o, 64));
        if (lane == 0) red[q][wave][c] = m[q][c];
      }
    __syncthreads();
    if (threadIdx.x < 3 * NC) {
      const int c = threadIdx.x % NC, q = threadIdx.x / NC;
      if (c0 + c < M.nrhs)
        part[((long long)q * nslots + M.norm0 + c0 + c) * nblk + blockIdx.x] =
            fmax(fmax(red[q][0][c], red[q][1][c]), fmax(red[q][2][c], red[q][3][c]));
    }
  }
}
// norms[s] = max of the workgroups' values part[s nblk ...]
__global__ __launch_bounds__(256) void k_norm_max(const double *__restrict__ part, int nblk,
                                                  double *__restrict__ norms) {
  __shared__ double red[4];
  double m = 0.0;
  for (int i = threadIdx.x; i < nblk; i += 256) m = fmax(m, part[(long long)blockIdx.x * nblk + i]);
  m = block_max(m, red);
  if (threadIdx.x == 0) norms[blockIdx.x] = m;
}
int residual_blocks(int nmat, int max_n) {
  const long long want = (8LL * max_n + 255) / 256;
  return (int)std::max(1LL, std::min(want, (long long)std::max(16, kResidualBlocks / std::max(1, nmat))));
}
template <typename T>
void launch_residual(const IrDev *tab, const VecDev *vd, int nmat, int max_n, T *bp, double *norms, int nslots,
                     hipStream_t st) {
  if (nmat <= 0 || max_n <= 0 || nslots <= 0) return;
  const int nblk = residual_blocks(nmat, max_n);
  double *part = norms + 3LL * nslots;
  hipLaunchKernelGGL(k_residual<T>, dim3(nblk, nmat), dim3(256), 0, st, tab, vd, bp, part, nslots);
  hipLaunchKernelGGL(k_norm_max, dim3(3 * nslots), dim3(256), 0, st, part, nblk, norms);
}
template void launch_residual<float>(const IrDev *, const VecDev *, int, int, float *, double *, int, hipStream_t);
// Plain streaming copy (16 B per lane per iteration): the reference kernel
// for scaling the HBM byte counters.
__global__ __launch_bounds__(256) void k_copy(const double2 *__restrict__ src,
                                              double2 *__restrict__ dst, long long n) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    dst[i] = src[i];
}
void launch_copy(const void *src, void *dst, long long bytes, hipStream_t st) {
  const long long n = bytes / 16;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_copy, dim3(4096), dim3(256), 0, st, (const double2 *)src, (double2 *)dst, n);
}
__global__ void k_zero_u64(unsigned long long *p, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0ull;
}
// out[matrix] = max_i sum_j |A_ij|
__global__ __launch_bounds__(256) void k_rowabs_max(const IrDev *__restrict__ tab,
                                                    unsigned long long *out) {
  __shared__ double red[4];
  const IrDev M = tab[blockIdx.y];
  const auto rowptr = gptr(M.rowptr);
  const auto val = gptr(M.val);
  double m = 0.0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < M.n;
       i += (long long)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int p = rowptr[i]; p < rowptr[i + 1]; p++) s += fabs(val[p]);
    m = fmax(m, s);
  }
  m = block_max(m, red);
  if (threadIdx.x == 0) atomicMax(out + blockIdx.y, (unsigned long long)__double_as_longlong(m));
}
void launch_rowabs_max(const IrDev *tab, int nmat, int max_n, unsigned long long *out,
                       hipStream_t st) {
  if (nmat <= 0) return;
  hipLaunchKernelGGL(k_zero_u64, dim3((nmat + 255) / 256), dim3(256), 0, st, out, nmat);
  if (max_n <= 0) return;
  hipLaunchKernelGGL(k_rowabs_max, dim3(ir_blocks(max_n), nmat), dim3(256), 0, st, tab, out);
}
// The scatter alone, for a set of matrices (one per blockIdx.y): zero the
// separators' blocks, then put A's separator entries into place.  (A
// factorization writes every tile of them in k_extend_add.)
template <typename T>
__global__ void k_prep_fill(const PrepDev *__restrict__ tab) {
  const PrepDev M = tab[blockIdx.y];
  const auto a = gptr((T *)M.arena);
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < M.arena_len; i += stride)
    a[i] = T(0);
}
template <typename T>
__global__ void k_prep_scatter(const PrepDev *__restrict__ tab) {
  const PrepDev M = tab[blockIdx.y];
  const auto a = gptr((T *)M.arena);
  const auto dest = gptr(M.adest);
  const auto src = gptr(M.asrc);
  const auto aval = gptr(M.aval);
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < M.nnz;
       i += (long long)gridDim.x * blockDim.x)
    a[dest[i]] = (T)aval[src[i]];
}
template <typename T>
void launch_prepare(const PrepDev *tab, int nmat, long long max_len, long long max_nnz,
                    hipStream_t st) {
  if (nmat <= 0) return;
  auto blocks = [](long long n) {
    return (unsigned)std::max(1LL, std::min((n + 255) / 256, 4096LL));
  };
  hipLaunchKernelGGL(k_prep_fill<T>, dim3(blocks(max_len), nmat), dim3(256), 0, st, tab);
  hipLaunchKernelGGL(k_prep_scatter<T>, dim3(blocks(max_nnz), nmat), dim3(256), 0, st, tab);
}



// ---- explicit instantiations: FP64 and FP32 value paths ----
#define SNU_INSTANTIATE(T)                                                                    \
  template void launch_fill<T>(T *, long long, hipStream_t);                                  \
  template void launch_prepare<T>(const PrepDev *, int, long long, long long, hipStream_t);   \
  template void launch_copy2d<T>(const GemmProbT<T> *, int, const GemmSegT<T> *, int, hipStream_t); \
  template void launch_gemm<T>(const GemmProbT<T> *, int, const GemmSegT<T> *, int, int,     \
                               hipStream_t);                                                  \
  template void launch_gemm128<T>(const GemmProbT<T> *, int, const GemmSegT<T> *, int, int,  \
                                  hipStream_t);                                               \
  template void launch_gemm_variant<T>(const GemmProbT<T> *, int, const GemmSegT<T> *, int,  \
                                       int, int, int, hipStream_t);                           \
  template void launch_diag_lu<T>(const DiagProbT<T> *, int, int, hipStream_t);
SNU_INSTANTIATE(double)
SNU_INSTANTIATE(float)
#undef SNU_INSTANTIATE

}  // namespace snu
