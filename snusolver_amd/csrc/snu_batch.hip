// Batches of independent matrices factorized and solved together: every
// step runs as one launch across all of them.  The leaves of all matrices
// share the leaf launches; separators of equal tree height (counted from
// the leaves, so trees of different depths align at the bottom) share one
// grouped launch per step of the dense level loop; solves pack the
// right-hand sides of all matrices, each with its own column count, into one
// buffer and run one launch per sweep step and tree height.
//
// No reference counterpart (the reference factorizes one matrix per MPI
// job); each matrix's arithmetic is unchanged, so its factors and solutions
// equal those of a standalone factorization and solve.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <string>
#include <vector>

#include "snu_engine.h"

using namespace snu;

struct snubatch {
  std::vector<snumat *> mats;
  int prec = SNU_FP64, device = 0;
  hipStream_t stream = nullptr;
  std::vector<void *> allocs;
  // factor set
  WorkDev wd;
  IrDev *d_ir_a = nullptr;  // |A| norm tables (FP32)
  unsigned long long *d_anorm = nullptr;
  int max_n = 0;
  DensePlan<double> f64;
  DensePlan<float> f32;
  FrontPlan<double> fr64;  // the members' leaf fronts, merged per height
  FrontPlan<float> fr32;
  // solves (sized for the last right-hand-side pattern)
  std::vector<int> pattern;  // nrhs per matrix of the current solve plan
  long long vec_cap = 0, y_cap = 0, w_cap = 0;
  int slot_cap = 0;
  void *bp = nullptr, *ys = nullptr, *wbuf = nullptr;
  double *norms = nullptr;
  int *d_active = nullptr;
  VecDev *d_vec = nullptr;
  PermDev *d_perm = nullptr;
  IrDev *d_ir = nullptr;
  GemvPlan<double> s64;
  GemvPlan<float> s32;
  std::vector<VecDev> h_vec;
  std::vector<double> anorm;
  int ir_steps = 0;
  std::vector<double> berr;
  std::vector<char> twin;  // members answered by FP64 factors
  double *stage = nullptr;  // host-pointer solves: packed b then x
  size_t stage_cap = 0;
  bool factor_plan = false;  // merged dense plan built (on first factorize)
  bool use_graph = false;
  FactorGraph graph;
  SideStream side;
  std::vector<hipEvent_t> ev;
  double t[16] = {0};
};

namespace {

int balloc(snubatch *b, void **p, size_t bytes) {
  *p = nullptr;
  const hipError_t e = bytes > b->mats[0]->alloc_limit ? hipErrorOutOfMemory : hipMalloc(p, std::max<size_t>(1, bytes));
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();  // (reported here; the next launch's check must not see it)
    return set_error(SNU_ERR_OOM, std::string("batch allocation failed: ") + hipGetErrorString(e));
  }
  b->allocs.push_back(*p);
  return SNU_OK;
}
template <class T>
int bupload(snubatch *b, T **p, const std::vector<T> &v) {
  int rc = balloc(b, (void **)p, v.size() * sizeof(T));
  if (rc) return rc;
  if (!v.empty()) HIPCHK(hipMemcpy(*p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return SNU_OK;
}
void bfree(snubatch *b, void *p) {
  if (!p) return;
  auto it = std::find(b->allocs.begin(), b->allocs.end(), p);
  if (it != b->allocs.end()) b->allocs.erase(it);
  (void)hipFree(p);
}
void free_batch(snubatch *b) {
  free_graph(b->graph);
  free_dense_plan(b->f64);
  free_dense_plan(b->f32);
  free_dense_plan(b->fr64.dense);
  free_dense_plan(b->fr32.dense);
  free_gemv_plan(b->s64);
  free_gemv_plan(b->s32);
  for (void *p : b->allocs) (void)hipFree(p);
  b->allocs.clear();
  for (hipEvent_t e : b->ev) (void)hipEventDestroy(e);
  b->ev.clear();
  free_side(b->side);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  b->stream = nullptr;
}

// What only factorizations need, on the first one: a batch that solves alone (a
// server forms them per pack) does without.
template <typename T>
int build_factor_set(snubatch *b) {
  std::vector<const DensePlan<T> *> parts;
  for (snumat *h : b->mats) parts.push_back(&vals<T>(h).fact);
  DensePlan<T> &out = std::is_same<T, double>::value ? (DensePlan<T> &)b->f64 : (DensePlan<T> &)b->f32;
  merge_dense(parts, out);
  int rc = upload_dense_plan(out);
  if (rc) return rc;
  // the members' leaf fronts, merged per height (descriptors point into the
  // members' own arrays)
  FrontPlan<T> &fp = std::is_same<T, double>::value ? (FrontPlan<T> &)b->fr64 : (FrontPlan<T> &)b->fr32;
  std::vector<const FrontPlan<T> *> fronts;
  for (snumat *h : b->mats) fronts.push_back(&vals<T>(h).fronts);
  merge_fronts(fronts, fp);
  if ((rc = upload_dense_plan(fp.dense)) || (rc = bupload(b, &fp.d_small, fp.small)) ||
      (rc = bupload(b, &fp.d_tiles, fp.tiles)) || (rc = bupload(b, &fp.d_src, fp.src)))
    return rc;
  // both streams anew, one after the other (see SideStream)
  if (b->stream) {
    HIPCHK(hipStreamSynchronize(b->stream));
    HIPCHK(hipStreamDestroy(b->stream));
    b->stream = nullptr;
  }
  HIPCHK(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
  return make_side<T>(parts, b->side);
}

// Solve plan and buffers for a right-hand-side pattern (columns per matrix;
// 0 skips a matrix).
template <typename T>
int ensure_pattern(snubatch *b, const std::vector<int> &nrhs) {
  if (b->pattern == nrhs) return SNU_OK;
  const int nm = (int)b->mats.size();
  // packed vectors (padded column groups; ys: separator rows), update rows
  long long tot = 0, ytot = 0, wtot = 0;
  int slots = 0;
  for (int m = 0; m < nm; m++) {
    const long long cols = (long long)vec_groups(nrhs[m]) * vec_width(nrhs[m]);
    tot += (long long)b->mats[m]->P.n * cols;
    ytot += (long long)b->mats[m]->sep_rows[b->mats[m]->P.np] * cols;
    wtot += (long long)b->mats[m]->wrows * cols;
    slots += nrhs[m];
  }
  int rc;
  b->pattern.clear();
  if (tot > b->vec_cap) {
    bfree(b, b->bp);
    b->bp = nullptr;
    b->vec_cap = 0;
    if ((rc = balloc(b, &b->bp, sizeof(T) * tot))) return rc;
    b->vec_cap = tot;
  }
  if (ytot > b->y_cap) {
    bfree(b, b->ys);
    b->ys = nullptr;
    b->y_cap = 0;
    if ((rc = balloc(b, &b->ys, sizeof(T) * ytot))) return rc;
    b->y_cap = ytot;
  }
  if (wtot > b->w_cap) {
    bfree(b, b->wbuf);
    b->wbuf = nullptr;
    b->w_cap = 0;
    if ((rc = balloc(b, &b->wbuf, sizeof(T) * (size_t)wtot))) return rc;
    b->w_cap = wtot;
  }
  if (slots > b->slot_cap) {
    bfree(b, b->norms);
    b->norms = nullptr;
    b->slot_cap = 0;
    if ((rc = balloc(b, (void **)&b->norms, sizeof(double) * norm_values(nm, b->max_n, slots)))) return rc;
    b->slot_cap = slots;
  }
  b->h_vec.assign(nm, VecDev());
  long long base = 0, wbase = 0;
  for (int m = 0; m < nm; m++) {
    const snumat *h = b->mats[m];
    const long long cols = (long long)vec_groups(nrhs[m]) * vec_width(nrhs[m]);
    b->h_vec[m] = VecDev{base, wbase, h->P.n, nrhs[m], h->wrows, 0};
    base += (long long)h->P.n * cols;
    wbase += (long long)h->wrows * cols;
  }
  HIPCHK(hipMemcpyAsync(b->d_vec, b->h_vec.data(), sizeof(VecDev) * nm, hipMemcpyHostToDevice, b->stream));
  GemvPlan<T> &out = std::is_same<T, double>::value ? (GemvPlan<T> &)b->s64 : (GemvPlan<T> &)b->s32;
  std::vector<GemvPlan<T>> parts(nm);
  std::vector<const GemvPlan<T> *> ptrs;
  T *bp = (T *)b->bp, *ys = (T *)b->ys;
  for (int m = 0; m < nm; m++) {
    if (!nrhs[m]) continue;
    build_solve_plan<T>(b->mats[m], bp + b->h_vec[m].base, ys, nrhs[m], parts[m]);
    ys += (long long)b->mats[m]->sep_rows[b->mats[m]->P.np] * vec_groups(nrhs[m]) * vec_width(nrhs[m]);
    ptrs.push_back(&parts[m]);
  }
  merge_gemv(ptrs, out);  // keeps out's device arrays, which grow only
  if ((rc = upload_gemv_plan(out, b->stream))) return rc;
  b->pattern = nrhs;
  return SNU_OK;
}

template <typename T>
int batch_factorize(snubatch *b) {
  FactorSet fs;
  fs.side = &b->side;
  fs.nmat = (int)b->mats.size();
  fs.ir = b->prec == SNU_FP32 ? b->d_ir_a : nullptr;
  fs.anorm_out = b->d_anorm;
  fs.max_n = b->max_n;
  fs.fronts = std::is_same<T, double>::value ? (const void *)&b->fr64 : (const void *)&b->fr32;
  fs.eps = b->mats[0]->opts.eps;
  fs.split = b->mats[0]->opts.fp32_gemm == SNU_GEMM_SPLIT;
  const DensePlan<T> &plan = std::is_same<T, double>::value ? (const DensePlan<T> &)b->f64
                                                            : (const DensePlan<T> &)b->f32;
  int rc = run_factor<T>(fs, plan, b->stream, &b->ev, false, nullptr, nullptr,
                         b->use_graph ? &b->graph : nullptr);
  if (rc) return rc;
  HIPCHK(hipEventSynchronize(b->ev[5]));
  for (int q = 0; q < 5; q++) b->t[q] = ev_ms(b->ev[q], b->ev[q + 1]);
  b->t[5] = ev_ms(b->ev[0], b->ev[5]);
  const int nm = (int)b->mats.size();
  b->anorm.assign(nm, 0.0);
  if (b->prec == SNU_FP32) {
    std::vector<unsigned long long> u(nm);
    HIPCHK(hipMemcpy(u.data(), b->d_anorm, sizeof(unsigned long long) * nm, hipMemcpyDeviceToHost));
    for (int m = 0; m < nm; m++) std::memcpy(&b->anorm[m], &u[m], sizeof(double));
  }
  for (int m = 0; m < nm; m++) {
    b->mats[m]->factored = true;
    b->mats[m]->scattered = false;
    b->mats[m]->fb64_current = false;  // an FP64 twin refactorizes on its next use
    b->mats[m]->anorm = b->anorm[m];
  }
  return SNU_OK;
}

// One pass over all members, on the buffers of ensure_pattern.
template <typename T>
int solve_pattern(snubatch *b, const double *const *d_b, double *const *d_x, const int *nrhs,
                  const int *ld) {
  const int nm = (int)b->mats.size();
  int rc = SNU_OK;
  hipStream_t st = b->stream;
  std::vector<PermDev> pd(nm);
  long long max_elems = 0;
  int max_groups = 0, max_n = 0;
  bool one = false, many = false;
  for (int m = 0; m < nm; m++) {
    const snumat *h = b->mats[m];
    const int n = h->P.n;
    pd[m] = PermDev{h->d_order, d_b[m], d_x[m], (long long)ld[m], (long long)ld[m], n, m};
    max_elems = std::max(max_elems, (long long)n * vec_groups(nrhs[m]));
    max_groups = std::max(max_groups, vec_groups(nrhs[m]));
    one |= nrhs[m] == 1;
    many |= nrhs[m] > 1;
    max_n = std::max(max_n, n);
  }
  HIPCHK(hipMemcpyAsync(b->d_perm, pd.data(), sizeof(PermDev) * pd.size(), hipMemcpyHostToDevice, st));
  SolveSet ss;
  ss.perm = b->d_perm;
  ss.vec = b->d_vec;
  ss.nmat = nm;
  ss.max_elems = max_elems;
  ss.max_groups = max_groups;
  ss.one = one;
  ss.many = many;
  ss.wd = &b->wd;
  HIPCHK(hipEventRecord(b->ev[6], st));
  if (b->prec == SNU_FP32) {
    std::vector<IrDev> ir(nm);
    std::vector<int> slot_mat;
    for (int m = 0; m < nm; m++) {
      const snumat *h = b->mats[m];
      IrDev &e = ir[m];
      std::memset(&e, 0, sizeof(e));
      e.rowptr = h->d_arow;
      e.colidx = h->d_acol;
      e.val = h->d_aval;
      e.b = d_b[m];
      e.x = d_x[m];
      e.order = h->d_order;
      e.vec = m;
      e.ldb = e.ldx = ld[m];
      e.n = h->P.n;
      e.nrhs = nrhs[m];
      e.norm0 = (int)slot_mat.size();
      for (int c = 0; c < nrhs[m]; c++) slot_mat.push_back(m);
    }
    HIPCHK(hipMemcpyAsync(b->d_ir, ir.data(), sizeof(IrDev) * nm, hipMemcpyHostToDevice, st));
    const snu_opts_t &o = b->mats[0]->opts;
    RefineSet rs;
    rs.sweep = ss;
    rs.ir = b->d_ir;
    rs.nmat = nm;
    rs.max_n = max_n;
    rs.norms = b->norms;
    rs.nslots = (int)slot_mat.size();
    rs.slot_mat = &slot_mat;
    b->anorm.assign(nm, 0.0);  // |A| of each member, from its last factorization
    for (int m = 0; m < nm; m++) b->anorm[m] = b->mats[m]->anorm;
    rs.anorm = &b->anorm;
    rs.d_active = b->d_active;
    rs.max_steps = o.ir_max_steps > 0 ? o.ir_max_steps : o.ir_max_steps < 0 ? 0 : 10;
    rs.tol = o.ir_tol > 0 ? o.ir_tol : 1e-15;
    rc = run_refined(rs, (float *)b->bp, (float *)b->wbuf, b->s32, st, &b->ir_steps, &b->berr);
    if (rc && rc != SNU_ERR_NOT_CONVERGED) return rc;
    if (rc == SNU_ERR_NOT_CONVERGED) {
      // members whose refinement stalled above 1e-12 are answered by FP64
      // factors of the same matrix (each member's FP64 twin); the batch's
      // own work is complete (run_refined has read the final norms back)
      for (int m = 0; m < nm; m++) {
        if (!nrhs[m] || b->berr[m] <= 1e-12) continue;
        if ((rc = fp64_fallback_solve(b->mats[m], d_b[m], ld[m], d_x[m], ld[m], nrhs[m]))) return rc;
        b->twin[m] = 1;
      }
      HIPCHK(hipSetDevice(b->device));
      rc = SNU_OK;
    }
  } else {
    run_solve<double>(ss, (double *)b->bp, (double *)b->wbuf, b->s64, st);
    b->ir_steps = 0;
    b->berr.assign(nm, 0.0);
  }
  HIPCHK(hipGetLastError());
  HIPCHK(hipEventRecord(b->ev[7], st));
  HIPCHK(hipEventSynchronize(b->ev[7]));
  b->t[6] = ev_ms(b->ev[6], b->ev[7]);
  return rc;
}
// Several columns of a member are padded to groups of 16 (vec_groups): where the
// memory for that is not there, one column of each member after the other.
template <typename T>
int batch_solve(snubatch *b, const double *const *d_b, double *const *d_x, const int *nrhs,
                const int *ld) {
  const int nm = (int)b->mats.size(), most = *std::max_element(nrhs, nrhs + nm);
  b->twin.assign(nm, 0);
  int rc = ensure_pattern<T>(b, std::vector<int>(nrhs, nrhs + nm)), steps = 0;
  double ms = 0;
  std::vector<double> berr(nm, 0.0);
  auto pass = [&](const double *const *pb, double *const *px, const int *k) -> int {
    const int r = solve_pattern<T>(b, pb, px, k, ld);
    steps = std::max(steps, b->ir_steps);
    for (int m = 0; m < nm && m < (int)b->berr.size(); m++) berr[m] = std::max(berr[m], b->berr[m]);
    ms += b->t[6];
    return r;
  };
  if (!rc) {
    rc = pass(d_b, d_x, nrhs);
  } else if (rc == SNU_ERR_OOM && most > 1) {
    std::vector<const double *> pb(d_b, d_b + nm);
    std::vector<double *> px(d_x, d_x + nm);
    std::vector<int> k(nm);
    for (int c = 0; c < most; c++) {
      for (int m = 0; m < nm; m++) {
        k[m] = nrhs[m] > c;
        if (k[m] && c) pb[m] += ld[m], px[m] += ld[m];
      }
      if ((rc = ensure_pattern<T>(b, k)) || (rc = pass(pb.data(), px.data(), k.data()))) return rc;
    }
  }
  if (rc) return rc;
  b->ir_steps = steps;
  b->berr = berr;
  b->t[6] = ms;
  b->t[13] = steps;
  b->t[14] = *std::max_element(berr.begin(), berr.end());
  b->t[15] = std::accumulate(b->twin.begin(), b->twin.end(), 0);
  return SNU_OK;
}

}  // namespace

extern "C" int snubatch_create(snumat_t *const *mats, int count, snubatch_t **out) {
  if (!out || !mats || count < 1) return set_error(SNU_ERR_BAD_INPUT, "bad batch arguments");
  *out = nullptr;
  for (int m = 0; m < count; m++) {
    if (!mats[m] || !mats[m]->on_device) return set_error(SNU_ERR_BAD_INPUT, "batch member not on a device");
    if (mats[m]->prec != mats[0]->prec || mats[m]->device != mats[0]->device ||
        (mats[m]->prec == SNU_FP32 && mats[m]->opts.fp32_gemm != mats[0]->opts.fp32_gemm))
      return set_error(SNU_ERR_BAD_INPUT, "batch members must share device, precision and FP32 GEMM form");
    for (int q = 0; q < m; q++)
      if (mats[q] == mats[m]) return set_error(SNU_ERR_BAD_INPUT, "matrix listed twice in a batch");
  }
  snubatch *b = new snubatch();
  b->mats.assign(mats, mats + count);
  b->prec = mats[0]->prec;
  b->device = mats[0]->device;
  auto fail = [&](int rc) {
    free_batch(b);
    delete b;
    return rc;
  };
  hipError_t he = hipSetDevice(b->device);
  if (he == hipSuccess) he = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking);
  if (he != hipSuccess) return fail(set_error(SNU_ERR_HIP, hipGetErrorString(he)));
  b->ev.resize(8);
  for (auto &e : b->ev)
    if (hipEventCreate(&e) != hipSuccess) return fail(set_error(SNU_ERR_HIP, "event creation failed"));
  // concatenated leaves and work lists
  std::vector<LeafDev> leaves;
  WorkLists W;
  std::vector<IrDev> ira;
  for (int m = 0; m < count; m++) {
    snumat *h = b->mats[m];
    const int sbase = (int)W.tsrc.size();
    for (LeafDev L : h->h_leaves) {
      L.vec = m;
      leaves.push_back(L);
    }
    const WorkLists &w = h->wl;
    for (TargetDev t : w.targets) W.targets.push_back(TargetDev{t.row, sbase + t.s0, sbase + t.s1, m});
    W.tsrc.insert(W.tsrc.end(), w.tsrc.begin(), w.tsrc.end());
    IrDev e;
    std::memset(&e, 0, sizeof(e));
    e.rowptr = h->d_arow;
    e.colidx = h->d_acol;
    e.val = h->d_aval;
    e.n = h->P.n;
    ira.push_back(e);
    b->max_n = std::max(b->max_n, h->P.n);
  }
  WorkDev &wd = b->wd;
  wd.nleaves = (int)leaves.size();
  wd.ntarget = (int)W.targets.size();
  int rc;
  if ((rc = bupload(b, &wd.leaves, leaves)) || (rc = bupload(b, &wd.targets, W.targets)) ||
      (rc = bupload(b, &wd.tsrc, W.tsrc)) ||
      (rc = bupload(b, &b->d_ir_a, ira)))
    return fail(rc);
  if ((rc = balloc(b, (void **)&b->d_anorm, sizeof(unsigned long long) * count)) ||
      (rc = balloc(b, (void **)&b->d_active, sizeof(int) * count)) ||
      (rc = balloc(b, (void **)&b->d_vec, sizeof(VecDev) * count)) ||
      (rc = balloc(b, (void **)&b->d_perm, sizeof(PermDev) * count)) ||
      (rc = balloc(b, (void **)&b->d_ir, sizeof(IrDev) * count)))
    return fail(rc);
  *out = b;
  return SNU_OK;
}

extern "C" int snubatch_factorize(snubatch_t *b) {
  if (!b) return set_error(SNU_ERR_BAD_INPUT, "null batch");
  HIPCHK(hipSetDevice(b->device));
  if (!b->factor_plan) {
    int rc = b->prec == SNU_FP32 ? build_factor_set<float>(b) : build_factor_set<double>(b);
    if (rc) return rc;
    b->factor_plan = true;
  }
  for (snumat *h : b->mats) h->factored = false;
  return b->prec == SNU_FP32 ? batch_factorize<float>(b) : batch_factorize<double>(b);
}

extern "C" int snubatch_solve_device(snubatch_t *b, const double *const *d_b, double *const *d_x,
                                     const int *nrhs, const int *ld) {
  if (!b || !d_b || !d_x || !nrhs || !ld) return set_error(SNU_ERR_BAD_INPUT, "bad batch solve arguments");
  const int nm = (int)b->mats.size();
  for (int m = 0; m < nm; m++) {
    if (nrhs[m] < 0 || (nrhs[m] > 0 && (!d_b[m] || !d_x[m] || ld[m] < b->mats[m]->P.n || d_b[m] == d_x[m])))
      return set_error(SNU_ERR_BAD_INPUT, "bad batch solve arguments for matrix " + std::to_string(m));
    if (nrhs[m] > 0 && !b->mats[m]->factored)
      return set_error(SNU_ERR_NOT_FACTORED, "batch member not factored");
  }
  HIPCHK(hipSetDevice(b->device));
  return b->prec == SNU_FP32 ? batch_solve<float>(b, d_b, d_x, nrhs, ld)
                             : batch_solve<double>(b, d_b, d_x, nrhs, ld);
}

extern "C" int snubatch_solve(snubatch_t *b, const double *const *hb, double *const *hx,
                              const int *nrhs, const int *ld) {
  if (!b || !hb || !hx || !nrhs || !ld) return set_error(SNU_ERR_BAD_INPUT, "bad batch solve arguments");
  const int nm = (int)b->mats.size();
  HIPCHK(hipSetDevice(b->device));
  size_t tot = 0;
  for (int m = 0; m < nm; m++) {
    if (nrhs[m] < 0 || (nrhs[m] > 0 && (!hb[m] || !hx[m] || ld[m] < b->mats[m]->P.n)))
      return set_error(SNU_ERR_BAD_INPUT, "bad batch solve arguments for matrix " + std::to_string(m));
    tot += (size_t)b->mats[m]->P.n * nrhs[m];
  }
  if (2 * tot > b->stage_cap) {
    bfree(b, b->stage);
    b->stage = nullptr;
    b->stage_cap = 0;
    int arc = balloc(b, (void **)&b->stage, sizeof(double) * 2 * std::max<size_t>(1, tot));
    if (arc) return arc;
    b->stage_cap = 2 * std::max<size_t>(1, tot);
  }
  double *stage = b->stage;
  std::vector<const double *> db(nm, nullptr);
  std::vector<double *> dx(nm, nullptr);
  std::vector<int> dld(nm);
  size_t off = 0;
  int rc = SNU_OK;
  for (int m = 0; m < nm && !rc; m++) {
    const int n = b->mats[m]->P.n;
    dld[m] = n;
    if (!nrhs[m]) continue;
    double *pb = stage + off, *px = stage + tot + off;
    off += (size_t)n * nrhs[m];
    if (hipMemcpy2DAsync(pb, sizeof(double) * n, hb[m], sizeof(double) * ld[m], sizeof(double) * n,
                         nrhs[m], hipMemcpyHostToDevice, b->stream) != hipSuccess)
      rc = set_error(SNU_ERR_HIP, "batch rhs upload failed");
    db[m] = pb;
    dx[m] = px;
  }
  if (!rc) rc = snubatch_solve_device(b, db.data(), dx.data(), nrhs, dld.data());
  if (!rc || rc == SNU_ERR_NOT_CONVERGED) {
    for (int m = 0; m < nm; m++) {
      if (!nrhs[m]) continue;
      const int n = b->mats[m]->P.n;
      if (hipMemcpy2DAsync(hx[m], sizeof(double) * ld[m], dx[m], sizeof(double) * n, sizeof(double) * n,
                           nrhs[m], hipMemcpyDeviceToHost, b->stream) != hipSuccess) {
        rc = set_error(SNU_ERR_HIP, "batch solution download failed");
        break;
      }
    }
    if (hipStreamSynchronize(b->stream) != hipSuccess) rc = set_error(SNU_ERR_HIP, "batch solve sync failed");
  }
  return rc;
}

extern "C" int snubatch_timings(const snubatch_t *b, double *t16) {
  if (!b || !t16) return set_error(SNU_ERR_BAD_INPUT, "null");
  std::memcpy(t16, b->t, sizeof(b->t));
  return SNU_OK;
}

extern "C" int snubatch_launches(const snubatch_t *b, int *factor_launches, int *solve_launches) {
  if (!b) return set_error(SNU_ERR_BAD_INPUT, "null");
  if (factor_launches)
    *factor_launches = (int)(b->prec == SNU_FP32 ? b->f32.launches.size() : b->f64.launches.size());
  if (solve_launches)
    *solve_launches = (int)(b->prec == SNU_FP32 ? b->s32.fwd.size() + b->s32.bwd.size()
                                                : b->s64.fwd.size() + b->s64.bwd.size());
  return SNU_OK;
}

extern "C" int snubatch_use_graph(snubatch_t *b, int on) {
  if (!b) return set_error(SNU_ERR_BAD_INPUT, "null");
  b->use_graph = on != 0;
  return SNU_OK;
}

extern "C" int snubatch_destroy(snubatch_t *b) {
  if (!b) return SNU_OK;
  (void)hipSetDevice(b->device);
  free_batch(b);
  delete b;
  return SNU_OK;
}
