// Packed solve of several tilt series of uneven width, thickness, tilt count
// and slice count in the same launches.
//
// The reference solves one slice at a time per device and derives the grid,
// window and node set per series (MainCode.cu:63-71, the slice loop
// MainCode.cu:113-162).  Here every series keeps its own plan (geometry
// tables, bins, per-slice buffers), and a batch enqueues each kernel of the
// iteration once per size class instead of once per series: the row kernels
// once per row length n1, the column kernels once per (n0, tile width,
// window), the node combine once for all series.  Each packed launch reads
// the argument block of a series from a device table and the (series, block)
// pair of each of its workgroups from an item table built at batch creation.
// The whole solve is captured into one HIP graph and replayed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>
#include <tuple>
#include <vector>

#include "icon_kernels.h"
#include "icon_plan.h"

using namespace icon;

namespace {

int bfail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  std::vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  set_last_error(buf);
  return code;
}

#define BCHK(expr)                                                                               \
  do {                                                                                           \
    hipError_t e_ = (expr);                                                                      \
    if (e_ != hipSuccess)                                                                        \
      return bfail(ICON_ERR_DEVICE, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, \
                   __LINE__);                                                                    \
  } while (0)

struct Items {
  int key0 = 0, key1 = 0, key2 = 0;  // size class (meaning per kernel)
  std::vector<int2> h;
  int2* d = nullptr;
  int n() const { return (int)h.size(); }
};

struct SolveKey {
  std::vector<const void*> ptrs;
  int pre = -1, icon = -1, post = -1, data_type = 0;
  float thr = 0;
  bool operator==(const SolveKey& o) const {
    return ptrs == o.ptrs && pre == o.pre && icon == o.icon && post == o.post && data_type == o.data_type &&
           thr == o.thr;
  }
};

}  // namespace

struct icon_batch {
  int device = 0;
  std::vector<icon_plan*> plans;
  std::vector<int> S;
  hipStream_t stream = nullptr;
  hipEvent_t ev_in = nullptr, ev_out = nullptr;
  // item tables per size class
  std::vector<Items> row_fwd, row_adj, sino, reproj;
  // the data adjoint's spread: items by their tile's entry count, largest first
  // across the class's series (each tile's blocks stay together)
  std::vector<Items> col_adj;
  std::vector<Items> normal;   // the normal operator's column kernels, by n0
  std::vector<Items> row_grad;
  // FP64 passes over up to S64 slices of a series (key2: which): rows (or pairs) and
  // columns; argument block pass * nseries + series
  std::vector<Items> row64, normal64;
  Items combine;
  // argument blocks, one per series (device copies written before each solve)
  std::vector<RowFwdArgs> h_rf;
  std::vector<RowAdjArgs> h_ra;
  std::vector<ColArgs> h_ca;
  std::vector<CombineArgs> h_cm;
  std::vector<SinoArgs> h_sa;
  std::vector<ReprojArgs> h_rp;
  std::vector<RowAdjArgs> h_rg, h_rg2;     // gradient; ... against the reference iterate
  std::vector<RowFwdArgs> h_rf2, h_rr;     // row pass against the reference iterate; of rhat
  std::vector<RefArgs> h_re;
  std::vector<ColArgs> h_c64;
  std::vector<ColArgs> h_cn, h_ce, h_cl;   // normal operator; energy; last forward pass
  std::vector<FinishArgs> h_fa;
  RowFwdArgs* d_rf = nullptr;
  RowAdjArgs* d_ra = nullptr;
  ColArgs* d_ca = nullptr;
  CombineArgs* d_cm = nullptr;
  SinoArgs* d_sa = nullptr;
  ReprojArgs* d_rp = nullptr;
  RowAdjArgs *d_rg = nullptr, *d_rg2 = nullptr;
  RowFwdArgs *d_rf2 = nullptr, *d_rr = nullptr;
  RefArgs* d_re = nullptr;
  ColArgs* d_c64 = nullptr;
  ColArgs *d_cn = nullptr, *d_ce = nullptr, *d_cl = nullptr;
  FinishArgs* d_fa = nullptr;
  hipGraphExec_t graph = nullptr;
  SolveKey graph_key;
};

namespace {

void free_items(std::vector<Items>& v) {
  for (auto& it : v)
    if (it.d) (void)hipFree(it.d);
  v.clear();
}

int upload_items(Items& it) {
  if (it.d) (void)hipFree(it.d);
  it.d = nullptr;
  if (it.h.empty()) return ICON_OK;
  BCHK(hipMalloc(&it.d, sizeof(int2) * it.h.size()));
  BCHK(hipMemcpy(it.d, it.h.data(), sizeof(int2) * it.h.size(), hipMemcpyHostToDevice));
  return ICON_OK;
}

// Slices that a series of S takes in one pass of its data adjoint and FP64
// gradient; kPasses passes at most.
constexpr int kPasses = 2;
int pass_slices(const icon_plan* p, int S) { return p->refreshes() ? p->S64 : S; }

// (series, block) items of every size class, built once: they depend on the
// tables that a plan keeps for its life.
int build_items(icon_batch* b) {
  const int ns = (int)b->plans.size();
  auto group = [](std::vector<Items>& v, int k0, int k1, int k2) -> Items& {
    for (auto& it : v)
      if (it.key0 == k0 && it.key1 == k1 && it.key2 == k2) return it;
    v.push_back(Items{});
    v.back().key0 = k0; v.back().key1 = k1; v.back().key2 = k2;
    return v.back();
  };
  for (int i = 0; i < ns; i++) {
    icon_plan* p = b->plans[i];
    const Geometry& g = p->g;
    const Bins& sb = p->spread().h;
    const int S = b->S[i];
    const int rows = S * g.N0;
    // the iteration's row kernels: key1 1 for real rows, two per transform
    const int half = p->half ? 1 : 0;
    // (key2 1: series that take FP64 gradients)
    const int r64ok = p->refreshes() ? 1 : 0;
    Items& rf = group(b->row_fwd, g.n1, half, r64ok);
    const int rpf = half ? 2 * half_row_pairs_per_block(g.n1) : row_fwd_rows_per_block(g.n1);
    for (int k = 0; k < (rows + rpf - 1) / rpf; k++) rf.h.push_back(make_int2(i, k));
    const int rpa = row_adj_rows_per_block(g.n1);
    if (!col_tile_ok(g.n0, g.n1, sb.C, sb.K))
      return bfail(ICON_ERR_ARG, "series %d: column tile %d unsupported for grid %d x %d", i, sb.C, g.n0, g.n1);
    // the data adjoint (key1 1: in FP64, one row per block) and the FP64 gradient
    for (int c = 0, s0 = 0; s0 < S; c++, s0 += pass_slices(p, S)) {
      const int n = std::min(pass_slices(p, S), S - s0), q = c * ns + i;
      Items& ra = group(b->row_adj, g.n1, r64ok, c);
      const int rpd = r64ok ? 1 : rpa;
      for (int k = 0; k < (n * g.N0 + rpd - 1) / rpd; k++) ra.h.push_back(make_int2(q, k));
      Items& cl = group(b->col_adj, g.n0, r64ok, c);
      for (int k = 0; k < n * (g.n1 / sb.C); k++) cl.h.push_back(make_int2(q, k));
      if (!r64ok) continue;
      Items& r64 = group(b->row64, g.n1, half, c);
      for (int k = 0; k < (half ? n * g.N0 / 2 : n * g.N0); k++) r64.h.push_back(make_int2(q, k));
      Items& n64 = group(b->normal64, g.n0, 0, c);
      for (int k = 0; k < n * (p->ncol / kNormalC); k++) n64.h.push_back(make_int2(q, k));
    }
    Items& rg = group(b->row_grad, g.n1, half, r64ok);
    const int rpg = half ? 2 * half_row_pairs_per_block(g.n1) : rpa;
    for (int k = 0; k < (rows + rpg - 1) / rpg; k++) rg.h.push_back(make_int2(i, k));
    Items& nm = group(b->normal, g.n0, r64ok, 0);
    for (int k = 0; k < S * (p->ncol / kNormalC); k++) nm.h.push_back(make_int2(i, k));
    Items& sn = group(b->sino, g.n0, 0, 0);
    const int rps = sino_rows_per_block(g.n0);
    for (int k = 0; k < (S * g.nz + rps - 1) / rps; k++) sn.h.push_back(make_int2(i, k));
    Items& rp = group(b->reproj, g.n0, 0, 0);
    for (int k = 0; k < S; k++) rp.h.push_back(make_int2(i, k));
    for (int k = 0; k < S; k++) b->combine.h.push_back(make_int2(i, k));
  }
  // the spread's order: a stable sort of each class's items by the entry
  // count of the tile the block runs (the plan's own largest-first tile order
  // maps a pass's block k to tile bins.order[k / its slices])
  for (Items& a : b->col_adj) {
    auto cnt = [&](const int2& q) {
      icon_plan* p = b->plans[q.x % ns];
      const Bins& sb = p->spread().h;
      const int S = b->S[q.x % ns], per = pass_slices(p, S), n = std::min(per, S - a.key2 * per);
      const int t = sb.order[q.y / n];
      return sb.off[t + 1] - sb.off[t];
    };
    std::stable_sort(a.h.begin(), a.h.end(), [&](const int2& u, const int2& v) { return cnt(u) > cnt(v); });
  }
  int rc;
  for (auto* v : {&b->row_fwd, &b->row_adj, &b->col_adj, &b->normal, &b->row_grad, &b->row64, &b->normal64, &b->sino,
                  &b->reproj})
    for (auto& it : *v)
      if ((rc = upload_items(it))) return rc;
  if ((rc = upload_items(b->combine))) return rc;
  const hipError_t e = set_col_adj_multi_attrs();
  if (e != hipSuccess) return bfail(ICON_ERR_DEVICE, "column kernel attributes: %s", hipGetErrorString(e));
  return ICON_OK;
}

void drop_batch_graph(icon_batch* b) {
  if (b->graph) (void)hipGraphExecDestroy(b->graph);
  b->graph = nullptr;
  b->graph_key = SolveKey{};
}

// Argument blocks of every series for a solve on the given buffers.
void fill_args(icon_batch* b, const float* const* sino, float* const* m, float* const* reproj, double* const* resid,
               double* const* alpha, int iters, bool any_resid) {
  const int ns = (int)b->plans.size();
  b->h_rf.assign(ns, RowFwdArgs{});
  b->h_cm.assign(ns, CombineArgs{});
  b->h_sa.assign(ns, SinoArgs{});
  b->h_rp.assign(ns, ReprojArgs{});
  for (auto* v : {&b->h_rg, &b->h_rg2}) v->assign(ns, RowAdjArgs{});
  for (auto* v : {&b->h_rf2, &b->h_rr}) v->assign(ns, RowFwdArgs{});
  b->h_ra.assign(kPasses * ns, RowAdjArgs{});
  b->h_re.assign(kPasses * ns, RefArgs{});
  for (auto* v : {&b->h_ca, &b->h_c64}) v->assign(kPasses * ns, ColArgs{});
  for (auto* v : {&b->h_cn, &b->h_ce, &b->h_cl}) v->assign(ns, ColArgs{});
  b->h_fa.assign(ns, FinishArgs{});
  for (int i = 0; i < ns; i++) {
    icon_plan* p = b->plans[i];
    const Geometry& g = p->g;
    const int S = b->S[i];
    RowFwdArgs& rf = b->h_rf[i];
    rf.rows = S * g.N0; rf.N0 = g.N0; rf.N1 = g.N1; rf.m = m[i]; rf.grad = p->d_grad; rf.alpha = p->d_alpha;
    rf.tw = p->d_tw1; rf.out = p->d_tmp;
    b->h_rg[i] = grad_args(p, S);
    b->h_rg2[i] = b->h_rg[i];
    b->h_rf2[i] = rf;
    if (p->refreshes()) {
      b->h_rg2[i].ahwb = p->d_base;
      b->h_rg2[i].ahwb_re = reinterpret_cast<const float*>(p->d_base);
      b->h_rf2[i].mref = p->d_mref;
    }
    b->h_rr[i] = rhat_row_args(p, S);
    // the adjoint of the data set-up and the FP64 gradient, by passes
    for (int s0 = 0, q = i; s0 < S; s0 += pass_slices(p, S), q += ns) {
      const int n = std::min(pass_slices(p, S), S - s0);
      b->h_ra[q] = data_row_args(p, s0, n);
      b->h_ca[q] = spread_args(p, s0, n);
      if (!p->refreshes()) continue;
      b->h_re[q] = ref_args(p, s0, n, m[i]);
      b->h_c64[q] = normal64_args(p, s0, n, any_resid);
    }
    CombineArgs& cm = b->h_cm[i];
    cm.S = S; cm.M = g.M; cm.N0 = g.N0; cm.nz = g.nz; cm.mode = 2; cm.E = b->h_ca[i].E;
    cm.w = p->d_w; cm.b = p->d_b; cm.fw = p->d_fw; cm.ent_of_node = p->spread().of_node; cm.bnorm = p->d_bnorm;
    b->h_cn[i] = normal_args(p, S, any_resid);
    b->h_ce[i] = energy_args(p, S);
    b->h_cl[i] = normal_args(p, S, true);
    FinishArgs& fa = b->h_fa[i];
    fa = finish_args(p, S);
    fa.beff = p->refreshes() ? p->d_beff : nullptr;
    fa.resid = resid ? resid[i] : nullptr; fa.resid_stride = iters + 1; fa.frep = p->d_frep;
    fa.alpha = p->d_alpha; fa.alpha_trace = alpha ? alpha[i] : nullptr; fa.alpha_stride = iters;
    SinoArgs& sa = b->h_sa[i];
    sa.rows = S * g.nz; sa.N0 = g.N0; sa.K = g.K; sa.nz = g.nz; sa.skip = g.cv_skip; sa.sino = sino[i];
    sa.ck1 = p->d_ck1; sa.phi1 = p->d_phi1; sa.i10 = p->d_i10; sa.tw = p->d_tw0; sa.b = p->d_b;
    b->h_rp[i] = reproj_args(p, S, reproj ? reproj[i] : nullptr);
  }
}

template <class T>
int upload_args(T* d, const std::vector<T>& h, hipStream_t st) {
  BCHK(hipMemcpyAsync(d, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice, st));
  return ICON_OK;
}

int ck(hipError_t e, const char* what) {
  if (e != hipSuccess) return bfail(ICON_ERR_DEVICE, "%s launch failed: %s", what, hipGetErrorString(e));
  return ICON_OK;
}

// The whole packed solve, enqueued on st (the order of enqueue_solve in the
// single-series path, each step once per size class).
int enqueue_batch(icon_batch* b, float* const* m, const float* const* m_init, bool any_resid, bool any_reproj,
                  const icon_solve_opts& o, hipStream_t st) {
  const int ns = (int)b->plans.size();
  const int iters = o.pre + o.icon + o.post;
  int rc;
  // which: series with (1) or without (0) FP64 gradients, -1: all
  auto row_fwd_all = [&](const RowFwdArgs* d, int update, int which) -> int {
    for (auto& it : b->row_fwd) {
      if (which >= 0 && it.key2 != which) continue;
      // rhat's row pass: complex images on full grids
      RowFwdLaunch L{d == b->d_rr && !it.key1 ? 1 : 0, update, o.data_type, o.threshold};
      if ((rc = ck(it.key1 ? launch_row_fwd_half_multi(it.key0, d, it.d, it.n(), L, st)
                           : launch_row_fwd_multi(it.key0, d, it.d, it.n(), L, st), "row_fwd")))
        return rc;
    }
    return ICON_OK;
  };
  auto gradient = [&](bool against_ref, int update, int which) -> int {
    if ((rc = row_fwd_all(against_ref ? b->d_rf2 : b->d_rf, update, which))) return rc;
    for (auto& nm : b->normal)
      if (which < 0 || nm.key1 == which)
        if ((rc = ck(launch_col_normal_multi(nm.key0, b->d_cn, nm.d, nm.n(), st), "col_normal"))) return rc;
    for (auto& it : b->row_grad) {
      if (which >= 0 && it.key2 != which) continue;
      const RowAdjArgs* d = against_ref ? b->d_rg2 : b->d_rg;
      if ((rc = ck(it.key1 ? launch_row_grad_half_multi(it.key0, d, it.d, it.n(), st)
                           : launch_row_adj_multi(it.key0, d, it.d, it.n(), true, st), "row_grad")))
        return rc;
    }
    return ICON_OK;
  };
  // the gradient in FP64 from the whole images (as in enqueue_solve), where a
  // series takes it
  auto reference = [&](int update) -> int {
    RowFwdLaunch L{0, update, o.data_type, o.threshold};
    for (int c = 0; c < kPasses; c++) {
      for (auto& it : b->row64)
        if (it.key2 == c && (rc = ck(launch_row_fwd64_multi(it.key0, it.key1, b->d_re, it.d, it.n(), L, st), "row_fwd64")))
          return rc;
      for (auto& nm : b->normal64)
        if (nm.key2 == c && (rc = ck(launch_col_normal64_multi(nm.key0, b->d_c64, nm.d, nm.n(), st), "col_normal64")))
          return rc;
      for (auto& it : b->row64)
        if (it.key2 == c && (rc = ck(launch_row_grad64_multi(it.key0, it.key1, b->d_re, it.d, it.n(), st), "row_grad64")))
          return rc;
    }
    if ((rc = row_fwd_all(b->d_rr, 0, 1))) return rc;
    return gradient(false, update, 0);
  };
  auto finish = [&](int ri, int ai, bool with_frep, int beff) -> int {
    FinishLaunch L{any_resid ? ri : -1, ai, with_frep ? 1 : 0, beff, 1};
    for (const FinishArgs& f : b->h_fa) L.blocks = std::max(L.blocks, f.blocks);
    return ck(launch_finish_multi(b->d_fa, b->combine.d, b->combine.n(), L, st), "finish");
  };
  // data set-up: b, w b, bnorm, A^H W b
  for (auto& it : b->sino)
    if ((rc = ck(launch_sino_multi(it.key0, b->d_sa, it.d, it.n(), st), "sino"))) return rc;
  if ((rc = ck(launch_combine_multi(b->d_cm, b->combine.d, b->combine.n(), st), "combine"))) return rc;
  for (int c = 0; c < kPasses; c++) {
    for (auto& it : b->col_adj)
      if (it.key2 == c &&
          (rc = ck(it.key1 ? launch_col_adj64_multi(it.key0, kSolveTile, b->d_ca, it.d, it.n(), st)
                           : launch_col_adj_multi(it.key0, b->d_ca, it.d, it.n(), st), "col_adj")))
        return rc;
    for (auto& it : b->row_adj)
      if (it.key2 == c && (rc = ck(it.key1 ? launch_row_adj64_multi(it.key0, b->d_ra, it.d, it.n(), st)
                                           : launch_row_adj_multi(it.key0, b->d_ra, it.d, it.n(), false, st), "row_adj")))
        return rc;
  }
  // m = 0 or the warm start
  for (int i = 0; i < ns; i++) {
    const size_t n = (size_t)b->S[i] * b->plans[i]->g.N0 * b->plans[i]->g.N1;
    hipError_t e = m_init && m_init[i] ? launch_copy(m[i], m_init[i], n, st) : launch_zero(m[i], n, st);
    if ((rc = ck(e, "init"))) return rc;
  }
  auto phase = [&](int it) { return (o.pre <= it && it < iters - o.post) ? 2 : 1; };
  bool referred = false;
  for (int it = 0; it < iters; it++) {
    const int update = it == 0 ? 0 : phase(it - 1);
    bool ref = false;
    for (const icon_plan* p : b->plans) ref |= refresh(p, o, it);
    if ((rc = ref ? reference(update) : gradient(referred, update, -1))) return rc;
    for (auto& nm : b->normal)
      if ((rc = ck(launch_col_energy_multi(nm.key0, b->d_ce, nm.d, nm.n(), st), "col_energy"))) return rc;
    if ((rc = finish(it, it, false, ref ? 1 : referred ? 2 : 0))) return rc;
    referred |= ref;
  }
  if (iters > 0 || any_resid || any_reproj)
    if ((rc = row_fwd_all(b->d_rf, iters > 0 ? phase(iters - 1) : 0, -1))) return rc;
  if (any_resid || any_reproj) {
    for (auto& nm : b->normal)
      if ((rc = ck(launch_col_fwd_nodes_multi(nm.key0, b->d_cl, nm.d, nm.n(), st), "col_fwd"))) return rc;
    if ((rc = finish(iters, -1, any_reproj, 0))) return rc;
    if (any_reproj)
      for (auto& it : b->reproj)
        if ((rc = ck(launch_reproj_multi(it.key0, b->d_rp, it.d, it.n(), st), "reproj"))) return rc;
  }
  return ICON_OK;
}

}  // namespace

extern "C" {

int icon_batch_destroy(icon_batch* b) {
  if (!b) return ICON_OK;
  int prev = -1;
  (void)hipGetDevice(&prev);
  (void)hipSetDevice(b->device);
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  drop_batch_graph(b);
  free_items(b->row_fwd);
  free_items(b->row_adj);
  free_items(b->col_adj);
  free_items(b->normal);
  free_items(b->row_grad);
  free_items(b->row64);
  free_items(b->normal64);
  free_items(b->sino);
  free_items(b->reproj);
  if (b->combine.d) (void)hipFree(b->combine.d);
  for (void* q : {(void*)b->d_rf, (void*)b->d_ra, (void*)b->d_ca, (void*)b->d_cm, (void*)b->d_sa, (void*)b->d_rp,
                  (void*)b->d_cn, (void*)b->d_ce, (void*)b->d_cl, (void*)b->d_rg, (void*)b->d_fa,
                  (void*)b->d_rg2, (void*)b->d_rf2, (void*)b->d_rr, (void*)b->d_re, (void*)b->d_c64})
    if (q) (void)hipFree(q);
  if (b->ev_in) (void)hipEventDestroy(b->ev_in);
  if (b->ev_out) (void)hipEventDestroy(b->ev_out);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
  if (prev >= 0) (void)hipSetDevice(prev);
  return ICON_OK;
}

int icon_batch_create(icon_batch** out, int nseries, icon_plan* const* plans, const int* slices) {
  if (!out || !plans || !slices || nseries < 1) return bfail(ICON_ERR_ARG, "icon_batch_create: bad argument");
  *out = nullptr;
  for (int i = 0; i < nseries; i++) {
    if (!plans[i]) return bfail(ICON_ERR_ARG, "icon_batch_create: series %d has no plan", i);
    if (plans[i]->device != plans[0]->device)
      return bfail(ICON_ERR_ARG, "icon_batch_create: series %d is on device %d, series 0 on %d", i,
                   plans[i]->device, plans[0]->device);
    if (slices[i] < 1 || slices[i] > plans[i]->S_max)
      return bfail(ICON_ERR_CAPACITY, "icon_batch_create: series %d: %d slices outside 1..%d", i, slices[i],
                   plans[i]->S_max);
    for (int j = 0; j < i; j++)
      if (plans[j] == plans[i]) return bfail(ICON_ERR_ARG, "icon_batch_create: series %d and %d share a plan", j, i);
  }
  auto* b = new icon_batch();
  b->device = plans[0]->device;
  b->plans.assign(plans, plans + nseries);
  b->S.assign(slices, slices + nseries);
  int prev = -1;
  (void)hipGetDevice(&prev);
  auto done = [&](int rc) {
    if (rc) icon_batch_destroy(b);
    else *out = b;
    if (prev >= 0) (void)hipSetDevice(prev);
    return rc;
  };
  if (hipSetDevice(b->device) != hipSuccess) return done(bfail(ICON_ERR_DEVICE, "icon_batch_create: hipSetDevice"));
  hipError_t e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&b->ev_in, hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&b->ev_out, hipEventDisableTiming);
  if (e == hipSuccess) e = hipMalloc(&b->d_rf, sizeof(RowFwdArgs) * nseries);
  if (e == hipSuccess) e = hipMalloc(&b->d_ra, sizeof(RowAdjArgs) * kPasses * nseries);
  if (e == hipSuccess) e = hipMalloc(&b->d_ca, sizeof(ColArgs) * kPasses * nseries);
  if (e == hipSuccess) e = hipMalloc(&b->d_cm, sizeof(CombineArgs) * nseries);
  if (e == hipSuccess) e = hipMalloc(&b->d_sa, sizeof(SinoArgs) * nseries);
  if (e == hipSuccess) e = hipMalloc(&b->d_rp, sizeof(ReprojArgs) * nseries);
  if (e == hipSuccess) e = hipMalloc(&b->d_rg, sizeof(RowAdjArgs) * nseries);
  if (e == hipSuccess) e = hipMalloc(&b->d_rg2, sizeof(RowAdjArgs) * nseries);
  if (e == hipSuccess) e = hipMalloc(&b->d_rf2, sizeof(RowFwdArgs) * nseries);
  if (e == hipSuccess) e = hipMalloc(&b->d_rr, sizeof(RowFwdArgs) * nseries);
  if (e == hipSuccess) e = hipMalloc(&b->d_re, sizeof(RefArgs) * kPasses * nseries);
  if (e == hipSuccess) e = hipMalloc(&b->d_c64, sizeof(ColArgs) * kPasses * nseries);
  for (ColArgs** q : {&b->d_cn, &b->d_ce, &b->d_cl})
    if (e == hipSuccess) e = hipMalloc(q, sizeof(ColArgs) * nseries);
  if (e == hipSuccess) e = hipMalloc(&b->d_fa, sizeof(FinishArgs) * nseries);
  if (e != hipSuccess) return done(bfail(ICON_ERR_DEVICE, "icon_batch_create: %s", hipGetErrorString(e)));
  return done(build_items(b));
}

int icon_batch_reconstruct(icon_batch* b, const void* const* d_sino, void* const* d_m, const void* const* d_m_init,
                           void* const* d_reproj, void* const* d_resid, void* const* d_alpha,
                           const icon_solve_opts* opts, void* stream) {
  if (!b || !d_sino || !d_m || !opts) return bfail(ICON_ERR_ARG, "icon_batch_reconstruct: null pointer");
  const icon_solve_opts& o = *opts;
  if (o.pre < 0 || o.icon < 0 || o.post < 0) return bfail(ICON_ERR_ARG, "negative iteration count");
  if (o.data_type != 1 && o.data_type != 2) return bfail(ICON_ERR_ARG, "data_type must be 1 or 2");
  if (o.reuse_data) return bfail(ICON_ERR_ARG, "icon_batch_reconstruct: reuse_data is not supported for batches");
  const int ns = (int)b->plans.size();
  for (int i = 0; i < ns; i++)
    if (!d_sino[i] || !d_m[i]) return bfail(ICON_ERR_ARG, "icon_batch_reconstruct: series %d has no sinograms or image", i);
  const int iters = o.pre + o.icon + o.post;
  bool any_resid = false, any_reproj = false;
  SolveKey key;
  key.pre = o.pre; key.icon = o.icon; key.post = o.post; key.data_type = o.data_type; key.thr = o.threshold;
  for (int i = 0; i < ns; i++) {
    any_resid |= d_resid && d_resid[i];
    any_reproj |= d_reproj && d_reproj[i];
    key.ptrs.push_back(d_sino[i]);
    key.ptrs.push_back(d_m[i]);
    key.ptrs.push_back(d_m_init ? d_m_init[i] : nullptr);
    key.ptrs.push_back(d_reproj ? d_reproj[i] : nullptr);
    key.ptrs.push_back(d_resid ? d_resid[i] : nullptr);
    key.ptrs.push_back(d_alpha ? d_alpha[i] : nullptr);
  }
  int prev = -1;
  (void)hipGetDevice(&prev);
  if (prev != b->device) BCHK(hipSetDevice(b->device));
  int rc = ICON_OK;
  hipStream_t user = (hipStream_t)stream;
  std::vector<float*> m(ns);
  std::vector<const float*> sino(ns), mi(ns);
  std::vector<float*> rp(ns);
  std::vector<double*> rs(ns), al(ns);
  for (int i = 0; i < ns; i++) {
    sino[i] = (const float*)d_sino[i];
    m[i] = (float*)d_m[i];
    mi[i] = d_m_init ? (const float*)d_m_init[i] : nullptr;
    rp[i] = d_reproj ? (float*)d_reproj[i] : nullptr;
    rs[i] = d_resid ? (double*)d_resid[i] : nullptr;
    al[i] = d_alpha ? (double*)d_alpha[i] : nullptr;
  }
  // the plans' own buffers are overwritten: their data reuse is void
  for (auto* p : b->plans) {
    p->data_sino = nullptr;
    p->data_S = 0;
  }
  do {
    hipError_t e = hipEventRecord(b->ev_in, user);
    if (e == hipSuccess) e = hipStreamWaitEvent(b->stream, b->ev_in, 0);
    if (e != hipSuccess) { rc = bfail(ICON_ERR_DEVICE, "icon_batch_reconstruct: %s", hipGetErrorString(e)); break; }
    if (!(b->graph && b->graph_key == key)) {
      drop_batch_graph(b);
      fill_args(b, sino.data(), m.data(), rp.data(), rs.data(), al.data(), iters, any_resid);
      if ((rc = upload_args(b->d_rf, b->h_rf, b->stream)) || (rc = upload_args(b->d_ra, b->h_ra, b->stream)) ||
          (rc = upload_args(b->d_ca, b->h_ca, b->stream)) || (rc = upload_args(b->d_cm, b->h_cm, b->stream)) ||
          (rc = upload_args(b->d_sa, b->h_sa, b->stream)) || (rc = upload_args(b->d_rp, b->h_rp, b->stream)) ||
          (rc = upload_args(b->d_rg, b->h_rg, b->stream)) || (rc = upload_args(b->d_rg2, b->h_rg2, b->stream)) ||
          (rc = upload_args(b->d_rf2, b->h_rf2, b->stream)) || (rc = upload_args(b->d_rr, b->h_rr, b->stream)) ||
          (rc = upload_args(b->d_re, b->h_re, b->stream)) || (rc = upload_args(b->d_c64, b->h_c64, b->stream)) ||
          (rc = upload_args(b->d_cn, b->h_cn, b->stream)) ||
          (rc = upload_args(b->d_ce, b->h_ce, b->stream)) || (rc = upload_args(b->d_cl, b->h_cl, b->stream)) || (rc = upload_args(b->d_fa, b->h_fa, b->stream)))
        break;
      e = hipStreamSynchronize(b->stream);
      if (e == hipSuccess) e = hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal);
      if (e != hipSuccess) { rc = bfail(ICON_ERR_DEVICE, "capture: %s", hipGetErrorString(e)); break; }
      rc = enqueue_batch(b, m.data(), mi.data(), any_resid, any_reproj, o, b->stream);
      hipGraph_t graph = nullptr;
      e = hipStreamEndCapture(b->stream, &graph);
      if (rc) {
        if (graph) (void)hipGraphDestroy(graph);
        break;
      }
      if (e == hipSuccess) e = hipGraphInstantiate(&b->graph, graph, nullptr, nullptr, 0);
      if (graph) (void)hipGraphDestroy(graph);
      if (e != hipSuccess) {
        b->graph = nullptr;
        rc = bfail(ICON_ERR_DEVICE, "graph: %s", hipGetErrorString(e));
        break;
      }
      b->graph_key = key;
    }
    e = hipGraphLaunch(b->graph, b->stream);
    if (e == hipSuccess) e = hipEventRecord(b->ev_out, b->stream);
    if (e == hipSuccess) e = hipStreamWaitEvent(user, b->ev_out, 0);
    if (e != hipSuccess) rc = bfail(ICON_ERR_DEVICE, "icon_batch_reconstruct: %s", hipGetErrorString(e));
  } while (0);
  if (prev >= 0 && prev != b->device) (void)hipSetDevice(prev);
  return rc;
}

int icon_batch_launches_per_iteration(const icon_batch* b, int* launches) {
  if (!b || !launches) return bfail(ICON_ERR_ARG, "icon_batch_launches_per_iteration: null pointer");
  *launches = (int)b->row_fwd.size() + (int)b->row_grad.size() + 2 * (int)b->normal.size() + 1;
  return ICON_OK;
}

// The column tile is the transforms' alone: a packed solve does not depend on it.
int icon_batch_autotune(icon_batch* b, int* col_blocks) {
  if (!b) return bfail(ICON_ERR_ARG, "icon_batch_autotune: null batch");
  BCHK(hipStreamSynchronize(b->stream));   // the plans' buffers are overwritten
  for (size_t i = 0; i < b->plans.size(); i++) {
    int c = 0;
    if (const int rc = icon_plan_autotune(b->plans[i], b->S[i], &c, nullptr))
      return bfail(rc, "icon_batch_autotune: series %d: %s", (int)i, icon_last_error());
    if (col_blocks) col_blocks[i] = c;
  }
  return ICON_OK;
}

}  // extern "C"
