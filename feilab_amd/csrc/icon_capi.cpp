// C ABI of the MI355X ICON core: plans, batched operators and the solve.
//
// Reference (tomography/ICON_GPU_v1.2.9/sourceCode/ICON-GPU/):
//   plan setup            MainCode.cu:38-109, nufft_gpu_v8.cu:281-556,1298-1391,1739-1771
//   per-slice solve       MainCode.cu:113-135, Iteration2.cu:33-146, alpha_new2.cu:28-114
//   reprojection          MainCode.cu:142, reProject_NFFT.cu:81-98
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "icon_kernels.h"
#include "icon_plan.h"

using namespace icon;

namespace {

thread_local std::string g_err;

int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  std::vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_err = buf;
  return code;
}

#define HIPCHK(expr)                                                                          \
  do {                                                                                        \
    hipError_t e_ = (expr);                                                                   \
    if (e_ != hipSuccess)                                                                     \
      return fail(ICON_ERR_DEVICE, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_),      \
                  __FILE__, __LINE__);                                                        \
  } while (0)

// Twiddle tables exp(-2 pi i q / n), q < n, per (device, n); computed in
// double and rounded to float.  Held for the life of the process.
std::mutex g_tw_mu;
std::map<std::pair<int, int>, float2*> g_tw;

// exp(-2 pi i q / n), q < n, in double, per (device, n).
std::map<std::pair<int, int>, double2*> g_w64;

int twiddles64(int n, const double2** out) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_tw_mu);
  auto key = std::make_pair(dev, n);
  auto it = g_w64.find(key);
  if (it != g_w64.end()) { *out = it->second; return ICON_OK; }
  std::vector<double2> w(n);
  for (int q = 0; q < n; q++) {
    const double a = -2.0 * M_PI * (double)q / (double)n;
    w[q] = make_double2(std::cos(a), std::sin(a));
  }
  double2* d = nullptr;
  HIPCHK(hipMalloc(&d, sizeof(double2) * n));
  HIPCHK(hipMemcpy(d, w.data(), sizeof(double2) * n, hipMemcpyHostToDevice));
  g_w64[key] = d;
  *out = d;
  return ICON_OK;
}

int twiddles(int n, const float2** out) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_tw_mu);
  auto key = std::make_pair(dev, n);
  auto it = g_tw.find(key);
  if (it != g_tw.end()) { *out = it->second; return ICON_OK; }
  // exp(-2 pi i q / n) in double, rounded to float
  std::vector<float2> w(n);
  for (int q = 0; q < n; q++) {
    const double a = -2.0 * M_PI * (double)q / (double)n;
    w[q] = make_float2((float)std::cos(a), (float)std::sin(a));
  }
  // layout read by load_twiddles (icon_fft.h): [dir][slot / 2][t][slot % 2]
  const int TH = n / 16;
  std::vector<float2> h((size_t)2 * TH * 32, make_float2(0.f, 0.f));
  for (int d = 0; d < 2; d++)
    for (int t = 0; t < TH; t++) {
      int ns = 1, P = 0;
      while (ns < n) {
        const int rp = n / ns >= 16 ? 16 : n / ns;
        if (ns > 1) {
          const int step = n / (ns * rp);
          for (int q = 0; q < 16 / rp; q++) {
            const int k = (t + q * TH) & (ns - 1);
            for (int r = 1; r < rp; r++) {
              float2 v = w[(size_t)r * k * step];
              if (d) v.y = -v.y;
              const int slot = P * 16 + q * (rp - 1) + r - 1;
              h[(((size_t)d * 16 + slot / 2) * TH + t) * 2 + slot % 2] = v;
            }
          }
          P++;
        }
        ns *= rp;
      }
    }
  float2* d = nullptr;
  HIPCHK(hipMalloc(&d, sizeof(float2) * h.size()));
  HIPCHK(hipMemcpy(d, h.data(), sizeof(float2) * h.size(), hipMemcpyHostToDevice));
  g_tw[key] = d;
  *out = d;
  return ICON_OK;
}

template <class T>
int dalloc(icon_plan* p, T** ptr, size_t count) {
  const size_t bytes = sizeof(T) * (count ? count : 1);
  HIPCHK(hipMalloc((void**)ptr, bytes));
  p->device_bytes += (int64_t)bytes;
  return ICON_OK;
}

template <class T>
int upload(icon_plan* p, T** ptr, const std::vector<T>& h) {
  int rc = dalloc(p, ptr, h.size());
  if (rc) return rc;
  if (!h.empty()) HIPCHK(hipMemcpy(*ptr, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice));
  return ICON_OK;
}

void free_bins(DevBins& b) {
  for (void* q : {(void*)b.ck, (void*)b.off, (void*)b.order, (void*)b.xoff, (void*)b.of_node, (void*)b.ent,
                  (void*)b.fent, (void*)b.parts, (void*)b.xt, (void*)b.px, (void*)b.py, (void*)b.fpx, (void*)b.fpy, (void*)b.nslot})
    if (q) (void)hipFree(q);
  b = DevBins{};
}

// Shares of the tiles' entries, a round of the block's threads each (8 at most):
// shares per tile, and (tile, share) of those past the first.
void dense_shares(const std::vector<int>& off, int round, std::vector<int>& parts, std::vector<int2>& xt) {
  for (size_t t = 0; t + 1 < off.size(); t++) {
    parts.push_back(std::max(1, std::min(8, (off[t + 1] - off[t] + round - 1) / round)));
    for (int k = 1; k < parts.back(); k++) xt.push_back(make_int2((int)t, k));
  }
}

// Blocks of a column tile of C columns resident on the device at once: 1024
// threads of up to 128 registers per CU.
long resident_tiles(const icon_plan* p, int C) { return (long)p->cus * std::max(1, 16384 / (C * p->g.n0)); }

// Slices up to which split_dense shares the dense tiles' entries.
int split_slices(const icon_plan* p) {
  if (!p->nd_nx || !p->refreshes()) return 0;
  return (int)std::min<long>(p->S_max, resident_tiles(p, kNormalC) / (p->ncol / kNormalC + p->nd_nx));
}

// Bins of a Kaiser-Bessel window of K taps in tiles of C columns; records and
// deapodisation are computed on the device.
int make_bins(icon_plan* p, DevBins& b, int C, int K) {
  const Geometry& g = p->g;
  build_bins(g, C, K, b.h);
  b.beta0 = kb_beta(g.sig0, K);
  b.beta1 = kb_beta(g.sig1, K);
  const size_t E = b.h.ent.size();
  std::vector<float> c(g.N0 + g.N1);
  kb_deapod(g.N0, g.sig0, b.beta0, K, c.data());
  kb_deapod(g.N1, g.sig1, b.beta1, K, c.data() + g.N0);
  int rc;
  std::vector<int> parts;
  std::vector<int2> xt;
  dense_shares(b.h.off, C * (g.n0 / 16), parts, xt);
  b.nx = (int)xt.size();
  if (b.nx && ((rc = upload(p, &b.parts, parts)) || (rc = upload(p, &b.xt, xt)))) return rc;
  if ((rc = upload(p, &b.off, b.h.off)) || (rc = upload(p, &b.order, b.h.order)) || (rc = upload(p, &b.ent, b.h.ent)) ||
      (rc = upload(p, &b.fent, b.h.fent)) || (rc = upload(p, &b.nslot, b.h.nslot)) ||
      (rc = upload(p, &b.xoff, b.h.xoff)) || (rc = upload(p, &b.of_node, b.h.of_node)) ||
      (rc = dalloc(p, &b.px, E * K)) || (rc = dalloc(p, &b.py, E * C)) || (rc = dalloc(p, &b.fpx, E * K)) ||
      (rc = dalloc(p, &b.fpy, E * C)) || (rc = dalloc(p, &b.ck, (size_t)g.N0 * g.N1)))
    return rc;
  float* dc = nullptr;
  HIPCHK(hipMalloc(&dc, sizeof(float) * c.size()));
  hipError_t e = hipMemcpy(dc, c.data(), sizeof(float) * c.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = launch_outer(dc, dc + g.N0, g.N0, g.N1, b.ck, p->stream);
  if (e == hipSuccess)
    e = launch_window_records(b.ent, b.off, p->d_nodes, (int)E, g.n0, g.n1, K, C, b.beta0, b.beta1, b.px, b.py, p->stream);
  if (e == hipSuccess)
    e = launch_window_records(b.fent, b.off, p->d_nodes, (int)E, g.n0, g.n1, K, C, b.beta0, b.beta1, b.fpx, b.fpy,
                              p->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(p->stream);
  (void)hipFree(dc);
  if (e != hipSuccess) return fail(ICON_ERR_DEVICE, "window tables: %s", hipGetErrorString(e));
  return ICON_OK;
}

int op_taps(const Geometry& g) { return g.window == ICON_WINDOW_KB6 ? kTapsKB : kTapsWide; }

// The transforms' bins at tile width C.  The solve keeps the bins that it was
// made with (accurate window, tiles of kSolveTile columns): its data set-up has
// an FP64 kernel for those alone, its results do not depend on a choice made by
// timing the transforms, and captured solves, of the plan and of batches that
// hold it, keep tables and buffers that live as long as the plan.
int make_op_bins(icon_plan* p, int C) {
  const int K = op_taps(p->g);
  DevBins t;
  int rc = ICON_OK;
  if (K == kTapsWide && C == kSolveTile && p->own_data) {
    free_bins(p->op);
    p->op = std::exchange(p->data, DevBins{});
    p->own_data = false;
  } else if ((rc = make_bins(p, t, C, K))) {
    free_bins(t);
    return rc;
  } else {
    if (p->op.ck && !p->own_data) {
      p->data = std::exchange(p->op, DevBins{});
      p->own_data = true;
    }
    free_bins(p->op);
    p->op = std::move(t);
  }
  return ICON_OK;
}

// Column-kernel arguments of a window's bins over S slices.
ColArgs window_args(icon_plan* p, const DevBins& b, int S) {
  const Geometry& g = p->g;
  ColArgs a{};
  a.K = b.h.K; a.S = S; a.N0 = g.N0; a.N1 = g.N1; a.M = g.M; a.n1 = g.n1; a.E = (int)b.h.ent.size();
  a.in = p->d_tmp; a.out = p->d_tmp; a.tw = p->d_tw0; a.ent_off = b.off; a.tile_order = b.order;
  a.split_min = split_min_entries(b.h); a.ent = b.ent; a.xoff = b.xoff; a.ent_px = b.px; a.ent_py = b.py;
  a.fent = b.fent; a.fent_px = b.fpx; a.fent_py = b.fpy; a.part = p->d_part; a.slots = kMaxSlot; a.fw = p->d_fw;
  zero_band(b.h, &a.zlo, &a.zhi);
  // few slices: the dense tiles' entries shared among further blocks, as in
  // split_dense (one 64^2 image, 21 tilts: 10.7 -> 4.7 us)
  if (b.nx && (long)S * (g.n1 / b.h.C + b.nx) <= resident_tiles(p, b.h.C)) {
    a.parts = b.parts;
    a.xt = b.xt;
    a.nx = b.nx;
  }
  return a;
}

void drop_graph(icon_plan* p) {
  for (int i = 0; i < kGraphCache; i++) {
    if (p->graph_exec[i]) (void)hipGraphExecDestroy(p->graph_exec[i]);
    p->graph_exec[i] = nullptr;
    p->graph_key[i] = GraphKey{};
    p->graph_used[i] = 0;
  }
  p->data_sino = nullptr;
  p->data_S = 0;
}

// Eight grid columns per tile: two blocks fit in one CU's LDS at n0 = 1024
// (measured faster than 16 columns at one block per CU).
int default_col_block(int n0) { (void)n0; return 8; }

struct DevGuard {
  int prev = -1;
  explicit DevGuard(int dev) {
    if (hipGetDevice(&prev) != hipSuccess) prev = -1;
    if (prev != dev) (void)hipSetDevice(dev);
  }
  ~DevGuard() {
    if (prev >= 0) (void)hipSetDevice(prev);
  }
};

int check_launch(hipError_t e, const char* what) {
  if (e != hipSuccess) return fail(ICON_ERR_DEVICE, "%s launch failed: %s", what, hipGetErrorString(e));
  return ICON_OK;
}

// ---------------------------------------------------------------- operators

int op_forward(icon_plan* p, int S, const void* img, int cplx, float2* out, hipStream_t st) {
  const Geometry& g = p->g;
  const ColArgs ca = window_args(p, p->op, S);
  RowFwdArgs ra{};
  ra.rows = S * g.N0; ra.N0 = g.N0; ra.N1 = g.N1; ra.cplx = cplx; ra.update = 0;
  ra.m = cplx ? nullptr : (float*)img;
  ra.rhat = cplx ? (const float2*)img : nullptr;
  ra.ck = p->op.ck; ra.tw = p->d_tw1; ra.out = p->d_tmp; ra.zlo = ca.zlo; ra.zhi = ca.zhi;
  int rc = check_launch(launch_row_fwd(g.n1, ra, st), "row_fwd");
  if (rc) return rc;
  if ((rc = check_launch(launch_col(g.n0, p->op.h.C, false, ca, st), "col_fwd"))) return rc;
  CombineArgs cb{};
  cb.S = S; cb.M = g.M; cb.N0 = g.N0; cb.nz = g.nz; cb.mode = 3; cb.part = p->d_part;
  cb.nslot = p->op.nslot; cb.w = p->d_w; cb.fw = out;
  return check_launch(launch_combine(cb, st), "combine");
}

// A^H of the per-entry weighted values already in p->d_fw (entries of b): the
// image, or its real part to img_re.
int op_adjoint_ent(icon_plan* p, const DevBins& b, int S, float2* img, hipStream_t st, float* img_re = nullptr) {
  const Geometry& g = p->g;
  const ColArgs ca = window_args(p, b, S);
  int rc = check_launch(launch_col(g.n0, b.h.C, true, ca, st), "col_adj");
  if (rc) return rc;
  RowAdjArgs ra{};
  ra.rows = S * g.N0; ra.N0 = g.N0; ra.N1 = g.N1; ra.in = p->d_tmp;
  ra.ck = b.ck; ra.tw = p->d_tw1; ra.img = img; ra.img_re = img_re; ra.zlo = ca.zlo; ra.zhi = ca.zhi;
  return check_launch(launch_row_adj(g.n1, ra, st), "row_adj");
}

// A^H of node vectors f [S][M].
int op_adjoint(icon_plan* p, int S, const float2* f, float2* img, hipStream_t st) {
  int rc = check_launch(launch_node_to_ent(f, p->d_fw, p->op.ent, S, p->g.M, (int)p->op.h.ent.size(), st),
                        "node_to_ent");
  if (rc) return rc;
  return op_adjoint_ent(p, p->op, S, img, st);
}

int op_sino(icon_plan* p, int S, const float* sino, float2* b, hipStream_t st) {
  const Geometry& g = p->g;
  SinoArgs sa{};
  sa.K = p->g.K;
  sa.rows = S * g.nz; sa.N0 = g.N0; sa.nz = g.nz; sa.skip = g.cv_skip; sa.sino = sino; sa.ck1 = p->d_ck1;
  sa.phi1 = p->d_phi1;
  sa.i10 = p->d_i10; sa.tw = p->d_tw0; sa.b = b;
  return check_launch(launch_sino(g.n0, sa, st), "sino");
}

// A^H of the data's weighted values in p->d_fw, as the gradient subtracts it
// (with paired nodes its real part), in FP64 where the plan takes FP64 gradients.
int op_adjoint_data(icon_plan* p, int S, hipStream_t st) {
  const DevBins& b = p->spread();
  float* re = p->half ? reinterpret_cast<float*>(p->d_ahwb) : nullptr;
  if (!p->refreshes()) return op_adjoint_ent(p, b, S, re ? nullptr : p->d_ahwb, st, re);
  for (int s0 = 0; s0 < S; s0 += p->S64) {
    const int n = std::min(p->S64, S - s0);
    int rc = check_launch(launch_col_adj64(p->g.n0, b.h.C, spread_args(p, s0, n), st), "col_adj64");
    if (!rc) rc = check_launch(launch_row_adj64(p->g.n1, data_row_args(p, s0, n), st), "row_adj64");
    if (rc) return rc;
  }
  return ICON_OK;
}

// An iteration's launches over S slices: with paired nodes the real-row
// kernels on half grids, otherwise the full ones.
hipError_t iter_row_fwd(icon_plan* p, const RowFwdArgs& a, hipStream_t st) {
  return p->half ? launch_row_fwd_half(p->g.n1, a, st) : launch_row_fwd(p->g.n1, a, st);
}
hipError_t iter_row_grad(icon_plan* p, const RowAdjArgs& a, hipStream_t st) {
  return p->half ? launch_row_grad_half(p->g.n1, a, st) : launch_row_adj(p->g.n1, a, st);
}

// The whole solve of S slices, enqueued on st (captured into a graph by the caller
// when requested).
int enqueue_solve(icon_plan* p, int S, const float* sino, float* m, const float* m_init, float* reproj,
                  double* resid, double* alpha_tr, const icon_solve_opts& o, hipStream_t st) {
  const Geometry& g = p->g;
  const int iters = o.pre + o.icon + o.post;
  int rc;
  if (!o.reuse_data) {
    // b = NFFT1D of every projection row; fw = w b; bnorm = sum w |b|^2
    if ((rc = op_sino(p, S, sino, p->d_b, st))) return rc;
    CombineArgs c0{};
    c0.S = S; c0.M = g.M; c0.N0 = g.N0; c0.nz = g.nz; c0.mode = 2; c0.b = p->d_b; c0.w = p->d_w;
    c0.fw = p->d_fw; c0.bnorm = p->d_bnorm;
    c0.E = (int)p->spread().h.ent.size(); c0.ent_of_node = p->spread().of_node;
    if ((rc = check_launch(launch_combine(c0, st), "combine_b"))) return rc;
    // A^H W b
    if ((rc = op_adjoint_data(p, S, st))) return rc;
  }
  // m = 0 (Iteration2.cu:33) or the warm start
  const size_t NN = (size_t)g.N0 * g.N1;
  if (m_init) rc = check_launch(launch_copy(m, m_init, (size_t)S * NN, st), "copy");
  else rc = check_launch(launch_zero(m, (size_t)S * NN, st), "zero");
  if (rc) return rc;

  RowFwdArgs rf{};
  rf.rows = S * g.N0; rf.N0 = g.N0; rf.N1 = g.N1; rf.data_type = o.data_type; rf.thr = o.threshold;
  rf.m = m; rf.grad = p->d_grad; rf.alpha = p->d_alpha; rf.tw = p->d_tw1; rf.out = p->d_tmp;
  ColArgs ca = normal_args(p, S, resid != nullptr);
  const ColArgs ce = energy_args(p, S);
  RowAdjArgs ra = grad_args(p, S);
  split_dense(p, S, ca, ra);
  FinishArgs fa = finish_args(p, S);
  fa.resid = resid; fa.resid_stride = iters + 1; fa.alpha = p->d_alpha; fa.alpha_trace = alpha_tr;
  fa.alpha_stride = iters;
  auto phase = [&](int it) { return (o.pre <= it && it < iters - o.post) ? 2 : 1; };

  for (int it = 0; it < iters; it++) {
    const int update = it == 0 ? 0 : phase(it - 1);
    const bool ref = refresh(p, o, it);
    if (ref) {
      // the iterate's gradient in FP64, from the whole image; from here on the
      // transforms take the difference from it
      for (int s0 = 0; s0 < S; s0 += p->S64) {
        const int n = std::min(p->S64, S - s0);
        RefArgs rr = ref_args(p, s0, n, m);
        rr.update = update; rr.data_type = o.data_type; rr.thr = o.threshold;
        const ColArgs c64 = normal64_args(p, s0, n, resid != nullptr);
        if ((rc = check_launch(launch_row_fwd64(g.n1, p->half, rr, st), "row_fwd64"))) return rc;
        if ((rc = check_launch(launch_col_normal64(g.n0, c64, st), "col_normal64"))) return rc;
        if ((rc = check_launch(launch_row_grad64(g.n1, p->half, rr, st), "row_grad64"))) return rc;
      }
      if ((rc = check_launch(iter_row_fwd(p, rhat_row_args(p, S), st), "row_fwd_rhat"))) return rc;
      rf.mref = p->d_mref;
      ra.ahwb = p->d_base;
      ra.ahwb_re = reinterpret_cast<const float*>(p->d_base);
      fa.b = p->d_b;
      fa.beff = p->d_beff;
    } else {
      // y FFT of m (with the previous iteration's update fused in front)
      rf.update = update;
      if ((rc = check_launch(iter_row_fwd(p, rf, st), "row_fwd"))) return rc;
      // A^H W A m up to its inverse y FFT, and A m at the nodes for R(m_it)
      if ((rc = check_launch(launch_col_normal(g.n0, ca, st), "col_normal"))) return rc;
      // rhat = A^H W A m - A^H W b, row sums of |rhat|^2, y FFT of rhat
      if ((rc = check_launch(iter_row_grad(p, ra, st), "row_adj"))) return rc;
    }
    // <rhat, A^H W A rhat> by column tile
    if ((rc = check_launch(launch_col_energy(g.n0, ce, st), "col_energy"))) return rc;
    // alpha = |rhat|^2 / <rhat, A^H W A rhat>, R(m_it)
    fa.resid_index = fa.alpha_index = it;
    if ((rc = check_launch(launch_finish(fa, st), "finish"))) return rc;
    if (ref) {
      fa.beff = nullptr;
      fa.b = p->d_beff;
    }
  }
  rf.mref = nullptr;
  fa.b = p->d_b;
  // last update, then A m_final for the final residual and the reprojection
  if (iters > 0 || resid || reproj) {
    rf.update = iters > 0 ? phase(iters - 1) : 0;
    if ((rc = check_launch(iter_row_fwd(p, rf, st), "row_fwd_final"))) return rc;
  }
  if (resid || reproj) {
    ca = normal_args(p, S, true);
    if ((rc = check_launch(launch_col_fwd_nodes(g.n0, ca, st), "col_fwd_final"))) return rc;
    fa.resid_index = iters;
    fa.alpha = nullptr;
    fa.frep = reproj ? p->d_frep : nullptr;
    if ((rc = check_launch(launch_finish(fa, st), "finish_final"))) return rc;
    if (reproj) {
      if ((rc = check_launch(launch_reproj(g.n0, reproj_args(p, S, reproj), st), "reproj"))) return rc;
    }
  }
  return ICON_OK;
}

// The normal operator's tables: interpolation entries and records, spectrum
// and, with paired nodes, the unpaired nodes' waves.  The spectrum takes
// 2 M n0 n1 FP64 operations on the matrix cores, in chunks of nodes whose
// factors fit the scratch.
int build_normal(icon_plan* p) {
  const Geometry& g = p->g;
  p->half = g.nz <= kMaxUnpaired && paired_nodes(g);
  p->nq = p->half ? g.nz : 0;
  p->rows = p->half ? g.nz * (g.N0 / 2 + 1) : g.M;
  p->ncol = p->half ? g.n1 / 2 + kNormalC : g.n1;
  NodeBins nb, ub;
  build_node_bins(g, p->half, nb);
  if (p->half) {
    unpaired_bins(g, nb, ub);
  } else {
    ub.off.assign(nb.off.size(), 0);   // no entries
  }
  std::vector<int4> entr = ub.ent;
  for (int4& e : entr) e.x /= g.N0 / 2 + 1;   // rows of d_rpart: the tilt line
  const size_t E = nb.ent.size(), U = ub.ent.size(), cells = (size_t)g.n0 * g.n1;
  const size_t S = (size_t)p->S_max;
  double chol[kInterpTaps * kInterpTaps];
  interp_factor(chol);
  int rc;
  std::vector<int> parts;
  std::vector<int2> xt;
  dense_shares(nb.off, kNormalC * (g.n0 / 16), parts, xt);
  p->nd_nx = (int)xt.size();
  if (p->nd_nx && ((rc = upload(p, &p->d_nd_parts, parts)) || (rc = upload(p, &p->d_nd_xt, xt)))) return rc;
  if ((rc = upload(p, &p->d_nd_off, nb.off)) || (rc = upload(p, &p->d_nd_ent, nb.ent)) ||
      (rc = upload(p, &p->d_nd_nslot, nb.nslot)) || (rc = dalloc(p, &p->d_nd_px, E * kInterpTaps)) ||
      (rc = dalloc(p, &p->d_nd_py, E * kNormalC)) || (rc = dalloc(p, &p->d_spec, (size_t)g.n0 * p->ncol)) ||
      (rc = dalloc(p, &p->d_epart, S * (p->ncol / kNormalC))) ||
      (rc = dalloc(p, &p->d_rsum, S * kFinishGroups)) || (rc = dalloc(p, &p->d_rcnt, S)) || (rc = upload(p, &p->d_nq_off, ub.off)))
    return rc;
  if (p->half &&
      ((rc = upload(p, &p->d_nq_ent, ub.ent)) || (rc = upload(p, &p->d_nq_entr, entr)) ||
       (rc = upload(p, &p->d_nq_nslot, ub.nslot)) || (rc = dalloc(p, &p->d_nq_px, U * kInterpTaps)) ||
       (rc = dalloc(p, &p->d_nq_py, U * kNormalC)) || (rc = dalloc(p, &p->d_rpart, S * p->nq * kNodeSlots)) ||
       (rc = dalloc(p, &p->d_gram, (size_t)8 * p->nq * p->nq))))
    return rc;
  constexpr int kChunk = 1024;
  const int ld = (2 * p->nq + 63) / 64 * 64;
  const size_t head = (sizeof(chol) + 255) / 256 * 256;
  const size_t acc_n = std::max(cells * spectrum_splits(g.n0, g.n1),
                                ld ? (size_t)ld * ld * spectrum_splits(ld, ld) : (size_t)0);
  const size_t fac_n = std::max((size_t)kChunk * (g.n0 + g.n1), (size_t)4 * kChunk * ld);
  char* scratch = nullptr;
  HIPCHK(hipMalloc(&scratch, head + sizeof(double) * (acc_n + fac_n)));
  const float2* nodes = p->d_nodes;
  auto* d_chol = reinterpret_cast<double*>(scratch);
  auto* acc = reinterpret_cast<double*>(scratch + head);
  double* fac = acc + acc_n;
  hipStream_t st = p->stream;
  const int half = p->half ? g.N0 / 2 : 0;
  hipError_t e = hipMemcpy(d_chol, chol, sizeof(chol), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = launch_zero(reinterpret_cast<float*>(p->d_rcnt), S, st);
  if (e == hipSuccess)
    e = launch_interp_records(p->d_nd_ent, p->d_nd_off, nodes, (int)E, g.n0, g.n1, half, d_chol, p->d_nd_px,
                              p->d_nd_py, st);
  if (e == hipSuccess && p->half)
    e = launch_interp_records(p->d_nq_ent, p->d_nq_off, nodes, (int)U, g.n0, g.n1, half, d_chol, p->d_nq_px,
                              p->d_nq_py, st);
  if (e == hipSuccess) e = launch_zero(reinterpret_cast<float*>(acc), 2 * acc_n, st);
  for (int j = 0; j < g.M && e == hipSuccess; j += kChunk)
    e = launch_spectrum_chunk(nodes, p->d_w, j, std::min(kChunk, g.M - j), g.N0, g.N1, g.n0, g.n1, fac,
                              fac + (size_t)kChunk * g.n0, acc, st);
  if (e == hipSuccess) e = launch_spectrum_store(acc, g.n0, g.n1, p->half, p->d_spec, st);
  if (e == hipSuccess && p->half) {
    e = launch_wave_gram(nodes, p->nq, g.N0, g.N1, p->d_gram, st);
    if (e == hipSuccess) e = launch_zero(reinterpret_cast<float*>(acc), 2 * acc_n, st);
    for (int j = 0; j < g.M && e == hipSuccess; j += kChunk)
      e = launch_wave_chunk(nodes, p->d_w, j, std::min(kChunk, g.M - j), p->nq, ld, g.N0, g.N1, fac,
                            fac + (size_t)2 * kChunk * ld, acc, st);
    if (e == hipSuccess) e = launch_wave_store(acc, p->nq, ld, p->d_gram + (size_t)4 * p->nq * p->nq, st);
  }
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  (void)hipFree(scratch);
  if (e == hipSuccess) e = set_normal_attrs(g.n0);
  if (e != hipSuccess) return fail(ICON_ERR_DEVICE, "normal operator: %s", hipGetErrorString(e));
  return ICON_OK;
}

int prepare_col(int n0, int n1, int C, int K) {
  // sets the LDS attribute outside any capture
  if (!col_tile_ok(n0, n1, C, K))
    return fail(ICON_ERR_ARG, "column tile %d unsupported for grid %d x %d with %d window taps", C, n0, n1, K);
  hipError_t e = set_col_attrs(n0, C, K);
  if (e != hipSuccess) return fail(ICON_ERR_DEVICE, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  return ICON_OK;
}

}  // namespace

void icon::set_last_error(const char* msg) { g_err = msg; }
int icon::fft_twiddles(int n, const float2** out) { return twiddles(n, out); }

// Arguments of the iteration's kernels over S slices of a plan.
ColArgs icon::normal_args(const icon_plan* p, int S, bool with_nodes) {
  const Geometry& g = p->g;
  ColArgs a{};
  a.S = S; a.N0 = g.N0; a.N1 = g.N1; a.M = p->rows; a.n1 = p->ncol; a.K = kInterpTaps; a.slots = kNodeSlots;
  a.in = p->d_tmp; a.out = p->d_tmp; a.tw = p->d_tw0; a.part = p->d_part; a.spec = p->d_spec;
  // all nodes for the residual; otherwise the unpaired ones (none on a full grid)
  a.ent_off = with_nodes ? p->d_nd_off : p->d_nq_off;
  a.fent = with_nodes ? p->d_nd_ent : p->d_nq_ent;
  a.fent_px = with_nodes ? p->d_nd_px : p->d_nq_px;
  a.fent_py = with_nodes ? p->d_nd_py : p->d_nq_py;
  return a;
}

ColArgs icon::energy_args(const icon_plan* p, int S) {
  ColArgs a = normal_args(p, S, false);
  a.M = p->nq; a.part = p->d_rpart; a.fent = p->d_nq_entr; a.epart = p->d_epart;
  a.nyq = p->half ? p->g.n1 / 2 : 0;
  return a;
}

ColArgs icon::normal64_args(const icon_plan* p, int s0, int S, bool with_nodes) {
  ColArgs a = normal_args(p, S, with_nodes);
  a.part += (size_t)s0 * a.M * a.slots;
  a.io64 = reinterpret_cast<double2*>(p->d_tmp);
  a.w64 = p->d_w640;
  return a;
}

RefArgs icon::ref_args(const icon_plan* p, int s0, int S, float* m) {
  const Geometry& g = p->g;
  const size_t o = (size_t)s0 * g.N0 * g.N1;
  RefArgs a{};
  a.rows = S * g.N0; a.N0 = g.N0; a.N1 = g.N1; a.ncol = p->ncol; a.m = m + o; a.mref = p->d_mref + o;
  a.alpha = p->d_alpha + s0; a.w64 = p->d_w641; a.io = reinterpret_cast<double2*>(p->d_tmp); a.grad = p->d_grad + o;
  a.rowpart = p->d_rowpart + (size_t)s0 * (p->half ? g.N0 / 2 : g.N0);
  if (p->half) {
    a.ahwb_re = reinterpret_cast<const float*>(p->d_ahwb) + o;
    a.base_re = reinterpret_cast<float*>(p->d_base) + o;
  } else {
    a.ahwb = p->d_ahwb + o;
    a.base = p->d_base + o;
  }
  return a;
}

// Phase of iteration it: 0 before, 1 in and 2 after the ICON iterations.
static int phase_of(const icon_solve_opts& o, int it) { return it < o.pre ? 0 : it < o.pre + o.icon ? 1 : 2; }

// Iterations whose gradient is computed in FP64: the iterates after 2, 8, 32,
// ... updates of each phase (the bound moves the image at once where it sets
// in or ends), where at least 6 more follow in the phase.
bool icon::refresh(const icon_plan* p, const icon_solve_opts& o, int it) {
  if (!p->refreshes() || it == 0) return false;
  const int ph = phase_of(o, it - 1);
  const int begin = ph == 0 ? 0 : ph == 1 ? o.pre : o.pre + o.icon;
  const int len = ph == 0 ? o.pre : ph == 1 ? o.icon : o.post;
  const int j = it - begin;   // updates of this phase so far
  for (int k = 2; k <= j; k *= 4)
    if (k == j) return j + 6 <= len;
  return false;
}

RowFwdArgs icon::rhat_row_args(const icon_plan* p, int S) {
  RowFwdArgs a{};
  a.rows = S * p->g.N0; a.N0 = p->g.N0; a.N1 = p->g.N1; a.tw = p->d_tw1; a.out = p->d_tmp;
  a.cplx = p->half ? 0 : 1;
  a.m = p->d_grad;
  a.rhat = p->d_base;   // -rhat: its energy is rhat's
  return a;
}

ColArgs icon::spread_args(icon_plan* p, int s0, int S) {
  ColArgs a = window_args(p, p->spread(), S);
  a.fw += (size_t)s0 * a.E;
  a.io64 = reinterpret_cast<double2*>(p->d_tmp);
  a.w64 = p->d_w640;
  return a;
}

RowAdjArgs icon::data_row_args(icon_plan* p, int s0, int S) {
  const Geometry& g = p->g;
  const size_t o = (size_t)s0 * g.N0 * g.N1;
  RowAdjArgs a{};
  a.rows = S * g.N0; a.N0 = g.N0; a.N1 = g.N1; a.in = p->d_tmp; a.ck = p->spread().ck; a.tw = p->d_tw1;
  a.in64 = reinterpret_cast<const double2*>(p->d_tmp); a.w64 = p->d_w641;
  if (p->half) a.img_re = reinterpret_cast<float*>(p->d_ahwb) + o;
  else a.img = p->d_ahwb + o;
  zero_band(p->spread().h, &a.zlo, &a.zhi);
  return a;
}

ReprojArgs icon::reproj_args(const icon_plan* p, int S, float* out) {
  ReprojArgs a{};
  a.S = S; a.N0 = p->g.N0; a.K = kTapsWide; a.sigma = p->g.sig0; a.frep = p->d_frep; a.ck = p->d_rck; a.phi = p->d_rphi;
  a.i0 = p->d_ri0; a.tw = p->d_tw0; a.out = out;
  return a;
}

RowAdjArgs icon::grad_args(const icon_plan* p, int S) {
  const Geometry& g = p->g;
  RowAdjArgs a{};
  a.rows = S * g.N0; a.N0 = g.N0; a.N1 = g.N1; a.in = p->d_tmp; a.tw = p->d_tw1; a.ahwb = p->d_ahwb;
  a.ahwb_re = reinterpret_cast<const float*>(p->d_ahwb); a.grad = p->d_grad; a.rowpart = p->d_rowpart;
  a.fwd_out = p->d_tmp;
  return a;
}

// Few slices leave CUs idle while the tiles around ky = 0, which all tilt lines
// cross, interpolate 6 and more rounds of entries (one 256^2 slice, 61 tilts:
// 22 us instead of 10 for a tile without): their entries are shared among
// further blocks, which transform the tile again.  The grid goes behind the rows
// in d_tmp, as those blocks read the rows that the tile's own would overwrite.
// Where all blocks are not resident at once they would cost more than the wait.
void icon::split_dense(const icon_plan* p, int S, ColArgs& ca, RowAdjArgs& ra) {
  const Geometry& g = p->g;
  if (ca.ent_off != p->d_nd_off || S > split_slices(p)) return;
  ca.parts = p->d_nd_parts;
  ca.xt = p->d_nd_xt;
  ca.nx = p->nd_nx;
  ca.out = p->d_tmp + (size_t)p->S_max * g.N0 * g.n1;
  ra.in = ca.out;
}

FinishArgs icon::finish_args(const icon_plan* p, int S) {
  const Geometry& g = p->g;
  FinishArgs a{};
  a.S = S; a.M = p->rows; a.Mb = g.M; a.N0 = g.N0; a.nblk = p->ncol / kNormalC; a.nrow = p->half ? g.N0 / 2 : g.N0;
  a.slots = kNodeSlots; a.part = p->d_part; a.nslot = p->d_nd_nslot;
  a.w = p->d_w; a.b = p->d_b; a.bnorm = p->d_bnorm; a.iomit = g.iomit;
  a.rowpart = p->d_rowpart; a.epart = p->d_epart;
  // one round of 4 rows per thread, and a block for each while blocks are fewer
  // than CUs (16 slices of 1007^2, 61400 nodes: 73 -> 17 us with 15 blocks per
  // slice; 256 slices of 512^2: 36 us with one, 41 with three)
  a.rsum = p->d_rsum; a.rcnt = p->d_rcnt;
  a.groups = std::max(1, std::min(kFinishGroups, (a.M + kFinishRows - 1) / kFinishRows));
  a.blocks = std::max(1, std::min(a.groups, p->cus / S));
  a.nq = p->nq; a.rpart = p->d_rpart; a.rslot = p->d_nq_nslot; a.gram = p->d_gram;
  return a;
}

// ====================================================================== ABI
extern "C" {

const char* icon_last_error(void) { return g_err.c_str(); }

const char* icon_version(void) { return "icon-mi355x 0.1 (gfx950)"; }

int icon_device_count(int* count) {
  if (!count) return fail(ICON_ERR_ARG, "icon_device_count: null pointer");
  HIPCHK(hipGetDeviceCount(count));
  return ICON_OK;
}

int icon_device_compute_units(int device, int* cus) {
  if (!cus) return fail(ICON_ERR_ARG, "icon_device_compute_units: null pointer");
  hipDeviceProp_t prop;
  HIPCHK(hipGetDeviceProperties(&prop, device));
  *cus = prop.multiProcessorCount;
  return ICON_OK;
}

int icon_set_device(int device) {
  HIPCHK(hipSetDevice(device));
  return ICON_OK;
}

int icon_get_device(int* device) {
  if (!device) return fail(ICON_ERR_ARG, "icon_get_device: null pointer");
  HIPCHK(hipGetDevice(device));
  return ICON_OK;
}

int icon_stream_create(void** stream) {
  if (!stream) return fail(ICON_ERR_ARG, "icon_stream_create: null pointer");
  hipStream_t st = nullptr;
  HIPCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  *stream = st;
  return ICON_OK;
}

int icon_stream_destroy(void* stream) {
  if (stream) HIPCHK(hipStreamDestroy((hipStream_t)stream));
  return ICON_OK;
}

int icon_stream_synchronize(void* stream) {
  HIPCHK(hipStreamSynchronize((hipStream_t)stream));
  return ICON_OK;
}

int icon_event_create(void** event) {
  if (!event) return fail(ICON_ERR_ARG, "icon_event_create: null pointer");
  hipEvent_t ev = nullptr;
  HIPCHK(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
  *event = ev;
  return ICON_OK;
}

int icon_event_destroy(void* event) {
  if (event) HIPCHK(hipEventDestroy((hipEvent_t)event));
  return ICON_OK;
}

int icon_event_record(void* event, void* stream) {
  if (!event) return fail(ICON_ERR_ARG, "icon_event_record: null event");
  HIPCHK(hipEventRecord((hipEvent_t)event, (hipStream_t)stream));
  return ICON_OK;
}

int icon_stream_wait_event(void* stream, void* event) {
  if (!event) return fail(ICON_ERR_ARG, "icon_stream_wait_event: null event");
  HIPCHK(hipStreamWaitEvent((hipStream_t)stream, (hipEvent_t)event, 0));
  return ICON_OK;
}

int icon_malloc(void** dptr, size_t bytes) {
  if (!dptr) return fail(ICON_ERR_ARG, "icon_malloc: null pointer");
  HIPCHK(hipMalloc(dptr, bytes ? bytes : 1));
  return ICON_OK;
}

int icon_free(void* dptr) {
  if (dptr) HIPCHK(hipFree(dptr));
  return ICON_OK;
}

int icon_memcpy_h2d(void* dst, const void* src, size_t bytes) {
  HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
  return ICON_OK;
}

int icon_memcpy_d2h(void* dst, const void* src, size_t bytes) {
  HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
  return ICON_OK;
}

int icon_memcpy_d2d_async(void* dst, const void* src, size_t bytes, void* stream) {
  if (!bytes) return ICON_OK;
  if (!dst || !src) return fail(ICON_ERR_ARG, "icon_memcpy_d2d_async: null pointer");
  HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, (hipStream_t)stream));
  return ICON_OK;
}

int icon_memset_d(void* dst, int value, size_t bytes) {
  HIPCHK(hipMemset(dst, value, bytes));
  return ICON_OK;
}

int icon_device_synchronize(void) {
  HIPCHK(hipDeviceSynchronize());
  return ICON_OK;
}

int icon_geometry_tables(int nx, int thickness, int nz, const float* tilt_deg, icon_plan_info* info,
                         float* nodes, float* weights, float* phix, float* phiy, int* ix0, int* iy0, float* ck,
                         float* ck1, float* phi1, int* i10) {
  if (!tilt_deg) return fail(ICON_ERR_ARG, "icon_geometry_tables: null tilt angles");
  Geometry g;
  std::string err;
  if (!build_geometry(g, nx, thickness > 0 ? thickness : nx, nz, tilt_deg, &err))
    return fail(ICON_ERR_ARG, "%s", err.c_str());
  auto put = [](auto* dst, const auto& v) {
    if (dst) std::memcpy(dst, v.data(), sizeof(v[0]) * v.size());
  };
  put(nodes, g.nodes); put(weights, g.w); put(phix, g.phix); put(phiy, g.phiy); put(ix0, g.ix0);
  put(iy0, g.iy0); put(ck, g.ck); put(ck1, g.ck1); put(phi1, g.phi1); put(i10, g.i10);
  if (info) {
    std::memset(info, 0, sizeof(*info));
    info->N0 = g.N0; info->N1 = g.N1; info->nz = g.nz; info->M = g.M; info->n0 = g.n0; info->n1 = g.n1;
    info->m = g.K == kTaps ? kWindowM : g.K / 2; info->window = g.window; info->iomit = g.iomit; info->sigma0 = g.sig0; info->sigma1 = g.sig1;
    info->b0 = g.b0; info->b1 = g.b1;
  }
  return ICON_OK;
}

namespace {
int plan_create(icon_plan** out, int device, int nx, int thickness, int nz, const float* tilt_deg, int max_slices,
                bool cv, int window = ICON_WINDOW_GAUSS);
}

int icon_plan_create(icon_plan** out, int device, int nx, int thickness, int nz, const float* tilt_deg,
                     int max_slices) {
  return plan_create(out, device, nx, thickness, nz, tilt_deg, max_slices, false);
}

int icon_plan_create_cv(icon_plan** out, int device, int nx, int thickness, int nz, const float* tilt_deg,
                        int max_slices) {
  return plan_create(out, device, nx, thickness, nz, tilt_deg, max_slices, true);
}

int icon_plan_create_window(icon_plan** out, int device, int nx, int thickness, int nz, const float* tilt_deg,
                            int max_slices, int cross_validation, int window) {
  return plan_create(out, device, nx, thickness, nz, tilt_deg, max_slices, cross_validation != 0, window);
}

}  // extern "C"

namespace {
int plan_create(icon_plan** out, int device, int nx, int thickness, int nz, const float* tilt_deg, int max_slices,
                bool cv, int window) {
  if (!out || !tilt_deg) return fail(ICON_ERR_ARG, "icon_plan_create: null pointer");
  *out = nullptr;
  if (max_slices < 1) return fail(ICON_ERR_ARG, "icon_plan_create: max_slices must be >= 1");
  int ndev = 0;
  HIPCHK(hipGetDeviceCount(&ndev));
  if (device < 0 || device >= ndev) return fail(ICON_ERR_ARG, "icon_plan_create: no device %d", device);
  DevGuard dg(device);
  HIPCHK(hipSetDevice(device));
  auto* p = new icon_plan();
  p->device = device;
  (void)hipDeviceGetAttribute(&p->cus, hipDeviceAttributeMultiprocessorCount, device);
  std::string err;
  if (!build_geometry(p->g, nx, thickness > 0 ? thickness : nx, nz, tilt_deg, &err, cv, window, false)) {
    delete p;
    return fail(ICON_ERR_ARG, "%s", err.c_str());
  }
  p->S_max = max_slices;
  const Geometry& g = p->g;
  int rc = ICON_OK;
  auto bail = [&](int code) {
    icon_plan_destroy(p);
    return code;
  };
  {
    hipError_t e = hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&p->ev_in, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&p->ev_out, hipEventDisableTiming);
    if (e != hipSuccess) return bail(fail(ICON_ERR_DEVICE, "stream/event create: %s", hipGetErrorString(e)));
  }
  if ((rc = dalloc(p, &p->d_nodes, (size_t)g.M))) return bail(rc);
  {
    hipError_t e = hipMemcpy(p->d_nodes, g.nodes.data(), sizeof(float2) * g.M, hipMemcpyHostToDevice);
    if (e != hipSuccess) return bail(fail(ICON_ERR_DEVICE, "node upload: %s", hipGetErrorString(e)));
  }
  if ((rc = upload(p, &p->d_ck1, g.ck1))) return bail(rc);
  if ((rc = upload(p, &p->d_w, g.w))) return bail(rc);
  if ((rc = upload(p, &p->d_phi1, g.phi1))) return bail(rc);
  if ((rc = upload(p, &p->d_i10, g.i10))) return bail(rc);
  if (2 * g.N0 != g.n0) {
    std::vector<float> ck, phi;
    std::vector<int> first;
    reproj_tables(g, ck, phi, first);
    if ((rc = upload(p, &p->d_rck, ck)) || (rc = upload(p, &p->d_rphi, phi)) || (rc = upload(p, &p->d_ri0, first)))
      return bail(rc);
  }
  // The solve subtracts A^H W b from the exact A^H W A m in every iteration, so
  // that an error of it in the directions that no tilt covers adds up over the
  // iterations: it needs the accurate window also where the transforms use the
  // 6-tap one (with it, and with the 14-tap Gaussian, a 100-iteration solve was
  // 4 to 5 times as far from the exact one as now).
  static_assert(kSolveTile == 8, "the tile of the FP64 data adjoint (COL64_CASES)");
  p->own_data = op_taps(g) != kTapsWide;
  if (p->own_data && (rc = make_bins(p, p->data, kSolveTile, kTapsWide))) return bail(rc);
  if ((rc = make_op_bins(p, default_col_block(g.n0)))) return bail(rc);
  if ((rc = twiddles(g.n0, &p->d_tw0))) return bail(rc);
  if ((rc = twiddles(g.n1, &p->d_tw1))) return bail(rc);
  if ((rc = twiddles64(g.n0, &p->d_w640))) return bail(rc);
  if ((rc = twiddles64(g.n1, &p->d_w641))) return bail(rc);
  const size_t S = (size_t)max_slices, M = (size_t)g.M, NN = (size_t)g.N0 * g.N1;
  if ((rc = dalloc(p, &p->d_b, S * M))) return bail(rc);
  if ((rc = dalloc(p, &p->d_grad, S * NN))) return bail(rc);
  if ((rc = dalloc(p, &p->d_frep, S * g.N0))) return bail(rc);
  if ((rc = dalloc(p, &p->d_rowpart, S * g.N0))) return bail(rc);
  if ((rc = dalloc(p, &p->d_bnorm, S))) return bail(rc);
  if ((rc = dalloc(p, &p->d_alpha, S))) return bail(rc);
  // alpha starts at 0 so an update before any step is a no-op
  {
    hipError_t e = hipMemset(p->d_alpha, 0, sizeof(double) * S);
    if (e != hipSuccess) return bail(fail(ICON_ERR_DEVICE, "hipMemset: %s", hipGetErrorString(e)));
  }
  if ((rc = prepare_col(g.n0, g.n1, p->op.h.C, p->op.h.K))) return bail(rc);
  if (p->own_data && (rc = prepare_col(g.n0, g.n1, p->data.h.C, p->data.h.K))) return bail(rc);
  if ((rc = build_normal(p))) return bail(rc);
  if ((rc = dalloc(p, &p->d_part, S * std::max(M * kMaxSlot, (size_t)p->rows * kNodeSlots)))) return bail(rc);
  // weighted values are spread before, and in other calls than, any interpolation;
  // a node has kMaxSlot entries at most, whatever the tile
  p->d_fw = p->d_part;
  if ((rc = dalloc(p, &p->d_ahwb, p->half ? (S * NN + 1) / 2 : S * NN))) return bail(rc);
  if (p->refreshes() && ((rc = dalloc(p, &p->d_base, p->half ? (S * NN + 1) / 2 : S * NN)) ||
                         (rc = dalloc(p, &p->d_mref, S * NN)) || (rc = dalloc(p, &p->d_beff, S * M))))
    return bail(rc);
  // the grid rows, in single precision or, for FP64 passes, in double: in two
  // passes where each still has slices for the whole device (64), so that a plan
  // for many takes no more for them
  p->S64 = max_slices < 128 ? max_slices : (max_slices + 1) / 2;
  const size_t grid = (size_t)g.N0 * g.n1;
  size_t tmp = S * grid + (size_t)split_slices(p) * g.N0 * p->ncol;
  if (p->refreshes()) tmp = std::max(tmp, 2 * p->S64 * grid);
  if ((rc = dalloc(p, &p->d_tmp, tmp))) return bail(rc);
  {
    const hipError_t e = set_adj64_attrs();
    if (e != hipSuccess) return bail(fail(ICON_ERR_DEVICE, "hipFuncSetAttribute: %s", hipGetErrorString(e)));
  }
  *out = p;
  return ICON_OK;
}
}  // namespace

extern "C" {

int icon_plan_destroy(icon_plan* p) {
  if (!p) return ICON_OK;
  DevGuard dg(p->device);
  if (p->stream) (void)hipStreamSynchronize(p->stream);
  drop_graph(p);
  void* ptrs[] = {p->d_nodes, p->d_ck1, p->d_w, p->d_phi1, p->d_i10, p->d_rck, p->d_rphi, p->d_ri0,
                  p->d_b, p->d_part, p->d_ahwb, p->d_grad, p->d_tmp, p->d_frep, p->d_rowpart,
                  p->d_bnorm, p->d_alpha, p->d_spec, p->d_nd_off, p->d_nd_ent, p->d_nd_parts, p->d_nd_xt, p->d_rsum, p->d_rcnt, p->d_nd_nslot, p->d_nd_px, p->d_nd_py,
                  p->d_epart, p->d_nq_off, p->d_nq_ent, p->d_nq_entr, p->d_nq_px, p->d_nq_py, p->d_nq_nslot,
                  p->d_rpart, p->d_gram, p->d_base, p->d_mref, p->d_beff};
  for (void* q : ptrs)
    if (q) (void)hipFree(q);
  free_bins(p->op);
  free_bins(p->data);
  if (p->ev_in) (void)hipEventDestroy(p->ev_in);
  if (p->ev_out) (void)hipEventDestroy(p->ev_out);
  if (p->stream) (void)hipStreamDestroy(p->stream);
  delete p;
  return ICON_OK;
}

int icon_plan_get_info(const icon_plan* p, icon_plan_info* info) {
  if (!p || !info) return fail(ICON_ERR_ARG, "icon_plan_get_info: null pointer");
  const Geometry& g = p->g;
  info->N0 = g.N0; info->N1 = g.N1; info->nz = g.nz; info->M = g.M; info->n0 = g.n0; info->n1 = g.n1;
  info->m = g.K == kTaps ? kWindowM : g.K / 2; info->window = g.window; info->iomit = g.iomit; info->sigma0 = g.sig0; info->sigma1 = g.sig1;
  info->b0 = g.b0; info->b1 = g.b1; info->max_slices = p->S_max; info->col_block = p->op.h.C;
  info->device_bytes = p->device_bytes;
  return ICON_OK;
}

int icon_plan_set_col_block(icon_plan* p, int C) {
  if (!p) return fail(ICON_ERR_ARG, "icon_plan_set_col_block: null plan");
  if (!col_tile_ok(p->g.n0, p->g.n1, C, op_taps(p->g)))
    return fail(ICON_ERR_ARG, "column tile %d unsupported for grid %d x %d", C, p->g.n0, p->g.n1);
  if (C == p->op.h.C) return ICON_OK;
  DevGuard dg(p->device);
  HIPCHK(hipStreamSynchronize(p->stream));
  drop_graph(p);
  const int rc = prepare_col(p->g.n0, p->g.n1, C, op_taps(p->g));
  return rc ? rc : make_op_bins(p, C);
}

int icon_nufft_forward_real(icon_plan* p, int S, const void* d_img, void* d_f, void* stream) {
  if (!p || !d_img || !d_f) return fail(ICON_ERR_ARG, "icon_nufft_forward_real: null pointer");
  if (S < 1 || S > p->S_max) return fail(ICON_ERR_CAPACITY, "batch %d outside 1..%d", S, p->S_max);
  DevGuard dg(p->device);
  return op_forward(p, S, d_img, 0, (float2*)d_f, (hipStream_t)stream);
}

int icon_nufft_forward_complex(icon_plan* p, int S, const void* d_img, void* d_f, void* stream) {
  if (!p || !d_img || !d_f) return fail(ICON_ERR_ARG, "icon_nufft_forward_complex: null pointer");
  if (S < 1 || S > p->S_max) return fail(ICON_ERR_CAPACITY, "batch %d outside 1..%d", S, p->S_max);
  DevGuard dg(p->device);
  return op_forward(p, S, d_img, 1, (float2*)d_f, (hipStream_t)stream);
}

int icon_nufft_adjoint(icon_plan* p, int S, const void* d_f, void* d_img, void* stream) {
  if (!p || !d_img || !d_f) return fail(ICON_ERR_ARG, "icon_nufft_adjoint: null pointer");
  if (S < 1 || S > p->S_max) return fail(ICON_ERR_CAPACITY, "batch %d outside 1..%d", S, p->S_max);
  DevGuard dg(p->device);
  return op_adjoint(p, S, (const float2*)d_f, (float2*)d_img, (hipStream_t)stream);
}

int icon_sino_to_b(icon_plan* p, int S, const void* d_sino, void* d_b, void* stream) {
  if (!p || !d_sino || !d_b) return fail(ICON_ERR_ARG, "icon_sino_to_b: null pointer");
  if (S < 1) return fail(ICON_ERR_ARG, "batch %d < 1", S);
  DevGuard dg(p->device);
  return op_sino(p, S, (const float*)d_sino, (float2*)d_b, (hipStream_t)stream);
}

int icon_fft_rows(int n, int rows, int sign, void* d_data, void* stream) {
  if (!d_data || rows < 0 || (sign != 1 && sign != -1)) return fail(ICON_ERR_ARG, "icon_fft_rows: bad argument");
  if (n != 128 && n != 256 && n != 512 && n != 1024 && n != 2048)
    return fail(ICON_ERR_ARG, "icon_fft_rows: n=%d unsupported", n);
  if (rows == 0) return ICON_OK;
  const float2* tw = nullptr;
  int rc = twiddles(n, &tw);
  if (rc) return rc;
  return check_launch(launch_fft_rows(n, (float2*)d_data, rows, sign, tw, (hipStream_t)stream), "fft_rows");
}

int icon_fft_2d(int n0, int n1, int count, int sign, void* d_data, void* stream) {
  if (!d_data || count < 0 || (sign != 1 && sign != -1)) return fail(ICON_ERR_ARG, "icon_fft_2d: bad argument");
  for (int n : {n0, n1})
    if (n != 128 && n != 256 && n != 512 && n != 1024 && n != 2048)
      return fail(ICON_ERR_ARG, "icon_fft_2d: n=%d unsupported", n);
  if (count == 0) return ICON_OK;
  const float2 *tw0 = nullptr, *tw1 = nullptr;
  int rc = twiddles(n0, &tw0);
  if (!rc) rc = twiddles(n1, &tw1);
  if (rc) return rc;
  const int C = default_col_block(n0);
  if ((rc = check_launch(launch_fft_rows(n1, (float2*)d_data, count * n0, sign, tw1, (hipStream_t)stream), "fft_rows")))
    return rc;
  return check_launch(launch_fft_cols(n0, C, (float2*)d_data, n1, count, sign, tw0, (hipStream_t)stream), "fft_cols");
}

int icon_reconstruct(icon_plan* p, int S, const void* d_sino, void* d_m, const void* d_m_init, void* d_reproj,
                     void* d_resid, void* d_alpha, const icon_solve_opts* opts, void* stream) {
  if (!p || !d_sino || !d_m || !opts) return fail(ICON_ERR_ARG, "icon_reconstruct: null pointer");
  if (S < 1 || S > p->S_max) return fail(ICON_ERR_CAPACITY, "batch %d outside 1..%d", S, p->S_max);
  const icon_solve_opts& o = *opts;
  if (o.pre < 0 || o.icon < 0 || o.post < 0) return fail(ICON_ERR_ARG, "negative iteration count");
  if (o.data_type != 1 && o.data_type != 2) return fail(ICON_ERR_ARG, "data_type must be 1 or 2");
  if (o.reuse_data && !(p->data_sino == d_sino && p->data_S == S))
    return fail(ICON_ERR_ARG, "reuse_data: the previous solve on this plan had other sinograms or batch");
  DevGuard dg(p->device);
  hipStream_t user = (hipStream_t)stream;
  HIPCHK(hipEventRecord(p->ev_in, user));
  HIPCHK(hipStreamWaitEvent(p->stream, p->ev_in, 0));
  int rc = ICON_OK;
  if (o.use_graph) {
    GraphKey key;
    key.S = S; key.sino = d_sino; key.m = d_m; key.m_init = d_m_init; key.reproj = d_reproj;
    key.resid = d_resid; key.alpha = d_alpha; key.pre = o.pre; key.icon = o.icon; key.post = o.post;
    key.data_type = o.data_type; key.reuse = o.reuse_data ? 1 : 0; key.thr = o.threshold;
    int slot = -1;
    for (int i = 0; i < kGraphCache; i++)
      if (p->graph_exec[i] && p->graph_key[i] == key) slot = i;
    if (slot < 0) {
      slot = 0;   // least recently used (empty slots have time 0)
      for (int i = 1; i < kGraphCache; i++)
        if (p->graph_used[i] < p->graph_used[slot]) slot = i;
      if (p->graph_exec[slot]) (void)hipGraphExecDestroy(p->graph_exec[slot]);
      p->graph_exec[slot] = nullptr;
      p->graph_key[slot] = GraphKey{};
      HIPCHK(hipStreamBeginCapture(p->stream, hipStreamCaptureModeThreadLocal));
      rc = enqueue_solve(p, S, (const float*)d_sino, (float*)d_m, (const float*)d_m_init, (float*)d_reproj,
                         (double*)d_resid, (double*)d_alpha, o, p->stream);
      hipGraph_t graph = nullptr;
      hipError_t e = hipStreamEndCapture(p->stream, &graph);
      if (rc) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc;
      }
      if (e != hipSuccess) return fail(ICON_ERR_DEVICE, "hipStreamEndCapture: %s", hipGetErrorString(e));
      e = hipGraphInstantiate(&p->graph_exec[slot], graph, nullptr, nullptr, 0);
      (void)hipGraphDestroy(graph);
      if (e != hipSuccess) {
        p->graph_exec[slot] = nullptr;
        return fail(ICON_ERR_DEVICE, "hipGraphInstantiate: %s", hipGetErrorString(e));
      }
      p->graph_key[slot] = key;
    }
    p->graph_used[slot] = ++p->graph_clock;
    HIPCHK(hipGraphLaunch(p->graph_exec[slot], p->stream));
  } else {
    rc = enqueue_solve(p, S, (const float*)d_sino, (float*)d_m, (const float*)d_m_init, (float*)d_reproj,
                       (double*)d_resid, (double*)d_alpha, o, p->stream);
    if (rc) return rc;
  }
  p->data_sino = d_sino;
  p->data_S = S;
  HIPCHK(hipEventRecord(p->ev_out, p->stream));
  HIPCHK(hipStreamWaitEvent(user, p->ev_out, 0));
  return rc;
}

int icon_reconstruct_host(icon_plan* p, int S, const float* sino, float* m, const float* m_init, float* reproj,
                          double* resid, double* alpha, const icon_solve_opts* opts) {
  if (!p || !sino || !m || !opts) return fail(ICON_ERR_ARG, "icon_reconstruct_host: null pointer");
  if (S < 1 || S > p->S_max) return fail(ICON_ERR_CAPACITY, "batch %d outside 1..%d", S, p->S_max);
  if (opts->reuse_data) return fail(ICON_ERR_ARG, "icon_reconstruct_host: reuse_data needs device buffers");
  DevGuard dg(p->device);
  const Geometry& g = p->g;
  const int iters = opts->pre + opts->icon + opts->post;
  const size_t nsino = (size_t)S * g.M, nimg = (size_t)S * g.N0 * g.N1;
  void *ds = nullptr, *dm = nullptr, *dmi = nullptr, *drp = nullptr, *drs = nullptr, *dal = nullptr;
  int rc = ICON_OK;
  auto cleanup = [&]() {
    for (void* q : {ds, dm, dmi, drp, drs, dal})
      if (q) (void)hipFree(q);
  };
#define TRY(expr)                                              \
  do {                                                         \
    hipError_t e_ = (expr);                                    \
    if (e_ != hipSuccess) {                                    \
      cleanup();                                               \
      return fail(ICON_ERR_DEVICE, "%s: %s", #expr, hipGetErrorString(e_)); \
    }                                                          \
  } while (0)
  TRY(hipMalloc(&ds, nsino * sizeof(float)));
  TRY(hipMalloc(&dm, nimg * sizeof(float)));
  if (m_init) TRY(hipMalloc(&dmi, nimg * sizeof(float)));
  if (reproj) TRY(hipMalloc(&drp, (size_t)S * g.N0 * sizeof(float)));
  if (resid) TRY(hipMalloc(&drs, (size_t)S * (iters + 1) * sizeof(double)));
  if (alpha && iters > 0) TRY(hipMalloc(&dal, (size_t)S * iters * sizeof(double)));
  TRY(hipMemcpy(ds, sino, nsino * sizeof(float), hipMemcpyHostToDevice));
  if (m_init) TRY(hipMemcpy(dmi, m_init, nimg * sizeof(float), hipMemcpyHostToDevice));
  rc = icon_reconstruct(p, S, ds, dm, dmi, drp, drs, dal, opts, nullptr);
  if (rc) { cleanup(); return rc; }
  TRY(hipDeviceSynchronize());
  TRY(hipMemcpy(m, dm, nimg * sizeof(float), hipMemcpyDeviceToHost));
  if (reproj) TRY(hipMemcpy(reproj, drp, (size_t)S * g.N0 * sizeof(float), hipMemcpyDeviceToHost));
  if (resid) TRY(hipMemcpy(resid, drs, (size_t)S * (iters + 1) * sizeof(double), hipMemcpyDeviceToHost));
  if (alpha && iters > 0) TRY(hipMemcpy(alpha, dal, (size_t)S * iters * sizeof(double), hipMemcpyDeviceToHost));
#undef TRY
  cleanup();
  return ICON_OK;
}

int icon_time_kernel(icon_plan* p, int kernel, int S, int reps, double* avg_ms) {
  if (!p || !avg_ms || reps < 1) return fail(ICON_ERR_ARG, "icon_time_kernel: bad argument");
  if (S < 1 || S > p->S_max) return fail(ICON_ERR_CAPACITY, "batch %d outside 1..%d", S, p->S_max);
  if (kernel < ICON_K_ROW_FWD || kernel > ICON_K_COL_ENERGY)
    return fail(ICON_ERR_ARG, "icon_time_kernel: unknown kernel %d", kernel);
  DevGuard dg(p->device);
  const Geometry& g = p->g;
  hipStream_t st = p->stream;
  p->data_sino = nullptr;   // the timed kernels overwrite the solve's data buffers
  RowFwdArgs rf{};
  // the row pass with the ICON update fused, as in every iteration after the
  // first; the image it updates lives in the (then stale) A^H W b buffer
  rf.rows = S * g.N0; rf.N0 = g.N0; rf.N1 = g.N1; rf.cplx = 0; rf.update = 2; rf.data_type = 1;
  rf.m = reinterpret_cast<float*>(p->d_ahwb); rf.grad = p->d_grad; rf.alpha = p->d_alpha;
  rf.tw = p->d_tw1; rf.out = p->d_tmp;
  rf.mref = p->d_mref;   // as in the iterations after the first FP64 gradient (n0 = 2048: null)
  ColArgs cn = normal_args(p, S, true);
  const ColArgs ce = energy_args(p, S);
  RowAdjArgs ra = grad_args(p, S);
  split_dense(p, S, cn, ra);
  // (the residuals of these stale values go to the bnorm buffer, rewritten by the next solve's set-up)
  FinishArgs fr = finish_args(p, S);
  fr.resid = p->d_bnorm; fr.resid_stride = 1; fr.alpha = p->d_alpha;
  FinishArgs fs = fr;
  fs.resid = nullptr;
  // the transforms' column kernels: interpolation and spread of the plan's window
  const ColArgs ca = window_args(p, p->op, S);
  SinoArgs sa{};
  sa.K = p->g.K;
  sa.rows = S * g.nz; sa.N0 = g.N0; sa.sino = reinterpret_cast<const float*>(p->d_b); sa.ck1 = p->d_ck1;
  sa.phi1 = p->d_phi1; sa.i10 = p->d_i10; sa.tw = p->d_tw0; sa.b = p->d_fw;
  auto launch = [&](int k) -> hipError_t {
    switch (k) {
      case ICON_K_ROW_FWD: return iter_row_fwd(p, rf, st);
      case ICON_K_COL_FWD: return launch_col(g.n0, p->op.h.C, false, ca, st);
      case ICON_K_COMBINE: return launch_finish(fr, st);
      case ICON_K_COL_ADJ: return launch_col(g.n0, p->op.h.C, true, ca, st);
      case ICON_K_ROW_ADJ: return iter_row_grad(p, ra, st);
      case ICON_K_SINO: return launch_sino(g.n0, sa, st);
      case ICON_K_COMBINE_ALPHA: return launch_finish(fs, st);
      case ICON_K_COL_NORMAL: return launch_col_normal(g.n0, cn, st);
      case ICON_K_COL_ENERGY: return launch_col_energy(g.n0, ce, st);
      default: return hipErrorInvalidValue;
    }
  };
  // The launch sequence of one iteration (with a residual), as the solve
  // enqueues it; the timed kernel runs inside it, so that each timed launch
  // finds its input as in a solve (just written by its predecessor, partly in
  // the caches) and the device busy (an idle gap before a launch lowers the
  // clock it starts at).  The transforms' column kernels are timed between the
  // row passes that precede them; the sinogram transform, which runs once per
  // solve, back to back.
  const int iter_seq[] = {ICON_K_ROW_FWD, ICON_K_COL_NORMAL, ICON_K_ROW_ADJ, ICON_K_COL_ENERGY, ICON_K_COMBINE};
  const int alpha_seq[] = {ICON_K_ROW_FWD, ICON_K_COL_NORMAL, ICON_K_ROW_ADJ, ICON_K_COL_ENERGY, ICON_K_COMBINE_ALPHA};
  const int op_seq[] = {ICON_K_ROW_FWD, ICON_K_COL_FWD, ICON_K_COL_ADJ, ICON_K_ROW_ADJ};
  const int sino_seq[] = {ICON_K_SINO};
  const int* seq = iter_seq;
  int nseq = 5;
  if (kernel == ICON_K_COMBINE_ALPHA) seq = alpha_seq;
  if (kernel == ICON_K_COL_FWD || kernel == ICON_K_COL_ADJ) seq = op_seq, nseq = 4;
  if (kernel == ICON_K_SINO) seq = sino_seq, nseq = 1;
  // Each timed launch carries events that take the kernel's own start and end
  // (hipExtLaunchKernel), not those of extra marker packets around it; all
  // launches are enqueued before one synchronisation.
  std::vector<hipEvent_t> ev(2 * (size_t)reps, nullptr);
  hipError_t e = hipSuccess;
  for (size_t i = 0; i < ev.size() && e == hipSuccess; i++) e = hipEventCreate(&ev[i]);
  for (int i = 0; i < nseq && e == hipSuccess; i++) e = launch(seq[i]);  // untimed warm-up pass
  for (int r = 0; r < reps && e == hipSuccess;) {
    for (int i = 0; i < nseq && e == hipSuccess; i++) {
      const bool timed = seq[i] == kernel && r < reps;
      if (timed) set_launch_events(ev[2 * r], ev[2 * r + 1]);
      e = launch(seq[i]);
      if (timed) {
        set_launch_events(nullptr, nullptr);
        r++;
      }
    }
  }
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  std::vector<float> t(reps, 0.f);
  for (int r = 0; r < reps && e == hipSuccess; r++) e = hipEventElapsedTime(&t[r], ev[2 * r], ev[2 * r + 1]);
  for (hipEvent_t x : ev)
    if (x) (void)hipEventDestroy(x);
  if (e != hipSuccess) return fail(ICON_ERR_DEVICE, "icon_time_kernel: %s", hipGetErrorString(e));
  // median launch duration: robust to a launch slowed by other work on the device
  std::sort(t.begin(), t.end());
  *avg_ms = reps % 2 ? t[reps / 2] : 0.5 * ((double)t[reps / 2 - 1] + t[reps / 2]);
  return ICON_OK;
}

int icon_plan_autotune(icon_plan* p, int S, int* col_block, double* ms_per_width) {
  if (!p || !col_block) return fail(ICON_ERR_ARG, "icon_plan_autotune: null pointer");
  const int widths[2] = {8, 16};
  double best = 0.0;
  int best_c = 0;
  for (int i = 0; i < 2; i++) {
    const int C = widths[i];
    if (ms_per_width) ms_per_width[i] = 0.0;
    if (!col_tile_ok(p->g.n0, p->g.n1, C, op_taps(p->g))) continue;
    int rc = icon_plan_set_col_block(p, C);
    double tf = 0.0, ta = 0.0;
    if (!rc) rc = icon_time_kernel(p, ICON_K_COL_FWD, S, 3, &tf);
    if (!rc) rc = icon_time_kernel(p, ICON_K_COL_ADJ, S, 3, &ta);
    if (rc) return rc;
    const double t = tf + ta;
    if (ms_per_width) ms_per_width[i] = t;
    if (best_c == 0 || t < best) { best = t; best_c = C; }
  }
  if (best_c == 0) return fail(ICON_ERR_ARG, "icon_plan_autotune: no supported column tile");
  if (p->op.h.C != best_c) {
    const int rc = icon_plan_set_col_block(p, best_c);
    if (rc) return rc;
  }
  *col_block = best_c;
  return ICON_OK;
}

int icon_copy_probe(void* d_dst, const void* d_src, size_t bytes, int reps, double* avg_ms) {
  if (!d_dst || !d_src || !avg_ms || reps < 1 || bytes % 16 != 0)
    return fail(ICON_ERR_ARG, "icon_copy_probe: bad argument (bytes must be a multiple of 16)");
  hipEvent_t e0, e1;
  HIPCHK(hipEventCreate(&e0));
  HIPCHK(hipEventCreate(&e1));
  hipError_t e = launch_copy4((float4*)d_dst, (const float4*)d_src, bytes / 16, nullptr);
  if (e == hipSuccess) e = hipEventRecord(e0, nullptr);
  for (int r = 0; r < reps && e == hipSuccess; r++) e = launch_copy4((float4*)d_dst, (const float4*)d_src, bytes / 16, nullptr);
  if (e == hipSuccess) e = hipEventRecord(e1, nullptr);
  if (e == hipSuccess) e = hipEventSynchronize(e1);
  float ms = 0.f;
  if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (e != hipSuccess) return fail(ICON_ERR_DEVICE, "icon_copy_probe: %s", hipGetErrorString(e));
  *avg_ms = (double)ms / reps;
  return ICON_OK;
}

}  // extern "C"
