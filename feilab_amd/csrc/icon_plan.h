// Internal plan state of the MI355X ICON core (host side).
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>
#include <string>
#include <vector>

#include "../../include/icon_mi355x.h"

namespace icon {

constexpr int kTaps = 14;      // Gaussian window: 2m+2, m = 6 (nufft_gpu_v8.cuh:5)
constexpr int kWindowM = 6;
constexpr int kTapsKB = 6;     // Kaiser-Bessel window of width 6
// The device's window of the default (Gaussian) plans: Kaiser-Bessel of width
// 10.  Its transforms are within 1e-9 of the exact ones before rounding (the
// 14-tap Gaussian: 7e-7 rms, 3.5e-6 at most) from fewer taps and column tiles.
constexpr int kTapsWide = 10;
constexpr int kSolveTile = 8;  // grid columns per tile of the solve's data set-up
constexpr int kMaxSlot = 3;    // node y-taps split over at most 3 column tiles (tile >= 8)

// Host-side geometry of one tilt series, computed exactly as the reference's
// setup does (float/double placement included).
struct Geometry {
  int N0 = 0, N1 = 0, nz = 0, M = 0, n0 = 0, n1 = 0;
  int window = ICON_WINDOW_GAUSS;  // ICON_WINDOW_GAUSS or ICON_WINDOW_KB6
  int K = kTaps;                  // taps per dimension of the window: 14 (Gaussian) or 6 (Kaiser-Bessel); the
                                  // projection rows' 1D transform uses it
  // window shape per dimension: Gaussian b and bf, or Kaiser-Bessel beta (b)
  float sig0 = 0, sig1 = 0, b0 = 0, b1 = 0, bf0 = 0, bf1 = 0;
  int iomit = 0;                  // tilt whose nodes give the reprojection
  float omit = 0;
  int cv_skip = -1;               // cross-validation plan: input row left out of the data, else -1
  std::vector<float> theta;       // negated angles (MainCode.cu:42)
  std::vector<float> nodes;       // 2*M, (x, y) per node j = i*N0 + k
  std::vector<float> w;           // M density weights
  std::vector<float> ck;          // N0*N1 deapodisation, index X*N1+Y
  std::vector<float> ck1;         // N0
  std::vector<float> phix, phiy;  // M*K window taps
  std::vector<int> ix0, iy0;      // M: wrapped first tap index
  std::vector<float> phi1;        // N0*K (1D plan)
  std::vector<int> i10;           // N0
};

// Column-tile bin lists for the spread / interpolation with a window of K taps.
// An entry is (node j, t0 | t1<<8 | slot<<16 | col0<<24, first x-tap x0, tile).
struct Bins {
  int C = 16;                     // grid columns per tile
  int K = 0;                      // window taps per dimension
  int nblk = 0;                   // n1 / C
  std::vector<int> off;           // nblk+1
  std::vector<int4> ent;          // a tile's entries are sorted by x0 (then node)
  std::vector<int> xoff;          // nblk*(n0+1): first entry of the tile with x0 >= x
  std::vector<int8_t> nslot;      // M
  std::vector<int> of_node;       // M*3: entries of node j by slot (-1: none)
  // The same entries in the interpolation's order: within a tile, groups of 16
  // entries whose first x-taps differ mod 16 where possible.
  std::vector<int4> fent;
  // Launch order of the spread's tiles: by entry count, largest first (ties
  // by index).  A spread block costs about its tile's entries, and the few
  // dense tiles around ky = 0 (up to 10x the median block) would otherwise
  // run at the start and the very end of the tile-major order, the last of
  // them alone on a nearly idle device.
  std::vector<int> order;
};

// Bins and their device tables.  The records (K x-taps of the entry's node, C
// y-taps, zero outside the run) are computed on the device, interleaved by
// field per tile.
struct DevBins {
  Bins h;
  float beta0 = 0, beta1 = 0;     // Kaiser-Bessel shape per dimension
  float* ck = nullptr;            // [N0][N1] deapodisation
  int* off = nullptr;
  int* order = nullptr;
  int* xoff = nullptr;
  int* of_node = nullptr;
  int4* ent = nullptr;
  int4* fent = nullptr;
  float *px = nullptr, *py = nullptr, *fpx = nullptr, *fpy = nullptr;
  int8_t* nslot = nullptr;
  int* parts = nullptr;           // shares of a tile's entries, and the further ones
  int2* xt = nullptr;
  int nx = 0;
};

// Entries of the solve's interpolation (16 taps, tiles of 8 columns): per tile
// (node row, t0 | t1<<8 | slot<<16 | col0<<24, first x-tap, tile and flags), in
// the interpolation's order (groups of 16 whose first x-taps differ mod 16
// where possible); the records are computed from them on the device.
// On a full grid every node is a row.  With paired nodes (paired_nodes) the
// grid holds columns 0..n1/2 of a real image's transform, the rows are those of
// node_of in icon_normal.hip (per tilt line the nodes N0/2..N0-1, then node 0),
// and an entry's w carries, beside the tile, bit 16: the node mirrored into the
// half that is stored, bit 17: columns that stand for their mirror images
// (descending, x-taps reversed), bit 31: the value is to be conjugated.
struct NodeBins {
  std::vector<int> off;           // tiles + 1
  std::vector<int4> ent;
  std::vector<int8_t> nslot;      // node rows
};
constexpr int kNodeSlots = 4;     // tiles (and mirrored runs) per node row, at most

// The grid columns [zlo, zhi) (FFT order, a multiple of C at both ends) of
// the run of column tiles without bin entries around column n1/2.  Every
// tilt line's nodes reach ky in [-k, k], so the tiles the nodes reach form a
// band around column 0 and the free ones a run around n1/2.  Spread grids
// are zero there and no interpolation reads a forward grid there, so the
// row kernels neither load nor store those columns and the spread kernel
// does not write them.  Empty (0, 0) when the tile holding column n1/2 is
// reached.
inline void zero_band(const Bins& b, int* zlo, int* zhi) {
  *zlo = *zhi = 0;
  const int mid = b.nblk / 2;
  auto empty = [&](int t) { return b.off[t] == b.off[t + 1]; };
  if (b.nblk < 2 || !empty(mid)) return;
  int lo = mid, hi = mid + 1;
  while (lo > 0 && empty(lo - 1)) lo--;
  while (hi < b.nblk && empty(hi)) hi++;
  *zlo = lo * b.C;
  *zhi = hi * b.C;
}

// Entry count from which a spread tile splits each row pair's entries
// between two threads: twice the median count of the tiles that have
// entries, so that only the dense tiles around ky = 0 reach it (22 of the
// 114 tiles with entries at 512^2, 41 tilts +-60 deg; 1.5x the median, 38
// tiles, and 3x, 8 tiles, measured slower).
inline int split_min_entries(const Bins& b) {
  std::vector<int> n;
  for (int t = 0; t < b.nblk; t++)
    if (b.off[t + 1] > b.off[t]) n.push_back(b.off[t + 1] - b.off[t]);
  if (n.empty()) return 0x7fffffff;
  std::nth_element(n.begin(), n.begin() + n.size() / 2, n.end());
  return std::max(1, 2 * n[n.size() / 2]);
}

// Fills g; returns false (with a message) on an invalid geometry.  Without
// tables the 2D window taps and deapodisation are left out (a plan computes
// its own on the device).
bool build_geometry(Geometry& g, int N0, int N1, int nz, const float* tilt_deg, std::string* err, bool cv = false,
                    int window = ICON_WINDOW_GAUSS, bool tables = true);
void build_bins(const Geometry& g, int C, int K, Bins& b);
// Kaiser-Bessel window of W taps: its shape for oversampling sigma, and its
// deapodisation over N samples.
float kb_beta(float sigma, int W);
void kb_deapod(int N, float sigma, float beta, int W, float* out);
// The reprojection's 1D window, kTapsWide taps: deapodisation [N0], taps [N0][K]
// and first taps [N0].
void reproj_tables(const Geometry& g, std::vector<float>& ck, std::vector<float>& phi, std::vector<int>& first);
// Every tilt line's nodes but the first in exact pairs (v, -v) of equal weight.
bool paired_nodes(const Geometry& g);
void build_node_bins(const Geometry& g, bool half, NodeBins& b);
// The entries of the unpaired nodes alone, rows renumbered to the tilt line.
void unpaired_bins(const Geometry& g, const NodeBins& b, NodeBins& u);
// Cholesky factor (16 x 16 row-major, the diagonal inverted) of the matrix
// sinc((p - q)/2)/2 of the interpolation's taps.
void interp_factor(double* l);
void grid_size(int N, float* sigma, int* n);
// Twiddle table of a power-of-two length (icon_fft.h) on the current device.
int fft_twiddles(int n, const float2** out);
// Sets the message icon_last_error() returns on the calling thread.
void set_last_error(const char* msg);

struct GraphKey {
  int S = -1;
  const void* sino = nullptr;
  void* m = nullptr;
  const void* m_init = nullptr;
  void* reproj = nullptr;
  void* resid = nullptr;
  void* alpha = nullptr;
  int pre = 0, icon = 0, post = 0, data_type = 0, reuse = 0;
  float thr = 0;
  bool operator==(const GraphKey& o) const {
    return S == o.S && sino == o.sino && m == o.m && m_init == o.m_init && reproj == o.reproj &&
           resid == o.resid && alpha == o.alpha && pre == o.pre && icon == o.icon &&
           post == o.post && data_type == o.data_type && reuse == o.reuse && thr == o.thr;
  }
};

// A few captured solves per plan (a warm-started solve alternates between two
// or three schedules); least recently used is replaced.
constexpr int kGraphCache = 4;

}  // namespace icon

// Opaque plan of the C ABI.
struct icon_plan {
  int device = 0;
  icon::Geometry g;
  int S_max = 0;
  hipStream_t stream = nullptr;     // plan-owned stream (capturable)
  hipEvent_t ev_in = nullptr, ev_out = nullptr;
  // the transforms' window: bins and tables; data: those of the solve's data
  // set-up (kTapsWide, kSolveTile) where the transforms' are others (else op's)
  icon::DevBins op, data;
  bool own_data = false;
  icon::DevBins& spread() { return own_data ? data : op; }
  // shared tables
  float2* d_nodes = nullptr;        // [M]
  float* d_ck1 = nullptr;
  float* d_w = nullptr;
  float* d_phi1 = nullptr;
  int* d_i10 = nullptr;
  float* d_rck = nullptr;           // the reprojection's window (null where N0 is a power of two: it needs none)
  float* d_rphi = nullptr;
  int* d_ri0 = nullptr;
  // the solve's normal operator (icon_normal.hip)
  bool half = false;                // paired nodes: real images on half grids
  int nq = 0;                       // ... and its unpaired nodes
  int rows = 0;                     // node rows of d_part
  int ncol = 0;                     // grid columns: n1, or n1/2 + 8
  // FP64 gradients: not at n0 = 2048, whose column kernel (1024 threads, 128
  // registers, 424 bytes of scratch per lane) ended in a memory aperture
  // violation inside a packed graph; its indexes are in bounds on the CPU
  bool refreshes() const { return g.n0 <= 1024; }
  // slices that an FP64 pass takes at once: the grid rows in double of half the
  // slices fit the room of all in single precision
  int S64 = 0;
  int* d_nq_off = nullptr;          // unpaired nodes: entries (rows of d_part / of d_rpart), records
  int4* d_nq_ent = nullptr;
  int4* d_nq_entr = nullptr;
  float* d_nq_px = nullptr;
  float* d_nq_py = nullptr;
  int8_t* d_nq_nslot = nullptr;
  float2* d_rpart = nullptr;        // [S][nq][kNodeSlots]
  float* d_gram = nullptr;          // [2][2 nq][2 nq]
  float* d_spec = nullptr;          // [ncol/8][n0][8] spectrum of A^H W A's kernel
  int* d_nd_off = nullptr;          // NodeBins and their records
  int4* d_nd_ent = nullptr;
  int* d_nd_parts = nullptr;        // shares of a tile's entries, and the further ones (split_dense)
  int2* d_nd_xt = nullptr;
  int nd_nx = 0;
  unsigned long long* d_rsum = nullptr;   // FinishArgs
  unsigned* d_rcnt = nullptr;
  int cus = 256;                    // compute units of the device
  int8_t* d_nd_nslot = nullptr;
  float* d_nd_px = nullptr;
  float* d_nd_py = nullptr;
  double* d_epart = nullptr;        // [S][ncol/8] energies of the gradient by column tile
  const float2* d_tw0 = nullptr;    // twiddles for n0 (shared cache)
  const float2* d_tw1 = nullptr;    // twiddles for n1
  // per-slice work buffers (capacity S_max)
  float2* d_b = nullptr;            // [S][M] Fourier-slice data
  float2* d_part = nullptr;         // [S][M][kMaxSlot] interpolation partials
  float2* d_fw = nullptr;           // the same room, [S][E]: weighted node value of every bin entry (op's or spread()'s)
  float2* d_ahwb = nullptr;         // [S][N0][N1]
  float* d_grad = nullptr;          // [S][N0][N1] Re(rhat), the gradient the update takes
  // [S][N0][n1] row-transform intermediate, or [S64][N0][n1] in double; then room
  // for the grid rows of few slices in split_dense
  float2* d_tmp = nullptr;
  // the reference iterate of the solve's differences: image, -rhat (half: real), b - A m
  float* d_mref = nullptr;
  float2* d_base = nullptr;
  float2* d_beff = nullptr;
  const double2* d_w640 = nullptr;  // FP64 twiddles for n0, n1 (shared cache)
  const double2* d_w641 = nullptr;
  float2* d_frep = nullptr;         // [S][N0] forward values at the omit tilt
  double* d_rowpart = nullptr;      // [S][N0] per-row partial sums
  double* d_bnorm = nullptr;        // [S]
  double* d_alpha = nullptr;        // [S]
  int64_t device_bytes = 0;
  // captured solves
  hipGraphExec_t graph_exec[icon::kGraphCache] = {};
  icon::GraphKey graph_key[icon::kGraphCache];
  int64_t graph_used[icon::kGraphCache] = {};
  int64_t graph_clock = 0;
  // sinograms whose b and A^H W b the per-slice buffers hold (reuse_data)
  const void* data_sino = nullptr;
  int data_S = 0;
};

#include "icon_kernels.h"

namespace icon {
// Arguments of the iteration's kernels over S slices of a plan (icon_capi.cpp).
ColArgs normal_args(const icon_plan* p, int S, bool with_nodes);
ColArgs energy_args(const icon_plan* p, int S);
RowAdjArgs grad_args(const icon_plan* p, int S);
void split_dense(const icon_plan* p, int S, ColArgs& ca, RowAdjArgs& ra);
// (of S slices from s0 on, at most S64: an FP64 pass)
ColArgs normal64_args(const icon_plan* p, int s0, int S, bool with_nodes);
RefArgs ref_args(const icon_plan* p, int s0, int S, float* m);
RowFwdArgs rhat_row_args(const icon_plan* p, int S);
bool refresh(const icon_plan* p, const icon_solve_opts& o, int it);
FinishArgs finish_args(const icon_plan* p, int S);
ReprojArgs reproj_args(const icon_plan* p, int S, float* out);
ColArgs spread_args(icon_plan* p, int s0, int S);   // of the data set-up
RowAdjArgs data_row_args(icon_plan* p, int s0, int S);
}  // namespace icon
