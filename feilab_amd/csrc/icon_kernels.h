// Kernel argument blocks and launchers of the ICON core (host + device view).
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>

namespace icon {

constexpr int kMaxSlotK = 3;

struct RowFwdArgs {
  int rows, N0, N1;
  int cplx;        // 0: real image m (with optional update), 1: complex rhat
  int update;      // 0 none, 1 INFR, 2 ICON (threshold)
  int data_type;
  float thr;
  float* m;
  const float2* rhat;   // cplx: the complex image
  const float* grad;    // update: Re(rhat) [S][N0][N1]
  const double* alpha;
  const float* ck;      // divides the image, or null (real image only)
  const float2* tw;
  float2* out;     // [S][N0][NR]
  const float* mref;    // real image: the reference iterate subtracted before the transform, or null
  int zlo, zhi;    // out columns [zlo, zhi) are not stored (no interpolation reads them)
};

struct RowAdjArgs {
  int rows, N0, N1;
  const float2* in;    // [S][N0][NR]
  const float* ck;     // adjoint transform: deapodisation
  const float2* tw;
  float2* img;         // adjoint transform (grad null): the image
  float* img_re;       // ... or, non-null, its real part alone
  const float2* ahwb;  // gradient: A^H W b; rhat = (A^H W A m) - ahwb
  const float* ahwb_re;  // gradient of real rows: Re(A^H W b) [S][N0][N1]
  float* grad;         // gradient: Re(rhat) [S][N0][N1], all the update reads
  double* rowpart;     // gradient: sum |rhat|^2 per row (real rows: per row pair)
  float2* fwd_out;     // gradient: y-FFT of rhat padded to NR, per row [S][N0][NR]
  int zlo, zhi;        // columns [zlo, zhi) of in are zero (not loaded)
  const double2* in64; // row_adj64: [S][N0][NR]
  const double2* w64;  // row_adj64: exp(-2 pi i q / NR)
};

struct ColArgs {
  int S, N0, N1, M, n1, E;
  int K;                   // window taps per dimension
  const float2* in;        // fwd: tmp [S][N0][n1]
  float2* out;             // adj: tmp [S][N0][n1]
  const float2* tw;
  const int* ent_off;
  const int* tile_order;   // adj: [nblk] tile of each block group (blocks bid / S), largest first
  const int4* ent;
  const int* xoff;         // adj: [nblk][n0+1] row offsets into ent
  const float* ent_px;     // [E][K], interleaved per tile
  const float* ent_py;     // [E][C], interleaved per tile
  // fwd: the entries and their records in the interpolation's order
  const int4* fent;
  const float* fent_px;
  const float* fent_py;
  float2* part;            // fwd: [S][M][3]
  const float2* fw;        // adj: [S][E] weighted value per bin entry
  int zlo, zhi;            // adj: tiles inside columns [zlo, zhi) store nothing (their zeros are implied)
  int split_min;           // adj: tiles with at least this many entries split their rows' entries in two
  // normal operator (col_normal, col_energy)
  const float* spec;       // [n1/C][n0][C] spectrum of A^H W A's kernel over n0 n1
  double* epart;           // col_energy: [S][n1/C] sums of spec |x|^2
  double2* io64;           // col_normal64: the grid rows [S][N0][n1], in place
  const double2* w64;      // col_normal64: exp(-2 pi i q / n0)
  int slots;               // partials per node in part
  int nyq;                 // half grid: its column n1/2; otherwise 0
  // col_normal, col_fwd, few slices: shares of the dense tiles' entries in blocks of
  // their own (col_normal: out then is not in): shares per tile, and (tile, share > 0) of
  // the nx further blocks per slice
  const int* parts;
  const int2* xt;
  int nx;
};

struct CombineArgs {
  int S, M, N0, nz, E;
  int mode;              // 2: initial b (weights, bnorm), 3: node values of a forward transform
  const float2* part;    // [S][M][3]
  const int8_t* nslot;
  const float* w;
  const float2* b;       // [S][M]
  float2* fw;            // mode 2: [S][E] weighted value per bin entry; mode 3: [S][M] sums
  const int* ent_of_node;  // [M][3] bin entries of each node
  double* bnorm;         // [S]
};

// An iterate's gradient in FP64 (k_row_fwd64, k_row_grad64): the update and the
// transform of the whole image, and the gradient, which becomes the reference of
// the iterations that follow.
struct RefArgs {
  int rows, N0, N1, ncol;
  int update, data_type;   // as RowFwdArgs
  float thr;
  float* m;
  float* mref;             // the iterate as the reference
  const double* alpha;
  const double2* w64;      // exp(-2 pi i q / n1)
  double2* io;             // grid rows [S][N0][ncol]
  const float2* ahwb;      // A^H W b (half: its real part)
  const float* ahwb_re;
  float* grad;             // Re(rhat): the update's gradient (in: of the last iterate)
  float2* base;            // -rhat (half: base_re, -Re(rhat))
  float* base_re;
  double* rowpart;
};

// Unpaired nodes (tilt lines) up to which a plan takes the real-gradient path.
constexpr int kMaxUnpaired = 256;

// End of an iteration: the data residual of the image (from the node partials
// of A m) and the step size of the gradient.
constexpr int kFinishGroups = 16;
constexpr int kFinishRows = 4096;   // rows of a group's round
struct FinishArgs {
  int S, M, N0, nblk, nrow;   // M: rows of part per slice
  int Mb;                // nodes per slice in b
  int slots;             // partials per node
  const float2* part;    // [S][M][slots]
  const int8_t* nslot;
  const float* w;
  const float2* b;       // [S][Mb]
  const double* bnorm;   // [S]
  unsigned long long* rsum;   // [S][kFinishGroups] sums of the residual's row groups (double bits)
  unsigned* rcnt;             // [S] blocks done, zero between launches
  int groups;                 // groups of the residual's rows, at most kFinishGroups
  int blocks;                 // blocks per slice that share them, at most groups
  double* resid;         // trace base or null
  int resid_stride, resid_index;
  float2* frep;          // [S][N0] values of A m at the omit tilt, or null
  int iomit;
  const double* rowpart; // [S][nrow] sums of |rhat|^2
  const double* epart;   // [S][nblk] sums of spec |rhat|^2
  double* alpha;         // [S]
  double* alpha_trace;   // [S][iters] or null
  int alpha_stride, alpha_index;
  // paired nodes (real gradient): the tilt lines, partials of A Re(rhat) at
  // their unpaired nodes, the waves' Gram matrix and their A^H W A products
  int nq;
  const float2* rpart;   // [S][nq][slots]
  const int8_t* rslot;
  const float* gram;     // [2][2 nq][2 nq]
  float2* beff;          // b - A m of these node values, for the iterations that follow, or null
};

struct SinoArgs {
  int rows, N0;
  int K;                 // window taps
  int nz, skip;          // tilts per slice; input row left out (cross validation), else -1
  const float* sino;     // [S][nz][N0]
  const float* ck1;
  const float* phi1;
  const int* i10;
  const float2* tw;
  float2* b;             // [S][nz*N0]
};

struct ReprojArgs {
  int S, N0;
  int K;                 // window taps (N0 a power of two: no window, its tables null)
  float sigma;
  const float2* frep;    // [S][N0]
  const float* ck;
  const float* phi;
  const int* i0;
  const float2* tw;
  float* out;            // [S][N0]
};

// Per-launch fields of a packed launch over several series (the argument
// blocks of the series are read from a device table).
struct RowFwdLaunch {
  int cplx, update, data_type;
  float thr;
};

struct FinishLaunch {
  int resid_index, alpha_index;   // < 0: no residual / no step size
  int with_frep;                  // 0: the series' frep pointers are ignored
  int beff;                       // 0: not used; 1: written; 2: read in place of b
  int blocks;                     // the largest of the series' blocks
};

// While set (non-null) on the calling thread, the next launches of the
// iteration kernels (row_fwd, col, combine, row_adj, sino) go through
// hipExtLaunchKernel with these events, which then hold the kernel's own start
// and end on the device clock. Used only for timing, never under capture.
void set_launch_events(hipEvent_t start, hipEvent_t stop);
extern thread_local hipEvent_t t_ev_start, t_ev_stop;
// hipLaunchKernelGGL, or, while timing events are set, hipExtLaunchKernelGGL
// with them (the events then bracket the kernel itself, not the enqueue)
#define LAUNCH_TIMED(KERNEL, GRID, BLOCK, SHM, ST, ...)                                          \
  do {                                                                                           \
    if (t_ev_start)                                                                              \
      hipExtLaunchKernelGGL(KERNEL, GRID, BLOCK, SHM, ST, t_ev_start, t_ev_stop, 0, __VA_ARGS__); \
    else                                                                                         \
      hipLaunchKernelGGL(KERNEL, GRID, BLOCK, SHM, ST, __VA_ARGS__);                             \
  } while (0)

hipError_t launch_row_fwd(int NR, const RowFwdArgs& a, hipStream_t st);
hipError_t launch_row_adj(int NR, const RowAdjArgs& a, hipStream_t st);
hipError_t launch_col(int NC, int C, bool adjoint, const ColArgs& a, hipStream_t st);
hipError_t launch_combine(const CombineArgs& a, hipStream_t st);
hipError_t launch_sino(int NR, const SinoArgs& a, hipStream_t st);
hipError_t launch_reproj(int NR, const ReprojArgs& a, hipStream_t st);
hipError_t launch_fft_rows(int NR, float2* data, int rows, int sign, const float2* tw, hipStream_t st);
hipError_t launch_fft_cols(int NC, int C, float2* data, int n1, int count, int sign, const float2* tw,
                           hipStream_t st);
hipError_t launch_zero(float* p, size_t n, hipStream_t st);
// fw_ent[s][e] = f[s][node of e]
hipError_t launch_node_to_ent(const float2* f, float2* fw_ent, const int4* ent, int S, int M, int E, hipStream_t st);
hipError_t launch_copy(float* dst, const float* src, size_t n, hipStream_t st);
hipError_t launch_copy4(float4* dst, const float4* src, size_t n, hipStream_t st);
// Packed launches: `n` blocks, block b running block items[b].y of the series
// descs[items[b].x] (both tables in device memory).  Rows per block of the
// row kernels (the unit of their items) by row length:
int row_fwd_rows_per_block(int NR);
int row_adj_rows_per_block(int NR);
int sino_rows_per_block(int NR);
hipError_t launch_row_fwd_multi(int NR, const RowFwdArgs* descs, const int2* items, int n, const RowFwdLaunch& L,
                                hipStream_t st);
hipError_t launch_row_adj_multi(int NR, const RowAdjArgs* descs, const int2* items, int n, bool grad,
                                hipStream_t st);
hipError_t launch_col_adj_multi(int NC, const ColArgs* descs, const int2* items, int n, hipStream_t st);
hipError_t launch_combine_multi(const CombineArgs* descs, const int2* items, int n, hipStream_t st);
hipError_t launch_sino_multi(int NR, const SinoArgs* descs, const int2* items, int n, hipStream_t st);
hipError_t launch_reproj_multi(int NR, const ReprojArgs* descs, const int2* items, int n, hipStream_t st);
// Normal operator of the solve (icon_normal.hip), tiles of kNormalC columns,
// in place on the grid rows: forward x FFT, the interpolation at the entries'
// nodes, the product with the spectrum, inverse x FFT.
constexpr int kNormalC = 8;
constexpr int kInterpTaps = 16;   // taps of the solve's interpolation
hipError_t launch_col_normal(int NC, const ColArgs& a, hipStream_t st);
// per column tile, sum of spec |x FFT|^2, and the interpolation at the entries' nodes
hipError_t launch_col_energy(int NC, const ColArgs& a, hipStream_t st);
hipError_t launch_finish(const FinishArgs& a, hipStream_t st);
hipError_t launch_col_normal_multi(int NC, const ColArgs* descs, const int2* items, int n, hipStream_t st);
hipError_t launch_col_energy_multi(int NC, const ColArgs* descs, const int2* items, int n, hipStream_t st);
hipError_t launch_finish_multi(const FinishArgs* descs, const int2* items, int n, const FinishLaunch& L,
                               hipStream_t st);
// The same iteration in FP64 from the whole image (its row kernels take full and half grids)
hipError_t launch_col_normal64(int NC, const ColArgs& a, hipStream_t st);
hipError_t launch_row_fwd64(int NR, bool half, const RefArgs& a, hipStream_t st);
hipError_t launch_row_grad64(int NR, bool half, const RefArgs& a, hipStream_t st);
hipError_t launch_col_normal64_multi(int NC, const ColArgs* descs, const int2* items, int n, hipStream_t st);
hipError_t launch_row_fwd64_multi(int NR, bool half, const RefArgs* descs, const int2* items, int n,
                                  const RowFwdLaunch& L, hipStream_t st);
hipError_t launch_row_grad64_multi(int NR, bool half, const RefArgs* descs, const int2* items, int n, hipStream_t st);
// Real rows, two per transform (half grids of n1/2 + 8 columns)
int half_row_pairs_per_block(int NR);
hipError_t launch_row_fwd_half(int NR, const RowFwdArgs& a, hipStream_t st);
hipError_t launch_row_grad_half(int NR, const RowAdjArgs& a, hipStream_t st);
hipError_t launch_row_fwd_half_multi(int NR, const RowFwdArgs* descs, const int2* items, int n, const RowFwdLaunch& L,
                                     hipStream_t st);
hipError_t launch_row_grad_half_multi(int NR, const RowAdjArgs* descs, const int2* items, int n, hipStream_t st);
hipError_t launch_col_fwd_nodes_multi(int NC, const ColArgs* descs, const int2* items, int n, hipStream_t st);
hipError_t launch_col_fwd_nodes(int NC, const ColArgs& a, hipStream_t st);
// A^H of the weighted data in FP64 (rows [S][N0][n1] in io64 / in64)
hipError_t set_adj64_attrs();
hipError_t launch_col_adj64(int NC, int C, const ColArgs& a, hipStream_t st);
hipError_t launch_row_adj64(int NR, const RowAdjArgs& a, hipStream_t st);
hipError_t launch_col_adj64_multi(int NC, int C, const ColArgs* descs, const int2* items, int n, hipStream_t st);
hipError_t launch_row_adj64_multi(int NR, const RowAdjArgs* descs, const int2* items, int n, hipStream_t st);
hipError_t set_normal_attrs(int NC);
hipError_t set_col_fwd_nodes_attrs(int NC);
// Records of the solve's interpolation for E entries (ent: node row, y-tap
// run, first x-tap, tile and flags) from the nodes: E x 16 x-taps and E x 8
// y-taps, interleaved by field per tile.  half: N0/2 where the node rows are
// those of paired nodes, else 0.  chol: interp_factor's.
hipError_t launch_interp_records(const int4* ent, const int* ent_off, const float2* nodes, int E, int n0, int n1,
                                 int half, const double* chol, float* px, float* py, hipStream_t st);
// Records of a Kaiser-Bessel window of K taps for E entries in tiles of C
// columns; out[X][Y] = cx[X] cy[Y].
hipError_t launch_window_records(const int4* ent, const int* ent_off, const float2* nodes, int E, int n0, int n1,
                                 int K, int C, float beta0, float beta1, float* px, float* py, hipStream_t st);
hipError_t launch_outer(const float* cx, const float* cy, int N0, int N1, float* out, hipStream_t st);
// acc[z][q0][q1] += sum over nodes j of [j0, j0 + cnt) of w_j D0(q0/n0 - x_j) D1(q1/n1 - y_j) in FP64,
// over spectrum_splits(n0, n1) splits z (scratch: d0 [cnt'][n0] and d1 [cnt'][n1], cnt' = cnt rounded up to 16)
int spectrum_splits(int n0, int n1);
hipError_t launch_spectrum_chunk(const float2* nodes, const float* w, int j0, int cnt, int N0, int N1, int n0, int n1,
                                 double* d0, double* d1, double* acc, hipStream_t st);
hipError_t launch_spectrum_store(const double* acc, int n0, int n1, bool half, float* spec, hipStream_t st);
// Waves of the nq unpaired nodes: their Gram matrix g, and h = their products
// under A^H W A, acc [splits][ld][ld] += over nodes (scratch fw, f: [2 cnt'][ld])
hipError_t launch_wave_gram(const float2* nodes, int nq, int N0, int N1, float* g, hipStream_t st);
hipError_t launch_wave_chunk(const float2* nodes, const float* w, int j0, int cnt, int nq, int ld, int N0, int N1,
                             double* fw, double* f, double* acc, hipStream_t st);
hipError_t launch_wave_store(const double* acc, int nq, int ld, float* h, hipStream_t st);
bool col_config_ok(int NC, int C, int K);
// A column tile of C grid columns usable on an n0 x n1 grid with K taps.
bool col_tile_ok(int NC, int n1, int C, int K);
hipError_t set_col_attrs(int NC, int C, int K);
hipError_t set_col_adj_multi_attrs();

}  // namespace icon
