// The solve's normal operator A^H W A as the convolution that it is.
//
// With nodes v_j and weights w_j, (A^H W A m)(x) = sum_x' k(x - x') m(x') with
// k(l) = sum_j w_j exp(2 pi i v_j l), a Hermitian kernel of the tilt geometry
// alone.  The lags of two N0 x N1 images fit the oversampled n0 x n1 grid
// (n >= 2 N), so the product with the kernel's (real) spectrum on that grid is
// the operator exactly, without the spread and the interpolation of a NUFFT
// pair and their window error:
//
//   spec(q) = 1/(n0 n1) sum_j w_j D0(q0/n0 - v_jx) D1(q1/n1 - v_jy),
//   D(t) = sum_{|l| < N} exp(-2 pi i t l) = sin((2N-1) pi t) / sin(pi t).
//
// The spectrum is computed once per plan in FP64 (k_dirichlet, k_spectrum) and
// stored in single precision.  Also <r, A^H W A r> = sum_q spec(q) |r^(q)|^2
// n0 n1 / (n0 n1), so the step size needs one forward transform of the gradient and
// no node values at all.
//
// Per iteration: k_row_fwd (update, y FFT of the image) -> k_col_normal (x FFT,
// product, inverse x FFT, in place; the values at the nodes for the data
// residual are interpolated from the same tile where a residual is asked for)
// -> k_row_adj (inverse y FFT, gradient, y FFT of the gradient) ->
// k_col_energy (x FFT, weighted energy) -> k_finish (residual, step size).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>

#include "icon_col.h"
#include "icon_fft.h"
#include "icon_kernels.h"

namespace icon {

// The spectrum's factors for thread (c, t): element in_index(t, r) of column
// c of tile blk, from the tile-contiguous spectrum (a wavefront reads 256
// consecutive bytes per slot, shared in L2 by the slices in flight).
template <int NC, int C>
__device__ __forceinline__ void load_spec(float (&sp)[16], const ColArgs& a, int blk, int c, int t) {
  const float* p = a.spec + (size_t)blk * NC * C + c;
#pragma unroll
  for (int r = 0; r < 16; r++) sp[r] = p[in_index<NC>(t, r) * C];
}

template <int NC, int C, int K>
__device__ __forceinline__ void col_normal_body(const ColArgs& a, int bid) {
  constexpr int LS = col_stride<NC, C>();
  extern __shared__ __align__(16) float2 tile[];   // col_lds<NC, C>()
  // tile-major order, as the transforms' column kernels: blocks in flight
  // together share the tile's spectrum and interpolation records in L2
  int blk = bid / a.S, part = 0, parts = 1;
  const int s = bid % a.S;
  if (a.parts) {
    // blocks past the tiles: a further share of a dense tile's entries
    if (blk >= a.n1 / C) {
      const int2 x = a.xt[blk - a.n1 / C];
      blk = x.x;
      part = x.y;
    }
    parts = a.parts[blk];
  }
  const int y0 = blk * C;
  const int c = threadIdx.x % C, t = threadIdx.x / C;
  float2 v[16];
  col_fft_fwd<NC, C>(v, a, tile, s, y0);
  // v[i] holds element out_index(t, i); the inverse takes element t + r NC/16
  // in slot r: the same elements, permuted
  constexpr int RL = last_radix<NC>();
  float2 u[16];
  if (a.ent_off[blk] != a.ent_off[blk + 1]) {
#pragma unroll
    for (int i = 0; i < 16; i++) tile[out_index<NC>(t, i) * LS + c] = v[i];
    __syncthreads();
    interp_tile<NC, C, K>(a, tile, blk, s, part, parts);
    if (part) return;
    // the column back from the tile rather than held through the interpolation
#pragma unroll
    for (int r = 0; r < 16; r++) u[r] = tile[in_index<NC>(t, r) * LS + c];
  } else {
#pragma unroll
    for (int i = 0; i < 16; i++) u[i / RL + (i % RL) * (16 / RL)] = v[i];
  }
  __syncthreads();   // the tile is consumed before the inverse's exchanges
  // nothing of the inverse is loaded earlier: with the spectrum and all
  // twiddles in flight above, the kernel spilled 60 registers (2.45 ms instead
  // of 1.22 at 512^2 x 256)
  __builtin_amdgcn_sched_barrier(0);
  float sp[16];
  load_spec<NC, C>(sp, a, blk, c, t);
#pragma unroll
  for (int r = 0; r < 16; r++) u[r] = make_float2(u[r].x * sp[r], u[r].y * sp[r]);
  FftTwiddles T;
  fft_from_lazy<NC, ColFftLay<C>, 1, 1>(u, tile + c, t, T, a.tw);
  const auto rs = slice_rows(a.out, a, s);
  typedef __attribute__((ext_vector_type(2))) unsigned u2v;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    if (out_slot_cropped<NC>(i)) continue;   // padding rows, as N0 <= NC/2
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2v, u[i]), rs,
                                          row_offset<NC>(a, t, out_offset<NC>(i), y0 + c), 0, 0);
  }
}

template <int NC, int C, int K>
__global__ __launch_bounds__(C * (NC / 16), 4) void k_col_normal(ColArgs a) {
  col_normal_body<NC, C, K>(a, blockIdx.x);
}

template <int NC, int C, int K>
__global__ __launch_bounds__(C * (NC / 16), 4) void k_col_normal_multi(const ColArgs* __restrict__ descs,
                                                                      const int2* __restrict__ items) {
  const int2 it = items[blockIdx.x];
  const ColArgs a = descs[it.x];
  col_normal_body<NC, C, K>(a, it.y);
}

template <int NC, int C, int K>
__device__ __forceinline__ void col_energy_body(const ColArgs& a, int bid) {
  constexpr int NT = C * (NC / 16);
  constexpr int LS = col_stride<NC, C>();
  extern __shared__ __align__(16) float2 tile[];
  const int blk = bid / a.S;
  const int s = bid % a.S;
  const int c = threadIdx.x % C, t = threadIdx.x / C;
  float2 v[16];
  col_fft_fwd<NC, C>(v, a, tile, s, blk * C);
  if (a.ent_off[blk] != a.ent_off[blk + 1]) {
    // real gradient: its values at the unpaired nodes
#pragma unroll
    for (int i = 0; i < 16; i++) tile[out_index<NC>(t, i) * LS + c] = v[i];
    __syncthreads();
    interp_tile<NC, C, K>(a, tile, blk, s);
    __syncthreads();
  }
  constexpr int RL = last_radix<NC>();
  float sp[16];
  load_spec<NC, C>(sp, a, blk, c, t);
  double acc = 0.0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const float2 x = v[i];
    acc += (double)sp[i / RL + (i % RL) * (16 / RL)] * ((double)x.x * (double)x.x + (double)x.y * (double)x.y);
  }
  // half grid: every column but 0 and n1/2 stands for its mirror image too
  const int y = blk * C + c;
  if (a.nyq && y != 0 && y != a.nyq) acc *= 2.0;
  // FP64 sum over the block in a fixed order: within each wavefront by lane
  // halves, then the wavefronts' sums in order
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) acc += __shfl_down(acc, h);
  double* red = reinterpret_cast<double*>(tile);
  constexpr int NW = (NT + 63) / 64;
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < NW; w++) sum += red[w];
    a.epart[(size_t)s * (a.n1 / C) + blk] = sum;
  }
}

template <int NC, int C, int K>
__global__ __launch_bounds__(C * (NC / 16), 4) void k_col_energy(ColArgs a) {
  col_energy_body<NC, C, K>(a, blockIdx.x);
}

template <int NC, int C, int K>
__global__ __launch_bounds__(C * (NC / 16), 4) void k_col_energy_multi(const ColArgs* __restrict__ descs,
                                                                      const int2* __restrict__ items) {
  const int2 it = items[blockIdx.x];
  const ColArgs a = descs[it.x];
  col_energy_body<NC, C, K>(a, it.y);
}

// ------------------------------------------------ real rows, two per transform
// Where the nodes of every tilt line come in exact pairs v, -v of equal weight
// (N a power of two: the radii k/N - 1/2 are then exact), only the line's first
// node, radius -1/2, is unpaired.  A^H W A of a real image then has the real
// part that the even half of the spectrum gives, and an imaginary part that
// lies in the span of the unpaired nodes' waves,
//   I(x) = sum_t w_t Im(exp(2 pi i v_t x) d_t),  d_t = (A m - b)_t,
// which enters the iteration only through the step size, as quadratic forms of
// the few d_t and (A Re rhat)_t (k_finish).  So the iteration transforms real
// images only: two rows per row FFT, and the grid columns 0..n1/2 (stored in
// n1/2 + 8 columns, a whole tile for column n1/2).

// Half spectra of the two real rows whose complex sum's transform a team holds
// in v (FFT output order): Z(y) and Z(NR - y) give row 0 as (Z + conj Z')/2 and
// row 1 as (Z - conj Z')/2i.  A thread's lower-half elements are its own; their
// mirrors come from the team through LDS.  Columns 0..NR/2 + 7, the last 7 zero.
// LDS address of the mirror NR - y of element y = t + k T.
template <int NR>
__device__ __forceinline__ int mirror_at(int t, int k) {
  constexpr int T = NR / 16;
  if constexpr (T % 32 == 0) return RowLay::at(NR - t) - RowLay::at(k * T);   // whole paddings apart
  else return RowLay::at(NR - t - k * T);
}

template <int NR>
__device__ __forceinline__ void half_store(const float2 (&v)[16], float2* L, int t, float2* o0, float2* o1,
                                           bool valid) {
  constexpr int T = NR / 16, RL = last_radix<NR>();
#pragma unroll
  for (int i = 0; i < 16; i++)
    if (i / RL + (i % RL) * (16 / RL) >= 8) L[RowLay::at(t, out_offset<NR>(i))] = v[i];
  __syncthreads();
  if (!valid) return;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int k = i / RL + (i % RL) * (16 / RL);   // element t + k T
    if (k < 8) {
      const int y = t + k * T;
      float2 z = v[i];
      if (y != 0) z = L[mirror_at<NR>(t, k)];
      o0[y] = make_float2(0.5f * (v[i].x + z.x), 0.5f * (v[i].y - z.y));
      o1[y] = make_float2(0.5f * (v[i].y + z.y), 0.5f * (z.x - v[i].x));
    } else if (k == 8) {
      // thread 0 holds element NR/2
      if (t < 8) {
        o0[NR / 2 + t] = make_float2(t == 0 ? v[i].x : 0.f, 0.f);
        o1[NR / 2 + t] = make_float2(t == 0 ? v[i].y : 0.f, 0.f);
      }
    }
  }
}

// The image update and the row pass of A m for row pairs of real images.
template <int NR, int RPB>
__device__ __forceinline__ void row_fwd_half_body(const RowFwdArgs& a, int bid) {
  constexpr int T = NR / 16;
  __shared__ float2 lds[RPB * RowLay::size(NR)];
  const int team = threadIdx.x / T, t = threadIdx.x % T;
  const int pair = bid * RPB + team;
  const bool valid = 2 * pair < a.rows;
  const int row = valid ? 2 * pair : 0;
  const int s = row / a.N0, h1 = a.N1 >> 1;
  const size_t r0 = (size_t)row * a.N1;   // rows are stored in order, s N0 + X
  float m0[8], m1[8], g0[8], g1[8];
  bool ok[8];
  int Yj[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const int Y = (in_index<NR>(t, j < 4 ? j : j + 8) + h1) & (NR - 1);
    ok[j] = valid && Y < a.N1;
    Yj[j] = ok[j] ? Y : 0;
    m0[j] = a.m[r0 + Yj[j]];
    m1[j] = a.m[r0 + a.N1 + Yj[j]];
  }
  if (a.update) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
      g0[j] = a.grad[r0 + Yj[j]];
      g1[j] = a.grad[r0 + a.N1 + Yj[j]];
    }
    const double al = a.alpha[s];
    auto upd = [&](float m, float g) {
      float nv = (float)__fma_rn(-al, (double)g, (double)m);
      if (a.update == 2) {
        if (a.data_type == 1) { if (nv > a.thr) nv = a.thr; }
        else { if (nv < a.thr) nv = a.thr; }
      }
      return nv;
    };
#pragma unroll
    for (int j = 0; j < 8; j++) {
      m0[j] = upd(m0[j], g0[j]);
      m1[j] = upd(m1[j], g1[j]);
      if (ok[j]) {
        a.m[r0 + Yj[j]] = m0[j];
        a.m[r0 + a.N1 + Yj[j]] = m1[j];
      }
    }
  }
  if (a.mref) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
      m0[j] -= a.mref[r0 + Yj[j]];
      m1[j] -= a.mref[r0 + a.N1 + Yj[j]];
    }
  }
  float2 v[16];
#pragma unroll
  for (int r = 0; r < 16; r++) v[r] = make_float2(0.f, 0.f);
#pragma unroll
  for (int j = 0; j < 8; j++)
    if (ok[j]) v[j < 4 ? j : j + 8] = make_float2(m0[j], m1[j]);
  FftTwiddles Tw;
  load_twiddles<NR, -1>(Tw, t, a.tw);
  float2* L = lds + team * RowLay::size(NR);
  fft_regs_half<NR, RowLay, -1>(v, L, t, Tw);
  constexpr int H = NR / 2 + kNormalC;
  half_store<NR>(v, L, t, a.out + (size_t)row * H, a.out + (size_t)(row + 1) * H, valid);
}

template <int NR, int RPB>
__global__ __launch_bounds__(RPB * (NR / 16)) void k_row_fwd_half(RowFwdArgs a) {
  row_fwd_half_body<NR, RPB>(a, blockIdx.x);
}

template <int NR, int RPB>
__global__ __launch_bounds__(RPB * (NR / 16)) void k_row_fwd_half_multi(const RowFwdArgs* __restrict__ descs,
                                                                       const int2* __restrict__ items,
                                                                       RowFwdLaunch L) {
  const int2 it = items[blockIdx.x];
  RowFwdArgs a = descs[it.x];
  a.cplx = L.cplx; a.update = L.update; a.data_type = L.data_type; a.thr = L.thr;
  row_fwd_half_body<NR, RPB>(a, it.y);
}

// Re(rhat) of row pairs from the half grid rows: inverse y FFT of the two rows'
// complex sum, minus Re(A^H W b), its square sums per pair, and the forward row
// pass of the result, in place.
template <int NR, int RPB>
__device__ __forceinline__ void row_grad_half_body(const RowAdjArgs& a, int bid) {
  constexpr int T = NR / 16, RL = last_radix<NR>(), H = NR / 2 + kNormalC;
  __shared__ float2 lds[RPB * RowLay::size(NR)];
  __shared__ double red[RPB * (T > 64 ? T / 64 : 1)];
  const int team = threadIdx.x / T, t = threadIdx.x % T;
  const int pair = bid * RPB + team;
  const bool valid = 2 * pair < a.rows;
  const int row = valid ? 2 * pair : 0;
  float2* L = lds + team * RowLay::size(NR);
  const float2 *i0 = a.in + (size_t)row * H, *i1 = i0 + H;
  float2 v[16];
  {
    float2 p[8], q[8];
#pragma unroll
    for (int r = 0; r < 8; r++) {
      p[r] = i0[t + r * T];
      q[r] = i1[t + r * T];
    }
    const float2 ph = i0[NR / 2], qh = i1[NR / 2];
    // Z(y) = P + iQ; Z(NR - y) = conj P + i conj Q, handed over through LDS
#pragma unroll
    for (int r = 0; r < 8; r++) {
      v[r] = make_float2(p[r].x - q[r].y, p[r].y + q[r].x);
      L[RowLay::at(t, r * T)] = make_float2(p[r].x + q[r].y, q[r].x - p[r].y);
    }
    __syncthreads();
#pragma unroll
    for (int r = 8; r < 16; r++) {
      const int y = (16 - r) * T - t;   // NR - (t + r T), in (0, NR/2]
      v[r] = y == NR / 2 ? make_float2(ph.x - qh.y, ph.y + qh.x) : L[mirror_at<NR>(t, r)];
    }
    __syncthreads();
  }
  FftTwiddles Tw;
  fft_from_lazy<NR, RowLay, 1, 1>(v, L, t, Tw, a.tw);
  const int h1 = a.N1 >> 1;
  const size_t r0 = (size_t)row * a.N1;
  double acc = 0.0;
  float2 u[16];   // forward input, slot r holds element t + r T
#pragma unroll
  for (int r = 0; r < 16; r++) u[r] = make_float2(0.f, 0.f);
  float c0[16], c1[16];
  int Yi[16];
  bool ok[16];
#pragma unroll
  for (int i = 0; i < 16; i++) {
    if (out_slot_cropped<NR>(i)) continue;
    const int Y = (out_index<NR>(t, i) + h1) & (NR - 1);
    ok[i] = valid && Y < a.N1;
    Yi[i] = ok[i] ? Y : 0;
    c0[i] = a.ahwb_re[r0 + Yi[i]];
    c1[i] = a.ahwb_re[r0 + a.N1 + Yi[i]];
  }
#pragma unroll
  for (int i = 0; i < 16; i++) {
    if (out_slot_cropped<NR>(i)) continue;
    if (!ok[i]) continue;
    const float x0 = v[i].x - c0[i], x1 = v[i].y - c1[i];
    a.grad[r0 + Yi[i]] = x0;
    a.grad[r0 + a.N1 + Yi[i]] = x1;
    acc += (double)x0 * (double)x0 + (double)x1 * (double)x1;
    u[i / RL + (i % RL) * (16 / RL)] = make_float2(x0, x1);
  }
  // FP64 sum over the team: lane halves within a wavefront, then the
  // wavefronts in order
  constexpr int W = T > 64 ? 64 : T;
#pragma unroll
  for (int h = W / 2; h > 0; h >>= 1) acc += __shfl_down(acc, h, W);
  if (t % W == 0) red[team * (T / W) + t / W] = acc;
  // (the forward transform's first barrier below orders red)
  fft_from_lazy<NR, RowLay, -1, 1, 0, true>(u, L, t, Tw, a.tw);
  if (valid && t == 0) {
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < T / W; w++) sum += red[team * (T / W) + w];
    a.rowpart[pair] = sum;
  }
  half_store<NR>(u, L, t, a.fwd_out + (size_t)row * H, a.fwd_out + (size_t)(row + 1) * H, valid);
}

template <int NR, int RPB>
__global__ __launch_bounds__(RPB * (NR / 16), 2) void k_row_grad_half(RowAdjArgs a) {
  row_grad_half_body<NR, RPB>(a, blockIdx.x);
}

template <int NR, int RPB>
__global__ __launch_bounds__(RPB * (NR / 16), 2) void k_row_grad_half_multi(const RowAdjArgs* __restrict__ descs,
                                                                           const int2* __restrict__ items) {
  const int2 it = items[blockIdx.x];
  const RowAdjArgs a = descs[it.x];
  row_grad_half_body<NR, RPB>(a, it.y);
}

// --------------------------------------------------- gradients in FP64
// Single-precision transforms leave a gradient error of ~4e-7 of A^H W A m.
// Steepest descent with a bound amplifies errors in some images (by a factor
// of 1.6 per iteration over tens of iterations, in a few of 256 slices), so
// the iterations work on differences: every few iterations (refresh in
// icon_capi.cpp) the gradient of the iterate m_ref is computed in FP64 from the
// whole image, and those between transform only m - m_ref in single precision:
//   rhat = A^H W A (m - m_ref) + rhat_ref,  A m - b = A (m - m_ref) + (A m_ref - b),
// whose rounding is that of the difference.

// Rows of the image: with `half` the pair 2 bid, 2 bid + 1 as one complex row.
template <int NR, bool HALF>
__device__ __forceinline__ void row_fwd64_body(const RefArgs& a, int bid) {
  constexpr int T = NR / 16, RL = last_radix<NR>();
  __shared__ double lds[RowLay::size(NR)];
  const int t = threadIdx.x;
  const int row = HALF ? 2 * bid : bid, s = row / a.N0, h1 = a.N1 >> 1;
  const size_t r0 = (size_t)row * a.N1;
  const double al = a.update ? a.alpha[s] : 0.0;
  auto pixel = [&](size_t p) {
    float nv = a.m[p];
    if (a.update) {
      nv = (float)__fma_rn(-al, (double)a.grad[p], (double)nv);
      if (a.update == 2) {
        if (a.data_type == 1) { if (nv > a.thr) nv = a.thr; }
        else { if (nv < a.thr) nv = a.thr; }
      }
      a.m[p] = nv;
    }
    a.mref[p] = nv;
    return (double)nv;
  };
  double2 v[16];
#pragma unroll
  for (int r = 0; r < 16; r++) {
    v[r] = make_double2(0.0, 0.0);
    if (r >= 4 && r < 12) continue;   // padding, as N1 <= NR/2
    const int Y = (in_index<NR>(t, r) + h1) & (NR - 1);
    if (Y < a.N1) v[r] = make_double2(pixel(r0 + Y), HALF ? pixel(r0 + a.N1 + Y) : 0.0);
  }
  fft64<NR, RowLay, -1>(v, lds, t, a.w64);
  double2* o0 = a.io + (size_t)row * a.ncol;
  if constexpr (!HALF) {
#pragma unroll
    for (int i = 0; i < 16; i++) o0[out_index<NR>(t, i)] = v[i];
  } else {
    // half spectra of the two rows, as half_store: the mirrors Z(NR - y) one
    // component at a time
    double2* o1 = o0 + a.ncol;
    double zx[16];
#pragma unroll
    for (int c = 0; c < 2; c++) {
#pragma unroll
      for (int i = 0; i < 16; i++)
        if (i / RL + (i % RL) * (16 / RL) >= 8) lds[RowLay::at(t, out_offset<NR>(i))] = c ? v[i].y : v[i].x;
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int k = i / RL + (i % RL) * (16 / RL), y = t + k * T;
        if (k >= 8) continue;
        const double z = y ? lds[mirror_at<NR>(t, k)] : (c ? v[i].y : v[i].x);
        if (c == 0) {
          zx[i] = z;
        } else {
          o0[y] = make_double2(0.5 * (v[i].x + zx[i]), 0.5 * (v[i].y - z));
          o1[y] = make_double2(0.5 * (v[i].y + z), 0.5 * (zx[i] - v[i].x));
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 16; i++)
      if (i / RL + (i % RL) * (16 / RL) == 8 && t < 8) {
        o0[NR / 2 + t] = make_double2(t == 0 ? v[i].x : 0.0, 0.0);
        o1[NR / 2 + t] = make_double2(t == 0 ? v[i].y : 0.0, 0.0);
      }
  }
}

template <int NR, bool HALF>
__global__ __launch_bounds__(NR / 16) void k_row_fwd64(RefArgs a) { row_fwd64_body<NR, HALF>(a, blockIdx.x); }

template <int NR, bool HALF>
__global__ __launch_bounds__(NR / 16) void k_row_fwd64_multi(const RefArgs* __restrict__ descs,
                                                             const int2* __restrict__ items, RowFwdLaunch L) {
  const int2 it = items[blockIdx.x];
  RefArgs a = descs[it.x];
  a.update = L.update; a.data_type = L.data_type; a.thr = L.thr;
  row_fwd64_body<NR, HALF>(a, it.y);
}

// rhat and its square sums from the grid rows of A^H W A m.
template <int NR, bool HALF>
__device__ __forceinline__ void row_grad64_body(const RefArgs& a, int bid) {
  constexpr int T = NR / 16;
  __shared__ double lds[RowLay::size(NR)];
  __shared__ double red[T > 64 ? T / 64 : 1];
  const int t = threadIdx.x;
  const int row = HALF ? 2 * bid : bid, h1 = a.N1 >> 1;
  const size_t r0 = (size_t)row * a.N1;
  const double2 *i0 = a.io + (size_t)row * a.ncol, *i1 = i0 + a.ncol;
  double2 v[16];
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int y = in_index<NR>(t, r);
    if constexpr (!HALF) {
      v[r] = i0[y];
    } else if (y <= NR / 2) {
      const double2 p = i0[y], q = i1[y];
      v[r] = make_double2(p.x - q.y, p.y + q.x);
    } else {
      const double2 p = i0[NR - y], q = i1[NR - y];
      v[r] = make_double2(p.x + q.y, q.x - p.y);
    }
  }
  fft64<NR, RowLay, 1>(v, lds, t, a.w64);
  double acc = 0.0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    if (out_slot_cropped<NR>(i)) continue;
    const int Y = (out_index<NR>(t, i) + h1) & (NR - 1);
    if (Y >= a.N1) continue;
    const size_t p = r0 + Y;
    if constexpr (HALF) {
      const float x0 = (float)(v[i].x - (double)a.ahwb_re[p]), x1 = (float)(v[i].y - (double)a.ahwb_re[p + a.N1]);
      a.grad[p] = x0;
      a.grad[p + a.N1] = x1;
      a.base_re[p] = -x0;
      a.base_re[p + a.N1] = -x1;
      acc += (double)x0 * (double)x0 + (double)x1 * (double)x1;
    } else {
      const float2 c = a.ahwb[p];
      const float2 r = make_float2((float)(v[i].x - (double)c.x), (float)(v[i].y - (double)c.y));
      a.grad[p] = r.x;
      a.base[p] = make_float2(-r.x, -r.y);
      acc += (double)r.x * (double)r.x + (double)r.y * (double)r.y;
    }
  }
  constexpr int W = T > 64 ? 64 : T;
#pragma unroll
  for (int h = W / 2; h > 0; h >>= 1) acc += __shfl_down(acc, h, W);
  if (t % W == 0) red[t / W] = acc;
  __syncthreads();
  if (t == 0) {
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < T / W; w++) sum += red[w];
    a.rowpart[bid] = sum;
  }
}

template <int NR, bool HALF>
__global__ __launch_bounds__(NR / 16) void k_row_grad64(RefArgs a) { row_grad64_body<NR, HALF>(a, blockIdx.x); }

template <int NR, bool HALF>
__global__ __launch_bounds__(NR / 16) void k_row_grad64_multi(const RefArgs* __restrict__ descs,
                                                              const int2* __restrict__ items) {
  const int2 it = items[blockIdx.x];
  const RefArgs a = descs[it.x];
  row_grad64_body<NR, HALF>(a, it.y);
}

// col_normal in FP64 on the rows io64; the node values are interpolated from
// the tile rounded to single precision.
template <int NC, int C, int K>
__device__ __forceinline__ void col_normal64_body(const ColArgs& a, int bid) {
  constexpr int LS = col_stride<NC, C>(), RL = last_radix<NC>();
  extern __shared__ __align__(16) float2 tile[];   // col_lds<NC, C>()
  double* lds = reinterpret_cast<double*>(tile);
  const int blk = bid / a.S;
  const int s = bid % a.S;
  const int c = threadIdx.x % C, t = threadIdx.x / C;
  double2* rows = a.io64 + (size_t)s * a.N0 * a.n1 + blk * C + c;
  const int h0 = a.N0 >> 1;
  double2 v[16];
#pragma unroll
  for (int r = 0; r < 16; r++) {
    v[r] = make_double2(0.0, 0.0);
    if (r >= 4 && r < 12) continue;   // padding rows, as N0 <= NC/2
    const int X = (in_index<NC>(t, r) + h0) & (NC - 1);
    if (X < a.N0) v[r] = rows[(size_t)X * a.n1];
  }
  fft64<NC, ColFftLay<C>, -1>(v, lds + c, t, a.w64);
  if (a.ent_off[blk] != a.ent_off[blk + 1]) {
#pragma unroll
    for (int i = 0; i < 16; i++) tile[out_index<NC>(t, i) * LS + c] = make_float2((float)v[i].x, (float)v[i].y);
    __syncthreads();
    interp_tile<NC, C, K>(a, tile, blk, s);
    __syncthreads();
  }
  float sp[16];
  load_spec<NC, C>(sp, a, blk, c, t);
  double2 u[16];
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int r = i / RL + (i % RL) * (16 / RL);
    u[r] = make_double2(v[i].x * (double)sp[r], v[i].y * (double)sp[r]);
  }
  fft64<NC, ColFftLay<C>, 1>(u, lds + c, t, a.w64);
#pragma unroll
  for (int i = 0; i < 16; i++) {
    if (out_slot_cropped<NC>(i)) continue;
    const int X = (out_index<NC>(t, i) + h0) & (NC - 1);
    if (X < a.N0) rows[(size_t)X * a.n1] = u[i];
  }
}

template <int NC, int C, int K>
__global__ __launch_bounds__(C * (NC / 16)) void k_col_normal64(ColArgs a) {
  col_normal64_body<NC, C, K>(a, blockIdx.x);
}

template <int NC, int C, int K>
__global__ __launch_bounds__(C * (NC / 16)) void k_col_normal64_multi(const ColArgs* __restrict__ descs,
                                                                     const int2* __restrict__ items) {
  const int2 it = items[blockIdx.x];
  const ColArgs a = descs[it.x];
  col_normal64_body<NC, C, K>(a, it.y);
}

// The node of a row of the node values: every node of a full plan; with paired
// nodes, per tilt line the nodes N0/2 .. N0-1 and last the unpaired node 0.
// *jm: the node whose value is the conjugate, or -1.
__device__ __forceinline__ int node_of(const FinishArgs& a, int r, int* jm) {
  *jm = -1;
  if (!a.nq) return r;
  const int per = a.N0 / 2 + 1, i = r / per, k = r - i * per;
  if (k == a.N0 / 2) return i * a.N0;
  if (k > 0) *jm = i * a.N0 + a.N0 / 2 - k;
  return i * a.N0 + a.N0 / 2 + k;
}

// role 0: alpha = |rhat|^2 / <rhat, A^H W A rhat>; role 1: the data residual
// R = sqrt(sum w |A m - b|^2 / sum w |b|^2) and the values at the omit tilt.
// One block per (slice, role); FP64 sums in a fixed order.
// Role 1 sums a.groups groups of rows, as many as the geometry asks for, and adds
// the groups' sums in order, whether one block takes all of them or a.blocks
// blocks per slice share them: the residual's bits do not depend on the number
// of slices.  Of several blocks the last to finish adds the sums (rsum) and
// leaves their counter (rcnt) at zero again.  The blocks exchange nothing but
// device-scope read-modify-writes, the store of a sum waited for before the
// count.
__device__ __forceinline__ void finish_body(const FinishArgs& a, int s, int role, int blk) {
  __shared__ double red[32];
  __shared__ double z[4 * kMaxUnpaired];
  const int tid = threadIdx.x;
  const float2* P = a.part + (size_t)s * a.M * a.slots;
  // One block per slice waits on its loads: each round issues those of several
  // elements together (one 256^2 slice, 61 tilts: 12.5 -> 8.2 us;
  // 256 slices of 512^2, 41 tilts: 48 -> 36 us)
  if (role == 0) {
    double sums[2] = {0.0, tid < a.nblk ? a.epart[(size_t)s * a.nblk + tid] : 0.0};
    for (int X = tid; X < a.nrow; X += 1024) sums[0] += a.rowpart[(size_t)s * a.nrow + X];
    if (a.nq) {
      // the gradient's imaginary part I = sum_a zd_a e_a over the waves e =
      // (cos, sin)(2 pi v_t x): |I|^2 = zd G zd, <I, A^H W A I> = zd H zd and
      // 2 <I, Im(A^H W A) Re rhat> = 2 zd G zr, with the coefficients z of the
      // residual d_t (zd) and of (A Re rhat)_t (zr)
      const int nf = 2 * a.nq, nn = nf * nf;
      double *zd = z, *zr = z + nf;
      for (int t = tid; t < a.nq; t += 1024) {
        const int j = t * a.N0;
        const double w = a.w[j];
        const float2 f = node_value(P, a.nslot, t * (a.N0 / 2 + 1) + a.N0 / 2, a.slots);
        const float2 bj = a.b[(size_t)s * a.Mb + j];
        const float2 r = node_value(a.rpart + (size_t)s * a.nq * a.slots, a.rslot, t, a.slots);
        // (where the residual is asked for, its blocks write beff)
        if (a.beff && !a.resid) a.beff[(size_t)s * a.Mb + j] = make_float2(bj.x - f.x, bj.y - f.y);
        zd[t] = w * ((double)f.y - (double)bj.y);
        zd[a.nq + t] = w * ((double)f.x - (double)bj.x);
        zr[t] = w * (double)r.y;
        zr[a.nq + t] = w * (double)r.x;
      }
      __syncthreads();
      // a wavefront takes rows 16 apart, its lanes the columns: no index
      // division (with one it was 40 instructions an element, all on one CU: 9.4
      // instead of 8.2 us)
      const int wave = tid >> 6, lane = tid & 63;
      constexpr int U = 8;   // rows whose loads are in flight together
      for (int c = lane; c < (nf + 63) / 64 * 64; c += 64) {
        const bool in = c < nf;
        const double dc = in ? zd[c] : 0.0, rc = in ? zr[c] : 0.0;
        for (int p0 = wave; p0 < nf; p0 += 16 * U) {
          float g[U], h[U];
#pragma unroll
          for (int u = 0; u < U; u++) {
            const int p = p0 + 16 * u;
            const bool ok = in && p < nf;
            g[u] = ok ? a.gram[p * nf + c] : 0.f;
            h[u] = ok ? a.gram[nn + p * nf + c] : 0.f;
          }
#pragma unroll
          for (int u = 0; u < U; u++) {
            const double q = zd[min(p0 + 16 * u, nf - 1)];
            sums[0] += q * ((double)g[u] * dc);
            sums[1] += q * ((double)h[u] * dc + 2.0 * (double)g[u] * rc);
          }
        }
      }
    }
    block_sums_1024(sums, red);
    if (tid == 0) {
      const double al = sums[1] != 0.0 ? sums[0] / sums[1] : 0.0;
      a.alpha[s] = al;
      if (a.alpha_trace) a.alpha_trace[(size_t)s * a.alpha_stride + a.alpha_index] = al;
    }
    return;
  }
  constexpr int U = 4, SL = 4;   // rows a round; partials loaded together (a.slots of them at most)
  double* gsum = z;              // [group][wavefront], then the groups' sums
  static_assert(kFinishRows == U * 1024 && 17 * kFinishGroups <= 4 * kMaxUnpaired, "a group's round; the sums fit z");
  for (int g = blk; g < a.groups; g += a.blocks) {
    double acc = 0.0;
    for (int r0 = g * U * 1024 + tid; r0 < a.M; r0 += a.groups * U * 1024) {
      float2 p[U][SL], b0[U], b1[U];
      float w0[U], w1[U];
      int j[U], jm[U], ns[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const bool in = r0 + u * 1024 < a.M;
        const int r = in ? r0 + u * 1024 : r0;
        j[u] = node_of(a, r, &jm[u]);
        if (!in) j[u] = jm[u] = -1;
        ns[u] = a.nslot[r];
#pragma unroll
        for (int q = 0; q < SL; q++) p[u][q] = P[(size_t)r * a.slots + min(q, a.slots - 1)];
        const int k0 = max(j[u], 0), k1 = max(jm[u], 0);
        w0[u] = a.w[k0];
        w1[u] = a.w[k1];
        if (a.resid) {
          b0[u] = a.b[(size_t)s * a.Mb + k0];
          b1[u] = a.b[(size_t)s * a.Mb + k1];
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        if (j[u] < 0) continue;
        // as node_value: the partials in slot order
        float2 f = p[u][0];
#pragma unroll
        for (int q = 1; q < SL; q++)
          if (q < ns[u]) {
            f.x += p[u][q].x;
            f.y += p[u][q].y;
          }
        if (a.resid) {
          const double dx = (double)f.x - (double)b0[u].x, dy = (double)f.y - (double)b0[u].y;
          acc += (double)w0[u] * (dx * dx + dy * dy);
          if (a.beff) a.beff[(size_t)s * a.Mb + j[u]] = make_float2((float)-dx, (float)-dy);
          if (jm[u] >= 0) {
            const double ex = (double)f.x - (double)b1[u].x, ey = (double)f.y + (double)b1[u].y;
            acc += (double)w1[u] * (ex * ex + ey * ey);
            if (a.beff) a.beff[(size_t)s * a.Mb + jm[u]] = make_float2((float)-ex, (float)ey);
          }
        }
        if (a.frep) {
          const int i = j[u] / a.N0;
          if (i == a.iomit) {
            a.frep[(size_t)s * a.N0 + (j[u] - i * a.N0)] = f;
            if (jm[u] >= 0) a.frep[(size_t)s * a.N0 + (jm[u] - i * a.N0)] = make_float2(f.x, -f.y);
          }
        }
      }
    }
#pragma unroll
    for (int h = 32; h > 0; h >>= 1) acc += __shfl_down(acc, h);
    if ((tid & 63) == 0) gsum[16 * g + (tid >> 6)] = acc;
  }
  if (!a.resid) return;
  __syncthreads();
  if (tid >= 64) return;
  // the first wavefront: thread g the sum of group g, thread 0 their sum
  double* sums = gsum + 16 * kFinishGroups;
  if (tid < a.groups && tid % a.blocks == blk) {
    double t = gsum[16 * tid];
#pragma unroll
    for (int w = 1; w < 16; w++) t += gsum[16 * tid + w];
    if (a.blocks > 1) {
      const unsigned long long old =
          atomicExch(a.rsum + (size_t)s * kFinishGroups + tid, (unsigned long long)__double_as_longlong(t));
      asm volatile("" ::"v"((unsigned)old) : "memory");
    } else {
      sums[tid] = t;
    }
  }
  line_sync<1>();
  if (tid == 0) {
    double tot = 0.0;
    if (a.blocks > 1) {
      unsigned long long* q = a.rsum + (size_t)s * kFinishGroups;
      if (atomicAdd(a.rcnt + s, 1u) != (unsigned)a.blocks - 1) return;
      unsigned long long v[kFinishGroups];
      for (int k = 0; k < a.groups; k++) v[k] = atomicAdd(q + k, 0ull);
      for (int k = 0; k < a.groups; k++) tot += __longlong_as_double((long long)v[k]);
      atomicExch(a.rcnt + s, 0u);
    } else {
      for (int k = 0; k < a.groups; k++) tot += sums[k];
    }
    const double bn = a.bnorm[s];
    a.resid[(size_t)s * a.resid_stride + a.resid_index] = bn > 0 ? sqrt(tot / bn) : 0.0;
  }
}

// blocks [0, S): the step size where asked for (alpha non-null); then a.blocks
// times S blocks for the residual's rows
__global__ __launch_bounds__(1024) void k_finish(FinishArgs a) {
  const int k = (int)blockIdx.x / a.S - (a.alpha ? 1 : 0);
  finish_body(a, blockIdx.x % a.S, k < 0 ? 0 : 1, k);
}

__global__ __launch_bounds__(1024) void k_finish_multi(const FinishArgs* __restrict__ descs,
                                                       const int2* __restrict__ items, int n, FinishLaunch L) {
  const int2 it = items[blockIdx.x % n];
  FinishArgs a = descs[it.x];
  a.resid_index = L.resid_index;
  a.alpha_index = L.alpha_index;
  if (L.resid_index < 0) a.resid = nullptr;
  if (!L.with_frep) a.frep = nullptr;
  if (L.beff == 2 && a.beff) a.b = a.beff;
  if (L.beff != 1) a.beff = nullptr;
  const int k = (int)blockIdx.x / n - (L.alpha_index >= 0 ? 1 : 0);
  if (k >= 0 && ((!a.resid && !a.frep) || k >= a.blocks)) return;
  finish_body(a, it.y, k < 0 ? 0 : 1, k);
}

// ------------------------------------------------------- plan-time kernels
// Taps of the solve's interpolation.  The image fills at most half of the
// grid (N <= n/2), so the grid values of its spectrum determine the values
// between the grid points: taps c_q over the 16 points around u with
// sum_q c_q exp(2 pi i xi (q - u)) ~ 1 for all |xi| <= 1/4, in the least-squares
// sense: S c = s, S_pq = sinc((p - q)/2)/2, s_q = sinc((q - u)/2)/2.  No
// deapodisation, so the tile that the normal operator transforms serves as it
// is.  Largest error 1.1e-6, rms 1.8e-7 of the spectrum's scale (the 14-tap
// Gaussian with deapodisation: 3.5e-6 and 7.1e-7).
//
// S's condition is 5e10, but the two triangular solves leave an error in c only
// along directions that no |xi| <= 1/4 sees (its explicit inverse would not).
__device__ __forceinline__ void interp_taps(double frac, const double* __restrict__ l, double (&c)[kInterpTaps]) {
  constexpr int K = kInterpTaps;
  constexpr double kPi = 3.14159265358979323846;
#pragma unroll
  for (int q = 0; q < K; q++) {
    const double x = 0.5 * (q - (K / 2 - 1) - frac);
    c[q] = x == 0.0 ? 0.5 : 0.5 * sinpi(x) / (kPi * x);
  }
#pragma unroll
  for (int p = 0; p < K; p++) {
#pragma unroll
    for (int q = 0; q < p; q++) c[p] -= l[p * K + q] * c[q];
    c[p] *= l[p * K + p];
  }
#pragma unroll
  for (int p = K - 1; p >= 0; p--) {
#pragma unroll
    for (int q = p + 1; q < K; q++) c[p] -= l[q * K + p] * c[q];
    c[p] *= l[p * K + p];
  }
}

// half: N0/2, the node rows of node_of with paired nodes; otherwise 0.  An entry's
// w: tile, bit 16: the node mirrored (-v), bit 17: columns of the grid's mirrored
// half (descending, x-taps reversed).
__global__ __launch_bounds__(256) void k_interp_records(const int4* ent, const int* ent_off, const float2* nodes,
                                                        int E, int n0, int n1, int half, const double* chol, float* px,
                                                        float* py) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= E) return;
  const int4 r = ent[e];
  const int tile = r.w & 0xffff;
  const bool mirror = (r.w >> 16) & 1, rev = (r.w >> 17) & 1;
  const int e0 = ent_off[tile], ne = ent_off[tile + 1] - e0;
  const int t0 = r.y & 0xff, t1 = (r.y >> 8) & 0xff, col0 = (r.y >> 24) & 0xff;
  int j = r.x;
  if (half) {
    const int i = r.x / (half + 1), k = r.x - i * (half + 1);
    j = i * 2 * half + (k < half ? half + k : 0);
  }
  float2 v = nodes[j];
  if (mirror) v = make_float2(-v.x, -v.y);
  double c[kInterpTaps];
  const double ux = (double)n0 * (double)v.x, uy = (double)n1 * (double)v.y;
  interp_taps(ux - floor(ux), chol, c);
  float* qx = px + (size_t)e0 * kInterpTaps + 2 * (e - e0);
#pragma unroll
  for (int t = 0; t < kInterpTaps; t++) {
    const int o = rev ? kInterpTaps - 1 - t : t;
    qx[(size_t)(o / 2) * ne * 2 + (o & 1)] = (float)c[t];
  }
  interp_taps(uy - floor(uy), chol, c);
  float* qy = py + (size_t)e0 * kNormalC + 4 * (e - e0);
#pragma unroll
  for (int k = 0; k < kNormalC; k++) {
    float p = 0.f;
#pragma unroll
    for (int t = 0; t < kInterpTaps; t++)
      if (t >= t0 && t <= t1 && (rev ? col0 - (t - t0) : col0 + t - t0) == k) p = (float)c[t];
    qy[(size_t)(k / 4) * ne * 4 + (k & 3)] = p;
  }
}

// Kaiser-Bessel taps I0(beta sqrt(1 - (2d/K)^2)) / Z, Z = K sinh(beta) / beta, at the
// grid points floor(u) - (K/2 - 1) .. + K/2 (I0 by its power series; arguments
// up to 24)
__device__ __forceinline__ double bessel_i0(double x) {
  double term = 1.0, sum = 1.0;
  const double q = 0.25 * x * x;
  for (int k = 1; k < 200 && term > 1e-17 * sum; k++) {
    term *= q / ((double)k * (double)k);
    sum += term;
  }
  return sum;
}

__device__ __forceinline__ float kb_tap(double frac, int t, int K, double beta) {
  const double d = frac + (double)(K / 2 - 1 - t);
  const double r = 1.0 - (2.0 * d / K) * (2.0 * d / K);
  return r > 0 ? (float)(bessel_i0(beta * sqrt(r)) * beta / (K * sinh(beta))) : 0.f;
}

// One thread per (entry, record value): its K x-taps, then its C y-taps.
__global__ __launch_bounds__(256) void k_window_records(const int4* ent, const int* ent_off, const float2* nodes,
                                                        int E, int n0, int n1, int K, int C, float beta0, float beta1,
                                                        float* px, float* py) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)E * (K + C)) return;
  const int e = (int)(i % E), q = (int)(i / E);
  const int4 r = ent[e];
  const int e0 = ent_off[r.w], ne = ent_off[r.w + 1] - e0;
  const float2 v = nodes[r.x];
  if (q < K) {
    const double u = (double)n0 * (double)v.x;
    px[(size_t)e0 * K + ((size_t)(q / 2) * ne + (e - e0)) * 2 + (q & 1)] = kb_tap(u - floor(u), q, K, (double)beta0);
    return;
  }
  const int c = q - K, t0 = r.y & 0xff, t1 = (r.y >> 8) & 0xff, col0 = (r.y >> 24) & 0xff;
  const int t = t0 + c - col0;
  const double u = (double)n1 * (double)v.y;
  py[(size_t)e0 * C + ((size_t)(c / 4) * ne + (e - e0)) * 4 + (c & 3)] =
      t >= t0 && t <= t1 ? kb_tap(u - floor(u), t, K, (double)beta1) : 0.f;
}

__global__ __launch_bounds__(256) void k_outer(const float* cx, const float* cy, int N0, int N1, float* out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < N0 * N1) out[i] = cx[i / N1] * cy[i % N1];
}

// d[k][q] = (w_j or 1) D(q/n - v_j), j = j0 + k; rows k in [cnt, cntp) zero.
// q/n - v is exact in double (n a power of two, v single precision).
__global__ __launch_bounds__(256) void k_dirichlet(const float* nodes, const float* w, int j0, int cnt, int cntp, int N,
                                                   int n, double* d) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)cntp * n) return;
  const int k = (int)(i / n), q = (int)(i % n);
  double v = 0.0;
  if (k < cnt) {
    const double th = (double)q / (double)n - (double)nodes[2 * (size_t)(j0 + k)];
    const double den = sinpi(th);
    v = den == 0.0 ? (double)(2 * N - 1) : sinpi((double)(2 * N - 1) * th) / den;
    if (w) v *= (double)w[j0 + k];
  }
  d[i] = v;
}

// acc[q0][q1] += sum_k d0[k][q0] d1[k][q1] on v_mfma_f64_16x16x4_f64.  A block
// of 4 wavefronts takes 64 x 64 outputs, a wavefront 32 x 32 (2 x 2 result
// tiles); the operands come straight from L1/L2 (k-major rows, 16 consecutive
// doubles per quarter wavefront), 4 loads per 4 matrix instructions.  Lane l
// feeds A[l % 16][k = l / 16] and B[k = l / 16][l % 16] and receives
// D[4 r + l / 16][l % 16] in register r.
typedef __attribute__((ext_vector_type(4))) double d4;
__global__ __launch_bounds__(256) void k_spectrum(const double* __restrict__ d0, const double* __restrict__ d1,
                                                  int cntp, int n0, int n1, double* acc) {
  // gridDim.z splits of the node rows (multiples of 16), each into its own acc
  const int per = (cntp / 16 + gridDim.z - 1) / gridDim.z * 16;
  const int k0 = blockIdx.z * per, k1 = min(cntp, k0 + per);
  acc += (size_t)blockIdx.z * n0 * n1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int i0 = blockIdx.x * 64 + 32 * (wave >> 1), j0 = blockIdx.y * 64 + 32 * (wave & 1);
  const double* pa = d0 + (size_t)g * n0 + i0 + l16;
  const double* pb = d1 + (size_t)g * n1 + j0 + l16;
  d4 s[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) s[i][j] = d4{0., 0., 0., 0.};
  for (int k = k0; k < k1; k += 16) {
    // 16 nodes a round, their loads in flight together
    double va[4][2], vb[4][2];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        va[q][h] = pa[(size_t)(k + 4 * q) * n0 + 16 * h];
        vb[q][h] = pb[(size_t)(k + 4 * q) * n1 + 16 * h];
      }
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          s[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(va[q][i], vb[q][j], s[i][j], 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        acc[(size_t)(i0 + 16 * i + 4 * r + g) * n1 + j0 + 16 * j + l16] += s[i][j][r];
}

// spec[tile][q0][c] = acc[q0][tile C + c] / (n0 n1), acc summed over its splits.
// half: the columns 0..n1/2 of the even part (acc(q) + acc(-q)) / 2, and zero
// columns up to n1/2 + 7.
__global__ __launch_bounds__(256) void k_spectrum_store(const double* acc, int splits, int n0, int n1, int half,
                                                        float* spec) {
  const int ncol = half ? n1 / 2 + kNormalC : n1;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)n0 * ncol) return;
  const int c = (int)(i % kNormalC), q0 = (int)((i / kNormalC) % n0), tile = (int)(i / kNormalC / n0);
  const int q1 = tile * kNormalC + c;
  double v = 0.0;
  if (!half || q1 <= n1 / 2)
    for (int z = 0; z < splits; z++) {
      const double* p = acc + (size_t)z * n0 * n1;
      const double x = p[(size_t)q0 * n1 + q1];
      v += half ? 0.5 * (x + p[(size_t)((n0 - q0) % n0) * n1 + (n1 - q1) % n1]) : x;
    }
  spec[i] = (float)(v / ((double)n0 * (double)n1));
}

// sum_{x = -h}^{N-1-h} exp(2 pi i th x), h = N/2
__device__ __forceinline__ double2 box_sum(double th, int N) {
  const double den = sinpi(th);
  const double r = den == 0.0 ? (double)N : sinpi((double)N * th) / den;
  // integer th: every term is 1 (N terms); the phase below covers even N's odd centre
  if (den == 0.0) return make_double2((double)N, 0.0);
  const int o = N - 1 - 2 * (N / 2);   // 0 for odd N, -1 for even
  return make_double2(r * cospi(o * th), r * sinpi(o * th));
}

// E(v) = sum over the image's pixels of exp(2 pi i v x)
__device__ __forceinline__ double2 image_sum(double vx, double vy, int N0, int N1) {
  const double2 p = box_sum(vx, N0), q = box_sum(vy, N1);
  return make_double2(p.x * q.x - p.y * q.y, p.x * q.y + p.y * q.x);
}

// The waves' inner products over the image, G_ab = <e_a, e_b>, e = cos (a < nq)
// or sin (a >= nq) of 2 pi v_t x, v_t the unpaired node (node t N0) of line t.
__global__ __launch_bounds__(256) void k_wave_gram(const float2* nodes, int nq, int N0, int N1, float* g) {
  const int i = blockIdx.x * 256 + threadIdx.x, nf = 2 * nq;
  if (i >= nf * nf) return;
  const int a = i / nf, b = i - a * nf;
  const float2 u = nodes[(size_t)(a % nq) * N0], w = nodes[(size_t)(b % nq) * N0];
  const double2 em = image_sum((double)u.x - (double)w.x, (double)u.y - (double)w.y, N0, N1);
  const double2 ep = image_sum((double)u.x + (double)w.x, (double)u.y + (double)w.y, N0, N1);
  double v;
  if (a < nq && b < nq) v = em.x + ep.x;
  else if (a >= nq && b >= nq) v = em.x - ep.x;
  else if (a < nq) v = ep.y - em.y;   // cos_a sin_b
  else v = ep.y + em.y;               // sin_a cos_b
  g[i] = (float)(0.5 * v);
}

// The waves' values at the nodes, f[2k][a] + i f[2k+1][a] = sum_x e_a(x)
// exp(-2 pi i v_j x), j = j0 + k, ld columns (zero from 2 nq on and for k >=
// cnt); weighted by w_j in fw.
__global__ __launch_bounds__(256) void k_wave_nodes(const float2* nodes, const float* w, int j0, int cnt, int cntp,
                                                    int nq, int ld, int N0, int N1, double* fw, double* f) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)cntp * ld) return;
  const int k = (int)(i / ld), a = (int)(i % ld);
  double2 v = make_double2(0.0, 0.0);
  double wj = 0.0;
  if (k < cnt && a < 2 * nq) {
    const float2 n = nodes[j0 + k], u = nodes[(size_t)(a % nq) * N0];
    const double2 em = image_sum((double)u.x - (double)n.x, (double)u.y - (double)n.y, N0, N1);
    const double2 ep = image_sum(-(double)u.x - (double)n.x, -(double)u.y - (double)n.y, N0, N1);
    // cos: (em + ep)/2; sin: (em - ep)/2i
    v = a < nq ? make_double2(0.5 * (em.x + ep.x), 0.5 * (em.y + ep.y))
               : make_double2(0.5 * (em.y - ep.y), -0.5 * (em.x - ep.x));
    wj = (double)w[j0 + k];
  }
  const size_t o = (size_t)(2 * k) * ld + a;
  f[o] = v.x;
  f[o + ld] = v.y;
  fw[o] = wj * v.x;
  fw[o + ld] = wj * v.y;
}

// h[a][b] = sum over the splits of acc[a][b] (ld columns)
__global__ __launch_bounds__(256) void k_wave_store(const double* acc, int splits, int nf, int ld, float* h) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= nf * nf) return;
  const int a = i / nf, b = i - a * nf;
  double v = 0.0;
  for (int z = 0; z < splits; z++) v += acc[((size_t)z * ld + a) * ld + b];
  h[i] = (float)v;
}

// ================================================================ launchers

#define NC_CASES(X) X(128) X(256) X(512) X(1024) X(2048)

namespace {

template <int NC>
constexpr int lds_bytes() { return col_lds<NC, kNormalC>() * (int)sizeof(float2); }

template <int NC>
hipError_t normal_attr() {
  constexpr int C = kNormalC, K = kInterpTaps;
  const void* f[] = {(const void*)k_col_normal<NC, C, K>, (const void*)k_col_normal_multi<NC, C, K>,
                     (const void*)k_col_energy<NC, C, K>, (const void*)k_col_energy_multi<NC, C, K>};
  for (const void* p : f) {
    const hipError_t e = hipFuncSetAttribute(p, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes<NC>());
    if (e != hipSuccess) return e;
  }
  if constexpr (NC <= 1024) {
    for (const void* p : {(const void*)k_col_normal64<NC, C, K>, (const void*)k_col_normal64_multi<NC, C, K>}) {
      const hipError_t e = hipFuncSetAttribute(p, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes<NC>());
      if (e != hipSuccess) return e;
    }
  }
  return hipSuccess;
}

// Row pairs per block of the half row kernels: 128 threads, as the full
// gradient kernel.
template <int NR>
constexpr int pairs_per_block() { return 128 / (NR / 16) > 1 ? 128 / (NR / 16) : 1; }

}  // namespace

hipError_t set_normal_attrs(int NC) {
  const hipError_t e = set_col_fwd_nodes_attrs(NC);
  if (e != hipSuccess) return e;
  switch (NC) {
#define CASE(N) case N: return normal_attr<N>();
    NC_CASES(CASE)
#undef CASE
    default: return hipErrorInvalidValue;
  }
}

#define COL_CASE(N, KERNEL, GRID, ...)                                                                              \
  case N:                                                                                                          \
    LAUNCH_TIMED((KERNEL<N, kNormalC, kInterpTaps>), dim3(GRID), dim3(N / 2), lds_bytes<N>(), st, __VA_ARGS__); \
    break;
#define LAUNCH_COL_1024(KERNEL, GRID, ...)                                                              \
  COL_CASE(128, KERNEL, GRID, __VA_ARGS__)                                                              \
  COL_CASE(256, KERNEL, GRID, __VA_ARGS__)                                                              \
  COL_CASE(512, KERNEL, GRID, __VA_ARGS__)                                                              \
  COL_CASE(1024, KERNEL, GRID, __VA_ARGS__)                                                             \
  default: return hipErrorInvalidValue;
#define LAUNCH_COL(KERNEL, GRID, ...)                                                                   \
  switch (NC) {                                                                                         \
    COL_CASE(2048, KERNEL, GRID, __VA_ARGS__)                                                           \
    LAUNCH_COL_1024(KERNEL, GRID, __VA_ARGS__)                                                          \
  }                                                                                                     \
  return hipGetLastError()

hipError_t launch_col_normal(int NC, const ColArgs& a, hipStream_t st) {
  LAUNCH_COL(k_col_normal, a.S * (a.n1 / kNormalC + a.nx), a);
}
hipError_t launch_col_energy(int NC, const ColArgs& a, hipStream_t st) {
  LAUNCH_COL(k_col_energy, a.S * (a.n1 / kNormalC), a);
}
hipError_t launch_col_normal_multi(int NC, const ColArgs* descs, const int2* items, int n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  LAUNCH_COL(k_col_normal_multi, n, descs, items);
}
hipError_t launch_col_energy_multi(int NC, const ColArgs* descs, const int2* items, int n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  LAUNCH_COL(k_col_energy_multi, n, descs, items);
}

int half_row_pairs_per_block(int NR) {
  switch (NR) {
#define CASE(N) case N: return pairs_per_block<N>();
    NC_CASES(CASE)
#undef CASE
    default: return 0;
  }
}

#define LAUNCH_HALF(KERNEL, GRID, ...)                                                                          \
  switch (NR) {                                                                                                 \
    case 128: LAUNCH_TIMED((KERNEL<128, pairs_per_block<128>()>), dim3(GRID), dim3(128), 0, st, __VA_ARGS__); break;    \
    case 256: LAUNCH_TIMED((KERNEL<256, pairs_per_block<256>()>), dim3(GRID), dim3(128), 0, st, __VA_ARGS__); break;    \
    case 512: LAUNCH_TIMED((KERNEL<512, pairs_per_block<512>()>), dim3(GRID), dim3(128), 0, st, __VA_ARGS__); break;    \
    case 1024: LAUNCH_TIMED((KERNEL<1024, pairs_per_block<1024>()>), dim3(GRID), dim3(128), 0, st, __VA_ARGS__); break; \
    case 2048: LAUNCH_TIMED((KERNEL<2048, pairs_per_block<2048>()>), dim3(GRID), dim3(128), 0, st, __VA_ARGS__); break; \
    default: return hipErrorInvalidValue;                                                                       \
  }                                                                                                             \
  return hipGetLastError()

hipError_t launch_row_fwd_half(int NR, const RowFwdArgs& a, hipStream_t st) {
  const int per = half_row_pairs_per_block(NR);
  LAUNCH_HALF(k_row_fwd_half, (a.rows / 2 + per - 1) / per, a);
}
hipError_t launch_row_grad_half(int NR, const RowAdjArgs& a, hipStream_t st) {
  const int per = half_row_pairs_per_block(NR);
  LAUNCH_HALF(k_row_grad_half, (a.rows / 2 + per - 1) / per, a);
}
hipError_t launch_row_fwd_half_multi(int NR, const RowFwdArgs* descs, const int2* items, int n, const RowFwdLaunch& L,
                                     hipStream_t st) {
  if (n <= 0) return hipSuccess;
  LAUNCH_HALF(k_row_fwd_half_multi, n, descs, items, L);
}
hipError_t launch_row_grad_half_multi(int NR, const RowAdjArgs* descs, const int2* items, int n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  LAUNCH_HALF(k_row_grad_half_multi, n, descs, items);
}

hipError_t launch_col_normal64(int NC, const ColArgs& a, hipStream_t st) {
  switch (NC) { LAUNCH_COL_1024(k_col_normal64, a.S * (a.n1 / kNormalC), a) }
  return hipGetLastError();
}
hipError_t launch_col_normal64_multi(int NC, const ColArgs* descs, const int2* items, int n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  switch (NC) { LAUNCH_COL_1024(k_col_normal64_multi, n, descs, items) }
  return hipGetLastError();
}

#define LAUNCH_REF(KERNEL, GRID, ...)                                                                              \
  if (half) {                                                                                                      \
    switch (NR) {                                                                                                  \
      case 128: hipLaunchKernelGGL((KERNEL<128, true>), dim3(GRID), dim3(8), 0, st, __VA_ARGS__); break;           \
      case 256: hipLaunchKernelGGL((KERNEL<256, true>), dim3(GRID), dim3(16), 0, st, __VA_ARGS__); break;          \
      case 512: hipLaunchKernelGGL((KERNEL<512, true>), dim3(GRID), dim3(32), 0, st, __VA_ARGS__); break;          \
      case 1024: hipLaunchKernelGGL((KERNEL<1024, true>), dim3(GRID), dim3(64), 0, st, __VA_ARGS__); break;        \
      case 2048: hipLaunchKernelGGL((KERNEL<2048, true>), dim3(GRID), dim3(128), 0, st, __VA_ARGS__); break;       \
      default: return hipErrorInvalidValue;                                                                        \
    }                                                                                                              \
  } else {                                                                                                         \
    switch (NR) {                                                                                                  \
      case 128: hipLaunchKernelGGL((KERNEL<128, false>), dim3(GRID), dim3(8), 0, st, __VA_ARGS__); break;          \
      case 256: hipLaunchKernelGGL((KERNEL<256, false>), dim3(GRID), dim3(16), 0, st, __VA_ARGS__); break;         \
      case 512: hipLaunchKernelGGL((KERNEL<512, false>), dim3(GRID), dim3(32), 0, st, __VA_ARGS__); break;         \
      case 1024: hipLaunchKernelGGL((KERNEL<1024, false>), dim3(GRID), dim3(64), 0, st, __VA_ARGS__); break;       \
      case 2048: hipLaunchKernelGGL((KERNEL<2048, false>), dim3(GRID), dim3(128), 0, st, __VA_ARGS__); break;      \
      default: return hipErrorInvalidValue;                                                                        \
    }                                                                                                              \
  }                                                                                                                \
  return hipGetLastError()

hipError_t launch_row_fwd64(int NR, bool half, const RefArgs& a, hipStream_t st) {
  LAUNCH_REF(k_row_fwd64, half ? a.rows / 2 : a.rows, a);
}
hipError_t launch_row_grad64(int NR, bool half, const RefArgs& a, hipStream_t st) {
  LAUNCH_REF(k_row_grad64, half ? a.rows / 2 : a.rows, a);
}
hipError_t launch_row_fwd64_multi(int NR, bool half, const RefArgs* descs, const int2* items, int n,
                                  const RowFwdLaunch& L, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  LAUNCH_REF(k_row_fwd64_multi, n, descs, items, L);
}
hipError_t launch_row_grad64_multi(int NR, bool half, const RefArgs* descs, const int2* items, int n,
                                   hipStream_t st) {
  if (n <= 0) return hipSuccess;
  LAUNCH_REF(k_row_grad64_multi, n, descs, items);
}

hipError_t launch_finish(const FinishArgs& a, hipStream_t st) {
  const int roles = (a.alpha ? 1 : 0) + (a.resid || a.frep ? a.blocks : 0);
  if (!roles) return hipSuccess;
  LAUNCH_TIMED(k_finish, dim3(roles * a.S), dim3(1024), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_finish_multi(const FinishArgs* descs, const int2* items, int n, const FinishLaunch& L,
                               hipStream_t st) {
  const int roles = (L.alpha_index >= 0 ? 1 : 0) + (L.resid_index >= 0 || L.with_frep ? L.blocks : 0);
  if (n <= 0 || !roles) return hipSuccess;
  LAUNCH_TIMED(k_finish_multi, dim3(roles * n), dim3(1024), 0, st, descs, items, n, L);
  return hipGetLastError();
}

hipError_t launch_interp_records(const int4* ent, const int* ent_off, const float2* nodes, int E, int n0, int n1,
                                 int half, const double* chol, float* px, float* py, hipStream_t st) {
  if (E <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_interp_records, dim3((E + 255) / 256), dim3(256), 0, st, ent, ent_off, nodes, E, n0, n1, half,
                     chol, px, py);
  return hipGetLastError();
}

hipError_t launch_window_records(const int4* ent, const int* ent_off, const float2* nodes, int E, int n0, int n1,
                                 int K, int C, float beta0, float beta1, float* px, float* py, hipStream_t st) {
  if (E <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_window_records, dim3((unsigned)(((long)E * (K + C) + 255) / 256)), dim3(256), 0, st, ent,
                     ent_off, nodes, E, n0, n1, K, C, beta0, beta1, px, py);
  return hipGetLastError();
}

hipError_t launch_outer(const float* cx, const float* cy, int N0, int N1, float* out, hipStream_t st) {
  hipLaunchKernelGGL(k_outer, dim3((N0 * N1 + 255) / 256), dim3(256), 0, st, cx, cy, N0, N1, out);
  return hipGetLastError();
}

int spectrum_splits(int n0, int n1) { return std::max(1, std::min(16, 256 / ((n0 / 64) * (n1 / 64)))); }

hipError_t launch_spectrum_chunk(const float2* nodes, const float* w, int j0, int cnt, int N0, int N1, int n0, int n1,
                                 double* d0, double* d1, double* acc, hipStream_t st) {
  if (n0 % 64 || n1 % 64 || cnt < 1) return hipErrorInvalidValue;
  const int cntp = (cnt + 15) / 16 * 16;
  const float* xy = reinterpret_cast<const float*>(nodes);
  hipLaunchKernelGGL(k_dirichlet, dim3((unsigned)(((long)cntp * n0 + 255) / 256)), dim3(256), 0, st, xy, w, j0, cnt,
                     cntp, N0, n0, d0);
  hipLaunchKernelGGL(k_dirichlet, dim3((unsigned)(((long)cntp * n1 + 255) / 256)), dim3(256), 0, st, xy + 1,
                     (const float*)nullptr, j0, cnt, cntp, N1, n1, d1);
  hipLaunchKernelGGL(k_spectrum, dim3(n0 / 64, n1 / 64, spectrum_splits(n0, n1)), dim3(256), 0, st, d0, d1, cntp, n0,
                     n1, acc);
  return hipGetLastError();
}

hipError_t launch_spectrum_store(const double* acc, int n0, int n1, bool half, float* spec, hipStream_t st) {
  const size_t n = (size_t)n0 * (half ? n1 / 2 + kNormalC : n1);
  hipLaunchKernelGGL(k_spectrum_store, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, acc,
                     spectrum_splits(n0, n1), n0, n1, half ? 1 : 0, spec);
  return hipGetLastError();
}

hipError_t launch_wave_gram(const float2* nodes, int nq, int N0, int N1, float* g, hipStream_t st) {
  const int n = 4 * nq * nq;
  hipLaunchKernelGGL(k_wave_gram, dim3((n + 255) / 256), dim3(256), 0, st, nodes, nq, N0, N1, g);
  return hipGetLastError();
}

hipError_t launch_wave_chunk(const float2* nodes, const float* w, int j0, int cnt, int nq, int ld, int N0, int N1,
                             double* fw, double* f, double* acc, hipStream_t st) {
  if (ld % 64 || ld < 2 * nq || cnt < 1) return hipErrorInvalidValue;
  const int cntp = (cnt + 15) / 16 * 16;
  hipLaunchKernelGGL(k_wave_nodes, dim3((unsigned)(((long)cntp * ld + 255) / 256)), dim3(256), 0, st, nodes, w, j0,
                     cnt, cntp, nq, ld, N0, N1, fw, f);
  hipLaunchKernelGGL(k_spectrum, dim3(ld / 64, ld / 64, spectrum_splits(ld, ld)), dim3(256), 0, st, fw, f, 2 * cntp,
                     ld, ld, acc);
  return hipGetLastError();
}

hipError_t launch_wave_store(const double* acc, int nq, int ld, float* h, hipStream_t st) {
  const int n = 4 * nq * nq;
  hipLaunchKernelGGL(k_wave_store, dim3((n + 255) / 256), dim3(256), 0, st, acc, spectrum_splits(ld, ld), 2 * nq, ld, h);
  return hipGetLastError();
}

}  // namespace icon
