// Column tiles of the oversampled grid: the n0 x C tile's layouts in LDS, its
// x FFT from global memory and the interpolation at the tile's nodes (device
// code shared by the transforms and the solve).
#pragma once
#include <hip/hip_runtime.h>

#include "icon_fft.h"
#include "icon_kernels.h"

namespace icon {

// LDS rows of the row kernels carry one float2 of padding after every 32
// elements: the first pass stores 16 consecutive elements per thread, which
// without it would put every second thread of a wavefront on the same banks.
using RowLay = Lay<1, 5, 1>;

// Row stride (float2) of the LDS tile: C + 2 keeps rows 16-byte aligned for
// vector reads while two blocks still share a CU's LDS; otherwise C + 1.
template <int NC, int C>
__host__ __device__ constexpr int col_stride() {
  return NC * (C + 2) * 8 <= 81920 ? C + 2 : C + 1;
}

// Layouts of the tile during the x FFT's exchanges.  A wavefront holds 64/C
// threads per column; at C = 8 each of its 8-byte loads and stores touches 8
// rows of the C columns at once, and the layout puts those rows on disjoint
// banks (2 cycles per 64-lane access, the minimum):
// * interpolation: row stride C, 8 float2 of padding after every 16 rows;
// * spread: row stride C, 1 float2 of padding after every 4 rows, which also
//   keeps the spread's own stores conflict-free (each thread writes its two
//   whole rows, 2 apart across lanes, where the padding every 16 rows would
//   put 4 lanes on one bank).
// The stride C + 1 used before took 3 cycles for most FFT accesses.
template <int C>
using ColFftLayFwd = Lay<C, 4, 8>;
template <int C>
using ColFftLay = Lay<C, 2, 1>;

// float2 of LDS per column block: the tile, or an FFT layout if larger
template <int NC, int C>
__host__ __device__ constexpr int col_lds() {
  constexpr int tile = NC * col_stride<NC, C>();
  constexpr int fwd = ColFftLayFwd<C>::at(NC - 1) + C, adj = ColFftLay<C>::at(NC - 1) + C;
  return tile > fwd ? (tile > adj ? tile : adj) : (fwd > adj ? fwd : adj);
}

// Buffer over the N0 grid rows of slice s, and the byte offset in it of grid
// row x = t + c (x FFT order, thread t < NC/16, slot constant c outside [NC/4,
// 3NC/4); image row X = x + N0/2 mod NC) and column y: past the buffer where the
// row is padding, so that its load gives 0 and its store is dropped.  32-bit
// offsets from one scalar base (the rows of a slice are at most 16 MiB) keep
// the kernels' addresses in few registers; the slots' offsets differ by scalars.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t slice_rows(const float2* p, const ColArgs& a, int s) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float2*>(p + (size_t)s * a.N0 * a.n1), (short)0,
                                           a.N0 * a.n1 * (int)sizeof(float2), 0x00020000);
}
template <int NC>
__device__ __forceinline__ unsigned row_offset(const ColArgs& a, int t, int c, int y) {
  const int X0 = t + (a.N0 >> 1), d = c < NC / 2 ? c : c - NC;
  return (unsigned)(X0 + d) < (unsigned)a.N0 ? (unsigned)((X0 * a.n1 + y) * 8 + d * a.n1 * 8) : 0x80000000u;
}

// x FFT of column c = tid % C of slice s: the first pass takes its 16 inputs
// (grid rows t + r NC/16; zero padding outside the N0 non-zero rows) straight
// from global memory, all loads in flight together; the output stays in
// registers in the FFT's output order.  Ends past the last exchange's barrier:
// the tile's LDS can be overwritten.
template <int NC, int C, bool LAZY = false>
__device__ __forceinline__ void col_fft_fwd(float2 (&v)[16], const ColArgs& a, float2* tile, int s, int y0) {
  const int c = threadIdx.x % C, t = threadIdx.x / C;
  // rows x in [NC/4, 3NC/4) (inputs 4..11) are padding, as N0 <= NC/2; the
  // other inputs are buffer loads over the slice's grid rows, at offsets past
  // its end for rows past N0 (only when N0 < NC/2), which read as 0
  const auto rs = slice_rows(a.in, a, s);
  float2 g[8];
#pragma unroll
  for (int j = 0; j < 8; j++)
    g[j] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(
                                          rs, row_offset<NC>(a, t, (j < 4 ? j : j + 8) * (NC / 16), y0 + c), 0, 0));
  // the twiddles (first used after the first pass) are requested after
  // the grid rows, so that the first pass waits for the rows only
  FftTwiddles T;
  if constexpr (!LAZY) load_twiddles<NC, -1>(T, t, a.tw);
#pragma unroll
  for (int j = 0; j < 8; j++) v[j < 4 ? j : j + 8] = g[j];
  if constexpr (LAZY) fft_from_lazy<NC, ColFftLayFwd<C>, -1, 1, 0, true>(v, tile + c, t, T, a.tw);
  else fft_regs_half<NC, ColFftLayFwd<C>, -1>(v, tile + c, t, T);
}

// Interpolation partials of tile blk of slice s, whose x-transformed grid
// columns lie in the LDS tile (row stride col_stride<NC, C>()); of its entries
// those of share `part` of `parts`.
template <int NC, int C, int K>
__device__ __forceinline__ void interp_tile(const ColArgs& a, const float2* tile, int blk, int s, int part = 0,
                                            int parts = 1) {
  constexpr int NT = C * (NC / 16);
  constexpr int LS = col_stride<NC, C>();
  const int tid = threadIdx.x;
  // interpolation partials of this tile's nodes: one bin entry per thread;
  // the entry's record (first x-tap, K x-taps, C y-taps) comes in with
  // vector loads and the thread sums its K x C cells from the LDS tile
  const int e0 = a.ent_off[blk], e1 = a.ent_off[blk + 1], ne = e1 - e0;
  for (int e = e0 + part * NT + tid; e < e1; e += parts * NT) {
    const int4 en = a.fent[e];
    float px[K];
    const float2* pxv = reinterpret_cast<const float2*>(a.fent_px + (size_t)e0 * K) + (e - e0);
#pragma unroll
    for (int q = 0; q < K / 2; q++) {
      const float2 p = pxv[q * ne];
      px[2 * q] = p.x;
      px[2 * q + 1] = p.y;
    }
    float py[C];
    const float4* pyv = reinterpret_cast<const float4*>(a.fent_py + (size_t)e0 * C) + (e - e0);
#pragma unroll
    for (int c4 = 0; c4 < C / 4; c4++) {
      const float4 v = pyv[c4 * ne];
      py[4 * c4] = v.x; py[4 * c4 + 1] = v.y; py[4 * c4 + 2] = v.z; py[4 * c4 + 3] = v.w;
    }
    // separable window: each grid row is first reduced over its C y-taps,
    // then weighted by its x-tap
    float ax = 0.f, ay = 0.f;
    auto add_row = [&](const float2* row, int q) {
      float2 gv[C];
      if constexpr (LS % 2 == 0) {
#pragma unroll
        for (int c2 = 0; c2 < C / 2; c2++) {
          const float4 g4 = reinterpret_cast<const float4*>(row)[c2];
          gv[2 * c2] = make_float2(g4.x, g4.y);
          gv[2 * c2 + 1] = make_float2(g4.z, g4.w);
        }
      } else {
#pragma unroll
        for (int c = 0; c < C; c++) gv[c] = row[c];
      }
      float tx = 0.f, ty = 0.f;
#pragma unroll
      for (int c = 0; c < C; c++) {
        tx = __fmaf_rn(gv[c].x, py[c], tx);
        ty = __fmaf_rn(gv[c].y, py[c], ty);
      }
      ax = __fmaf_rn(tx, px[q], ax);
      ay = __fmaf_rn(ty, px[q], ay);
    };
    // Entries whose taps wrap past row NC-1 have the largest first taps and
    // come last in the tile's order: only the last wavefronts can hold them;
    // the others take the fully unrolled loop with one base address and
    // constant row offsets.
    if (__builtin_amdgcn_ballot_w64(en.z > NC - K) == 0) {
      const float2* base = tile + en.z * LS;
#pragma unroll
      for (int q = 0; q < K; q++) add_row(base + q * LS, q);
    } else {
#pragma unroll 2
      for (int q = 0; q < K; q++) add_row(tile + ((en.z + q) & (NC - 1)) * LS, q);
    }
    // bit 31 of w: the value is the conjugate (mirrored half of the grid)
    a.part[((size_t)s * a.M + en.x) * a.slots + ((en.y >> 16) & 0xff)] =
        make_float2(ax, __int_as_float(__float_as_int(ay) ^ (en.w & (int)0x80000000)));
  }
}

// FP64 sums of N values over a block of 1024 threads, in a fixed order: by lane
// halves within each wavefront, then the wavefronts in order.  red: 16 N doubles.
template <int N>
__device__ __forceinline__ void block_sums_1024(double (&v)[N], double* red) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int k = 0; k < N; k++) {
#pragma unroll
    for (int h = 32; h > 0; h >>= 1) v[k] += __shfl_down(v[k], h);
    if ((tid & 63) == 0) red[16 * k + (tid >> 6)] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; k++) {
    double r = red[16 * k];
#pragma unroll
    for (int w = 1; w < 16; w++) r += red[16 * k + w];
    v[k] = r;
  }
  __syncthreads();
}
__device__ __forceinline__ double block_sum_1024(double v, double* red) {
  double x[1] = {v};
  block_sums_1024(x, red);
  return x[0];
}

// Value of node j: its partials of up to `slots` column tiles, in slot order.
__device__ __forceinline__ float2 node_value(const float2* part, const int8_t* nslot, int j, int slots) {
  const int ns = nslot[j];
  float2 f = part[(size_t)j * slots];
  for (int q = 1; q < ns; q++) {
    const float2 p = part[(size_t)j * slots + q];
    f.x += p.x;
    f.y += p.y;
  }
  return f;
}

}  // namespace icon
