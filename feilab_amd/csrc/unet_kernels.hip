// CDNA4 kernels of the learned warm start: a 2D U-Net on BF16 MFMA.
//
// Tensors are NHWC.  Forward activations are BF16 (stored as uint16), the
// gradients FP32; weights keep an FP32 master copy and a BF16 compute copy in
// the layout [tap][c_out][c_in] (c_in fastest), taps ky*3 + kx.
//
// The 3x3 (and 1x1) convolution is an implicit GEMM on
// v_mfma_f32_16x16x32_bf16: M = output channels, N = pixels, K = taps x
// input channels in groups of 32.  Lane l feeds A[channel slot l%16][8 input
// channels 8*(l/16)...] (weights) and B[8 input channels 8*(l/16)...][pixel
// l%16] as 16-byte vectors from LDS-staged tiles and receives D[slots
// 4*(l/16)+i][pixel l%16], the slots ordered so that they are consecutive
// output channels.  The same kernel computes the input gradient with the
// spatially flipped, channel-transposed weights; the weight gradient is a
// split-K GEMM over pixels whose operands are transposed through LDS.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "unet_kernels.h"

namespace unet {

typedef __attribute__((ext_vector_type(4))) float f4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf8;

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
// round to nearest even
__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);   // inf / nan
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

union V8 {
  uint4 u;
  uint16_t h[8];
  bf8 v;
};

// Sum of the 1x1 head over one group of 8 channels, in channel order,
// starting from s0.  The head adds the groups' sums in group order:
// out = ((b + S_0) + S_1) + ... with S_g the group sum started from 0 (g > 0),
// the order that the fused head of the convolution epilogue also follows.
__device__ __forceinline__ float head_group(const V8& v, const float* w, float s0) {
  float s = s0;
#pragma unroll
  for (int k = 0; k < 8; k++) s = fmaf(bf2f(v.h[k]), w[k], s);
  return s;
}



// ----------------------------------------------------------------- conv
// Block: 256 threads = 4 waves on a 4R x 16 pixel tile of one image and COB
// output channels.  Per 32-channel chunk of the input the block stages the
// tile with its one-pixel halo ((4R + 2) x 18 pixels) and the chunk's
// weights for all taps in LDS (64-byte rows with a bank swizzle, kLdsRow);
// wave w then multiplies the COB/16 weight tiles by tile rows Rw..Rw+R-1 (R
// MFMA column tiles of 16 pixels) for every tap, reading both operands from
// LDS.
//
// The weights are the MFMA's A operand and the pixels its B operand: lane l
// receives rows 4(l/16)..4(l/16)+3 of every weight tile's result for pixel
// l % 16.  The weight rows are staged in the order that makes those rows the
// COB/4 consecutive output channels (COB/4)(l/16)... (slot_channel), so each
// lane holds whole 16-byte runs of channels of its pixels: the epilogue adds
// the bias, applies the ReLU, rounds to BF16 and stores, pools (the pixel
// pair x, x+1 sits in neighbouring lanes) or evaluates the fused head
// straight from registers.
//
// The grid is persistent: a block walks the work items (tile, chunk) of its
// output-channel block, tiles blockIdx.x, blockIdx.x + gridDim.x, ..., and
// loads the next item's input and weights into registers while the MFMAs of
// the current one run; the weights are loaded once when the input has a
// single chunk.  The input pieces (8 channels of one halo pixel) are buffer
// loads over the tile's image, at per-thread offsets fixed for the launch
// plus one offset per tile; a piece outside the image (or the channels) is
// given an offset past the image's end, which the buffer load returns as 0.
constexpr int kTile = 16;
constexpr int kHalo = kTile + 2;
// LDS rows of staged pixels and weights: 64 bytes (32 BF16), the 16-byte
// piece c of LDS row p stored at position c ^ swz(p), swz(p) = (p / 2) % 4.
// The operand reads and the staging writes (ds_read_b128, ds_write_b128)
// take 16 consecutive rows x pieces g = l / 16 per wavefront; measured on
// gfx950, plain 64- or 80-byte rows read at half the rate of consecutive
// memory (80-byte rows write at full rate), 64-byte rows with this swizzle
// read and write at full rate.  A staged halo row is kPitch = 24 LDS rows
// (18 used), so that swz of a pixel depends on its column only.
constexpr int kLdsRow = 32;
constexpr int kPitch = 24;
__device__ __forceinline__ int swz(int x) { return (x >> 1) & 3; }
constexpr unsigned kOutside = 0x80000000u;         // a byte offset past every image

// Output channel (within the block's COB) of result slot s = 16 j + m, m the
// row of weight tile j's 16 x 16 result: lane group m / 4 holds channels
// (COB/4)(m/4) ... (COB/4)(m/4) + COB/4 - 1, in the order 4 j + m % 4.
template <int COB>
__device__ __forceinline__ int slot_channel(int s) {
  return (COB / 4) * ((s & 15) >> 2) + 4 * (s >> 4) + (s & 3);
}

// Buffer resource over `bytes` bytes at p: loads at larger offsets return 0.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t image_rsrc(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// s_waitcnt vmcnt(0).  A load whose value is stored under a per-lane
// condition is waited for only on the branch that stores it; without this
// wait on every path the compiler makes the next writes of the load's
// registers (the MFMA operands' LDS reads) wait for all loads in flight,
// the next item's prefetch included.
__device__ __forceinline__ void vm_wait_all() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// two floats rounded to BF16 (nearest even, as f2bf) in one dword, lo first
// (one v_cvt_pk_bf16_f32)
typedef __attribute__((ext_vector_type(2))) float f2v;
typedef __attribute__((ext_vector_type(2))) __bf16 bf2v;
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2v){lo, hi}, bf2v));
}
// max(v, 0) as an integer max of the bits (one instruction; the float max
// is preceded by a NaN-quieting copy): equal for every non-NaN v
__device__ __forceinline__ float relu(float v) { return __int_as_float(max(__float_as_int(v), 0)); }
__device__ __forceinline__ float bf_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf_hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }

template <typename TX, typename TY, int COB, int R, bool FIRST>
__global__ __launch_bounds__(256, COB == 32 && R <= 4 ? 3 : 2) void k_conv(ConvArgs<TX, TY> a) {
  constexpr int CT = COB / 16;
  constexpr int CL = COB / 4;                        // consecutive output channels per lane
  constexpr int PW = sizeof(TX) / 2;                 // 16-byte loads per input piece
  // the next chunk's weights are prefetched into registers with its input
  // FIRST: the input is computed from the FP32 images (a single chunk whose
  // weights are staged once, no prefetch)
  constexpr bool kWPrefetch = !FIRST;
  constexpr int kTH = 4 * R;       // tile rows: R per wave
  constexpr int kHY = kTH + 2;     // halo rows
  // FIRST: the BF16 image over the halo's own halo (kRY x kRX pixels), per
  // pixel its row of three taps (the pixel and the next two) in 8 bytes;
  // one more zero entry
  constexpr int kRY = FIRST ? kHY + 2 : 1, kRX = kHalo + 2, kRawPer = (kRY * kRX + 255) / 256;
  __shared__ __align__(16) uint16_t s_in[kHY * kPitch * kLdsRow];
  __shared__ __align__(16) uint16_t s_w[9 * COB * kLdsRow];
  __shared__ __align__(16) uint2 s_raw3[FIRST ? kRY * kRX + 1 : 1];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, g = lane >> 4;
  const int tiles_x = (a.W + kTile - 1) / kTile, tiles_y = (a.H + kTH - 1) / kTH;
  const int ntiles = a.N * tiles_x * tiles_y;
  const int nck = (a.Cin + 31) / 32;
  const int co0 = blockIdx.y * COB;
  const int cl0 = co0 + CL * g;   // this lane's first output channel
  const int taps = a.taps;
  int tt = blockIdx.x;
  if (tt >= ntiles) return;
  float bl[CL];
#pragma unroll
  for (int k = 0; k < CL; k++) bl[k] = a.bias && cl0 + k < a.Cout ? a.bias[cl0 + k] : 0.f;
  // the fused head's weights of this lane's channels (COB 32 only), loaded
  // here: a load in the epilogue would wait for the prefetch in flight
  constexpr int HW = COB == 32 ? CL : 1;
  float hw[HW], hb = 0.f;
  if constexpr (COB == 32) {
    if (a.head_out) {
#pragma unroll
      for (int k = 0; k < HW; k++) hw[k] = a.head_w[cl0 + k];
      hb = g == 0 ? a.head_b[0] : 0.f;
    }
  }
  // ---- staging.  One wave instruction moves 16 consecutive pixels (or
  // weight rows) x 4 pieces of 8 channels: lane l takes pixel / row l % 16
  // and piece (l / 16) % 4, so each 32 lanes write 16 consecutive LDS rows
  // x 2 pieces (distinct banks, kLdsRow) and the wave reads 1 KB of
  // consecutive memory.  Offsets that do not change during the launch are
  // computed here once; a piece outside the image or the tensor is given
  // the offset kOutside, which the buffer load returns as 0.
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  const int lx = lane & 15, lc8 = 8 * ((lane >> 4) & 3);
  // Input, main part: halo rows 0..kHY-1 x halo columns 0..15; wave w takes
  // the rows w, w + 4, ... (kRounds rounds, the last one waves 0 and 1 only).
  // Byte offset of this lane's piece from halo column 0 of a row, in x and
  // in the half-size tensor up:
  constexpr int kRounds = (kHY + 3) / 4;
  const unsigned lo_x = (unsigned)((lx * a.ldx + lc8) * (int)sizeof(TX));
  const unsigned lo_u = (unsigned)((((lx + 1) >> 1) * a.ldu + lc8) * 2);
  // Input, extra part: halo columns 16 and 17 of every row, 8 kHY pieces in
  // kExR rounds; piece e = t + 256 round: row e / 8, column 16 + (e / 4) % 2,
  // piece e % 4.
  constexpr int kExR = (8 * kHY + 255) / 256;
  const int ex_x = kTile + ((tid >> 2) & 1), ex_c8 = 8 * (tid & 3);
  // LDS element offsets of this lane's pieces (main: round 0; round r is
  // 4 r halo rows further)
  const int la_in = (wave * kPitch + lx) * kLdsRow + 8 * (((lane >> 4) & 3) ^ swz(lx));
  const int la_ex = ((tid >> 3) * kPitch + ex_x) * kLdsRow + 8 * ((tid & 3) ^ swz(ex_x));   // round e: + 32 e halo rows
  // Weights: slot row r = tap * COB + slot; round k covers rows 64 k ... 64 k
  // + 63, wave w the rows 64 k + 16 w + (0..15), so the tap (64 k + 16 w) /
  // COB of a round is uniform and the lane's slot (16 w + lx) % COB fixed.
  constexpr int kWRounds = (9 * COB + 63) / 64;
  const int wco = co0 + slot_channel<COB>((16 * wave + lx) % COB);
  const unsigned lo_w = wco < a.Cout ? (unsigned)((wco * a.Cin + lc8) * 2) : kOutside;
  const int la_w = (16 * wave + lx) * kLdsRow + 8 * (((lane >> 4) & 3) ^ swz(lx));
  uint4 pin[FIRST ? 1 : kRounds + kExR][PW];
  uint4 wreg[kWRounds];
  // loads the chunk's weights into registers
  const uint16_t* const Wt0 = a.w;
  const long wtap = (long)a.Cout * a.Cin;   // elements per tap
  auto wfetch = [&](int ck) {
    const uint16_t* wck = Wt0 + 32 * ck;
#pragma unroll
    for (int k = 0; k < kWRounds; k++) {
      const int t = (64 * k + 16 * wv) / COB;
      wreg[k] = make_uint4(0, 0, 0, 0);
      if (t < taps) {
        const auto rs = image_rsrc(wck + t * wtap, 0x7fffffffu);
        wreg[k] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, lo_w, 0, 0));
      }
    }
  };
  auto wput = [&]() {
#pragma unroll
    for (int k = 0; k < kWRounds; k++)
      if ((64 * k + 16 * wv) / COB < taps) *reinterpret_cast<uint4*>(&s_w[la_w + 64 * k * kLdsRow]) = wreg[k];
    vm_wait_all();
  };
  // loads the input tile + halo of work item (tile, chunk) into registers
  const TX* const X = a.x;
  const uint16_t* const UP = a.up;
  const int H = a.H, W = a.W, H2 = a.H >> 1, W2 = a.W >> 1, ldx = a.ldx, ldu = a.ldu;
  // FIRST: this thread's image pixels p = tid + 256 i of the kRY x kRX
  // region at image (y0 - 2, x0 - 2) and the two after each; the first
  // convolution's weights as MFMA A operands, K position 4 ty + tx for tap
  // (ty, tx) (positions 4 ty + 3 and from 12 on zero), and its bias as the
  // MFMA's C operand, per lane as the second convolution's own slots
  float rawv[FIRST ? kRawPer : 1][3];
  bf8 w1a[FIRST ? CT : 1];
  f4 b1c[FIRST ? CT : 1];
  if constexpr (FIRST) {
#pragma unroll
    for (int j = 0; j < CT; j++) {
      const int ch = slot_channel<COB>(16 * j + r16);
      V8 v;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const int ty = 2 * g + k / 4, tx = k % 4;
        v.h[k] = tx < 3 && ty < 3 ? a.w1[((long)(3 * ty + tx) * COB + ch) * a.w1_cin] : (uint16_t)0;
      }
      w1a[j] = v.v;
      // result rows 4 g + r of weight tile j: channels cl0 + 4 j + r
      b1c[j] = f4{a.b1[cl0 + 4 * j], a.b1[cl0 + 4 * j + 1], a.b1[cl0 + 4 * j + 2], a.b1[cl0 + 4 * j + 3]};
    }
    if (tid == 0) s_raw3[kRY * kRX] = make_uint2(0, 0);
  }
  auto fetch = [&](int tile, int ck) {
    const int tx = tile % tiles_x, rest = tile / tiles_x;
    const int y0 = (rest % tiles_y) * kTH, x0 = tx * kTile, n = rest / tiles_y;
    if constexpr (FIRST) {
      const auto rs = image_rsrc(a.x1 + (long)n * a.H * a.W, 0x7fffffffu);
#pragma unroll
      for (int i = 0; i < kRawPer; i++) {
        const int p = tid + 256 * i, ry = p / kRX, rx = p - kRX * ry;
        const int yy = y0 - 2 + ry, xx = x0 - 2 + rx;
        const bool oky = p < kRY * kRX && (unsigned)yy < (unsigned)a.H;
#pragma unroll
        for (int d = 0; d < 3; d++) {
          const bool ok = oky && (unsigned)(xx + d) < (unsigned)a.W;
          rawv[i][d] = __uint_as_float(
              __builtin_amdgcn_raw_buffer_load_b32(rs, ok ? (unsigned)((yy * a.W + xx + d) * 4) : kOutside, 0, 0));
        }
      }
      return;
    }
    const int ci0 = 32 * ck;
    bool from_up = false;
    if constexpr (sizeof(TX) == 2) from_up = ci0 < a.Cup;   // Cup is a multiple of 32
    // halo row wv (image row y0 - 1 + wv) from halo column 0 (image column
    // x0 - 1; its offset is not used where that column is outside the
    // image), and the step of 4 halo rows (2 rows of up), in bytes
    const int yw = y0 - 1 + wv;
    const char* row0;
    long step;
    if (from_up) {
      row0 = reinterpret_cast<const char*>(UP + (((long)n * H2 + (yw >> 1)) * W2 + (x0 >> 1) - 1) * ldu + a.cu0 + ci0);
      step = 2L * W2 * ldu * 2;
    } else {
      row0 = reinterpret_cast<const char*>(X + (((long)n * H + yw) * W + x0 - 1) * ldx + a.cx0 + ci0);
      step = 4L * W * ldx * (long)sizeof(TX);
    }
    const unsigned lo = (unsigned)(x0 - 1 + lx) < (unsigned)W ? (from_up ? lo_u : lo_x) : kOutside;
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
#pragma unroll
      for (int h = 0; h < PW; h++) pin[r][h] = make_uint4(0, 0, 0, 0);
      if ((r < kRounds - 1 || wv + 4 * r < kHY) && (unsigned)(yw + 4 * r) < (unsigned)H) {
        const auto rs = image_rsrc(row0 + r * step, 0x7fffffffu);
#pragma unroll
        for (int h = 0; h < PW; h++)
          pin[r][h] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, lo + 16 * h, 0, 0));
      }
    }
#pragma unroll
    for (int e = 0; e < kExR; e++) {
      const int yy = y0 - 1 + (tid >> 3) + 32 * e, xx = x0 - 1 + ex_x;
      const bool ok = tid + 256 * e < 8 * kHY && (unsigned)yy < (unsigned)H && (unsigned)xx < (unsigned)W;
      const char* img;
      unsigned off;
      if (from_up) {
        img = reinterpret_cast<const char*>(UP + (long)n * H2 * W2 * ldu + a.cu0 + ci0);
        off = (unsigned)((((yy >> 1) * W2 + (xx >> 1)) * ldu + ex_c8) * 2);
      } else {
        img = reinterpret_cast<const char*>(X + (long)n * H * W * ldx + a.cx0 + ci0);
        off = (unsigned)(((yy * W + xx) * ldx + ex_c8) * (int)sizeof(TX));
      }
      const auto rs = image_rsrc(img, 0x7fffffffu);
#pragma unroll
      for (int h = 0; h < PW; h++)
        pin[kRounds + e][h] =
            __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, ok ? off + 16 * h : kOutside, 0, 0));
    }
  };
  // FIRST: the staged input is the first convolution over the halo, from the
  // image rows in LDS: per 16 halo pixels one MFMA per 16 channels, K = the
  // taps (lane group 0 tap rows 0 and 1, group 1 row 2, the rest zero); zero
  // outside the image (the input's padding); the tile's own pixels also to
  // a1_out
  auto put_first = [&](int tile) {
    const int tx = tile % tiles_x, rest = tile / tiles_x;
    const int y0 = (rest % tiles_y) * kTH, x0 = tx * kTile, n = rest / tiles_y;
    const float sc = a.x1_scale ? a.x1_scale[n] : 1.f;
#pragma unroll
    for (int i = 0; i < kRawPer; i++) {
      const int p = tid + 256 * i;
      // as the input conversion rounds the image
      if (p < kRY * kRX)
        s_raw3[p] = make_uint2((uint32_t)f2bf(rawv[i][0] / sc) | ((uint32_t)f2bf(rawv[i][1] / sc) << 16),
                               (uint32_t)f2bf(rawv[i][2] / sc));
    }
    __syncthreads();
    constexpr int kHP = kHY * kHalo, kPT = (kHP + 15) / 16, kZero = kRY * kRX;
    // every halo pixel inside the image (most tiles): no per-pixel test
    const bool interior = y0 >= 1 && y0 + kTH + 1 <= a.H && x0 >= 1 && x0 + kTile + 1 <= a.W;
    // halo pixel q = 16 pt + r16, pt = wv, wv + 4, ...: q grows by 64 = 3 rows + 10 columns
    int hy = (16 * wv + r16) / kHalo, hx = (16 * wv + r16) - kHalo * hy;
#pragma unroll 1
    for (int pt = wv; pt < kPT; pt += 4) {
      const bool valid = 16 * pt + r16 < kHP;
      const int rb = hy * kRX + hx;   // image pixel of tap (0, 0)
      const int i0 = !valid ? kZero : g == 0 ? rb : g == 1 ? rb + 2 * kRX : kZero;
      const int i1 = valid && g == 0 ? rb + kRX : kZero;
      const uint2 lo = s_raw3[i0], hi = s_raw3[i1];
      V8 b;
      b.u = make_uint4(lo.x, lo.y, hi.x, hi.y);
      f4 d[CT];
#pragma unroll
      for (int j = 0; j < CT; j++) d[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1a[j], b.v, b1c[j], 0, 0, 0);
      // channels cl0 + k = 8 g + k of halo pixel (hy, hx)
      const int yy = y0 - 1 + hy, xx = x0 - 1 + hx;
      const bool inside = valid && (interior || ((unsigned)yy < (unsigned)a.H && (unsigned)xx < (unsigned)a.W));
      uint4 o;
      uint32_t* po = reinterpret_cast<uint32_t*>(&o);
#pragma unroll
      for (int k = 0; k < CL; k += 2)
        po[k / 2] = pack_bf16(relu(d[k >> 2][k & 3]), relu(d[(k + 1) >> 2][(k + 1) & 3]));
      if (!inside) o = make_uint4(0, 0, 0, 0);
      if (valid) *reinterpret_cast<uint4*>(&s_in[(hy * kPitch + hx) * kLdsRow + 8 * (g ^ swz(hx))]) = o;
      if (a.a1_out && inside && hy >= 1 && hy <= kTH && hx >= 1 && hx <= kTile)
        *reinterpret_cast<uint4*>(a.a1_out + (((long)n * a.H + yy) * a.W + xx) * COB + cl0) = o;
      hx += 10;
      hy += 3;
      if (hx >= kHalo) {
        hx -= kHalo;
        hy += 1;
      }
    }
  };
  // stores the prefetched input and, when they change, the chunk's weights
  // (read straight from L2: every block of the launch reads the same ones)
  auto put = [&](int tile, int ck, bool with_w) {
    auto bf = [&](const uint4* p) {
      if constexpr (PW == 1) {
        return p[0];
      } else {
        // FP32 input: 8 channels rounded to BF16
        uint4 v;
        v.x = pack_bf16(__uint_as_float(p[0].x), __uint_as_float(p[0].y));
        v.y = pack_bf16(__uint_as_float(p[0].z), __uint_as_float(p[0].w));
        v.z = pack_bf16(__uint_as_float(p[1].x), __uint_as_float(p[1].y));
        v.w = pack_bf16(__uint_as_float(p[1].z), __uint_as_float(p[1].w));
        return v;
      }
    };
    if constexpr (FIRST) {
      put_first(tile);
    } else {
#pragma unroll
      for (int r = 0; r < kRounds; r++)
        if (r < kRounds - 1 || wv + 4 * r < kHY)
          *reinterpret_cast<uint4*>(&s_in[la_in + 4 * r * kPitch * kLdsRow]) = bf(pin[r]);
#pragma unroll
      for (int e = 0; e < kExR; e++)
        if (tid + 256 * e < 8 * kHY)
          *reinterpret_cast<uint4*>(&s_in[la_ex + 32 * e * kPitch * kLdsRow]) = bf(pin[kRounds + e]);
      vm_wait_all();
    }
    if (with_w) {
      if constexpr (!kWPrefetch) wfetch(ck);
      wput();
    }
  };
  f4 acc[R][CT];
#pragma unroll
  for (int i = 0; i < R; i++)
#pragma unroll
    for (int j = 0; j < CT; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  int ck = 0;
  bool w_in = true;   // the weights in LDS are not this chunk's
  fetch(tt, 0);
  if constexpr (kWPrefetch) wfetch(0);
  for (;;) {
    put(tt, ck, w_in);
    __syncthreads();
    // the next work item; its loads are in flight during this item's MFMAs
    int tt2 = tt, ck2 = ck + 1;
    if (ck2 == nck) {
      ck2 = 0;
      tt2 = tt + gridDim.x;
    }
    const bool more = tt2 < ntiles;
    w_in = nck > 1;
    if (more) {
      fetch(tt2, ck2);
      if constexpr (kWPrefetch)
        if (w_in) wfetch(ck2);
    }
    if (taps == 9) {
      // for a column offset dx the B operand of tile row i at row offset dy
      // is halo row R w + i + dy: R + 2 halo rows serve all three dy
#pragma unroll 1
      for (int dx = 0; dx < 3; dx++) {
        // scheduling hint: interleave the LDS operand reads with the MFMAs
        // (single-wave small-GEMM strategy; measured 1.7 % faster, same
        // code otherwise)
        __builtin_amdgcn_iglp_opt(1);
        bf8 P[R + 2];
        const int pc = 8 * (g ^ swz(r16 + dx));
#pragma unroll
        for (int h = 0; h < R + 2; h++) {
          V8 v;
          v.u = *reinterpret_cast<const uint4*>(&s_in[((R * wave + h) * kPitch + r16 + dx) * kLdsRow + pc]);
          P[h] = v.v;
        }
#pragma unroll
        for (int dy = 0; dy < 3; dy++) {
          const int t = dy * 3 + dx;
          bf8 Wt[CT];
#pragma unroll
          for (int j = 0; j < CT; j++) {
            V8 v;
            v.u = *reinterpret_cast<const uint4*>(&s_w[(t * COB + 16 * j + r16) * kLdsRow + 8 * (g ^ swz(r16))]);
            Wt[j] = v.v;
          }
#pragma unroll
          for (int i = 0; i < R; i++)
#pragma unroll
            for (int j = 0; j < CT; j++)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Wt[j], P[i + dy], acc[i][j], 0, 0, 0);
        }
      }
    } else {
      // 1x1: the centre of the halo
      bf8 Wt[CT];
#pragma unroll
      for (int j = 0; j < CT; j++) {
        V8 v;
        v.u = *reinterpret_cast<const uint4*>(&s_w[(16 * j + r16) * kLdsRow + 8 * (g ^ swz(r16))]);
        Wt[j] = v.v;
      }
#pragma unroll
      for (int i = 0; i < R; i++) {
        V8 v;
        v.u = *reinterpret_cast<const uint4*>(&s_in[((R * wave + i + 1) * kPitch + r16 + 1) * kLdsRow + 8 * (g ^ swz(r16 + 1))]);
#pragma unroll
        for (int j = 0; j < CT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Wt[j], v.v, acc[i][j], 0, 0, 0);
      }
    }
    if (ck == nck - 1) {
      // epilogue: acc[i][k / 4][k % 4] is channel cl0 + k of pixel
      // (y0 + R wave + i, x0 + r16)
      const int tx = tt % tiles_x, rest = tt / tiles_x;
      const int y0 = (rest % tiles_y) * kTH, x0 = tx * kTile, n = rest / tiles_y;
      const int x = x0 + r16;
      if constexpr (sizeof(TY) == 2) {
#pragma unroll
        for (int i0 = 0; i0 < R; i0 += 2) {
          // rows i0, i0 + 1: bias, ReLU and the rounding to BF16 once (the
          // stores, the pool and the head all use the rounded values)
          uint32_t pk[2][CL / 2];
#pragma unroll
          for (int h = 0; h < 2; h++) {
            const int i = i0 + h;
#pragma unroll
            for (int k = 0; k < CL; k += 2) {
              float v0 = acc[i][k >> 2][k & 3] + bl[k];
              float v1 = acc[i][(k + 1) >> 2][(k + 1) & 3] + bl[k + 1];
              if (a.relu) {
                v0 = relu(v0);
                v1 = relu(v1);
              }
              pk[h][k / 2] = pack_bf16(v0, v1);
            }
            const int y = y0 + R * wave + i;
            if (COB == 32 && a.head_out) {
              // lane group g holds the head's channel group g (COB = Cout
              // = 32): its sum in channel order, then the groups' sums in
              // group order, as k_head_fwd adds them
              float s = hb;
#pragma unroll
              for (int k = 0; k < HW; k += 2) {
                s = fmaf(bf_lo(pk[h][k / 2]), hw[k], s);
                s = fmaf(bf_hi(pk[h][k / 2]), hw[k + 1], s);
              }
              const float s1 = __shfl(s, r16 + 16), s2 = __shfl(s, r16 + 32), s3 = __shfl(s, r16 + 48);
              if (g == 0 && y < a.H && x < a.W) a.head_out[((long)n * a.H + y) * a.W + x] = ((s + s1) + s2) + s3;
            } else if (y < a.H && x < a.W) {
              uint16_t* dst = a.y + (((long)n * a.H + y) * a.W + x) * a.ldy + a.cy0 + cl0;
#pragma unroll
              for (int h8 = 0; h8 < CL / 8; h8++)
                if (cl0 + 8 * h8 < a.Cout)
                  *reinterpret_cast<uint4*>(dst + 8 * h8) =
                      make_uint4(pk[h][4 * h8], pk[h][4 * h8 + 1], pk[h][4 * h8 + 2], pk[h][4 * h8 + 3]);
            }
          }
          if (a.pool) {
            // 2x2 average of the rounded values, summed in the order
            // (y, x), (y, x+1), (y+1, x), (y+1, x+1); pixel x + 1 is the
            // next lane's (DPP row_shl:1 reads lane l + 1 of the 16-lane row)
            uint32_t nb[2][CL / 2];
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
              for (int k = 0; k < CL / 2; k++)
                nb[h][k] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)pk[h][k], 0x101, 0xf, 0xf, true);
            const int y = y0 + R * wave + i0;
            if (!(r16 & 1) && y + 1 < a.H && x + 1 < a.W) {
              uint32_t po[CL / 2];
#pragma unroll
              for (int k = 0; k < CL / 2; k++) {
                const float lo = 0.25f * (((bf_lo(pk[0][k]) + bf_lo(nb[0][k])) + bf_lo(pk[1][k])) + bf_lo(nb[1][k]));
                const float hi = 0.25f * (((bf_hi(pk[0][k]) + bf_hi(nb[0][k])) + bf_hi(pk[1][k])) + bf_hi(nb[1][k]));
                po[k] = pack_bf16(lo, hi);
              }
              uint16_t* dst =
                  a.pool + (((long)n * (a.H >> 1) + (y >> 1)) * (a.W >> 1) + (x >> 1)) * a.ldp + a.cp0 + cl0;
#pragma unroll
              for (int h8 = 0; h8 < CL / 8; h8++)
                if (cl0 + 8 * h8 < a.Cout)
                  *reinterpret_cast<uint4*>(dst + 8 * h8) =
                      make_uint4(po[4 * h8], po[4 * h8 + 1], po[4 * h8 + 2], po[4 * h8 + 3]);
            }
          }
        }
      } else {
        // FP32 output (an input gradient), in whole 16-byte accesses, with
        // what the backward pass does next to it: the ReLU mask, and instead
        // of a pass of its own each
        //   usum: channels below Cus go to the half-size gradient of the
        //         upsampled tensor, as 2x2 sums
        //   pgrad: a pooled gradient goes to the four full-size pixels
        const bool up2 = co0 < a.Cus;
#pragma unroll
        for (int i0 = 0; i0 < R; i0 += 2) {
          float v[2][CL];
          const bool inx = x < a.W;
#pragma unroll
          for (int h = 0; h < 2; h++) {
            const int i = i0 + h, y = y0 + R * wave + i;
            const bool in = inx && y < a.H;
            const long p = ((long)n * a.H + y) * a.W + x;
#pragma unroll
            for (int k = 0; k < CL; k++) v[h][k] = acc[i][k >> 2][k & 3];
            if (a.mask && in) {
#pragma unroll
              for (int h8 = 0; h8 < CL / 8; h8++) {
                if (cl0 + 8 * h8 >= a.Cout) continue;
                V8 m;
                m.u = *reinterpret_cast<const uint4*>(a.mask + p * a.ldm + a.cm0 + cl0 + 8 * h8);
#pragma unroll
                for (int k = 0; k < 8; k++)
                  if (!(bf2f(m.h[k]) > 0.f)) v[h][8 * h8 + k] = 0.f;
              }
            }
            if (!in || up2 || a.pgrad) continue;
            f4* dst = reinterpret_cast<f4*>(a.y + p * a.ldy + a.cy0 + cl0 - a.Cus);
#pragma unroll
            for (int k = 0; k < CL; k += 4)
              if (cl0 + k < a.Cout) dst[k / 4] = f4{v[h][k], v[h][k + 1], v[h][k + 2], v[h][k + 3]};
          }
          const int y = y0 + R * wave + i0;
          if (up2) {
            // (y, x) + (y, x+1) + (y+1, x) + (y+1, x+1); pixel x + 1 is the
            // next lane's (DPP row_shl:1)
            f4 o[CL / 4];
#pragma unroll
            for (int k = 0; k < CL; k++) {
              const float r0 = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v[0][k]), 0x101, 0xf, 0xf, true));
              const float r1 = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v[1][k]), 0x101, 0xf, 0xf, true));
              o[k >> 2][k & 3] = ((v[0][k] + r0) + v[1][k]) + r1;
            }
            if (!(r16 & 1) && y + 1 < a.H && x + 1 < a.W) {
              f4* dst = reinterpret_cast<f4*>(
                  a.usum + (((long)n * (a.H >> 1) + (y >> 1)) * (a.W >> 1) + (x >> 1)) * a.ldus + cl0);
#pragma unroll
              for (int k = 0; k < CL / 4; k++) dst[k] = o[k];
            }
          } else if (a.pgrad) {
            // pgrad = (pgrad + v / 4) where its forward value (pmask) is positive
#pragma unroll
            for (int h = 0; h < 2; h++) {
              if (!inx || y + h >= a.H) continue;
#pragma unroll
              for (int q = 0; q < 4; q++) {
                const long p = ((long)n * (2 * a.H) + 2 * (y + h) + (q >> 1)) * (2 * a.W) + 2 * x + (q & 1);
#pragma unroll
                for (int h8 = 0; h8 < CL / 8; h8++) {
                  const int c = cl0 + 8 * h8;
                  if (c >= a.Cout) continue;
                  f4* d = reinterpret_cast<f4*>(a.pgrad + p * a.ldpg + c);
                  V8 m;
                  m.u = *reinterpret_cast<const uint4*>(a.pmask + p * a.ldpm + a.cpm0 + c);
                  f4 g[2] = {d[0], d[1]};
#pragma unroll
                  for (int k = 0; k < 8; k++)
                    g[k >> 2][k & 3] = bf2f(m.h[k]) > 0.f ? g[k >> 2][k & 3] + 0.25f * v[h][8 * h8 + k] : 0.f;
                  d[0] = g[0];
                  d[1] = g[1];
                }
              }
            }
          }
        }
      }
#pragma unroll
      for (int i = 0; i < R; i++)
#pragma unroll
        for (int j = 0; j < CT; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();   // the LDS operands are consumed before the next put
    if (!more) break;
    tt = tt2;
    ck = ck2;
  }
}

// ------------------------------------------------------------ weight grad
// dW[tap][co][ci] = sum_p dY[p][co] X[p + off(tap)][ci] and dbias[co] = sum_p
// dY[p][co] of all layers in one launch.  A GEMM whose long dimension is the
// pixels: bound by the matrix cores on the inner layers (286,000 units of 9
// MFMAs of 32 cycles on 1024 SIMDs, 16 images of 128^2: 34 us) and by the FP32
// gradients' bytes on the full-size ones.
//
// A wavefront holds a 32 x 32 (co, ci) tile of all 9 taps in registers (144
// accumulators) and walks the pixel rows of a 16-pixel-wide strip:
// v_mfma_f32_32x32x16_bf16 takes the 16 pixels of a row as its K.  An input row
// is read once, shifted in registers for the three column offsets, and
// multiplied with the three gradient rows in flight.  The block's 4 wavefronts
// are 2 x 2 tiles of 64 x 64 channels on the same rows, or fewer tiles times
// several row segments where the layer has only 32 channels (reduced through
// LDS at the end).
//
// MFMA operands are 8 consecutive pixels of one channel, tensors are channel
// fastest: a thread loads 8 channels of 2 neighbouring pixels and writes one
// dword (the pixel pair) per channel.  LDS holds per pixel row 32 bytes per
// channel; the channels of a group of 8 are rotated (slot = channel ^ group) so
// that a wavefront's 64 dword writes fall on 64 banks; the operand reads take
// 8 whole consecutive channels (256 bytes) per cycle pair either way.
//
// One launch for all layers: each needs only as many pixel splits as its share
// of the device, so the partial sums are 2 blocks per CU x 64 x 64 x 9 floats
// at most.  Measured, 14 layers of 16 images of 128^2: 131 us and 16 us for
// their reduction (one launch per layer, 64 x 64 x 1 tap tiles, gradients and
// inputs re-read for every tap, the sums and the bias gradients by kernels of
// their own: 3056 us).
typedef __attribute__((ext_vector_type(16))) float f16v;
// gradient rows per wavefront and pixel tile
__host__ __device__ constexpr int wgrad_rows(int co, int ci) { return ci == 2 ? 4 : 2; }
constexpr int kWgLds = 2 * 9 * 16 * 64 * 4;   // the segments' sums of two tiles; the staged rows take less

template <int CO, int CI>
__device__ __forceinline__ void wgrad_block(const WgradLayer& L, int bt, int split, char* lds) {
  constexpr int kWgR = wgrad_rows(CO, CI), KS = 4 / (CO * CI), TR = kWgR * KS;
  constexpr int DYB = CO * 1024, XB = CI * 1024;        // bytes of a pixel row
  char* const s_dy = lds;
  char* const s_x = s_dy + TR * DYB;
  char* const s_h = s_x + (TR + 2) * XB;                // [row][side][channel] dwords
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int co_t = wave % CO, ci_t = wave / CO % CI, ks = wave / (CO * CI);
  const int co0 = 32 * CO * (bt % L.nco), ci0 = 32 * CI * (bt / L.nco);
  const bool bias = ci0 == 0;
  const int H = L.H, W = L.W;
  f16v acc[9];
#pragma unroll
  for (int t = 0; t < 9; t++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[t][r] = 0.f;
  float bs[8];
#pragma unroll
  for (int i = 0; i < 8; i++) bs[i] = 0.f;
  // staging: lanes take the channel groups fastest (whole lines of a pixel),
  // then the pixel pairs of a row, then rows
  constexpr int GO = 4 * CO, GI = 4 * CI;
  const int go = tid % GO, po = tid / GO % 8, ro = tid / (8 * GO);
  const int gi = tid % GI, pi = tid / GI % 8, ri = tid / (8 * GI);
  constexpr int RO = 256 / (8 * GO), RI = 256 / (8 * GI);   // rows per round of the block
  // rotation of a channel group (and, with 4 groups, the row's parity: a
  // wavefront then writes two rows)
  auto rot = [](int g, int row, int G) { return G == 8 ? g : (g | (row & 1) << 2); };
  const int h = lane >> 5, c32 = lane & 31;
  const int t_end = min(L.tiles, (split + 1) * L.per);
  // the next tile's loads are in flight during this one's MFMAs: a tile's rows
  // are few enough that they fit the registers beside the accumulators (8 rows
  // per wavefront, loaded when staged: 172 us instead of 131)
  constexpr int ND = TR / RO, NX = (TR + 2 + RI - 1) / RI;
  static_assert(TR % RO == 0 && (TR + 2) * 2 * GI <= 256, "one halo piece per thread");
  f4 da[ND][2], db[ND][2];
  V8 xa[NX], xb[NX], xh;
  const int gh = tid % GI, sh = tid / GI & 1, rh = tid / (2 * GI);   // halo piece: group, side, row
  auto fetch = [&](int tile) {
    const int tx = tile % L.tiles_x, rest = tile / L.tiles_x;
    const int x0 = 16 * tx, y0 = TR * (rest % L.tiles_y), n = rest / L.tiles_y;
    const auto rdy = image_rsrc(L.dy + (long)n * H * W * L.lddy + L.cdy0 + co0, 0x7fffffffu);
    const auto rx = image_rsrc(L.x + (long)n * H * W * L.ldx + L.cx0 + ci0, 0x7fffffffu);
#pragma unroll
    for (int k = 0; k < ND; k++) {
      const int x = x0 + 2 * po, y = y0 + ro + RO * k;
      const unsigned o = (unsigned)(((y * W + x) * L.lddy + 8 * go) * 4);
      const unsigned o0 = x < W && y < H ? o : kOutside, o1 = x + 1 < W && y < H ? o + 4u * L.lddy : kOutside;
#pragma unroll
      for (int q = 0; q < 2; q++) {
        da[k][q] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rdy, o0 + 16 * q, 0, 0));
        db[k][q] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rdy, o1 + 16 * q, 0, 0));
      }
    }
    // input rows y0 - 1 .. y0 + TR
#pragma unroll
    for (int k = 0; k < NX; k++) {
      const int x = x0 + 2 * pi, row = ri + RI * k, y = y0 - 1 + row;
      const bool ok = ci0 + 8 * gi < L.Cin && row < TR + 2 && (unsigned)y < (unsigned)H;
      const unsigned o = (unsigned)(((y * W + x) * L.ldx + 8 * gi) * 2);
      xa[k].u = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rx, ok && x < W ? o : kOutside, 0, 0));
      xb[k].u = __builtin_bit_cast(
          uint4, __builtin_amdgcn_raw_buffer_load_b128(rx, ok && x + 1 < W ? o + 2u * L.ldx : kOutside, 0, 0));
    }
    // their neighbours: pixels x0 - 1 and x0 + 16
    {
      const int x = sh ? x0 + 16 : x0 - 1, y = y0 - 1 + rh;
      const bool ok = rh < TR + 2 && ci0 + 8 * gh < L.Cin && (unsigned)x < (unsigned)W && (unsigned)y < (unsigned)H;
      xh.u = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
                                           rx, ok ? (unsigned)(((y * W + x) * L.ldx + 8 * gh) * 2) : kOutside, 0, 0));
    }
  };
  auto put = [&]() {
    // gradient rows, FP32 to BF16 (nearest even) with the transposition
#pragma unroll
    for (int k = 0; k < ND; k++) {
      const int row = ro + RO * k, ro8 = rot(go, row, GO);
      char* d = s_dy + row * DYB + go * 256 + po * 4;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float u = da[k][i >> 2][i & 3], v = db[k][i >> 2][i & 3];
        bs[i] += u + v;
        *reinterpret_cast<uint32_t*>(d + ((i ^ ro8) & 7) * 32) = pack_bf16(u, v);
      }
    }
#pragma unroll
    for (int k = 0; k < NX; k++) {
      const int row = ri + RI * k, ro8 = rot(gi, row, GI);
      char* d = s_x + row * XB + gi * 256 + pi * 4;
      if (row < TR + 2) {
#pragma unroll
        for (int i = 0; i < 8; i++)
          *reinterpret_cast<uint32_t*>(d + ((i ^ ro8) & 7) * 32) = (uint32_t)xa[k].h[i] | (uint32_t)xb[k].h[i] << 16;
      }
    }
    // pixel x0 - 1 in the high half of side 0, x0 + 16 in the low half of side
    // 1 (the other halves are not used)
    if (rh < TR + 2) {
      uint32_t* d = reinterpret_cast<uint32_t*>(s_h) + (rh * 2 + sh) * 32 * CI + 8 * gh;
#pragma unroll
      for (int i = 0; i < 8; i++) d[i] = sh ? (uint32_t)xh.h[i] : (uint32_t)xh.h[i] << 16;
    }
    // (as in k_conv: the loads are waited for on every path)
    vm_wait_all();
  };
  if (split * L.per < t_end) fetch(split * L.per);
  for (int tile = split * L.per; tile < t_end; tile++) {
    put();
    __syncthreads();
    if (tile + 1 < t_end) fetch(tile + 1);
    {
      bf8 D[kWgR];
      const int co = 32 * co_t + c32, ci = 32 * ci_t + c32;
#pragma unroll
      for (int xr = 0; xr < kWgR + 2; xr++) {
        const int row = kWgR * ks + xr;
        const uint4 m = *reinterpret_cast<const uint4*>(
            s_x + row * XB + (ci >> 3) * 256 + (((ci & 7) ^ rot(ci >> 3, row, GI)) & 7) * 32 + 16 * h);
        const uint32_t hal = reinterpret_cast<const uint32_t*>(s_h)[(row * 2 + h) * 32 * CI + ci];
        if (xr < kWgR) {
          V8 v;
          v.u = *reinterpret_cast<const uint4*>(
              s_dy + row * DYB + (co >> 3) * 256 + (((co & 7) ^ rot(co >> 3, row, GO)) & 7) * 32 + 16 * h);
          D[xr] = v.v;
        }
        // lanes l and l + 32 hold the row's two halves: the last pixels of the
        // left half and the first of the right half change places
        const auto sw = __builtin_amdgcn_permlane32_swap(m.x, m.w, false, false);
        const uint32_t prev = h ? (uint32_t)sw[0] : hal, next = h ? hal : (uint32_t)sw[1];
        const uint32_t e01 = __builtin_amdgcn_alignbit(m.y, m.x, 16), e12 = __builtin_amdgcn_alignbit(m.z, m.y, 16),
                       e23 = __builtin_amdgcn_alignbit(m.w, m.z, 16);
        V8 X[3];
        X[0].u = make_uint4(__builtin_amdgcn_alignbit(m.x, prev, 16), e01, e12, e23);
        X[1].u = m;
        X[2].u = make_uint4(e01, e12, e23, __builtin_amdgcn_alignbit(next, m.w, 16));
#pragma unroll
        for (int ky = 0; ky < 3; ky++) {
          const int dr = xr - ky;   // gradient row of this input row at tap row ky
          if (dr < 0 || dr >= kWgR) continue;
#pragma unroll
          for (int kx = 0; kx < 3; kx++)
            acc[3 * ky + kx] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(D[dr], X[kx].v, acc[3 * ky + kx], 0, 0, 0);
        }
      }
    }
    __syncthreads();
  }
  // the segments' sums, in order
  if constexpr (KS > 1) {
    float* red = reinterpret_cast<float*>(lds) + (co_t + CO * ci_t) * 9 * 16 * 64 + lane;
    for (int k = 1; k < KS; k++) {
      if (ks == k) {
#pragma unroll
        for (int t = 0; t < 9; t++)
#pragma unroll
          for (int r = 0; r < 16; r++) red[(t * 16 + r) * 64] = acc[t][r];
      }
      __syncthreads();
      if (ks == 0) {
#pragma unroll
        for (int t = 0; t < 9; t++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[t][r] += red[(t * 16 + r) * 64];
      }
      __syncthreads();
    }
  }
  // result row 8 (r / 4) + 4 h + r % 4, column lane % 32
  const int ci = ci0 + 32 * ci_t + c32;
  if (ks == 0 && ci < L.Cin) {
    float* dst = L.part + (long)split * 9 * L.Cout * L.Cin + (co0 + 32 * co_t + 4 * h) * L.Cin + ci;
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
      for (int r = 0; r < 16; r++) dst[(t * L.Cout + 8 * (r >> 2) + (r & 3)) * L.Cin] = acc[t][r];
  }
  if (bias) {
    // [thread][8] in LDS, then channel c adds its group's threads in order
    float* red = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < 8; i++) red[i * 256 + tid] = bs[i];
    __syncthreads();
    if (tid < 32 * CO) {
      float s = 0.f;
      for (int k = 0; k < 256 / GO; k++) s += red[(tid & 7) * 256 + (tid >> 3) + GO * k];
      L.bpart[(long)split * L.Cout + co0 + tid] = s;
    }
  }
}

__global__ __launch_bounds__(256, 2) void k_wgrad(WgradGroup a) {
  __shared__ __align__(16) char lds[kWgLds];
  int l = 0;
  while (l + 1 < a.n && (int)blockIdx.x >= a.l[l + 1].first) l++;
  const WgradLayer& L = a.l[l];
  const int r = blockIdx.x - L.first, bt = r / L.splits, split = r - bt * L.splits;
  if (L.co == 2 && L.ci == 2) wgrad_block<2, 2>(L, bt, split, lds);
  else if (L.co == 2) wgrad_block<2, 1>(L, bt, split, lds);
  else if (L.ci == 2) wgrad_block<1, 2>(L, bt, split, lds);
  else wgrad_block<1, 1>(L, bt, split, lds);
}

// out[i] = part[0][i] + part[1][i] + ... (in that order) of every tensor of the
// group.  Weights: 4 consecutive elements per thread, 1024 per block.  The few
// biases with many parts: a wavefront per element, lanes over the parts, then
// by lane halves.
__global__ __launch_bounds__(256) void k_grad_reduce(ReduceGroup a) {
  int k = 0;
  while (k + 1 < a.n && (int)blockIdx.x >= a.t[k + 1].first) k++;
  const ReduceItem& T = a.t[k];
  const int b = blockIdx.x - T.first;
  if (T.wide) {
    const long i = ((long)b * 256 + threadIdx.x) * 4;
    if (i >= T.n) return;
    f4 s = *reinterpret_cast<const f4*>(T.part + i);
#pragma unroll 4
    for (int z = 1; z < T.nparts; z++) s += *reinterpret_cast<const f4*>(T.part + (long)z * T.n + i);
    *reinterpret_cast<f4*>(T.out + i) = s;
    return;
  }
  const long i = (long)b * 4 + (threadIdx.x >> 6);
  if (i >= T.n) return;
  float s = 0.f;
  for (int z = threadIdx.x & 63; z < T.nparts; z += 64) s += T.part[(long)z * T.n + i];
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) s += __shfl_down(s, h);
  if ((threadIdx.x & 63) == 0) T.out[i] = s;
}

// ------------------------------------------------------------ small ops

// nearest 2x upsample (bf16): out[2y+u][2x+v] = in[y][x]; 8 channels per thread
__global__ void k_up_fwd(PoolArgs a) {
  const int C8 = a.C / 8;
  const long n = (long)a.N * (2 * a.H) * (2 * a.W) * C8;   // H, W of the input
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const int c = 8 * (int)(i % C8);
    const long q = i / C8;
    const int x = (int)(q % (2 * a.W)), y = (int)((q / (2 * a.W)) % (2 * a.H));
    const long nn = q / ((long)(2 * a.W) * (2 * a.H));
    *reinterpret_cast<uint4*>(a.out + q * a.ldo + a.co0 + c) =
        *reinterpret_cast<const uint4*>(a.in + ((nn * a.H + y / 2) * a.W + x / 2) * a.ldi + a.ci0 + c);
  }
}

// 1x1 head: out[p] = b + sum_c x[p][c] w[c]  (fp32 out); C a multiple of 8
__global__ void k_head_fwd(const uint16_t* x, int ldx, const float* w, const float* b, int C, long P, float* out) {
  for (long p = (long)blockIdx.x * blockDim.x + threadIdx.x; p < P; p += (long)gridDim.x * blockDim.x) {
    float s = 0.f;
    for (int c = 0; c < C; c += 8) {
      V8 v;
      v.u = *reinterpret_cast<const uint4*>(x + p * ldx + c);
      const float g = head_group(v, w + c, c == 0 ? b[0] : 0.f);
      s = c == 0 ? g : s + g;
    }
    out[p] = s;
  }
}

// head backward, 32 channels: dX[p][c] = dout[p] w[c] (masked by ReLU of x);
// each block's sums of dw and db to part[block] (added in block order
// afterwards).  4 threads per pixel, 8 channels each, whole 16-byte accesses
// (one thread per pixel and scalar accesses: 100 us instead of 11 at 16 images
// of 128^2, a memory pass over 6 bytes per channel).
__global__ __launch_bounds__(256) void k_head_bwd(const uint16_t* x, int ldx, const float* w, long P, const float* dout,
                                                 float* dx, int lddx, float* part) {
  __shared__ float red[9][257];
  const int c0 = 8 * (threadIdx.x & 3);
  float wc[8], gw[8], gb = 0.f;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    wc[k] = w[c0 + k];
    gw[k] = 0.f;
  }
#pragma unroll 4
  for (long p = (long)blockIdx.x * 64 + (threadIdx.x >> 2); p < P; p += (long)gridDim.x * 64) {
    const float d = dout[p];
    V8 v;
    v.u = *reinterpret_cast<const uint4*>(x + p * ldx + c0);
    gb += d;
    f4 o[2];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const float xv = bf2f(v.h[k]);
      gw[k] = fmaf(d, xv, gw[k]);
      o[k >> 2][k & 3] = xv > 0.f ? d * wc[k] : 0.f;
    }
    f4* q = reinterpret_cast<f4*>(dx + p * lddx + c0);
    q[0] = o[0];
    q[1] = o[1];
  }
#pragma unroll
  for (int k = 0; k < 8; k++) red[k][threadIdx.x] = gw[k];
  red[8][threadIdx.x] = gb;
  __syncthreads();
  // channel c (32: db): the 64 threads of its group, in order
  if (threadIdx.x < 33) {
    const int c = threadIdx.x, k = c < 32 ? c & 7 : 8, g = c < 32 ? c >> 3 : 0;
    float s = 0.f;
    for (int t = 0; t < 64; t++) s += red[k][4 * t + g];
    part[(long)blockIdx.x * 33 + c] = s;
  }
}

// dgrad weights: wt[tap'][ci][co] = w[8 - tap'][co][ci]  (bf16)
__global__ void k_flip_weights(const uint16_t* w, uint16_t* wt, int taps, int Cout, int Cin) {
  const long n = (long)taps * Cout * Cin;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const int co = (int)(i % Cout);
    const int ci = (int)((i / Cout) % Cin);
    const int tp = (int)(i / ((long)Cout * Cin));
    wt[i] = w[((long)(taps - 1 - tp) * Cout + co) * Cin + ci];
  }
}

// Adam step on fp32 master weights, refreshes the bf16 copy.
__global__ void k_adam(float* w, uint16_t* w16, const float* g, float* m, float* v, long n, float lr, float b1,
                       float b2, float eps, float c1, float c2, float gscale) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const float gi = g[i] * gscale;
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
    w[i] = wi;
    if (w16) w16[i] = f2bf(wi);
  }
}

__global__ void k_f32_to_bf16(const float* in, uint16_t* out, long n, int ldo, int co0, int C) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const long p = i / C;
    const int c = (int)(i % C);
    out[p * ldo + co0 + c] = f2bf(in[i]);
  }
}

// MSE loss on scaled residual targets: d = pred - target; loss partial sums
__global__ __launch_bounds__(256) void k_mse(const float* pred, const float* target, long P, float* dpred,
                                            double* loss, float scale) {
  __shared__ double red[256];
  double s = 0.0;
  for (long p = (long)blockIdx.x * blockDim.x + threadIdx.x; p < P; p += (long)gridDim.x * blockDim.x) {
    const float d = pred[p] - target[p];
    s += (double)d * d;
    dpred[p] = scale * d;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}

// Per-image scale of the warm start: s = RMS of the image (1 for a zero image),
// accumulated in FP64: kRmsParts blocks per image write partial sums, then one
// thread per image adds them in a fixed order.
constexpr int kRmsParts = 64;

__global__ __launch_bounds__(256) void k_image_rms_part(const float* in, long P, double* part) {
  __shared__ double red[256];
  const float* x = in + (long)blockIdx.y * P;
  double s = 0.0;
  for (long p = (long)blockIdx.x * blockDim.x + threadIdx.x; p < P; p += (long)gridDim.x * blockDim.x)
    s += (double)x[p] * x[p];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[(long)blockIdx.y * kRmsParts + blockIdx.x] = red[0];
}

__global__ void k_image_rms_final(const double* part, long P, int B, float* scale) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  double s = 0.0;
  for (int k = 0; k < kRmsParts; k++) s += part[(long)b * kRmsParts + k];
  const double r = sqrt(s / (double)P);
  scale[b] = r > 0.0 ? (float)r : 1.f;
}

// out[p][0] = bf16(in[p] / scale[image]) into an 8-channel NHWC buffer
__global__ void k_to_bf16_scaled(const float* in, const float* scale, long P, long n, uint16_t* out) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    out[i * 8] = f2bf(in[i] / scale[i / P]);
}

// out = m + scale[image] * y
__global__ void k_residual_add(const float* m, const float* y, const float* scale, long P, long n, float gain,
                               float* out) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    out[i] = gain * fmaf(scale[i / P], y[i], m[i]);
}

// ================================================================ launchers

static int blocks_for(long n, int per = 256) { return (int)std::min<long>((n + per - 1) / per, 65536); }

// Blocks of a convolution's tiles of 4 R x 16 pixels and COB output channels.
static long conv_blocks(int N, int H, int W, int Cout, int COB, int R) {
  return (long)N * ((H + 4 * R - 1) / (4 * R)) * ((W + kTile - 1) / kTile) * ((Cout + COB - 1) / COB);
}

template <typename TX, typename TY, int COB, int R, bool FIRST = false>
void launch_conv_tiles(const ConvArgs<TX, TY>& a, int cus, hipStream_t st) {
  // LDS per block: the staged halo tile and one chunk's weights
  constexpr long lds = ((4L * R + 2) * kPitch + 9L * COB) * kLdsRow * 2 + (FIRST ? ((4L * R + 4) * (kHalo + 2) + 1) * 8 : 0);
  constexpr long per_cu = std::min<long>(COB == 32 && R <= 4 ? 3 : 2, (160L * 1024) / lds);
  const long tiles = (long)a.N * ((a.H + 4 * R - 1) / (4 * R)) * ((a.W + kTile - 1) / kTile);
  const int cb = (a.Cout + COB - 1) / COB;
  const long gx = std::max<long>(1, std::min<long>(tiles, per_cu * cus / cb));
  hipLaunchKernelGGL((k_conv<TX, TY, COB, R, FIRST>), dim3((unsigned)gx, (unsigned)cb), dim3(256), 0, st, a);
}

template <typename TX, typename TY>
hipError_t launch_conv(const ConvArgs<TX, TY>& a, hipStream_t st) {
  if (a.taps != 9 && a.taps != 1) return hipErrorInvalidValue;
  // the fused head needs all 32 output channels in one block's BF16 epilogue
  if (a.head_out && (sizeof(TY) != 2 || a.Cout != 32 || a.mask || a.pool || a.ldy % 8 ||
                     a.cy0 % 8 || !a.head_w || !a.head_b))
    return hipErrorInvalidValue;
  // BF16 output is plain (no mask) and stored 8 channels at a time, as is its
  // optional pool; FP32 output has no bias, ReLU or pool
  if (sizeof(TY) == 2 && (a.mask || a.usum || a.pgrad || a.Cout % 8 || a.ldy % 8 || a.cy0 % 8)) return hipErrorInvalidValue;
  if (sizeof(TY) == 4 &&
      (a.bias || a.relu || a.Cout % 8 || a.ldy % 4 || a.cy0 % 4 || (a.mask && (a.ldm % 8 || a.cm0 % 8)) ||
       (a.usum ? a.Cus % 64 || a.Cus < 1 || a.ldus % 4 || a.H % 2 || a.W % 2 || a.pgrad : a.Cus) ||
       (a.pgrad && (!a.pmask || a.ldpg % 4 || a.ldpm % 8 || a.cpm0 % 8))))
    return hipErrorInvalidValue;
  if (a.pool && (sizeof(TY) != 2 || a.ldp % 8 || a.cp0 % 8)) return hipErrorInvalidValue;
  // the input is staged in whole 32-channel chunks, each from x or from up;
  // one image's bytes are addressed by 32-bit buffer offsets
  if (a.Cin % 32 || (a.up && (a.Cup % 32 || a.H % 2 || a.W % 2)) || (!a.up && a.Cup) ||
      (long)a.H * a.W * a.ldx * (long)sizeof(TX) >= (1L << 31) || (long)a.H * a.W * a.ldu * 2 >= (1L << 31))
    return hipErrorInvalidValue;
  if (sizeof(TX) != 2 && a.up) return hipErrorInvalidValue;
  // persistent grid: the blocks that fit the device at once (LDS-bound), over
  // all output-channel blocks
  static int cus = 0;
  if (!cus) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      cus = 256;
  }
  if (a.x1) {
    // the input computed from the images: one 32-channel chunk, plain 3x3
    if (sizeof(TX) != 2 || sizeof(TY) != 2 || a.Cin != 32 || a.Cout != 32 || a.taps != 9 || a.up || !a.w1 ||
        !a.b1 || a.w1_cin < 1 || (long)a.N * a.H * a.W * 4 >= (1L << 31))
      return hipErrorInvalidValue;
    if constexpr (sizeof(TX) == 2 && sizeof(TY) == 2) launch_conv_tiles<TX, TY, 32, 8, true>(a, cus, st);
    return hipGetLastError();
  }
  // Tile shape.  Large problems: 64 channels x 16 x 16 pixels, or 32 channels x
  // 32 x 16 (BF16 input) for 32 output channels and from 4 input chunks on
  // (measured faster).  Where those blocks leave CUs idle, smaller ones: the
  // shape with the smallest blocks per CU x (MFMA cycles of a chunk + its
  // staging, in the same unit).  16 images of 128^2: the forward pass's
  // convolutions 250 -> 215 us, the input gradients' 670 -> 320 us (with the
  // weights' prefetch and without the passes that their epilogue took over,
  // 153 us).
  const bool wide = a.Cout > 32 && !(sizeof(TX) == 2 && a.Cin >= 128);
  auto cost = [&](int COB, int R, long chunk) { return (conv_blocks(a.N, a.H, a.W, a.Cout, COB, R) + cus - 1) / cus * chunk; };
  const long big = wide ? cost(64, 4, 3000) : sizeof(TX) == 2 ? cost(32, 8, 3000) : cost(32, 4, 1650);
  const long mid = cost(32, 4, 1650), small = cost(32, 2, 1000);
  if (small < mid && small < big) {
    launch_conv_tiles<TX, TY, 32, 2>(a, cus, st);
  } else if (mid < big || (!wide && sizeof(TX) != 2)) {
    launch_conv_tiles<TX, TY, 32, 4>(a, cus, st);
  } else if (wide) {
    launch_conv_tiles<TX, TY, 64, 4>(a, cus, st);
  } else {
    if constexpr (sizeof(TX) == 2) launch_conv_tiles<TX, TY, 32, 8>(a, cus, st);
  }
  return hipGetLastError();
}
template hipError_t launch_conv<uint16_t, uint16_t>(const ConvArgs<uint16_t, uint16_t>&, hipStream_t);
template hipError_t launch_conv<float, float>(const ConvArgs<float, float>&, hipStream_t);

// Channel tiles (units of 32) of a layer's block, 4 / (co ci) row segments.
static void wgrad_shape(WgradLayer& L) {
  L.co = L.Cout % 64 == 0 ? 2 : 1;
  L.ci = L.Cin % 64 == 0 ? 2 : 1;
  const int rows = wgrad_rows(L.co, L.ci), tr = rows * 4 / (L.co * L.ci);
  L.nco = L.Cout / (32 * L.co);
  L.nci = (L.Cin + 32 * L.ci - 1) / (32 * L.ci);
  L.tiles_x = (L.W + 15) / 16;
  L.tiles_y = (L.H + tr - 1) / tr;
  L.tiles = L.N * L.tiles_x * L.tiles_y;
  // cost of a pixel tile: the rows' MFMAs, and the staging of the rows of 4 KB
  // of gradient and 2 KB of input per 64 channels
  L.cost = rows * 4 + (tr * L.co * 2 + (tr + 2) * L.ci) / 2;
}

// Splits of every layer's pixels: the smallest largest cost per block such that
// the blocks are resident at once.
int plan_wgrad(WgradGroup& g, int blocks) {
  long hi = 1;
  for (int l = 0; l < g.n; l++) {
    wgrad_shape(g.l[l]);
    hi = std::max(hi, (long)g.l[l].tiles * g.l[l].cost);
  }
  auto plan = [&](long T) {
    long total = 0;
    for (int l = 0; l < g.n; l++) {
      WgradLayer& L = g.l[l];
      L.per = (int)std::min<long>(L.tiles, std::max<long>(1, T / L.cost));
      L.splits = (L.tiles + L.per - 1) / L.per;
      L.first = (int)total;
      total += (long)L.nco * L.nci * L.splits;
    }
    return total;
  };
  long lo = 1;
  while (lo < hi) {
    const long mid = (lo + hi) / 2;
    if (plan(mid) <= blocks) hi = mid;
    else lo = mid + 1;
  }
  return (int)plan(lo);
}

long wgrad_part_floats(const WgradGroup& g) {
  long n = 0;
  for (int l = 0; l < g.n; l++) n += (long)g.l[l].splits * (9L * g.l[l].Cout * g.l[l].Cin + g.l[l].Cout);
  return n;
}

hipError_t launch_wgrad(WgradGroup& g, int blocks, float* part, ReduceGroup& r, hipStream_t st) {
  for (int l = 0; l < g.n; l++) {
    WgradLayer& L = g.l[l];
    // 16-byte accesses of 8 channels; 32-bit byte offsets within an image
    if (L.Cout % 32 || L.Cin % 8 || (L.Cin > 32 && L.Cin % 32) || L.ldx % 8 || L.cx0 % 8 || L.lddy % 4 || L.cdy0 % 4 ||
        (long)L.H * L.W * L.ldx * 2 >= (1L << 31) || (long)L.H * L.W * L.lddy * 4 >= (1L << 31))
      return hipErrorInvalidValue;
    L.part = part;
    part += (long)L.splits * 9 * L.Cout * L.Cin;
    L.bpart = part;
    part += (long)L.splits * L.Cout;
    add_reduce(r, L.part, L.splits, 9L * L.Cout * L.Cin, L.dw, true);
    add_reduce(r, L.bpart, L.splits, L.Cout, L.db, false);
  }
  hipLaunchKernelGGL(k_wgrad, dim3(blocks), dim3(256), 0, st, g);
  return hipGetLastError();
}

void add_reduce(ReduceGroup& r, const float* part, int nparts, long n, float* out, bool wide) {
  ReduceItem& t = r.t[r.n++];
  t = ReduceItem{part, out, n, nparts, r.blocks, wide ? 1 : 0};
  r.blocks += (int)(wide ? (n + 1023) / 1024 : (n + 3) / 4);
}

hipError_t launch_grad_reduce(const ReduceGroup& r, hipStream_t st) {
  if (!r.blocks) return hipSuccess;
  hipLaunchKernelGGL(k_grad_reduce, dim3(r.blocks), dim3(256), 0, st, r);
  return hipGetLastError();
}

hipError_t launch_up_fwd(const PoolArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(k_up_fwd, dim3(blocks_for((long)a.N * a.H * a.W * a.C / 2)), dim3(256), 0, st, a);
  return hipGetLastError();
}
hipError_t launch_head_fwd(const uint16_t* x, int ldx, const float* w, const float* b, int C, long P, float* out,
                           hipStream_t st) {
  hipLaunchKernelGGL(k_head_fwd, dim3(blocks_for(P)), dim3(256), 0, st, x, ldx, w, b, C, P, out);
  return hipGetLastError();
}
hipError_t launch_head_bwd(const uint16_t* x, int ldx, const float* w, long P, const float* dout, float* dx, int lddx,
                           float* part, hipStream_t st) {
  hipLaunchKernelGGL(k_head_bwd, dim3(kHeadGradParts), dim3(256), 0, st, x, ldx, w, P, dout, dx, lddx, part);
  return hipGetLastError();
}
hipError_t launch_flip_weights(const uint16_t* w, uint16_t* wt, int taps, int Cout, int Cin, hipStream_t st) {
  hipLaunchKernelGGL(k_flip_weights, dim3(blocks_for((long)taps * Cout * Cin)), dim3(256), 0, st, w, wt, taps,
                     Cout, Cin);
  return hipGetLastError();
}
hipError_t launch_adam(float* w, uint16_t* w16, const float* g, float* m, float* v, long n, float lr, float b1,
                       float b2, float eps, float c1, float c2, float gscale, hipStream_t st) {
  hipLaunchKernelGGL(k_adam, dim3(blocks_for(n)), dim3(256), 0, st, w, w16, g, m, v, n, lr, b1, b2, eps, c1, c2,
                     gscale);
  return hipGetLastError();
}
hipError_t launch_f32_to_bf16(const float* in, uint16_t* out, long n, int ldo, int co0, int C, hipStream_t st) {
  hipLaunchKernelGGL(k_f32_to_bf16, dim3(blocks_for(n)), dim3(256), 0, st, in, out, n, ldo, co0, C);
  return hipGetLastError();
}
hipError_t launch_mse(const float* pred, const float* target, long P, float* dpred, double* loss, float scale,
                      hipStream_t st) {
  hipLaunchKernelGGL(k_mse, dim3(blocks_for(P, 1024)), dim3(256), 0, st, pred, target, P, dpred, loss, scale);
  return hipGetLastError();
}
hipError_t launch_image_rms(const float* in, long P, int B, double* part, float* scale, hipStream_t st) {
  hipLaunchKernelGGL(k_image_rms_part, dim3(kRmsParts, B), dim3(256), 0, st, in, P, part);
  hipLaunchKernelGGL(k_image_rms_final, dim3((B + 63) / 64), dim3(64), 0, st, part, P, B, scale);
  return hipGetLastError();
}
int image_rms_parts() { return kRmsParts; }
hipError_t launch_to_bf16_scaled(const float* in, const float* scale, long P, int B, uint16_t* out, hipStream_t st) {
  hipLaunchKernelGGL(k_to_bf16_scaled, dim3(blocks_for(P * B)), dim3(256), 0, st, in, scale, P, P * B, out);
  return hipGetLastError();
}
hipError_t launch_residual_add(const float* m, const float* y, const float* scale, long P, int B, float gain,
                               float* out, hipStream_t st) {
  hipLaunchKernelGGL(k_residual_add, dim3(blocks_for(P * B)), dim3(256), 0, st, m, y, scale, P, P * B, gain, out);
  return hipGetLastError();
}

}  // namespace unet
