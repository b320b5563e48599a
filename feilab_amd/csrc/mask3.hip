// ICONMask3 (sourceCode/ICONMask3/ICONCrossVMaskIn2D_weightOnlyOnSampled.cu):
// combine the reconstructed slices midYYYYY.mrc into a volume, each slice
// filtered in 2D Fourier space by
//   realMask  1 inside the FRC-0.5 radius; outside, the angular sampling
//             mask (the union of the tilt lines), raised to a Gaussian edge
//             between the FRC-0.5 and FRC-0.3 radii;
//   weighting |k| / r_full on sampled frequencies beyond r_full (the radius
//             where neighbouring tilt lines stop overlapping), else 1;
// then cropped to the specimen thickness.
//
// The masks are built on the host exactly as the reference builds them
// (float/double placement included).  The filtering runs batched on the
// device with this library's own transforms: for a real slice f with spectrum
// F, the reference's R2C -> (half-spectrum mask M) -> C2R / N^2 equals
// Re(IFFT2(F * Mfull)) / N^2 with Mfull(ky, kx) = M(ky, kx) for kx <= N/2
// and M(-ky, N-kx) otherwise; for the columns kx = 0 and N/2, which are their
// own mirrors, the real part leaves the even part of M.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <strings.h>
#include <vector>

#include "../../include/icon_mi355x.h"
#include "icon_col.h"
#include "icon_fft.h"
#include "icon_plan.h"
#include "mrc_io.h"

using namespace icon;

namespace {

constexpr double kPi180 = 0.01745329252;   // PI_180 of the reference

thread_local std::string g_merr;

int merr(int code, const std::string& m) {
  g_merr = m;
  return code;
}

// The angular sampling mask (main, lines 958-1000): the central column of an
// N x N image rotated by -theta-90 degrees for every tilt with bilinear
// splatting, summed and clipped to 1.  Index j1*N + i1, centred at N/2.
void sampling_mask(int N, const float* thita, int ang_num, std::vector<float>& origmask) {
  const long nx = N, ny = N;
  std::vector<float> line(nx * ny, 0.f), rot(nx * ny);
  origmask.assign(nx * ny, 0.f);
  for (long j = 0; j < nx; j++) line[j * nx + nx / 2] = 1.f;
  for (int k = 0; k < ang_num; k++) {
    const float c = (float)std::cos((-thita[k] - 90) * kPi180);
    const float s = (float)std::sin((-thita[k] - 90) * kPi180);
    std::fill(rot.begin(), rot.end(), 0.f);
    for (long j = 0; j < ny; j++)
      for (long i = 0; i < nx; i++) {
        const float lv = line[j * nx + i];
        if (lv == 0.f) continue;
        const float xf = (float)(i - nx / 2) * c - (float)(j - ny / 2) * s + (float)(nx / 2);
        const float yf = (float)(i - nx / 2) * s + (float)(j - ny / 2) * c + (float)(ny / 2);
        const int xi = (int)xf, yi = (int)yf;
        const float dx = xf - xi, dy = yf - yi;
        if (xi >= 0 && xi < nx && yi >= 0 && yi < ny) rot[yi * nx + xi] += lv * (1 - dx) * (1 - dy);
        if (xi >= 0 && xi < nx && yi + 1 >= 0 && yi + 1 < ny) rot[(yi + 1) * nx + xi] += lv * (1 - dx) * dy;
        if (xi + 1 >= 0 && xi + 1 < nx && yi >= 0 && yi < ny) rot[yi * nx + xi + 1] += lv * dx * (1 - dy);
        if (xi + 1 >= 0 && xi + 1 < nx && yi + 1 >= 0 && yi + 1 < ny) rot[(yi + 1) * nx + xi + 1] += lv * dx * dy;
      }
    for (long i = 0; i < nx * ny; i++) origmask[i] += rot[i];
  }
  for (auto& v : origmask)
    if (v > 1) v = 1;
}

// ------------------------------------------------------------------ filtering
// Three passes over the stack, in place: a row pass (spectra of the real
// rows), a column pass (forward transform, mask, inverse transform) and a row
// pass back.  The spectrum of a real row of N samples is N floats: F_0, for even
// N F_{N/2}, and the pairs F_k, 0 < k < N/2, so it replaces the row in the stack
// and no other buffer is needed.  Two real rows of a slice share one complex
// transform (an odd slice's last row has one alone: rows of two slices in one
// would mix their rounding, and spread a NaN from one to the next).
//
// Lengths that are not powers of two (or below 128) use Bluestein's chirp-z
// transform on a power-of-two transform of length M >= 2N - 1.  With
// c_n = exp(-i pi n^2 / N),
//   X_k = c_k sum_n (x_n c_n) conj(c_{k-n}),
// a circular convolution of length M, inside registers and LDS; the inverse is
// the same with every factor conjugated (the kernel is even, so its spectrum's
// conjugate is the conjugate kernel's spectrum).
//
// Bound by the transforms' arithmetic (two of length M per row pair and four
// per column), not by memory (24 N^2 bytes per slice).  64 slices of 464^2 (M =
// 1024): rows 60 us, columns 160 us, rows back 72 us, 341 us for the call with
// the mask's upload and the device's 17 us copy of the input before it, against
// 4440 us as separate passes over a complex stack in a chirp's buffer of its
// own, the chirp's spectrum summed on the host and six allocations.

struct FiltArgs {
  float* data;            // [rows][N] in place
  const float* half;      // mask [N][N/2 + 1]
  const float2* chirp;    // c_n, n < N (chirp transforms)
  const float2* bhat;     // spectrum of the conj(c) kernel over M
  const float2* tw;       // twiddles of the length-M transform
  int N;
  long rows;              // N x slices
};

// Spectrum entry k (0 <= k <= N/2) of a packed row.
__device__ __forceinline__ float2 spec_get(const float* p, int k, int N) {
  if (k == 0) return make_float2(p[0], 0.f);
  if (2 * k == N) return make_float2(p[1], 0.f);
  const int o = N % 2 ? 2 * k - 1 : 2 * k;
  return make_float2(p[o], p[o + 1]);
}
__device__ __forceinline__ void spec_put(float* p, int k, int N, float2 v) {
  if (k == 0) { p[0] = v.x; return; }
  if (2 * k == N) { p[1] = v.x; return; }
  const int o = N % 2 ? 2 * k - 1 : 2 * k;
  p[o] = v.x;
  p[o + 1] = v.y;
}

__device__ __forceinline__ float2 conj_if(bool c, float2 a) { return c ? make_float2(a.x, -a.y) : a; }

// Transform of length N (direction DIR) of the line that a team of M/16 threads
// holds in v: in, slot r element t + r M/16 (for a chirp transform already
// times its chirp factor, and zero from N on); out, slot i element
// out_index<M>(t, i) (without the chirp factor of the output).
template <int M, typename L, int DIR, bool CHIRP>
__device__ __forceinline__ void line_fft(float2 (&v)[16], float2* lds, int t, const FiltArgs& a) {
  FftTwiddles T;
  if constexpr (!CHIRP) {
    fft_from_lazy<M, L, DIR, 1>(v, lds, t, T, a.tw);
  } else {
    fft_from_lazy<M, L, -1, 1>(v, lds, t, T, a.tw);
    constexpr int RL = last_radix<M>();
    float2 u[16];
#pragma unroll
    for (int i = 0; i < 16; i++)
      u[i / RL + (i % RL) * (16 / RL)] = c_mul(v[i], conj_if(DIR > 0, a.bhat[out_index<M>(t, i)]));
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = u[i];
    fft_from_lazy<M, L, 1, 1>(v, lds, t, T, a.tw);
  }
}

// Row pairs: INV 0, spectra of the two real rows; INV 1, the rows back, over N^2.
template <int M, int RPB, bool CHIRP, bool INV>
__global__ __launch_bounds__(RPB * (M / 16)) void k_filt_rows(FiltArgs a) {
  constexpr int T = M / 16;
  __shared__ float2 lds[RPB * RowLay::size(M)];
  const int team = threadIdx.x / T, t = threadIdx.x % T;
  const int N = a.N, pairs = (N + 1) / 2;   // row pairs of a slice
  const long p = (long)blockIdx.x * RPB + team, slice = p / pairs;
  const int y = 2 * (int)(p - slice * pairs);
  const long row = slice * N + y;
  float2* L = lds + team * RowLay::size(M);
  const bool v0 = row < a.rows, v1 = v0 && y + 1 < N;
  float *p0 = a.data + (v0 ? row : 0) * N, *p1 = a.data + (v1 ? row + 1 : 0) * N;
  float2 v[16];
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int n = in_index<M>(t, r);
    v[r] = make_float2(0.f, 0.f);
    if (n >= N) continue;
    if constexpr (!INV) {
      v[r] = make_float2(v0 ? p0[n] : 0.f, v1 ? p1[n] : 0.f);
    } else {
      // Z = A + iB of the rows' spectra; beyond N/2 their mirrors' conjugates
      const bool up = 2 * n > N;
      const int k = up ? N - n : n;
      const float2 A = v0 ? conj_if(up, spec_get(p0, k, N)) : make_float2(0.f, 0.f);
      const float2 B = v1 ? conj_if(up, spec_get(p1, k, N)) : make_float2(0.f, 0.f);
      v[r] = make_float2(A.x - B.y, A.y + B.x);
    }
    if constexpr (CHIRP) v[r] = c_mul(v[r], conj_if(INV, a.chirp[n]));
  }
  line_fft<M, RowLay, INV ? 1 : -1, CHIRP>(v, L, t, a);
  if constexpr (CHIRP) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int k = out_index<M>(t, i);
      if (k < N) v[i] = c_mul(v[i], conj_if(INV, a.chirp[k]));
    }
  }
  if constexpr (INV) {
    // (the last exchange's barrier was passed after every load of the rows)
    const double f = 1.0 / ((double)N * (double)N);
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int n = out_index<M>(t, i);
      if (n >= N) continue;
      if (v0) p0[n] = (float)((double)v[i].x * f);
      if (v1) p1[n] = (float)((double)v[i].y * f);
    }
  } else {
    // A_k = (Z_k + conj Z_{N-k})/2, B_k = (Z_k - conj Z_{N-k})/2i
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int k = out_index<M>(t, i);
      if (k < N) L[RowLay::at(k)] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int k = out_index<M>(t, i);
      if (2 * k > N) continue;
      const float2 z = v[i], y = L[RowLay::at(k ? N - k : 0)];
      if (v0) spec_put(p0, k, N, make_float2(0.5f * (z.x + y.x), 0.5f * (z.y - y.y)));
      if (v1) spec_put(p1, k, N, make_float2(0.5f * (z.y + y.y), 0.5f * (y.x - z.x)));
    }
  }
}

// Tiles of C spectrum columns of one slice: column transform, mask, inverse.
// Column 0 of an even width carries F_0 + i F_{N/2} (both columns are real
// before the transform), separated by the mirror k -> N - k.
template <int M, int C, bool CHIRP>
__global__ __launch_bounds__(C * (M / 16)) void k_filt_cols(FiltArgs a, int ntiles) {
  using Lo = ColFftLayFwd<C>;
  extern __shared__ __align__(16) float2 tile[];   // Lo::at(M - 1) + C
  const int N = a.N, H = N / 2 + 1, ncol = (N + 1) / 2;
  const int c = threadIdx.x % C, t = threadIdx.x / C;
  const int k0 = (blockIdx.x % ntiles) * C + c;      // spectrum column, 0: special
  const bool ok = k0 < ncol;
  float* base = a.data + (long)(blockIdx.x / ntiles) * N * N;
  const int o = k0 == 0 ? 0 : N % 2 ? 2 * k0 - 1 : 2 * k0;
  const bool two = k0 != 0 || N % 2 == 0;            // an odd width's column 0 is real
  float2 v[16];
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int n = in_index<M>(t, r);
    v[r] = make_float2(0.f, 0.f);
    if (ok && n < N) v[r] = make_float2(base[(long)n * N + o], two ? base[(long)n * N + o + 1] : 0.f);
    if constexpr (CHIRP)
      if (n < N) v[r] = c_mul(v[r], a.chirp[n]);
  }
  line_fft<M, Lo, -1, CHIRP>(v, tile + c, t, a);
  // the mask; the output's and the inverse's input's chirp factors cancel
  if (blockIdx.x % ntiles == 0 && N % 2 == 0) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int k = out_index<M>(t, i);
      if (k >= N) continue;
      if (CHIRP && c == 0) v[i] = c_mul(v[i], a.chirp[k]);
      tile[Lo::at(k) + c] = v[i];
    }
    __syncthreads();
    if (c == 0) {
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int k = out_index<M>(t, i), km = (N - k) % N;
        if (k >= N) continue;
        // the real part keeps the masks' even parts: Re over columns 0 and N/2
        const float m0 = 0.5f * (a.half[(long)k * H] + a.half[(long)km * H]);
        const float mn = 0.5f * (a.half[(long)k * H + N / 2] + a.half[(long)km * H + N / 2]);
        const float s = 0.5f * (m0 + mn), d = 0.5f * (m0 - mn);
        const float2 z = v[i], y = tile[Lo::at(km)];
        v[i] = make_float2(s * z.x + d * y.x, s * z.y - d * y.y);
        if (CHIRP) v[i] = c_mul(v[i], conj_if(true, a.chirp[k]));
      }
    }
    __syncthreads();
  } else if (k0 == 0) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int k = out_index<M>(t, i);
      if (k >= N) continue;
      const float m = 0.5f * (a.half[(long)k * H] + a.half[(long)((N - k) % N) * H]);
      v[i] = make_float2(v[i].x * m, v[i].y * m);
    }
  }
  constexpr int RL = last_radix<M>();
  float2 u[16];
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int k = out_index<M>(t, i);
    const float m = k0 == 0 || !ok || k >= N ? 1.f : a.half[(long)k * H + k0];
    u[i / RL + (i % RL) * (16 / RL)] = k < N ? make_float2(v[i].x * m, v[i].y * m) : make_float2(0.f, 0.f);
  }
  line_fft<M, Lo, 1, CHIRP>(u, tile + c, t, a);
  if (!ok) return;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int n = out_index<M>(t, i);
    if (n >= N) continue;
    float2 x = u[i];
    if constexpr (CHIRP) x = c_mul(x, conj_if(true, a.chirp[n]));
    base[(long)n * N + o] = x.x;
    if (two) base[(long)n * N + o + 1] = x.y;
  }
}

// Chirp and its kernel's spectrum, in FP64 with exact phases: block k sums
// bhat_k = (1 + 2 sum_{0<j<N} exp(i pi j^2 / N) cos(2 pi j k / M)) / M (the 1/M
// of the inverse transform folded in).
__global__ __launch_bounds__(64) void k_chirp(int N, int M, float2* chirp, float2* bhat) {
  const int k = blockIdx.x, t = threadIdx.x;
  double x = 0.0, y = 0.0;
  for (int j = 1 + t; j < N; j += 64) {
    const double ph = (double)(((long)j * j) % (2L * N)) / (double)N;
    const double f = 2.0 * cospi(2.0 * (double)(((long)j * k) % M) / (double)M);
    x += f * cospi(ph);
    y += f * sinpi(ph);
  }
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) {
    x += __shfl_down(x, h);
    y += __shfl_down(y, h);
  }
  if (t == 0) {
    bhat[k] = make_float2((float)((1.0 + x) / M), (float)(y / M));
    if (k < N) {
      const double ph = (double)(((long)k * k) % (2L * N)) / (double)N;
      chirp[k] = make_float2((float)cospi(ph), (float)-sinpi(ph));
    }
  }
}

template <int M, bool CHIRP>
hipError_t launch_filter(const FiltArgs& a, int count, hipStream_t st) {
  // columns per tile: 8 (64 bytes of each row); 4 at M = 2048, whose 8 would
  // need 1024 threads, and so 128 registers each and scratch memory
  constexpr int RPB = 256 / (M / 16) > 16 ? 16 : 256 / (M / 16), C = M >= 2048 ? 4 : 8;
  constexpr int lds = (ColFftLayFwd<C>::at(M - 1) + C) * (int)sizeof(float2);
  const hipError_t e = hipFuncSetAttribute((const void*)k_filt_cols<M, C, CHIRP>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  const long pairs = (long)count * ((a.N + 1) / 2);
  const unsigned blocks = (unsigned)((pairs + RPB - 1) / RPB);
  const int ntiles = ((a.N + 1) / 2 + C - 1) / C;
  hipLaunchKernelGGL((k_filt_rows<M, RPB, CHIRP, false>), dim3(blocks), dim3(RPB * (M / 16)), 0, st, a);
  hipLaunchKernelGGL((k_filt_cols<M, C, CHIRP>), dim3((unsigned)ntiles * count), dim3(C * (M / 16)), lds, st, a, ntiles);
  hipLaunchKernelGGL((k_filt_rows<M, RPB, CHIRP, true>), dim3(blocks), dim3(RPB * (M / 16)), 0, st, a);
  return hipGetLastError();
}

}  // namespace

extern "C" {

const char* icon_mask3_error(void) { return g_merr.c_str(); }

int icon_mask3_weights(int N, const float* tilt_deg, int ang_num, float radius05_rate, float radius03_rate,
                       int radius_given, int gauss_width, float mean_ang_step, float* half_mask) {
  if (N < 2 || !tilt_deg || ang_num < 1 || !half_mask) return merr(ICON_ERR_ARG, "icon_mask3_weights: bad argument");
  std::vector<float> origmask;
  sampling_mask(N, tilt_deg, ang_num, origmask);
  // genMask (lines 369-455)
  const int r_full = (int)std::ceil(2.0 / (mean_ang_step / 360.0 * 2 * 3.1415926));
  const int radius05 = (int)((float)N / 2.0 * radius05_rate);
  const int radius03 = (int)((float)N / 2.0 * radius03_rate);
  const int nx = N, ny = N;
  long gaussianlenMax;
  const int radius = radius05;
  if (!radius_given)
    gaussianlenMax = gauss_width >= 0 ? gauss_width : radius03 - radius05;
  else
    gaussianlenMax = gauss_width >= 0 ? gauss_width : (long)(10.0 * (N / 150.0));
  if (gaussianlenMax < 10.0 * (N / 150.0)) gaussianlenMax = (long)(10.0 * (N / 150.0));
  const long gaussianradius = radius + gaussianlenMax;
  const long gaussianlen = gaussianradius - radius;
  const double c = (double)gaussianlen / 3.0;
  const double e_end = std::exp(-(double)(gaussianlen * gaussianlen) / (2 * c * c));
  for (int j = 0; j < ny; j++)
    for (int i = 0; i < nx / 2 + 1; i++) {
      const int i1 = (i + nx / 2) % nx, j1 = (j + ny / 2) % ny;
      const long rr = (long)std::sqrt((double)((i1 - nx / 2) * (i1 - nx / 2) + (j1 - ny / 2) * (j1 - ny / 2)));
      const float om = origmask[(size_t)j1 * nx + i1];
      float real;
      if (rr >= radius) {
        if (rr <= gaussianradius) {
          double w = om;
          const double xxx = (double)(rr - radius);
          const double w2 = (std::exp(-(xxx * xxx) / (2 * c * c)) - e_end) / (1 - e_end);
          w = w > w2 ? w : w2;
          real = (float)w;
        } else {
          real = om;
        }
      } else {
        real = 1.f;
      }
      const float weighting = (rr > r_full && std::fabs(om) > 0.00001) ? (float)rr / (float)r_full : 1.f;
      half_mask[(size_t)j * (nx / 2 + 1) + i] = real * weighting;
    }
  return ICON_OK;
}

int icon_mask3_filter(int device, float* d_slices, int N, int count, const float* half_mask, void* stream) {
  if (!d_slices || !half_mask || count < 1 || N < 8 || N > 2048)
    return merr(ICON_ERR_ARG, "icon_mask3_filter: slices must be N x N with N in 8..2048");
  const bool pow2 = N >= 128 && (N & (N - 1)) == 0;
  if (!pow2 && N > 1024)
    return merr(ICON_ERR_ARG, "icon_mask3_filter: widths above 1024 must be powers of two");
  if (hipSetDevice(device) != hipSuccess) return merr(ICON_ERR_ARG, "icon_mask3_filter: no such device");
  hipStream_t st = (hipStream_t)stream;
  int M = 128;
  while (pow2 ? M < N : M < 2 * N - 1) M *= 2;
  const float2* tw = nullptr;
  if (int rc = fft_twiddles(M, &tw)) return merr(rc, std::string("icon_mask3_filter: ") + icon_last_error());
  // one buffer: the mask and, for a chirp transform, its tables
  const size_t hb = (sizeof(float) * (size_t)N * (N / 2 + 1) + 255) / 256 * 256;
  char* buf = nullptr;
  hipError_t e = hipMalloc(&buf, hb + (pow2 ? 0 : sizeof(float2) * (size_t)(M + N)));
  if (e == hipSuccess)
    e = hipMemcpy(buf, half_mask, sizeof(float) * (size_t)N * (N / 2 + 1), hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    float2 *bhat = reinterpret_cast<float2*>(buf + hb), *chirp = bhat + M;
    FiltArgs a{d_slices, reinterpret_cast<const float*>(buf), chirp, bhat, tw, N, (long)count * N};
    if (!pow2) {
      hipLaunchKernelGGL(k_chirp, dim3(M), dim3(64), 0, st, N, M, chirp, bhat);
      e = hipGetLastError();
    }
    if (e == hipSuccess) {
      switch (M) {
#define CASE(MM) \
  case MM: e = pow2 ? launch_filter<MM, false>(a, count, st) : launch_filter<MM, true>(a, count, st); break;
        CASE(128) CASE(256) CASE(512) CASE(1024) CASE(2048)
#undef CASE
        default: e = hipErrorInvalidValue;
      }
    }
  }
  const hipError_t es = hipStreamSynchronize(st);
  if (e == hipSuccess) e = es;
  if (buf) (void)hipFree(buf);
  if (e != hipSuccess) return merr(ICON_ERR_DEVICE, std::string("icon_mask3_filter: ") + hipGetErrorString(e));
  return ICON_OK;
}

int icon_mask3(int device, const char* input_dir, int slice_begin, int slice_end, int thickness,
               const char* tilt_path, const char* out_path, int radius, const char* crossv_frc,
               const char* fullrec_frc, int zshift, int gauss_width, int no_mask) {
  if (!input_dir || !tilt_path || !out_path || slice_end < slice_begin || thickness < 1)
    return merr(ICON_ERR_ARG, "parameter error! '-inputPath' or '-slice' or '-thickness' or '-tiltfile' or "
                              "'-output' are missed!");
  auto mid = [&](int z) {
    char b[4096];
    std::snprintf(b, sizeof b, "%s/mid%05d.mrc", input_dir, z);
    return std::string(b);
  };
  // geometry of the slices
  MrcHeader head;
  {
    FILE* fp = std::fopen(mid(slice_begin).c_str(), "rb");
    if (!fp || !mrc::read_header(fp, &head)) {
      if (fp) std::fclose(fp);
      return merr(ICON_ERR_IO, "Can not open infile " + mid(slice_begin) + "!");
    }
    std::fclose(fp);
  }
  const int Sx = head.nx, Sy = head.ny;
  const int ystart = Sy / 2 - thickness / 2 + zshift;
  if (ystart < 0 || ystart + thickness > Sy)
    return merr(ICON_ERR_ARG, "zshift & thickness make the size of volume out of limitation!");
  const int nslice = slice_end - slice_begin + 1;
  std::vector<float> out((size_t)nslice * thickness * Sx);
  std::vector<float> half;
  if (!no_mask) {
    if (Sx != Sy)
      return merr(ICON_ERR_ARG, "icon_mask3: the filtering needs square slices (thickness of the ICON run = width)");
    // tilt file (main, lines 803-822): numbers split by " ;,\n\r\t", up to "END"
    std::vector<float> thita;
    {
      FILE* fa = std::fopen(tilt_path, "r");
      if (!fa) return merr(ICON_ERR_IO, std::string("Cannot open file ") + tilt_path);
      char line[800];
      bool stop = false;
      while (!stop && std::fgets(line, sizeof line, fa)) {
        char* p = std::strtok(line, " ;,\n\r\t");
        if (!p || strncasecmp(p, "END", 3) == 0) break;
        while (p) {
          thita.push_back((float)std::atof(p));
          p = std::strtok(nullptr, " ;,\n\r\t");
        }
      }
      std::fclose(fa);
    }
    if (thita.size() < 2) return merr(ICON_ERR_ARG, "icon_mask3: the tilt file needs at least two angles");
    float biggest = -1, smallest = 1;
    for (float t : thita) {
      if (biggest < t) biggest = t;
      if (smallest > t) smallest = t;
    }
    const float big_step = biggest - smallest;
    const int big_step_radius = (int)std::ceil(2 * 180.0 / 3.1415926 / big_step);
    float mean_step = 0.f;
    for (size_t i = 0; i + 1 < thita.size(); i++) mean_step += std::fabs(thita[i + 1] - thita[i]);
    mean_step /= (float)(thita.size() - 1);
    // radii from the FRC files (lines 866-940)
    bool radius_given = radius > 0;
    float r05 = 0.f, r03 = 0.f;
    if (!radius_given) {
      auto read_frc = [](const char* path, std::vector<float>& v) {
        FILE* f = path ? std::fopen(path, "r") : nullptr;
        if (!f) return false;
        float a, b;
        while (std::fscanf(f, "%f %f", &a, &b) == 2) v.push_back(b);
        std::fclose(f);
        return true;
      };
      std::vector<float> cv, fr;
      if (!read_frc(crossv_frc, cv)) return merr(ICON_ERR_IO, std::string("Cannot open file '") + (crossv_frc ? crossv_frc : "") + "'");
      bool valid = (int)cv.size() >= Sx / 2 - 1;
      if (valid) {
        if (!read_frc(fullrec_frc, fr)) return merr(ICON_ERR_IO, std::string("Cannot open file '") + (fullrec_frc ? fullrec_frc : "") + "'");
        valid = (int)fr.size() >= Sx / 2 - 1;
      }
      if (valid) {
        const int sz = (int)fr.size();
        for (int i = 0; i < sz && i < (int)cv.size(); i++)
          if (fr[i] != 0) cv[i] /= fr[i];
        auto last_at_least = [&](float th) {
          int i = sz - 1;
          for (; i >= 0; i--)
            if (cv[i] >= th) break;
          return i;
        };
        const int radius05 = last_at_least(0.5f), radius03 = last_at_least(0.3f);
        std::printf("the calculated radius of frc0.5 is %d\nthe calculated radius of frc0.3 is %d\n", radius05, radius03);
        if (radius05 > radius03 || radius03 == 0) {
          valid = false;
        } else {
          r05 = (float)radius05 / (float)sz;
          r03 = (float)radius03 / (float)sz;
        }
      }
      if (!valid) {
        std::printf("the FRC files are not valid\nAssign radius : %d\n", big_step_radius);
        radius_given = true;
        radius = big_step_radius;
      }
    }
    if (radius_given) {
      r05 = (float)((float)radius / ((float)Sx / 2.0));
      r03 = 0.f;
    }
    half.resize((size_t)Sx * (Sx / 2 + 1));
    int rc = icon_mask3_weights(Sx, thita.data(), (int)thita.size(), r05, r03, radius_given ? 1 : 0, gauss_width,
                                mean_step, half.data());
    if (rc) return rc;
  }
  // slices in batches of up to 64 on the device
  const int B = 64;
  std::vector<float> buf((size_t)B * Sx * Sy);
  float* d = nullptr;
  if (!no_mask && (hipSetDevice(device) != hipSuccess || hipMalloc(&d, sizeof(float) * buf.size()) != hipSuccess))
    return merr(ICON_ERR_DEVICE, "icon_mask3: device allocation failed");
  int rc = ICON_OK;
  std::string err;
  for (int z0 = 0; z0 < nslice && rc == ICON_OK; z0 += B) {
    const int cnt = std::min(B, nslice - z0);
    for (int q = 0; q < cnt && rc == ICON_OK; q++) {
      FILE* fp = std::fopen(mid(slice_begin + z0 + q).c_str(), "rb");
      MrcHeader h;
      if (!fp || !mrc::read_header(fp, &h) || h.nx != Sx || h.ny != Sy ||
          !mrc::read_z_section(fp, h, 0, buf.data() + (size_t)q * Sx * Sy, &err))
        rc = merr(ICON_ERR_IO, "Can not open infile " + mid(slice_begin + z0 + q) + "!");
      if (fp) std::fclose(fp);
    }
    if (rc) break;
    if (!no_mask) {
      if (hipMemcpy(d, buf.data(), sizeof(float) * cnt * Sx * Sy, hipMemcpyHostToDevice) != hipSuccess) {
        rc = merr(ICON_ERR_DEVICE, "icon_mask3: upload failed");
        break;
      }
      if ((rc = icon_mask3_filter(device, d, Sx, cnt, half.data(), nullptr))) break;
      if (hipMemcpy(buf.data(), d, sizeof(float) * cnt * Sx * Sy, hipMemcpyDeviceToHost) != hipSuccess) {
        rc = merr(ICON_ERR_DEVICE, "icon_mask3: download failed");
        break;
      }
    }
    for (int q = 0; q < cnt; q++)
      std::memcpy(&out[(size_t)(z0 + q) * thickness * Sx], &buf[((size_t)q * Sy + ystart) * Sx],
                  sizeof(float) * thickness * Sx);
  }
  if (d) (void)hipFree(d);
  if (rc) return rc;
  // header of the first slice with nx, ny = thickness, nz = slices, float
  if (!mrc::write_float(out_path, head, out.data(), Sx, thickness, nslice, &err)) return merr(ICON_ERR_IO, err);
  return ICON_OK;
}

}  // extern "C"
