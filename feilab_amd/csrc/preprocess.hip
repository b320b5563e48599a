// Tilt-series pre-processing on the device (ICONPreProcess,
// sourceCode/ICONPreProcess/ICONPreProcess.c:31-86,256-302): per projection
// image, subtract the histogram mode of its central region and, given the
// tilt angles and the specimen thickness, scale it to variance
// 0.33 thickness / cos(theta).  This fixes the input scale that ICON's
// threshold (-thr) assumes.
//
// Three passes over the stack, each image shared by several blocks so that a
// short stack fills the device too: min / max of the central region and the
// sum; the histogram (LDS, then integer atomics) and the squared deviations;
// the pointwise update.  Bound by memory: four passes over the images, three
// reading and one writing.  61 images of 928 x 960 (217 MB): 46 + 95 + 101 us
// (4.7 TB/s read; the histogram bound by its FP64 divisions; the update moves
// 4.3 TB/s), against 1944 us in one block of 1024 threads per image, which left
// three quarters of the CUs idle.  Partial sums are added in a fixed order, in
// FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/icon_mi355x.h"
#include "mrc_io.h"

namespace {

constexpr int kThreads = 256;
constexpr int kBins = 256;
constexpr int kUnroll = 8;   // independent loads per thread
constexpr int kMaxBlocks = 64;

// Blocks per image: enough for ~2048 in all (8 per CU), at least 2048 pixels each.
int blocks_per_image(int nz, long size) {
  const long want = (2048 + nz - 1) / nz, most = (size + 2047) / 2048;
  return (int)std::max(1L, std::min({want, most, (long)kMaxBlocks}));
}

// Device scratch of a call over nz images in nb blocks each.
struct PreScratch {
  double* sum;    // [nz][nb]
  double* dev;    // [nz][nb] squared deviations
  float2* range;  // [nz][nb] central min, max
  int* hist;      // [nz][kBins]
  double* modes;  // [nz]
  float* tilt;    // [nz]
};

struct PreArgs {
  float* stack;
  int nx, ny, nb, thickness;
  PreScratch w;
  const float* tilt;   // null: mode subtraction only
};

size_t scratch_bytes(long nz, long blocks) { return blocks * (8 + 8 + 8) + nz * (4L * kBins + 8 + 4); }

PreScratch carve(unsigned char* p, long nz, long blocks) {
  PreScratch w;
  w.sum = reinterpret_cast<double*>(p); p += 8 * blocks;
  w.dev = reinterpret_cast<double*>(p); p += 8 * blocks;
  w.range = reinterpret_cast<float2*>(p); p += 8 * blocks;
  w.modes = reinterpret_cast<double*>(p); p += 8 * nz;
  w.hist = reinterpret_cast<int*>(p); p += 4L * kBins * nz;
  w.tilt = reinterpret_cast<float*>(p);
  return w;
}

// Sum over the block in a fixed order.
__device__ __forceinline__ double block_sum(double v, double* red) {
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) v += __shfl_down(v, h);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < kThreads / 64; w++) s += red[w];
  return s;
}

__device__ __forceinline__ float2 min_max(float2 a, float2 b) {
  return make_float2(b.x < a.x ? b.x : a.x, b.y > a.y ? b.y : a.y);
}

// Calls f(value, central) for the pixels of block blk of the image's nb: pixels
// blk * kThreads + threadIdx.x + k nb * kThreads, kUnroll loads in flight at a time, the row and column carried along instead of divided out.
template <typename F>
__device__ __forceinline__ void for_pixels(const float* in, int nx, int ny, int blk, int nb, F f) {
  const int xe = (int)(nx * 0.1), ye = (int)(ny * 0.1);
  const long size = (long)nx * ny, step = (long)nb * kThreads;
  long i = (long)blk * kThreads + threadIdx.x;
  int y = (int)(i / nx), x = (int)(i % nx);
  const int sy = (int)(step / nx), sx = (int)(step % nx);
  for (; i < size; i += kUnroll * step) {
    float v[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; u++) v[u] = i + u * step < size ? in[i + u * step] : 0.f;
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      if (i + u * step < size) f(v[u], x >= xe && x < nx - xe && y >= ye && y < ny - ye);
      x += sx;
      y += sy;
      if (x >= nx) { x -= nx; y++; }
    }
  }
}

// Per block: the sum, and min / max of the central region (starting, as the
// reference, from its first pixel); clears the image's histogram.
__global__ __launch_bounds__(kThreads) void k_pre_stats(PreArgs a) {
  __shared__ double red[kThreads / 64];
  __shared__ float2 rr[kThreads / 64];
  const int k = blockIdx.x / a.nb, blk = blockIdx.x % a.nb;
  const float* in = a.stack + (size_t)k * a.nx * a.ny;
  const float first = in[(size_t)(int)(a.ny * 0.1) * a.nx + (int)(a.nx * 0.1)];
  float2 r = make_float2(first, first);
  double s = 0.0;
  for_pixels(in, a.nx, a.ny, blk, a.nb, [&](float v, bool central) {
    s += (double)v;
    if (central) r = min_max(r, make_float2(v, v));
  });
  s = block_sum(s, red);
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) r = min_max(r, make_float2(__shfl_down(r.x, h), __shfl_down(r.y, h)));
  if ((threadIdx.x & 63) == 0) rr[threadIdx.x >> 6] = r;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < kThreads / 64; w++) r = min_max(r, rr[w]);
    a.w.sum[(size_t)k * a.nb + blk] = s;
    a.w.range[(size_t)k * a.nb + blk] = r;
  }
  if (blk == 0) a.w.hist[(size_t)k * kBins + threadIdx.x] = 0;
}

// The image's central min and the histogram's bin width, from the blocks' ranges.
__device__ __forceinline__ void bin_range(const PreArgs& a, int k, double* mn, double* step) {
  float2 r = a.w.range[(size_t)k * a.nb];
  for (int b = 1; b < a.nb; b++) r = min_max(r, a.w.range[(size_t)k * a.nb + b]);
  *mn = (double)r.x;
  *step = ((double)r.y - (double)r.x) / (double)kBins;
}

__global__ __launch_bounds__(kThreads) void k_pre_hist(PreArgs a) {
  __shared__ double red[kThreads / 64];
  __shared__ int hist[kThreads / 64][kBins];   // per wavefront
  const int k = blockIdx.x / a.nb, blk = blockIdx.x % a.nb;
  const float* in = a.stack + (size_t)k * a.nx * a.ny;
  double mn, step;
  bin_range(a, k, &mn, &step);
  double sum = 0.0;
  for (int b = 0; b < a.nb; b++) sum += a.w.sum[(size_t)k * a.nb + b];
  const double mean = sum / (double)((long)a.nx * a.ny);
#pragma unroll
  for (int w = 0; w < kThreads / 64; w++) hist[w][threadIdx.x] = 0;
  __syncthreads();
  int* mine = hist[threadIdx.x >> 6];
  const bool bins = step > 0;
  double v2 = 0.0;
  for_pixels(in, a.nx, a.ny, blk, a.nb, [&](float v, bool central) {
    const double d = (double)v - mean;
    v2 += d * d;
    if (bins && central) {
      const int b = (int)floor(((double)v - mn) / step);
      if (b >= 0 && b < kBins) atomicAdd(&mine[b], 1);   // the maximum (b == 256) is not counted
    }
  });
  v2 = block_sum(v2, red);
  if (threadIdx.x == 0) a.w.dev[(size_t)k * a.nb + blk] = v2;
  __syncthreads();
  int n = 0;
#pragma unroll
  for (int w = 0; w < kThreads / 64; w++) n += hist[w][threadIdx.x];
  if (n) atomicAdd(&a.w.hist[(size_t)k * kBins + threadIdx.x], n);
}

// in <- (float)(in - mode), and with tilts scaled to the variance that the
// thickness asks for.
__global__ __launch_bounds__(kThreads) void k_pre_scale(PreArgs a) {
  __shared__ long best[kThreads / 64];
  const int k = blockIdx.x / a.nb, blk = blockIdx.x % a.nb;
  float* in = a.stack + (size_t)k * a.nx * a.ny;
  double mn, step;
  bin_range(a, k, &mn, &step);
  // first bin of the largest count
  long key = ((long)a.w.hist[(size_t)k * kBins + threadIdx.x] << 32) | (kBins - 1 - (int)threadIdx.x);
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) {
    const long o = __shfl_down(key, h);
    key = o > key ? o : key;
  }
  if ((threadIdx.x & 63) == 0) best[threadIdx.x >> 6] = key;
  __syncthreads();
  key = best[0];
#pragma unroll
  for (int w = 1; w < kThreads / 64; w++) key = best[w] > key ? best[w] : key;
  const int bi = kBins - 1 - (int)(key & 0xffffffff);
  double mode = mn;
  if (step > 0) mode = bi * step + mn;
  if (blk == 0 && threadIdx.x == 0) a.w.modes[k] = mode;
  const long size = (long)a.nx * a.ny, stride = (long)a.nb * kThreads;
  double f = 1.0;
  if (a.tilt) {
    double v2 = 0.0;
    for (int b = 0; b < a.nb; b++) v2 += a.w.dev[(size_t)k * a.nb + b];
    const double var = v2 / (double)size;
    const double angle = -(double)a.tilt[k];
    const double factor = 0.33 * a.thickness / cos(angle / 180.0 * 3.1415926);
    f = sqrt(factor) / sqrt(var);
  }
  for (long i = (long)blk * kThreads + threadIdx.x; i < size; i += kUnroll * stride) {
    float v[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; u++) v[u] = i + u * stride < size ? in[i + u * stride] : 0.f;
#pragma unroll
    for (int u = 0; u < kUnroll; u++)
      if (i + u * stride < size) {
        const float d = (float)((double)v[u] - mode);
        in[i + u * stride] = a.tilt ? (float)((double)d * f) : d;
      }
  }
}

hipError_t run_passes(const PreArgs& a, int nz, hipStream_t st) {
  static_assert(kThreads == kBins, "one bin per thread");
  const dim3 grid((unsigned)((long)a.nb * nz));
  hipLaunchKernelGGL(k_pre_stats, grid, dim3(kThreads), 0, st, a);
  hipLaunchKernelGGL(k_pre_hist, grid, dim3(kThreads), 0, st, a);
  hipLaunchKernelGGL(k_pre_scale, grid, dim3(kThreads), 0, st, a);
  return hipGetLastError();
}

thread_local std::string g_perr;

int perr(int code, const std::string& m) {
  g_perr = m;
  return code;
}

// Device memory of icon_preprocess_noalloc, in place of the buffer that
// icon_preprocess allocates per call.  Each device holds its own copy until the
// process ends.  nz images take nz ceil(2048 / nz) < 2048 + nz blocks at most.
constexpr long kNoAllocMaxImages = 4096;
constexpr long kNoAllocMaxBlocks = 2048 + kNoAllocMaxImages;
constexpr size_t kScratchBytes = kNoAllocMaxBlocks * (8 + 8 + 8) + kNoAllocMaxImages * (4L * kBins + 8 + 4);

}  // namespace

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

// `scratch` of each device: its address, resolved once with that device current
// (the array's name in host code is only a stand-in), and a lock held by the
// call that uses it until its last kernel has ended, so that calls that overlap
// on one device take turns.
struct DeviceScratch {
  unsigned char* p = nullptr;
  std::mutex busy;
};
std::mutex g_scratch_mu;
std::map<int, DeviceScratch> g_scratch;

hipError_t scratch_on_current_device(DeviceScratch** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  DeviceScratch& d = g_scratch[dev];
  if (!d.p) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    d.p = static_cast<unsigned char*>(p);
  }
  *out = &d;
  return hipSuccess;
}

}  // namespace

extern "C" {

const char* icon_preprocess_error(void) { return g_perr.c_str(); }

int icon_preprocess(int device, float* d_stack, int nx, int ny, int nz, const float* tilt_deg, int thickness,
                    double* modes, void* stream) {
  if (!d_stack || nx < 1 || ny < 1 || nz < 1) return perr(ICON_ERR_ARG, "icon_preprocess: bad argument");
  if (hipSetDevice(device) != hipSuccess) return perr(ICON_ERR_ARG, "icon_preprocess: no such device");
  hipStream_t st = (hipStream_t)stream;
  const bool norm = tilt_deg && thickness > 0;
  PreArgs a{};
  a.stack = d_stack; a.nx = nx; a.ny = ny; a.thickness = thickness;
  a.nb = blocks_per_image(nz, (long)nx * ny);
  unsigned char* buf = nullptr;
  hipError_t e = hipMalloc(&buf, scratch_bytes(nz, (long)nz * a.nb));
  if (e == hipSuccess) {
    a.w = carve(buf, nz, (long)nz * a.nb);
    if (norm) {
      a.tilt = a.w.tilt;
      e = hipMemcpy(a.w.tilt, tilt_deg, sizeof(float) * nz, hipMemcpyHostToDevice);
    }
  }
  if (e == hipSuccess) e = run_passes(a, nz, st);
  if (e == hipSuccess && modes) e = hipMemcpyAsync(modes, a.w.modes, sizeof(double) * nz, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (buf) (void)hipFree(buf);
  if (e != hipSuccess) return perr(ICON_ERR_DEVICE, std::string("icon_preprocess: ") + hipGetErrorString(e));
  return ICON_OK;
}

int icon_preprocess_noalloc(int device, float* d_stack, int nx, int ny, int nz, const float* tilt_deg, int thickness,
                            double* modes, void* stream) {
  if (!d_stack || nx < 1 || ny < 1 || nz < 1) return perr(ICON_ERR_ARG, "icon_preprocess_noalloc: bad argument");
  if (nz > kNoAllocMaxImages)
    return perr(ICON_ERR_CAPACITY, "icon_preprocess_noalloc: " + std::to_string(nz) + " images exceed the " +
                                       std::to_string(kNoAllocMaxImages) + " its device scratch holds per call");
  if (hipSetDevice(device) != hipSuccess) return perr(ICON_ERR_ARG, "icon_preprocess_noalloc: no such device");
  DeviceScratch* d = nullptr;
  hipError_t e = scratch_on_current_device(&d);
  if (e != hipSuccess)
    return perr(ICON_ERR_DEVICE, std::string("icon_preprocess_noalloc: hipGetSymbolAddress: ") + hipGetErrorString(e));
  std::lock_guard<std::mutex> busy(d->busy);
  hipStream_t st = (hipStream_t)stream;
  const bool norm = tilt_deg && thickness > 0;
  // every call writes what it reads of the scratch, so nothing left in it by
  // an earlier call is read
  PreArgs a{};
  a.stack = d_stack; a.nx = nx; a.ny = ny; a.thickness = thickness;
  a.nb = blocks_per_image(nz, (long)nx * ny);
  a.w = carve(d->p, nz, (long)nz * a.nb);
  if (norm) {
    a.tilt = a.w.tilt;
    e = hipMemcpyAsync(a.w.tilt, tilt_deg, sizeof(float) * nz, hipMemcpyHostToDevice, st);
  }
  if (e == hipSuccess) e = run_passes(a, nz, st);
  if (e == hipSuccess && modes) e = hipMemcpyAsync(modes, a.w.modes, sizeof(double) * nz, hipMemcpyDeviceToHost, st);
  const hipError_t es = hipStreamSynchronize(st);   // (also after an error: nothing uses the scratch past the lock)
  if (e == hipSuccess) e = es;
  if (e != hipSuccess) return perr(ICON_ERR_DEVICE, std::string("icon_preprocess_noalloc: ") + hipGetErrorString(e));
  return ICON_OK;
}

int icon_preprocess_file(int device, const char* in_path, const char* out_path, const char* tilt_path,
                         int thickness) {
  if (!in_path || !out_path) return perr(ICON_ERR_ARG, "icon_preprocess_file: input or output missing");
  FILE* fp = std::fopen(in_path, "rb");
  if (!fp) return perr(ICON_ERR_IO, std::string("Cannot open file '") + in_path + "'");
  MrcHeader h;
  std::string err;
  if (!mrc::read_header(fp, &h)) {
    std::fclose(fp);
    return perr(ICON_ERR_IO, "cannot read the MRC header");
  }
  const size_t sec = (size_t)h.nx * h.ny;
  std::vector<float> stack(sec * h.nz);
  for (int k = 0; k < h.nz; k++)
    if (!mrc::read_z_section(fp, h, k, stack.data() + k * sec, &err)) {
      std::fclose(fp);
      return perr(ICON_ERR_IO, err);
    }
  std::fclose(fp);
  std::vector<float> tilts;
  if (tilt_path && thickness > 0) {
    tilts.assign(1000, 0.f);
    int n = 0;
    if (icon_read_tilts(tilt_path, tilts.data(), (int)tilts.size(), &n) != ICON_OK)
      return perr(ICON_ERR_IO, std::string("Cannot open file '") + tilt_path + "'");
    if (n < h.nz) return perr(ICON_ERR_ARG, "tilt file has fewer angles than the stack has sections");
  }
  float* d = nullptr;
  if (hipSetDevice(device) != hipSuccess || hipMalloc(&d, sizeof(float) * stack.size()) != hipSuccess)
    return perr(ICON_ERR_DEVICE, "icon_preprocess_file: device allocation failed");
  int rc = ICON_OK;
  if (hipMemcpy(d, stack.data(), sizeof(float) * stack.size(), hipMemcpyHostToDevice) != hipSuccess) {
    rc = perr(ICON_ERR_DEVICE, "icon_preprocess_file: upload failed");
  } else {
    rc = icon_preprocess(device, d, h.nx, h.ny, h.nz, tilts.empty() ? nullptr : tilts.data(), thickness, nullptr,
                         nullptr);
    if (rc == ICON_OK && hipMemcpy(stack.data(), d, sizeof(float) * stack.size(), hipMemcpyDeviceToHost) != hipSuccess)
      rc = perr(ICON_ERR_DEVICE, "icon_preprocess_file: download failed");
  }
  (void)hipFree(d);
  if (rc) return rc;
  // header copied from the input, mode float, statistics recomputed
  if (!mrc::write_float(out_path, h, stack.data(), h.nx, h.ny, h.nz, &err)) return perr(ICON_ERR_IO, err);
  return ICON_OK;
}

}  // extern "C"
