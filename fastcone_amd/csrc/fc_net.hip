// The network's element-wise kernels between its convolutions (gfx950): 2x2x2 average pooling,
// nearest upsampling with channel concatenation, their gradients, and the ReLU mask with the bias
// gradient. Activations are N x D x H x W x C, BF16; arithmetic is FP32, rounded once per stored
// value, in the order of the operations they stand for.
//
// All are bound by memory: a thread moves 16 bytes (8 channels of a voxel) per access, every tensor
// is read or written once, and one launch takes the place of a chain of element-wise operations
// that stored FP32 or strided copies in between. At 256^3 (inference) the pooling takes 0.12 ms; the
// concatenation at full size would take 0.44 ms (1.6 GB written, 0.8 GB read), so it is formed only
// for planes of 2^31 elements and more, and the convolutions load its parts elsewhere. At 4 x 128^3
// (training) the mask with the bias gradient takes 0.14 ms a layer (0.8 GB) and all steps 1.3 instead
// of 6.6 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "fc_device.h"
#include "fc_internal.h"

namespace fc {
namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// The two channels of word q of a 16-byte unit as FP32.
__device__ __forceinline__ float lo_bf16(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi_bf16(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// Sum over the 2 x 2 x 2 voxels of a coarse voxel, FP32: units p + dz sz + dy sy + dx sx.
__device__ __forceinline__ void sum8(const u32x4* p, size_t sx, size_t sy, size_t sz, float s[8]) {
#pragma unroll
  for (int q = 0; q < 8; ++q) s[q] = 0.0f;
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const u32x4 v = p[(d >> 2) * sz + (d >> 1 & 1) * sy + (d & 1) * sx];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      s[2 * q] += lo_bf16(v[q]);
      s[2 * q + 1] += hi_bf16(v[q]);
    }
  }
}

// Grid of the kernels below: x covers the 16-byte units of one row, y strides over the rows
// (n, z, y), so a row's decomposition is scalar work.

// y = mean over 2 x 2 x 2 voxels; D, H, W are the fine sizes.
template <int C8>
__global__ __launch_bounds__(256) void pool_kernel(const u32x4* __restrict__ x,
                                                   u32x4* __restrict__ y, long long rows, int H,
                                                   int W) {
  const int u = blockIdx.x * 256 + threadIdx.x, w2 = W / 2, h2 = H / 2;
  if (u >= w2 * C8) return;
  const int xx = u / C8, c = u - xx * C8;
  for (long long r = blockIdx.y; r < rows; r += gridDim.y) {
    const long long nz = r / h2, yy = r - nz * h2;  // n D/2 + z: the fine plane is 2 nz
    const size_t sy = (size_t)W * C8, sz = sy * H;
    float s[8];
    sum8(x + 2 * nz * sz + 2 * yy * sy + (size_t)2 * xx * C8 + c, C8, sy, sz, s);
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = pack_bf16(0.125f * s[2 * q], 0.125f * s[2 * q + 1]);
    y[r * w2 * C8 + u] = o;
  }
}

// out = (a upsampled by 2 in every direction, b) along the channels.
template <int CA8, int CB8>
__global__ __launch_bounds__(256) void up_cat_kernel(const u32x4* __restrict__ a,
                                                     const u32x4* __restrict__ b,
                                                     u32x4* __restrict__ out, long long rows,
                                                     int H, int W) {
  constexpr int C8 = CA8 + CB8;
  const int u = blockIdx.x * 256 + threadIdx.x;
  if (u >= W * C8) return;
  const int xx = u / C8, c = u - xx * C8;
  for (long long r = blockIdx.y; r < rows; r += gridDim.y) {
    const long long nz = r / H, yy = r - nz * H;
    const u32x4 v = c < CA8
                        ? a[(((nz >> 1) * (H / 2) + (yy >> 1)) * (W / 2) + (xx >> 1)) * CA8 + c]
                        : b[(r * W + xx) * CB8 + (c - CA8)];
    out[r * W * C8 + u] = v;
  }
}

// Gradient of up_cat with respect to a: the sum over each coarse voxel's 2 x 2 x 2 fine voxels.
template <int CA8, int CB8>
__global__ __launch_bounds__(256) void up_cat_grad_kernel(const u32x4* __restrict__ g,
                                                          u32x4* __restrict__ ga, long long rows,
                                                          int H, int W) {
  constexpr int C8 = CA8 + CB8;
  const int u = blockIdx.x * 256 + threadIdx.x, w2 = W / 2, h2 = H / 2;
  if (u >= w2 * CA8) return;
  const int xx = u / CA8, c = u - xx * CA8;
  for (long long r = blockIdx.y; r < rows; r += gridDim.y) {
    const long long nz = r / h2, yy = r - nz * h2;
    const size_t sy = (size_t)W * C8, sz = sy * H;
    float s[8];
    sum8(g + 2 * nz * sz + 2 * yy * sy + (size_t)2 * xx * C8 + c, C8, sy, sz, s);
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = pack_bf16(s[2 * q], s[2 * q + 1]);
    ga[r * w2 * CA8 + u] = o;
  }
}

// Gradient of a tensor that goes into a skip connection and into the pooling: gs (channels
// [0, C) of voxels `pitch` channels apart) + gp / 8 of the voxel's coarse voxel, each term and the
// sum rounded to BF16.
template <int C8>
__global__ __launch_bounds__(256) void skip_pool_grad_kernel(const u32x4* __restrict__ gs,
                                                             int pitch8,
                                                             const u32x4* __restrict__ gp,
                                                             u32x4* __restrict__ g,
                                                             long long rows, int H, int W) {
  const int u = blockIdx.x * 256 + threadIdx.x;
  if (u >= W * C8) return;
  const int xx = u / C8, c = u - xx * C8;
  for (long long r = blockIdx.y; r < rows; r += gridDim.y) {
    const long long nz = r / H, yy = r - nz * H;
    const u32x4 p = gp[(((nz >> 1) * (H / 2) + (yy >> 1)) * (W / 2) + (xx >> 1)) * C8 + c];
    const u32x4 s = gs[(r * W + xx) * pitch8 + c];
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t e = pack_bf16(0.125f * lo_bf16(p[q]), 0.125f * hi_bf16(p[q]));
      o[q] = pack_bf16(lo_bf16(s[q]) + lo_bf16(e), hi_bf16(s[q]) + hi_bf16(e));
    }
    g[r * W * C8 + u] = o;
  }
}

// gm = gy (y > 0) and the sums over voxels of gm. A thread keeps its 8 channels: the stride of its
// units is a multiple of C8. Every block stores its sums in `part` (bias_sum adds them in order, so
// that equal inputs give equal bits), or adds them to db with one float atomic per channel if part is
// null.
template <int C8>
__global__ __launch_bounds__(256) void relu_grad_kernel(const u32x4* __restrict__ gy,
                                                        const u32x4* __restrict__ y,
                                                        u32x4* __restrict__ gm,
                                                        float* __restrict__ part,
                                                        float* __restrict__ db, long long units) {
  __shared__ float red[4][8 * C8];
  float s[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) s[q] = 0.0f;
  const long long stride = (long long)gridDim.x * 256;
  for (long long u = (long long)blockIdx.x * 256 + threadIdx.x; u < units; u += stride) {
    const u32x4 g = gy[u], v = y[u];
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // a product, so an infinite or NaN gradient of a masked value is NaN
      const float a = lo_bf16(g[q]) * (lo_bf16(v[q]) > 0.0f ? 1.0f : 0.0f);
      const float b = hi_bf16(g[q]) * (hi_bf16(v[q]) > 0.0f ? 1.0f : 0.0f);
      s[2 * q] += a;
      s[2 * q + 1] += b;
      o[q] = pack_bf16(a, b);
    }
    gm[u] = o;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    for (int off = 32; off >= C8; off >>= 1) s[q] += __shfl_xor(s[q], off, 64);
    if (lane < C8) red[wave][lane * 8 + q] = s[q];
  }
  __syncthreads();
  if (threadIdx.x < 8 * C8) {
    const float v = red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] +
                    red[3][threadIdx.x];
    if (part) part[(size_t)blockIdx.x * (8 * C8) + threadIdx.x] = v;
    else unsafeAtomicAdd(db + threadIdx.x, v);
  }
}

// db[c] = sum over the rows of part, in an order that depends on their number only. A block sums
// sixteen channels with 64 rows at a time; bound by its latency.
__global__ __launch_bounds__(1024) void bias_sum(const float* __restrict__ part, int rows, int c,
                                                 float* __restrict__ db) {
  __shared__ float red[16][16];
  const int ch = threadIdx.x & 15;
  const float* p = part + blockIdx.x * 16 + ch;
  float s = 0.0f;
  for (int r = threadIdx.x >> 4; r < rows; r += 64) s += p[(size_t)r * c];
  s += __shfl_xor(s, 16, 64);
  s += __shfl_xor(s, 32, 64);
  if ((threadIdx.x & 63) < 16) red[threadIdx.x >> 6][ch] = s;
  __syncthreads();
  if (threadIdx.x < 16) {
    s = red[0][ch];
    for (int w = 1; w < 16; ++w) s += red[w][ch];
    db[blockIdx.x * 16 + ch] = s;
  }
}

// Blocks of relu_grad_kernel at most: four per CU.
constexpr int kReluRows = 1024;

dim3 row_grid(long long units_per_row, long long rows) {
  return dim3((unsigned)((units_per_row + 255) / 256),
              (unsigned)std::max(1LL, std::min(rows, 65535LL)));
}

// Checks shared by the entry points: positive even sizes (odd where `even` is false), a device.
int net_check(int device, int N, int D, int H, int W, bool even) {
  FC_CHECK_ARG(N > 0 && D > 0 && H > 0 && W > 0 && W <= (1 << 24), "bad activation shape");
  FC_CHECK_ARG(!even || (D % 2 == 0 && H % 2 == 0 && W % 2 == 0), "sides must be even");
  return select_device(device);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// The network's weights as the convolutions read them: up to kMaxTensors FP32 tensors rounded to
// BF16 into one buffer, a column of blocks per tensor. 0.4 M elements: bound by its launch. In
// place of a launch per tensor an inference takes 254 instead of 274 us at 64^3 and 361 instead of
// 382 at 96^3; at 256^3 the difference is 0.3 %.
constexpr int kMaxTensors = 16;

struct WeightArgs {
  const float* src[kMaxTensors];
  long long begin[kMaxTensors + 1];
};

__global__ __launch_bounds__(256) void round_weights(WeightArgs a, uint16_t* __restrict__ out) {
  const float* src = a.src[blockIdx.y];
  uint16_t* dst = out + a.begin[blockIdx.y];
  const long long n = a.begin[blockIdx.y + 1] - a.begin[blockIdx.y];
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += gridDim.x * 256ll)
    dst[i] = f32_to_bf16_bits(src[i]);
}

}  // namespace
}  // namespace fc

using namespace fc;

extern "C" {

int fc_net_pool_dev(int device, const void* x, void* y, int N, int D, int H, int W, int c,
                    void* stream) {
  clear_error();
  FC_CHECK_ARG(x && y, "null pointer argument");
  FC_CHECK_ARG(aligned16(x) && aligned16(y), "activations must be 16-byte aligned");
  FC_CHECK_ARG(c == 16 || c == 32, "unsupported channel count %d", c);
  int rc = net_check(device, N, D, H, W, true);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long long rows = (long long)N * (D / 2) * (H / 2);
  const dim3 grid = row_grid((long long)W / 2 * (c / 8), rows);
  const u32x4* xi = static_cast<const u32x4*>(x);
  u32x4* yo = static_cast<u32x4*>(y);
  if (c == 16) pool_kernel<2><<<grid, 256, 0, s>>>(xi, yo, rows, H, W);
  else pool_kernel<4><<<grid, 256, 0, s>>>(xi, yo, rows, H, W);
  FC_HIP(hipGetLastError());
  return FC_OK;
}

int fc_net_up_cat_dev(int device, const void* a, const void* b, void* out, int N, int D, int H,
                      int W, int ca, int cb, void* stream) {
  clear_error();
  FC_CHECK_ARG(a && b && out, "null pointer argument");
  FC_CHECK_ARG(aligned16(a) && aligned16(b) && aligned16(out),
               "activations must be 16-byte aligned");
  FC_CHECK_ARG((ca == 64 && cb == 32) || (ca == 32 && cb == 16),
               "unsupported channel counts %d + %d", ca, cb);
  int rc = net_check(device, N, D, H, W, true);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long long rows = (long long)N * D * H;
  const dim3 grid = row_grid((long long)W * ((ca + cb) / 8), rows);
  const u32x4 *pa = static_cast<const u32x4*>(a), *pb = static_cast<const u32x4*>(b);
  u32x4* po = static_cast<u32x4*>(out);
  if (ca == 64) up_cat_kernel<8, 4><<<grid, 256, 0, s>>>(pa, pb, po, rows, H, W);
  else up_cat_kernel<4, 2><<<grid, 256, 0, s>>>(pa, pb, po, rows, H, W);
  FC_HIP(hipGetLastError());
  return FC_OK;
}

int fc_net_up_cat_grad_dev(int device, const void* g, void* ga, int N, int D, int H, int W,
                           int ca, int cb, void* stream) {
  clear_error();
  FC_CHECK_ARG(g && ga, "null pointer argument");
  FC_CHECK_ARG(aligned16(g) && aligned16(ga), "activations must be 16-byte aligned");
  FC_CHECK_ARG((ca == 64 && cb == 32) || (ca == 32 && cb == 16),
               "unsupported channel counts %d + %d", ca, cb);
  int rc = net_check(device, N, D, H, W, true);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long long rows = (long long)N * (D / 2) * (H / 2);
  const dim3 grid = row_grid((long long)W / 2 * (ca / 8), rows);
  const u32x4* pg = static_cast<const u32x4*>(g);
  u32x4* po = static_cast<u32x4*>(ga);
  if (ca == 64) up_cat_grad_kernel<8, 4><<<grid, 256, 0, s>>>(pg, po, rows, H, W);
  else up_cat_grad_kernel<4, 2><<<grid, 256, 0, s>>>(pg, po, rows, H, W);
  FC_HIP(hipGetLastError());
  return FC_OK;
}

int fc_net_skip_pool_grad_dev(int device, const void* gs, int gs_pitch, const void* gp, void* g,
                              int N, int D, int H, int W, int c, void* stream) {
  clear_error();
  FC_CHECK_ARG(gs && gp && g, "null pointer argument");
  FC_CHECK_ARG(aligned16(gs) && aligned16(gp) && aligned16(g),
               "activations must be 16-byte aligned");
  FC_CHECK_ARG((c == 16 || c == 32) && gs_pitch >= c && gs_pitch % 8 == 0,
               "unsupported channel count %d (pitch %d)", c, gs_pitch);
  int rc = net_check(device, N, D, H, W, true);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long long rows = (long long)N * D * H;
  const dim3 grid = row_grid((long long)W * (c / 8), rows);
  const u32x4 *ps = static_cast<const u32x4*>(gs), *pp = static_cast<const u32x4*>(gp);
  u32x4* po = static_cast<u32x4*>(g);
  if (c == 16)
    skip_pool_grad_kernel<2><<<grid, 256, 0, s>>>(ps, gs_pitch / 8, pp, po, rows, H, W);
  else
    skip_pool_grad_kernel<4><<<grid, 256, 0, s>>>(ps, gs_pitch / 8, pp, po, rows, H, W);
  FC_HIP(hipGetLastError());
  return FC_OK;
}

// fc_net_relu_grad_dev and fc_net_relu_grad_parts_dev: `rows` is the most blocks that `part` holds.
static int relu_grad(int device, const void* gy, const void* y, void* gm, float* part, long long rows,
                     float* db, long long voxels, int c, void* stream) {
  clear_error();
  FC_CHECK_ARG(gy && y && gm && db, "null pointer argument");
  FC_CHECK_ARG(aligned16(gy) && aligned16(y) && aligned16(gm),
               "activations must be 16-byte aligned");
  FC_CHECK_ARG(voxels > 0, "bad activation shape");
  FC_CHECK_ARG(c == 16 || c == 32 || c == 64, "unsupported channel count %d", c);
  int rc = select_device(device);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long long units = voxels * (c / 8);
  // at least 16 units per thread, so that a block's sums are few beside its loads
  const unsigned blocks = (unsigned)std::max(1LL, std::min(rows, units / (256 * 16)));
  const u32x4 *pg = static_cast<const u32x4*>(gy), *py = static_cast<const u32x4*>(y);
  u32x4* po = static_cast<u32x4*>(gm);
  if (c == 16) relu_grad_kernel<2><<<blocks, 256, 0, s>>>(pg, py, po, part, db, units);
  else if (c == 32) relu_grad_kernel<4><<<blocks, 256, 0, s>>>(pg, py, po, part, db, units);
  else relu_grad_kernel<8><<<blocks, 256, 0, s>>>(pg, py, po, part, db, units);
  if (part) bias_sum<<<c / 16, 1024, 0, s>>>(part, (int)blocks, c, db);
  FC_HIP(hipGetLastError());
  return FC_OK;
}

int fc_net_relu_grad_dev(int device, const void* gy, const void* y, void* gm, float* db,
                         long long voxels, int c, void* stream) {
  return relu_grad(device, gy, y, gm, nullptr, kReluRows, db, voxels, c, stream);
}

int fc_net_relu_grad_parts_dev(int device, const void* gy, const void* y, void* gm, float* part,
                               int rows, float* db, long long voxels, int c, void* stream) {
  clear_error();
  FC_CHECK_ARG(part && rows > 0, "null or empty scratch");
  return relu_grad(device, gy, y, gm, part, std::min(rows, kReluRows), db, voxels, c, stream);
}

int fc_net_weights_dev(int device, const float* const* src, const long long* counts, int n,
                       void* dst, void* stream) {
  clear_error();
  FC_CHECK_ARG(src && counts && dst, "null pointer argument");
  FC_CHECK_ARG(n > 0 && n <= kMaxTensors, "1 to %d tensors", kMaxTensors);
  WeightArgs a;
  a.begin[0] = 0;
  long long most = 0;
  for (int q = 0; q < n; ++q) {
    FC_CHECK_ARG(src[q] && counts[q] > 0, "empty tensor %d", q);
    a.src[q] = src[q];
    a.begin[q + 1] = a.begin[q] + counts[q];
    most = std::max(most, counts[q]);
  }
  int rc = select_device(device);
  if (rc) return rc;
  const dim3 grid((unsigned)std::min(256LL, (most + 255) / 256), n);
  round_weights<<<grid, 256, 0, static_cast<hipStream_t>(stream)>>>(a, static_cast<uint16_t*>(dst));
  FC_HIP(hipGetLastError());
  return FC_OK;
}

}  // extern "C"
