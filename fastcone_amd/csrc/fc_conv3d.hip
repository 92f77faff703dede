// 3x3x3 convolution kernels for the CGLS warm-start network (gfx950, MFMA).
//
// Layout: activations N x D x H x W x C (channels last), BF16; weights [Cout][27][Cin] BF16
// (tap = 9 dz + 3 dy + dx, zero padding 1); accumulation FP32.
//
//  * forward (and input gradient): implicit GEMM  Y[voxel][co] = sum_k P[voxel][k] Wt[k][co],
//    k = tap * Cin + ci, with v_mfma_f32_16x16x32_bf16 on input planes staged in LDS; each lane
//    feeds 8 consecutive k (8 channels of one tap). Bias and ReLU are fused in the epilogue. The
//    input gradient is the same kernel on dY with the flipped, transposed weights
//    W'[ci][26 - tap][co] = W[co][tap][ci].
//  * weight gradient: dW[co][tap][ci] = sum_voxel dY[voxel][co] x[voxel + tap][ci] with
//    v_mfma_f32_16x16x32_bf16 fed the raw BF16 bits (products exact in FP32), voxels as k: a wave
//    per 16 x 16 channels and x segment, walking rows. Each block adds its sums to the FP32 master
//    gradient with float atomics.
//  * 1-channel layers (first layer Cin = 1, last layer Cout = 1): forward passes and the last
//    layer's input gradient are FP32 FMAs in ascending order of k; both weight gradients are MFMAs
//    over the voxels.
//
// Operand / result lane layouts of the MFMA form used (checked by fc_mfma_layout_probe, which also
// checks the 16x16x4 FP32 form):
//   16x16x32 bf16: A lane l holds A[l % 16][8 (l / 16) + 0..7], B lane l holds
//   B[8 (l / 16) + 0..7][l % 16]; 16x16x4 f32: A[l % 16][l / 16], B[l / 16][l % 16];
//   result D lane l, register r holds D[4 (l / 16) + r][l % 16].
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>
#include <utility>

#include "fc_device.h"
#include "fc_internal.h"

namespace fc {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
// the caller's buffers may start at any element
typedef unsigned int u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
typedef unsigned int u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// ---- forward / input-gradient implicit GEMM --------------------------------------------------
// A block owns a tile of XT x YT voxels in x and y and walks a chunk of z planes. Three input planes
// (the tile with its one-voxel halo, zero outside the volume) are resident in LDS; the next one is
// loaded into registers while a plane is computed. A wave owns V groups of 16 consecutive x voxels
// and all output channels: the weights are the MFMA's A operand (16 channels x 32 k), the patches
// its B operand (32 k x 16 voxels, one 16-byte LDS read per lane), so a lane ends with four
// consecutive channels of one voxel, an 8-byte store. The order of every output's sum is k
// ascending, 32 per instruction.
//
// Each weight fragment feeds V instructions; where the whole weight set fits (kWReg) it stays in
// registers over the walk, otherwise it comes from L1 once per V instructions. A voxel's channels
// are padded by 16 bytes in LDS: the pitch is an odd number of 16-byte units, so the eight voxels of
// a quarter of a read lie in different banks.
//
// Bound by the LDS reads of the patches (1 KB per instruction) in the 16- and 48-channel layers and
// by the weights' way from L1 in the 64- and 96-channel ones. Before, a wave owned one group and
// read patches and weights from L1 for every instruction. Time at 256^3: 16 -> 16 channels 1.49 ->
// 0.32 ms (1.07 GB of activations: 0.23 ms at the rate of a large copy), 48 -> 16 5.29 -> 0.98 ms;
// at 128^3: 96 -> 32 2.26 -> 0.96 ms, 32 -> 32 0.64 -> 0.17 ms; at 64^3: 64 -> 64 0.47 -> 0.21 ms
// (the layers with whole 32-channel steps have since got a kernel of their own for large inputs,
// conv_fwd_stream).
template <int CIN, int COUT>
struct ConvTile {
  static constexpr int XT = (CIN == 16 && COUT <= 32) || (CIN == 32 && COUT >= 32) ? 32 : 16;
  static constexpr int YT = 8;
  static constexpr int V = XT * YT / 16 / 4;          // groups of 16 voxels per wave
  static constexpr int PITCH = 2 * CIN + 16;          // bytes per voxel
  static constexpr int ROWB = (XT + 2) * PITCH, PLANEB = (YT + 2) * ROWB;
  static constexpr int K = 27 * CIN, KSTEPS = (K + 31) / 32, NB = COUT / 16;
  static constexpr bool kWReg = KSTEPS * NB <= 42;    // 168 VGPRs
  static constexpr int G = NB <= 2 ? 4 : (NB <= 4 ? 2 : 1);  // steps of weights loaded ahead
  // LDS offset of k's tap and channel in its plane, and its plane
  static constexpr int off(int k) {
    const int tap = k / CIN;
    return ((tap / 3) % 3 * (XT + 2) + tap % 3) * PITCH + 2 * (k % CIN);
  }
  static constexpr int dz(int k) { return k / CIN / 9; }
};

// UPCAT: the input is the concatenation (x upsampled by 2 in every direction, skip) of 2/3 and 1/3 of
// the channels, which never exists in memory: a plane's units are loaded from where they are. At
// 256^3, 48 -> 16 channels 0.98 -> 0.90 ms, and the 0.44 ms that forming it took are gone.
template <int CIN, int COUT, bool RELU, bool UPCAT>
__global__ __launch_bounds__(256, 2) void conv_fwd_mfma(const uint16_t* __restrict__ x,
                                                        const uint16_t* __restrict__ skip,
                                                        const uint16_t* __restrict__ w,
                                                        const float* __restrict__ bias,
                                                        uint16_t* __restrict__ y, int D, int H,
                                                        int W, int tx, int ty, int zc, int nzc) {
  static_assert(CIN % 16 == 0 && COUT % 16 == 0, "channel counts must be multiples of 16");
  using T = ConvTile<CIN, COUT>;
  constexpr int XT = T::XT, YT = T::YT, V = T::V, PITCH = T::PITCH, ROWB = T::ROWB;
  constexpr int K = T::K, KSTEPS = T::KSTEPS, NB = T::NB, CA = 2 * CIN / 3;
  constexpr int C8 = CIN / 8, UNITS = (XT + 2) * (YT + 2) * C8, NU = (UNITS + 255) / 256;
  __shared__ __align__(16) char ring[3 * T::PLANEB];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, g = lane >> 4;
  const bool hi = g >= 2;
  int b = xcd_remap(blockIdx.x, gridDim.x);
  const int bx = b % tx; b /= tx;
  const int by = b % ty; b /= ty;
  const int bz = b % nzc, n = b / nzc;
  const int xb = bx * XT, yb = by * YT, z0 = bz * zc, z1 = min(D, z0 + zc);

  // this thread's 16-byte units of a plane: voxel offset from the tile's corner (-1: outside the
  // volume in x or y, or no unit) and LDS address
  int vox[NU], dst[NU], ch[NU];
#pragma unroll
  for (int q = 0; q < NU; ++q) {
    const int u = (int)threadIdx.x + 256 * q;
    const int v = u / C8, c8 = u - v * C8, yy = v / (XT + 2), xx = v - yy * (XT + 2);
    const int gx = xb + xx - 1, gy = yb + yy - 1;
    vox[q] = u < UNITS && gx >= 0 && gx < W && gy >= 0 && gy < H ? (yy * W + xx) : -1;
    dst[q] = u < UNITS ? v * PITCH + 16 * c8 : -1;
    ch[q] = 8 * c8;
    if (UPCAT && vox[q] >= 0)  // element of its tensor's plane
      vox[q] = ch[q] < CA ? ((gy >> 1) * (W >> 1) + (gx >> 1)) * CA + ch[q]
                          : (gy * W + gx) * (CIN - CA) + ch[q] - CA;
  }
  u32x4 pf[NU];
  auto fetch = [&](int z) {
    // element (z, yb - 1, xb - 1) of batch n; only units inside the volume are read
    const uint16_t* p = x + ((((long long)n * D + z) * H + (yb - 1)) * W + (xb - 1)) * CIN;
    const bool zin = z >= 0 && z < D;
    const uint16_t *pa = nullptr, *pb = nullptr;
    if constexpr (UPCAT) {
      const long long plane = (long long)n * D + z;  // D is even
      pa = x + (plane >> 1) * (H >> 1) * (W >> 1) * CA;
      pb = skip + plane * H * W * (CIN - CA);
    }
#pragma unroll
    for (int q = 0; q < NU; ++q) {
      pf[q] = u32x4{0u, 0u, 0u, 0u};
      if (zin && vox[q] >= 0)
        pf[q] = *reinterpret_cast<const u32x4_a2*>(
            UPCAT ? (ch[q] < CA ? pa : pb) + vox[q] : p + (long long)vox[q] * CIN + ch[q]);
    }
  };
  auto put = [&](int slot) {
#pragma unroll
    for (int q = 0; q < NU; ++q)
      if (dst[q] >= 0) *reinterpret_cast<u32x4*>(ring + slot * T::PLANEB + dst[q]) = pf[q];
  };
  // weight fragment (step s, block cb): row cb 16 + m, k = 32 s + 8 g; zero past K
  const int wlane = m * K + g * 8;
  auto wfrag = [&](int s, int cb, int from) {
    u32x4 q = u32x4{0u, 0u, 0u, 0u};
    if (K % 32 == 0 || s + 1 < KSTEPS || !hi)
      q = *reinterpret_cast<const u32x4_a2*>(w + from + cb * 16 * K + s * 32);
    return __builtin_bit_cast(bf16x8, q);
  };
  constexpr int G = T::kWReg ? KSTEPS : T::G;
  bf16x8 wr[T::kWReg ? KSTEPS * NB : 2 * G * NB];
  if constexpr (T::kWReg) {
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) wr[s * NB + cb] = wfrag(s, cb, wlane);
  }
  f32x4 bb[NB];
#pragma unroll
  for (int cb = 0; cb < NB; ++cb)
#pragma unroll
    for (int r = 0; r < 4; ++r) bb[cb][r] = bias ? bias[cb * 16 + 4 * g + r] : 0.0f;

  // group v of wave `wave`: row (wave V + v) 16 / XT, x offset 16 ((wave V + v) % (XT / 16))
  constexpr int GX = XT / 16;
  static_assert(V % GX == 0, "a wave owns whole rows");
  const int lane0 = (wave * (V / GX) * (XT + 2) + m) * PITCH + 16 * g;
  // weights not held in registers come G steps ahead, in alternating halves of wr; the empty asm
  // keeps the compiler from loading them earlier (it would hoist them all and spill)
  auto ahead = [&](int s0) {
    int from = wlane;
    asm volatile("" : "+v"(from));
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
      for (int cb = 0; cb < NB; ++cb)
        if (s0 + q < KSTEPS) wr[((s0 / G % 2) * G + q) * NB + cb] = wfrag(s0 + q, cb, from);
  };
  int slot[3] = {0, 1, 2};  // ring slots of planes z - 1, z, z + 1
  for (int d = 0; d < 3; ++d) {
    fetch(z0 - 1 + d);
    put(d);
  }
  __syncthreads();
  for (int z = z0; z < z1; ++z) {
    if (z + 1 < z1) fetch(z + 2);
    int base[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) base[d] = lane0 + slot[d] * T::PLANEB;
    f32x4 acc[V][NB];
#pragma unroll
    for (int v = 0; v < V; ++v)
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) acc[v][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (!T::kWReg) ahead(0);
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      if constexpr (!T::kWReg) {
        if (s % G == 0) {
          __builtin_amdgcn_sched_barrier(0);
          if (s + G < KSTEPS) ahead(s + G);
        }
      }
      // lanes g = 0, 1 hold k0 .. k0 + 15 and lanes g = 2, 3 k1 .. k1 + 15: the second half is
      // either the next 16 channels of the same tap, another tap, or past the end (zero)
      const int k0 = 32 * s, k1 = 32 * s + 16;
      const int o0 = T::off(k0), d0 = T::dz(k0);
      int addr = base[d0];
      if (k1 >= K) {
        addr -= hi ? 32 : 0;
      } else if (T::dz(k1) != d0) {
        addr = hi ? base[T::dz(k1)] + (T::off(k1) - 32 - o0) : addr;
      } else if (T::off(k1) - o0 != 32) {
        addr += hi ? T::off(k1) - 32 - o0 : 0;
      }
      bf16x8 a[NB];
#pragma unroll
      for (int cb = 0; cb < NB; ++cb)
        a[cb] = wr[(T::kWReg ? s : s / G % 2 * G + s % G) * NB + cb];
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const int gofs = (v / GX) * ROWB + (v % GX) * 16 * PITCH;
        u32x4 q = *reinterpret_cast<const u32x4*>(ring + addr + (o0 + gofs));
        if (k1 >= K && hi) q = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int cb = 0; cb < NB; ++cb)
          acc[v][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[cb], __builtin_bit_cast(bf16x8, q),
                                                               acc[v][cb], 0, 0, 0);
      }
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int vy = yb + wave * (V / GX) + v / GX, vx = xb + (v % GX) * 16 + m;
      if (vy < H && vx < W) {
        uint16_t* o = y + ((((size_t)n * D + z) * H + vy) * W + vx) * COUT + 4 * g;
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) {
          float f[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            f[r] = acc[v][cb][r] + bb[cb][r];
            if (RELU) f[r] = fmaxf(f[r], 0.0f);
          }
          *reinterpret_cast<u32x2_a2*>(o + cb * 16) =
              u32x2_a2{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3])};
        }
      }
    }
    __syncthreads();  // plane z - 1 is no longer read
    if (z + 1 < z1) {
      put(slot[0]);
      const int s0 = slot[0];
      slot[0] = slot[1];
      slot[1] = slot[2];
      slot[2] = s0;
      __syncthreads();
    }
  }
}

// The same convolution for whole 32-channel steps (Cin a multiple of 32) and many tiles, plane by
// plane: one input plane is in LDS, and a patch read from it feeds the three output planes z - 1, z,
// z + 1 at once (their dz = 2, 1, 0 weights), whose sums are all in registers. Every output still
// adds its terms in ascending order of k, 32 per instruction: dz = 0 comes with its first plane. A
// wave owns one block of 16 output channels and V rows of 16 voxels, so a step's three weight
// fragments (from L1, a step ahead) feed 3 V instructions; the next plane is loaded into registers
// meanwhile.
//
// conv_fwd_mfma is bound by the weights' way from L1 in these layers: two instructions per fragment
// of 1 KB, which takes L1 16 clocks for each wave as the instruction takes its SIMD. Here it is 24
// (12 for 96 channels, whose next plane needs the registers), and a third of the patch reads. Time
// before and now: 96 -> 32 channels at 128^3 0.92 -> 0.58 ms, 64 -> 64 at 64^3 0.20 -> 0.09, 32 -> 32
// at 128^3 0.15 -> 0.12, 64 -> 32 at 4 x 32^3 0.055 -> 0.037 ms. With all of a row's channel blocks
// in one wave (6 or 12 fragments a step) it was slower than before. (64 -> 32 channels spill 23 of 256
// registers, and are 1.5 times as fast as conv_fwd_mfma all the same.)
template <int CIN, int COUT>
struct StreamTile {
  static constexpr int NB = COUT / 16;          // channel blocks; a wave owns one
  static constexpr int V = CIN == 96 ? 4 : 8;    // and this many rows of 16 voxels
  static constexpr int XT = 16, YT = 4 / NB * V, PITCH = 2 * CIN + 16;
  static constexpr int ROWB = (XT + 2) * PITCH, PLANEB = (YT + 2) * ROWB;
  static constexpr int C32 = CIN / 32, STEPS = 9 * C32, K = 27 * CIN;
};

template <int CIN, int COUT, bool RELU, bool UPCAT>
__global__ __launch_bounds__(256, 2) void conv_fwd_stream(const uint16_t* __restrict__ x,
                                                          const uint16_t* __restrict__ skip,
                                                          const uint16_t* __restrict__ w,
                                                          const float* __restrict__ bias,
                                                          uint16_t* __restrict__ y, int D, int H,
                                                          int W, int tx, int ty, int zc, int nzc) {
  using T = StreamTile<CIN, COUT>;
  constexpr int XT = T::XT, YT = T::YT, V = T::V, PITCH = T::PITCH, ROWB = T::ROWB, NB = T::NB;
  constexpr int C8 = CIN / 8, UNITS = (XT + 2) * (YT + 2) * C8, NU = (UNITS + 255) / 256;
  constexpr int CA = 2 * CIN / 3, STEPS = T::STEPS, K = T::K;
  __shared__ __align__(16) char plane[T::PLANEB];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, g = lane >> 4;
  int b = xcd_remap(blockIdx.x, gridDim.x);
  const int bx = b % tx; b /= tx;
  const int by = b % ty; b /= ty;
  const int bz = b % nzc, n = b / nzc;
  const int xb = bx * XT, yb = by * YT, z0 = bz * zc, z1 = min(D, z0 + zc);

  // plane units as in conv_fwd_mfma
  int vox[NU];
#pragma unroll
  for (int q = 0; q < NU; ++q) {
    const int u = (int)threadIdx.x + 256 * q;
    const int v = u / C8, ch = 8 * (u - v * C8), yy = v / (XT + 2), xx = v - yy * (XT + 2);
    const int gx = xb + xx - 1, gy = yb + yy - 1;
    vox[q] = -1;
    if (u < UNITS && gx >= 0 && gx < W && gy >= 0 && gy < H)
      vox[q] = !UPCAT    ? yy * W + xx
               : ch < CA ? ((gy >> 1) * (W >> 1) + (gx >> 1)) * CA + ch
                         : (gy * W + gx) * (CIN - CA) + ch - CA;
  }
  u32x4 pf[NU];
  auto fetch = [&](int z) {
    const uint16_t* p = x + ((((long long)n * D + z) * H + (yb - 1)) * W + (xb - 1)) * CIN;
    const bool zin = z >= 0 && z < D;
    const long long pl = (long long)n * D + z;
    const uint16_t *pa = nullptr, *pb = nullptr;
    if constexpr (UPCAT) {
      pa = x + (pl >> 1) * (H >> 1) * (W >> 1) * CA;  // D is even
      pb = skip + pl * H * W * (CIN - CA);
    }
#pragma unroll
    for (int q = 0; q < NU; ++q) {
      const int ch = 8 * (((int)threadIdx.x + 256 * q) % C8);
      pf[q] = u32x4{0u, 0u, 0u, 0u};
      if (zin && vox[q] >= 0)
        pf[q] = *reinterpret_cast<const u32x4_a2*>(UPCAT ? (ch < CA ? pa : pb) + vox[q]
                                                         : p + (long long)vox[q] * CIN + ch);
    }
  };
  auto put = [&]() {
#pragma unroll
    for (int q = 0; q < NU; ++q) {
      const int u = (int)threadIdx.x + 256 * q, v = u / C8;
      if (u < UNITS) *reinterpret_cast<u32x4*>(plane + v * PITCH + 16 * (u - v * C8)) = pf[q];
    }
  };
  const int cb = wave % NB, rows = wave / NB * V;  // this wave's channel block and first row
  f32x4 bb;
#pragma unroll
  for (int r = 0; r < 4; ++r) bb[r] = bias ? bias[cb * 16 + 4 * g + r] : 0.0f;
  const char* lane0 = plane + (rows * (XT + 2) + m) * PITCH + 16 * g;
  const uint32_t wlane = 2u * (uint32_t)((cb * 16 + m) * K + g * 8);
  bf16x8 wr[2][3];
  auto weights = [&](int s) {
    uint32_t from = wlane;
    const uint16_t* ws = w;
    asm volatile("" : "+v"(from), "+s"(ws));  // loads and addresses not earlier than a step ahead
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const char* at = reinterpret_cast<const char*>(ws + (d * 9 * CIN + s * 32));
      wr[s & 1][d] =
          __builtin_bit_cast(bf16x8, (u32x4)*reinterpret_cast<const u32x4_a2*>(at + from));
    }
  };
  f32x4 acc[3][V];  // output planes p - 1, p, p + 1
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int v = 0; v < V; ++v) acc[d][v] = f32x4{0.f, 0.f, 0.f, 0.f};
  fetch(z0 - 1);
  put();
  __syncthreads();
  for (int p = z0 - 1; p <= z1; ++p) {
    if (p < z1) fetch(p + 1);
    // planes at the ends of the chunk serve one or two outputs
    const bool use[3] = {p + 1 < z1, p >= z0 && p < z1, p > z0};
    weights(0);
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      if (s + 1 < STEPS) weights(s + 1);
      const int tap = s / T::C32, o = (tap / 3 * (XT + 2) + tap % 3) * PITCH + s % T::C32 * 64;
      bf16x8 f[V];
#pragma unroll
      for (int v = 0; v < V; ++v)
        f[v] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(lane0 + o + v * ROWB));
#pragma unroll
      for (int d = 0; d < 3; ++d)
        if (use[d])
#pragma unroll
          for (int v = 0; v < V; ++v)
            acc[2 - d][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[s & 1][d], f[v],
                                                                    acc[2 - d][v], 0, 0, 0);
    }
    if (p > z0) {
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const int vy = yb + rows + v, vx = xb + m;
        if (vy < H && vx < W) {
          float f[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            f[r] = acc[0][v][r] + bb[r];
            if (RELU) f[r] = fmaxf(f[r], 0.0f);
          }
          uint16_t* o = y + ((((size_t)n * D + (p - 1)) * H + vy) * W + vx) * COUT + cb * 16 + 4 * g;
          *reinterpret_cast<u32x2_a2*>(o) = u32x2_a2{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3])};
        }
      }
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
      acc[0][v] = acc[1][v];
      acc[1][v] = acc[2][v];
      acc[2][v] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();  // the plane is no longer read
    if (p < z1) {
      put();
      __syncthreads();
    }
  }
}

// W'[ci][(26 - tap) * COUT + co] = W[co][tap * CIN + ci]
__global__ __launch_bounds__(256) void flip_transpose_weights(const uint16_t* __restrict__ w,
                                                              uint16_t* __restrict__ wt, int cin,
                                                              int cout) {
  int q = blockIdx.x * 256 + threadIdx.x;
  int total = cout * 27 * cin;
  if (q >= total) return;
  int co = q / (27 * cin), rem = q - co * 27 * cin;
  int tap = rem / cin, ci = rem - tap * cin;
  wt[((size_t)ci * 27 + (26 - tap)) * cout + co] = w[q];
}

// ---- weight gradient -------------------------------------------------------------------------
// dW[co][tap][ci] for 16 output and 16 input channels per wave: 27 accumulators of 16 x 16, one per
// tap, with the voxels as the MFMA's k. A wave owns 32 consecutive x voxels of the input and walks
// rows y at fixed (n, z); per row of the output gradient it stages three new input rows (z - 1, z,
// z + 1) and the gradient row in its own LDS, as they lie in memory (16 channels per voxel), and
// reads them back transposed (ds_read_b64_tr_b16: four voxels of one channel per lane). The taps'
// shift along x is applied to the gradient row (three fragments), so an input fragment serves its
// three dx; along y it is kept in registers for the three rows that use it. A row then costs 27
// instructions, 6 KB of LDS reads and no barrier. The waves of a block add their sums in LDS and the
// block adds them to dW with float atomics.
//
// Bound by the matrix instructions (27 x 16 clocks per row and wave) with two waves per SIMD (108
// accumulator registers). Before, every lane gathered its eight voxels one by one for each tap:
// a training step's seven layers (4 x 128^3) took 19.1 ms; 48 -> 16 channels at 4 x 128^3 7.88 ->
// 0.52 ms, 16 -> 16 2.24 -> 0.17 ms, 96 -> 32 at 4 x 64^3 2.12 -> 0.22 ms.
// A block's input channels are one aligned group of 16, so for the decoder's layers they lie in one
// of the two tensors that are concatenated, and the rows are loaded from there: with the forward
// pass doing the same, a training step at 4 x 128^3 forms none of its 1.0 GB of concatenations (6.17
// -> 5.68 ms).
constexpr int kWgSeg = 32;                        // input voxels per wave and row
constexpr int kWgWaveB = 3 * kWgSeg * 32 + 34 * 32;  // LDS bytes per wave: three rows, gradient row
constexpr int kWgRed = 4;                         // accumulators reduced at once

struct WgArgs {
  const uint16_t* x;     // the input, or its first ca channels at half the size (skip: the others)
  const uint16_t* skip;
  int ca;                // 0: x is the input
  const uint16_t* dy;
  float* dw;
  long long units;  // (n, z, y chunk, x segment)
  int D, H, W, cin, cout;
  int nseg, nyc, yc;
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
// Eight voxels of one channel per lane from voxels of 32 bytes (16 channels): lane (m, g) gets
// channel m of voxels 8 g .. 8 g + 7. A transposed read takes, per 16 lanes, four voxels: lane j
// addresses voxel j / 4, channels 4 (j % 4) .. + 3, and receives channel j of all four.
__device__ __forceinline__ bf16x8 read_channel(const char* row, int lane) {
  typedef __attribute__((address_space(3))) s16x4* lds_p;
  const char* p = row + (8 * (lane >> 4) + ((lane & 15) >> 2)) * 32 + (lane & 3) * 8;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_p)p);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_p)(p + 4 * 32));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Orders a wave's LDS writes before its lanes' later reads, and reads before later writes. LDS
// operations of one wave execute in order; this only keeps the compiler from moving them.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Mask of the eight BF16 voxels x .. x + 7 of a fragment that lie in [0, W), as do those `shift` on.
__device__ __forceinline__ u32x4 pairs_inside(int x, int shift, int W) {
  u32x4 in;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int v = x + 2 * q;
    const bool lo = v < W && v + shift >= 0 && v + shift < W;
    const bool hi = v + 1 < W && v + 1 + shift >= 0 && v + 1 + shift < W;
    in[q] = (lo ? 0xffffu : 0u) | (hi ? 0xffff0000u : 0u);
  }
  return in;
}
__device__ __forceinline__ bf16x8 masked(bf16x8 v, u32x4 mask) {
  return __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, v) & mask);
}

__global__ __launch_bounds__(256, 2) void conv_wgrad_mfma(WgArgs a) {
  __shared__ __align__(16) char lds[4 * kWgWaveB];
  static_assert(4 * kWgRed * 1024 <= 4 * kWgWaveB, "the reduction reuses the rows' LDS");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, g = lane >> 4;
  const int ncb = a.cin / 16, nco = a.cout / 16;
  int b = xcd_remap(blockIdx.x, gridDim.x);
  const int ci0 = b % ncb * 16; b /= ncb;
  const int co0 = b % nco * 16; b /= nco;
  const long long unit = (long long)b * 4 + wave;
  f32x4 acc[3][3][3];  // [dz][dy][dx]
#pragma unroll
  for (int q = 0; q < 27; ++q) acc[q / 9][q / 3 % 3][q % 3] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (unit < a.units) {
    long long u = unit;
    const int x0 = (int)(u % a.nseg) * kWgSeg; u /= a.nseg;
    const int y0 = (int)(u % a.nyc) * a.yc; u /= a.nyc;
    const int z = (int)(u % a.D);
    const long long n = u / a.D;
    const int y1 = min(a.H, y0 + a.yc);
    char* xr = lds + wave * kWgWaveB;
    char* gr = xr + 3 * kWgSeg * 32;
    const int xv = x0 + (lane >> 1);                     // input voxel of this lane's 16 bytes
    const int gv0 = x0 - 1 + (lane >> 1), gv1 = gv0 + 32;  // gradient voxels (gv1: lanes 0 - 3)
    const bool xok = xv < a.W, g0ok = gv0 >= 0 && gv0 < a.W, g1ok = lane < 4 && gv1 < a.W;
    // where this block's input channels are: in x, or of a concatenation (x upsampled, skip)
    const int up = a.ca && ci0 < a.ca, xc = !a.ca ? a.cin : (up ? a.ca : a.cin - a.ca);
    const uint16_t* xp = !a.ca || up ? a.x + ci0 : a.skip + (ci0 - a.ca);
    const long long xh = a.H >> up, xw = a.W >> up;
    u32x4 px[3], pg0, pg1;
    // input rows yy of the three planes, and gradient row yg, as zeros outside the volume
    auto fetch_x = [&](int yy) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const int zz = z + d - 1;
        px[d] = u32x4{0u, 0u, 0u, 0u};
        if (xok && zz >= 0 && zz < a.D && yy >= 0 && yy < a.H)
          px[d] = *reinterpret_cast<const u32x4_a2*>(
              xp + ((((n * a.D + zz) >> up) * xh + (yy >> up)) * xw + (xv >> up)) * xc + 8 * (lane & 1));
      }
    };
    auto fetch_g = [&](int yg) {
      const uint16_t* p = a.dy + ((n * a.D + z) * a.H + yg) * a.W * a.cout + co0 + 8 * (lane & 1);
      pg0 = pg1 = u32x4{0u, 0u, 0u, 0u};
      if (g0ok) pg0 = *reinterpret_cast<const u32x4_a2*>(p + (long long)gv0 * a.cout);
      if (g1ok) pg1 = *reinterpret_cast<const u32x4_a2*>(p + (long long)gv1 * a.cout);
    };
    auto put_x = [&]() {
#pragma unroll
      for (int d = 0; d < 3; ++d)
        *reinterpret_cast<u32x4*>(xr + d * kWgSeg * 32 + lane * 16) = px[d];
    };
    bf16x8 B[3][3];  // [dz][row mod 3]
    auto read_x = [&](int slot) {
#pragma unroll
      for (int d = 0; d < 3; ++d) B[d][slot] = read_channel(xr + d * kWgSeg * 32, lane);
    };
    fetch_x(y0 - 1);
    put_x();
    wave_sync();
    read_x(0);
    fetch_x(y0);
    wave_sync();
    put_x();
    wave_sync();
    read_x(1);
    wave_sync();
    fetch_x(y0 + 1);
    fetch_g(y0);
    for (int y = y0; y < y1;) {
#pragma unroll
      for (int r = 0; r < 3; ++r) {  // rows y - 1, y, y + 1 are in slots r, r + 1, r + 2 mod 3
        if (y >= y1) break;
        put_x();
        *reinterpret_cast<u32x4*>(gr + lane * 16) = pg0;
        if (lane < 4) *reinterpret_cast<u32x4*>(gr + (64 + lane) * 16) = pg1;
        wave_sync();
        if (y + 1 < y1) {
          fetch_x(y + 2);
          fetch_g(y + 1);
        }
        read_x((r + 2) % 3);
        bf16x8 A[3];
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) A[dx] = read_channel(gr + (2 - dx) * 32, lane);
#pragma unroll
        for (int dy = 0; dy < 3; ++dy)
#pragma unroll
          for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int dx = 0; dx < 3; ++dx)
              acc[d][dy][dx] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  A[dx], B[d][(r + dy) % 3], acc[d][dy][dx], 0, 0, 0);
        wave_sync();
        ++y;
      }
    }
    // A product of a padding zero with an infinite value is NaN, where the sum has no such term: sums
    // with a NaN are formed once more, with both factors of these products zero, row by row.
    float sum = 0.0f;
#pragma unroll
    for (int q = 0; q < 27 * 4; ++q) sum += 0.0f * acc[q / 36][q / 12 % 3][q / 4 % 3][q % 4];
    if (__any(sum != 0.0f)) {
#pragma unroll
      for (int q = 0; q < 27; ++q) acc[q / 9][q / 3 % 3][q % 3] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int y = y0; y < y1; ++y) {
        fetch_g(y);
        *reinterpret_cast<u32x4*>(gr + lane * 16) = pg0;
        if (lane < 4) *reinterpret_cast<u32x4*>(gr + (64 + lane) * 16) = pg1;
#pragma unroll
        for (int dy = 0; dy < 3; ++dy) {
          const int yy = y + dy - 1;
          if (yy < 0 || yy >= a.H) continue;
          fetch_x(yy);
          put_x();
          wave_sync();
#pragma unroll
          for (int dx = 0; dx < 3; ++dx) {
            int xs = x0 + 8 * g;
            asm volatile("" : "+v"(xs));  // a mask at a time in registers
            const u32x4 in = pairs_inside(xs, 1 - dx, a.W);
            const bf16x8 A = masked(read_channel(gr + (2 - dx) * 32, lane), in);
#pragma unroll
            for (int d = 0; d < 3; ++d)
              if (z + d - 1 >= 0 && z + d - 1 < a.D)
                acc[d][dy][dx] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    A, masked(read_channel(xr + d * kWgSeg * 32, lane), in), acc[d][dy][dx], 0, 0, 0);
          }
          wave_sync();
        }
      }
    }
  }
  // sum over the block's waves, kWgRed taps at a time: part[wave][tap][co][ci]
  float* part = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int q0 = 0; q0 < 27; q0 += kWgRed) {
    __syncthreads();
#pragma unroll
    for (int q = q0; q < q0 + kWgRed && q < 27; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        part[((wave * kWgRed + q - q0) * 16 + 4 * g + r) * 16 + m] = acc[q / 9][q / 3 % 3][q % 3][r];
    __syncthreads();
    for (int e = threadIdx.x; e < kWgRed * 256 && q0 + e / 256 < 27; e += 256) {
      const int co = co0 + e / 16 % 16, ci = ci0 + e % 16;
      const float v = part[e] + part[e + kWgRed * 256] + part[e + 2 * kWgRed * 256] +
                      part[e + 3 * kWgRed * 256];
      if (v != 0.0f)
        unsafeAtomicAdd(a.dw + ((size_t)co * 27 + (q0 + e / 256)) * a.cin + ci, v);
    }
  }
}

// ---- 1-channel layers ------------------------------------------------------------------------
// Sixteen channels from one: y[v][c] = act(b[c] + sum_tap w[c][tap] x[v + tap]) (the first layer) or,
// with FLIP, sum_tap w[tap][c] x[v - tap] (the input gradient of the last layer), FP32 FMAs in
// ascending order of the taps that lie in the volume. A thread computes kOneZ consecutive z of one
// (x, y): an input value serves three outputs and the weights of a tap, read from LDS for the whole
// wave, 16 kOneZ FMAs. Bound by the 432 FMAs per voxel (0.2 ms at 256^3; two, three or four waves per
// SIMD and kOneZ = 2 or 4 take the same time). With one voxel per thread, a branch per tap and the
// integer BF16 rounding it took 0.74 ms at 256^3, now 0.27 ms; the input gradient at 4 x 128^3 0.37
// -> 0.14 ms.
constexpr int kOneZ = 2;

template <bool FLIP>
struct OneIn {
  using T = uint16_t;
  static __device__ __forceinline__ float load(const T* p) { return bf2f(*p); }
};
template <>
struct OneIn<true> {
  using T = float;
  static __device__ __forceinline__ float load(const T* p) { return *p; }
};

template <bool FLIP, bool RELU>
__global__ __launch_bounds__(256) void conv_one_to_16(const void* __restrict__ xin,
                                                      const uint16_t* __restrict__ w,
                                                      const float* __restrict__ bias,
                                                      uint16_t* __restrict__ y, int D, int H,
                                                      int W, int nzc) {
  using In = OneIn<FLIP>;
  __shared__ __align__(16) float ws[27][16];
  bool finite = true;
  for (int q = threadIdx.x; q < 27 * 16; q += 256) {
    const float f = bf2f(w[q]);
    finite = finite && fabsf(f) <= 3.402823466e38f;
    if (FLIP) ws[q / 16][q % 16] = f;
    else ws[q % 27][q / 27] = f;
  }
  // a tap outside the volume is left out of the sum; its value is 0 here, so with finite weights it
  // may as well be added, and the taps need no branches
  finite = __syncthreads_and(finite);
  const long long plane = (long long)H * W;
  const long long p = (long long)blockIdx.x * 256 + threadIdx.x;
  if (p >= plane) return;
  const int n = blockIdx.y / nzc, z0 = (blockIdx.y - n * nzc) * kOneZ;
  const int yv = plane < (1ll << 31) ? (int)((uint32_t)p / (uint32_t)W) : (int)(p / W);
  const int xv = (int)(p - (long long)yv * W);
  const typename In::T* x = static_cast<const typename In::T*>(xin) + (long long)n * D * plane;
  // v[q][t]: plane z0 - 1 + q, offset t of the 3 x 3 neighbourhood; zero outside the volume (the
  // load then reads the thread's own voxel or the nearest plane)
  bool ok[9];
  float v[kOneZ + 2][9];
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const int yy = yv + t / 3 - 1, xx = xv + t % 3 - 1;
    ok[t] = yy >= 0 && yy < H && xx >= 0 && xx < W;
    const typename In::T* px = x + p + (ok[t] ? (long long)(t / 3 - 1) * W + (t % 3 - 1) : 0);
#pragma unroll
    for (int q = 0; q < kOneZ + 2; ++q) {
      const int zz = z0 - 1 + q;
      const float f = In::load(px + min(max(zz, 0), D - 1) * plane);
      v[q][t] = ok[t] && zz >= 0 && zz < D ? f : 0.0f;
    }
  }
  float acc[kOneZ][16];
#pragma unroll
  for (int r = 0; r < kOneZ; ++r)
#pragma unroll
    for (int c = 0; c < 16; ++c) acc[r][c] = bias ? bias[c] : 0.0f;
  auto taps = [&](auto tag) {
    constexpr bool CHECK = decltype(tag)::value;
#pragma unroll
    for (int tap = 0; tap < 27; ++tap) {
      const int dz = FLIP ? 2 - tap / 9 : tap / 9, t = FLIP ? 8 - tap % 9 : tap % 9;
      float wt[16];
#pragma unroll
      for (int c = 0; c < 16; ++c) wt[c] = ws[tap][c];
#pragma unroll
      for (int r = 0; r < kOneZ; ++r) {
        const int zz = z0 + r + dz - 1;
        if (CHECK && !(ok[t] && zz >= 0 && zz < D)) continue;
#pragma unroll
        for (int c = 0; c < 16; ++c) acc[r][c] = fmaf(wt[c], v[r + dz][t], acc[r][c]);
      }
    }
  };
  if (finite) taps(std::false_type{});
  else taps(std::true_type{});
#pragma unroll
  for (int r = 0; r < kOneZ; ++r) {
    if (z0 + r >= D) break;
    uint16_t* o = y + (((long long)n * D + z0 + r) * plane + p) * 16;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4_a2 q;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float f0 = acc[r][8 * h + 2 * e], f1 = acc[r][8 * h + 2 * e + 1];
        if (RELU) f0 = fmaxf(f0, 0.0f), f1 = fmaxf(f1, 0.0f);
        q[e] = pack_bf16(f0, f1);
      }
      *reinterpret_cast<u32x4_a2*>(o + 8 * h) = q;
    }
  }
}

template <bool FLIP, bool RELU>
void launch_one_to_16(const void* x, const void* w, const float* b, void* y, int N, int D, int H,
                      int W, hipStream_t s) {
  const int nzc = (D + kOneZ - 1) / kOneZ;
  const dim3 grid((unsigned)(((long long)H * W + 255) / 256), N * nzc);
  conv_one_to_16<FLIP, RELU><<<grid, 256, 0, s>>>(x, (const uint16_t*)w, b, (uint16_t*)y, D, H, W,
                                                  nzc);
}

// One FP32 channel from sixteen (the last layer): y[v] = b + sum_{tap, c} w[tap][c] x[v + tap][c], one
// chain of FMAs per voxel in ascending order over the taps that lie in the volume. A thread computes
// kOneY consecutive y of one (x, z): an input voxel is loaded and converted once per plane for the
// up to three outputs that use it, and the nine taps of a plane stay in registers (144) over the
// thread's rows; the next row's voxels are in flight meanwhile. Bound by its 432 FMAs and 216
// conversions per voxel: 0.33 ms at 256^3, 0.66 ms with one voxel per thread (every tap's weights
// from LDS and its input converted again). As an implicit GEMM with one used row it takes 0.25 ms,
// but the other order of the sums changes the loss gradient's last bits, and they the BF16
// gradients of all layers.
constexpr int kOneY = 4;

__global__ __launch_bounds__(256, 2) void conv_16_to_one(const uint16_t* __restrict__ x,
                                                         const uint16_t* __restrict__ w,
                                                         const float* __restrict__ bias,
                                                         float* __restrict__ y, int D, int H,
                                                         int W) {
  __shared__ __align__(16) float ws[27 * 16];
  for (int q = threadIdx.x; q < 27 * 16; q += 256) ws[q] = bf2f(w[q]);
  __syncthreads();
  const int hg = (H + kOneY - 1) / kOneY;
  const long long cols = (long long)hg * W;
  const long long p = (long long)blockIdx.x * 256 + threadIdx.x;
  if (p >= cols) return;
  const int yg = cols < (1ll << 31) ? (int)((uint32_t)p / (uint32_t)W) : (int)(p / W);
  const int xv = (int)(p - (long long)yg * W), y0 = yg * kOneY;
  const int n = blockIdx.y / D, z = blockIdx.y - n * D;
  const uint16_t* vol = x + (long long)n * D * H * W * 16;
  constexpr int NR = kOneY + 2;  // input rows per plane
  const bool xok[3] = {xv > 0, true, xv + 1 < W};
  u32x4 cur[3][2], nxt[3][2];
  // row j of plane z - 1 + d; voxels outside the volume read one inside (and are not used)
  auto fetch = [&](int d, int j) {
    const int zz = min(max(z - 1 + d, 0), D - 1), yy = min(max(y0 - 1 + j, 0), H - 1);
    const uint16_t* row = vol + (((long long)zz * H + yy) * W + xv) * 16;
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const u32x4_a2* q = reinterpret_cast<const u32x4_a2*>(row + (xok[t] ? (t - 1) * 16 : 0));
      nxt[t][0] = q[0];
      nxt[t][1] = q[1];
    }
  };
  float acc[kOneY];
#pragma unroll
  for (int r = 0; r < kOneY; ++r) acc[r] = bias ? bias[0] : 0.0f;
  fetch(0, 0);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    float wt[9][16];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int c = 0; c < 16; ++c) wt[t][c] = ws[(9 * d + t) * 16 + c];
    const bool zok = z - 1 + d >= 0 && z - 1 + d < D;  // uniform
#pragma unroll
    for (int j = 0; j < NR; ++j) {
#pragma unroll
      for (int t = 0; t < 3; ++t) cur[t][0] = nxt[t][0], cur[t][1] = nxt[t][1];
      if (d < 2 || j + 1 < NR) fetch(j + 1 < NR ? d : d + 1, j + 1 < NR ? j + 1 : 0);
      const int yy = y0 - 1 + j;
      if (!zok || yy < 0 || yy >= H) continue;
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        if (!xok[t]) continue;
        float f[16];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const uint32_t u = cur[t][q / 4][q % 4];
          f[2 * q] = __uint_as_float(u << 16);
          f[2 * q + 1] = __uint_as_float(u & 0xffff0000u);
        }
#pragma unroll
        for (int c = 0; c < 16; ++c)
#pragma unroll
          for (int r = 0; r < kOneY; ++r) {
            const int dy = j - r;  // output row y0 + r uses this row as its tap dy
            if (dy >= 0 && dy < 3) acc[r] = fmaf(wt[3 * dy + t][c], f[c], acc[r]);
          }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kOneY; ++r)
    if (y0 + r < H) y[(((long long)n * D + z) * H + y0 + r) * W + xv] = acc[r];
}

void launch_16_to_one(const void* x, const void* w, const float* b, float* y, int N, int D, int H,
                      int W, hipStream_t s) {
  const long long cols = (long long)((H + kOneY - 1) / kOneY) * W;
  conv_16_to_one<<<dim3((unsigned)((cols + 255) / 256), N * D), 256, 0, s>>>(
      (const uint16_t*)x, (const uint16_t*)w, b, y, D, H, W);
}

// Weight gradient of a 1-channel layer: one tensor has 16 channels per voxel ("wide", BF16), the
// other one ("narrow": the first layer's BF16 input, or with FLIP the last layer's FP32 output
// gradient). dW[tap][c] = sum over narrow voxels v of narrow[v] wide[v + shift(tap)][c], as MFMAs with
// the voxels as k: the rows of A are the narrow rows (dz, dy) around the wide row, B its 16 channels
// read transposed (as in conv_wgrad_mfma) at the three shifts along x. FP32 narrow values are split
// into three BF16 parts of eight significant bits each (their sum is exact), one row of A per part:
// the products are exact in FP32 and only the order of the sums differs from FP32 FMAs.
// A wave owns 32 narrow x voxels and walks rows y at fixed (n, z). Bound by the reading of the wide
// tensor (0.27 GB at 4 x 128^3: 0.06 ms at the rate of a large copy). Before, a block per tap read
// both tensors again: first layer 1.05 -> 0.11 ms, last layer 1.11 -> 0.07 ms there.
constexpr int kNrPitch = 80;  // bytes of 32 BF16 values, padded: rows four apart share no bank
constexpr int kNrWaves = 16;  // waves per block: few blocks keep the chain of atomic sums short

struct WgNarrowArgs {
  const uint16_t* wide;
  const void* narrow;
  float* dw;
  long long units;  // (n, z, y chunk, x segment)
  int D, H, W;
  int nseg, nyc, yc;
};

// Mask of a fragment's finite values.
__device__ __forceinline__ u32x4 finite_values(bf16x8 v) {
  const u32x4 u = __builtin_bit_cast(u32x4, v);
  u32x4 m;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    m[q] = ((u[q] & 0x7f80u) != 0x7f80u ? 0xffffu : 0u) |
           ((u[q] & 0x7f800000u) != 0x7f800000u ? 0xffff0000u : 0u);
  return m;
}

template <bool FLIP>
__global__ __launch_bounds__(64 * kNrWaves) void conv_wgrad_narrow(WgNarrowArgs a) {
  constexpr int PARTS = FLIP ? 3 : 1, ROWS = 9 * PARTS, MT = (ROWS + 15) / 16;
  constexpr int kNarrowB = 9 * PARTS * kNrPitch, kWaveB = kNarrowB + 34 * 32;
  constexpr int kRedB = kNrWaves * MT * 1024;  // one shift's accumulators
  __shared__ __align__(16) char lds[kNrWaves * kWaveB > kRedB ? kNrWaves * kWaveB : kRedB];
  __shared__ float sums[27 * 16];              // as dW lies in memory
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, g = lane >> 4;
  const long long unit = (long long)xcd_remap(blockIdx.x, gridDim.x) * kNrWaves + wave;
  f32x4 acc[MT][3];
#pragma unroll
  for (int q = 0; q < 3 * MT; ++q) acc[q / 3][q % 3] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (unit < a.units) {
    long long u = unit;
    const int x0 = (int)(u % a.nseg) * kWgSeg; u /= a.nseg;
    const int y0 = (int)(u % a.nyc) * a.yc; u /= a.nyc;
    const int z = (int)(u % a.D);
    const long long n = u / a.D;
    const int y1 = min(a.H, y0 + a.yc);
    char* nr = lds + wave * kWaveB;       // [plane z - 1 + d][row mod 3][part]
    char* wr = nr + kNarrowB;             // wide voxels x0 - 1 .. x0 + 32
    const int wv0 = x0 - 1 + (lane >> 1), wv1 = wv0 + 32;
    const bool w0ok = wv0 >= 0 && wv0 < a.W, w1ok = lane < 4 && wv1 < a.W;
    u32x4 pw0, pw1;
    float pn[2];
    auto fetch_w = [&](int yy) {
      const uint16_t* p = a.wide + ((n * a.D + z) * a.H + yy) * a.W * 16 + 8 * (lane & 1);
      pw0 = pw1 = u32x4{0u, 0u, 0u, 0u};
      if (w0ok) pw0 = *reinterpret_cast<const u32x4_a2*>(p + (long long)wv0 * 16);
      if (w1ok) pw1 = *reinterpret_cast<const u32x4_a2*>(p + (long long)wv1 * 16);
    };
    // value q of this lane: plane (lane + 64 q) / 32, voxel (lane + 64 q) % 32 of row yy
    auto fetch_n = [&](int yy) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int e = lane + 64 * q, zz = z - 1 + e / 32, xx = x0 + e % 32;
        pn[q] = 0.0f;
        if (e < 96 && zz >= 0 && zz < a.D && yy >= 0 && yy < a.H && xx < a.W) {
          const long long i = ((n * a.D + zz) * a.H + yy) * a.W + xx;
          pn[q] = FLIP ? static_cast<const float*>(a.narrow)[i]
                       : bf2f(static_cast<const uint16_t*>(a.narrow)[i]);
        }
      }
    };
    auto put_n = [&](int slot) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int e = lane + 64 * q;
        if (e >= 96) continue;
        uint16_t* o = reinterpret_cast<uint16_t*>(nr + ((e / 32 * 3 + slot) * PARTS) * kNrPitch) +
                      e % 32;
        uint32_t b = __float_as_uint(pn[q]);
        if constexpr (FLIP) {
          // parts by truncation; an infinite value has no further parts, a NaN stays one
          const bool fin = (b & 0x7f800000u) != 0x7f800000u;
          if ((b & 0x7fffffffu) > 0x7f800000u) b |= 0x400000u;
          const float r1 = fin ? pn[q] - __uint_as_float(b & 0xffff0000u) : 0.0f;
          const uint32_t b1 = __float_as_uint(r1) & 0xffff0000u;
          const float r2 = r1 - __uint_as_float(b1);
          o[kNrPitch / 2] = (uint16_t)(b1 >> 16);
          o[kNrPitch] = (uint16_t)(__float_as_uint(r2) >> 16);
        }
        o[0] = (uint16_t)(b >> 16);
      }
    };
    // A row m of tile i is row j = 16 i + m: part j / 9 of the narrow row (dz, dy) = j % 9. Its
    // address when rows y - 1, y, y + 1 are in slots r, r + 1, r + 2 mod 3; rows past the last are
    // not used and repeat the first
    int arow[MT][3];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int j = 16 * i + m < ROWS ? 16 * i + m : 0;
      const int part = j / 9, d = j % 9;
      const int zi = FLIP ? 2 - d / 3 : d / 3, yi = FLIP ? 2 - d % 3 : d % 3;
#pragma unroll
      for (int r = 0; r < 3; ++r)
        arow[i][r] = ((zi * 3 + (r + yi) % 3) * PARTS + part) * kNrPitch + 16 * g;
    }
    fetch_n(y0 - 1);
    put_n(0);
    fetch_n(y0);
    put_n(1);
    fetch_n(y0 + 1);
    fetch_w(y0);
    for (int y = y0; y < y1;) {
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        if (y >= y1) break;
        put_n((r + 2) % 3);
        *reinterpret_cast<u32x4*>(wr + lane * 16) = pw0;
        if (lane < 4) *reinterpret_cast<u32x4*>(wr + (64 + lane) * 16) = pw1;
        wave_sync();
        if (y + 1 < y1) {
          fetch_n(y + 2);
          fetch_w(y + 1);
        }
        bf16x8 B[3];
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) B[dx] = read_channel(wr + (FLIP ? dx : 2 - dx) * 32, lane);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const bf16x8 A =
              __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(nr + arow[i][r]));
#pragma unroll
          for (int dx = 0; dx < 3; ++dx)
            acc[i][dx] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B[dx], acc[i][dx], 0, 0, 0);
        }
        wave_sync();
        ++y;
      }
    }
    // As in conv_wgrad_mfma. A narrow row outside the volume is a row of A, so its products are left out
    // of the sums instead, and an infinite wide value is multiplied by a narrow value's first part only
    // (the others may be zero where the value is not).
    float sum = 0.0f;
#pragma unroll
    for (int q = 0; q < MT * 12; ++q) sum += 0.0f * acc[q / 12][q / 4 % 3][q % 4];
    if (__any(sum != 0.0f)) {
#pragma unroll
      for (int q = 0; q < 3 * MT; ++q) acc[q / 3][q % 3] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int y = y0; y < y1; ++y) {
#pragma unroll
        for (int r = 0; r < 3; ++r) {
          fetch_n(y + r - 1);
          put_n(r);
        }
        fetch_w(y);
        *reinterpret_cast<u32x4*>(wr + lane * 16) = pw0;
        if (lane < 4) *reinterpret_cast<u32x4*>(wr + (64 + lane) * 16) = pw1;
        wave_sync();
#pragma unroll
        for (int q = 0; q < 3 * MT; ++q) {
          const int dx = q / MT, i = q % MT;
          int xs = x0 + 8 * g;
          asm volatile("" : "+v"(xs));  // a mask at a time in registers
          const u32x4 in = pairs_inside(xs, FLIP ? dx - 1 : 1 - dx, a.W);
          const bf16x8 A =
              masked(__builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(nr + arow[i][0])), in);
          const bf16x8 B = masked(read_channel(wr + (FLIP ? dx : 2 - dx) * 32, lane), in);
          const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
          const f32x4 all = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B, zero, 0, 0, 0);
          const f32x4 fin = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, masked(B, finite_values(B)),
                                                                    zero, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = 16 * i + 4 * g + e, d = j % 9;
            const int zz = z + (FLIP ? 1 - d / 3 : d / 3 - 1),
                      yy = y + (FLIP ? 1 - d % 3 : d % 3 - 1);
            if (zz >= 0 && zz < a.D && yy >= 0 && yy < a.H) acc[i][dx][e] += j < 9 ? all[e] : fin[e];
          }
        }
        wave_sync();
      }
    }
  }
  // sum over the block's waves and the parts, one shift at a time: part[wave][row][channel]
  float* part = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int dx = 0; dx < 3; ++dx) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        part[((wave * MT + i) * 16 + 4 * g + r) * 16 + m] = acc[i][dx][r];
    __syncthreads();
    if (threadIdx.x < 9 * 16) {
      const int d = threadIdx.x / 16, c = threadIdx.x % 16;
      float v = 0.0f;
#pragma unroll
      for (int q = 0; q < PARTS; ++q)
#pragma unroll
        for (int k = 0; k < kNrWaves; ++k) v += part[(k * MT * 16 + q * 9 + d) * 16 + c];
      const int tap = 3 * d + dx;
      sums[FLIP ? tap * 16 + c : c * 27 + tap] = v;
    }
  }
  __syncthreads();
  if (threadIdx.x < 27 * 16) unsafeAtomicAdd(a.dw + threadIdx.x, sums[threadIdx.x]);
}

template <bool FLIP>
void launch_wgrad_narrow(const void* wide, const void* narrow, float* dw, int N, int D, int H,
                         int W, hipStream_t s) {
  WgNarrowArgs a;
  a.wide = (const uint16_t*)wide;
  a.narrow = narrow;
  a.dw = dw;
  a.D = D; a.H = H; a.W = W;
  a.nseg = (W + kWgSeg - 1) / kWgSeg;
  // about 4096 waves (a block of 16 per CU), at least sixteen rows each
  const long long columns = (long long)N * D * a.nseg;
  const int want = (int)std::min<long long>((H + 15) / 16, (4096 + columns - 1) / columns);
  a.yc = (H + want - 1) / want;
  a.nyc = (H + a.yc - 1) / a.yc;
  a.units = columns * a.nyc;
  conv_wgrad_narrow<FLIP>
      <<<(unsigned)((a.units + kNrWaves - 1) / kNrWaves), 64 * kNrWaves, 0, s>>>(a);
}

// MFMA lane-layout probe: D = A B for one 16x16x32 BF16 and one 16x16x4 FP32 product, with
// A and B given row-major; a single wave, every access in bounds.
__global__ __launch_bounds__(64) void mfma_probe(const uint16_t* __restrict__ A32,
                                                 const uint16_t* __restrict__ B32,
                                                 const float* __restrict__ A4,
                                                 const float* __restrict__ B4,
                                                 float* __restrict__ D32, float* __restrict__ D4) {
  const int l = threadIdx.x, m = l & 15, g = l >> 4;
  bf16x8 a, b;
  uint16_t* pa = reinterpret_cast<uint16_t*>(&a);
  uint16_t* pb = reinterpret_cast<uint16_t*>(&b);
  for (int q = 0; q < 8; ++q) {
    pa[q] = A32[m * 32 + g * 8 + q];   // A[16][32] row-major
    pb[q] = B32[(g * 8 + q) * 16 + m]; // B[32][16] row-major
  }
  f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  f32x4 e = __builtin_amdgcn_mfma_f32_16x16x4f32(A4[m * 4 + g], B4[g * 16 + m],
                                                  f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  for (int r = 0; r < 4; ++r) {
    D32[(g * 4 + r) * 16 + m] = d[r];
    D4[(g * 4 + r) * 16 + m] = e[r];
  }
}

template <int CIN, int COUT, bool UPCAT>
void launch_fwd_t(const void* x, const void* skip, const void* w, const float* b, void* y, int N,
                  int D, int H, int W, int relu, hipStream_t s) {
  const auto run = [&](auto tile, auto with_relu, auto without, int blocks, int zmin) {
    using T = decltype(tile);
    const int tx = (W + T::XT - 1) / T::XT, ty = (H + T::YT - 1) / T::YT;
    const long long tiles = (long long)tx * ty * N;
    const int zc = (int)std::max((long long)zmin, std::min(32LL, tiles * D / blocks));
    const int nzc = (D + zc - 1) / zc;
    (relu ? with_relu : without)<<<(unsigned)(tiles * nzc), 256, 0, s>>>(
        (const uint16_t*)x, (const uint16_t*)skip, (const uint16_t*)w, b, (uint16_t*)y, D, H, W, tx,
        ty, zc, nzc);
  };
  // conv_fwd_stream wants its 512 resident blocks (two per CU) and at least two planes per block (the
  // two halo planes are loaded besides): below 512 tile planes the smaller tiles of conv_fwd_mfma are
  // faster (us, before / stream): 96 -> 32 at 32^3 (256 tile planes) 18 / 32, 32 -> 32 at 48^3 (432)
  // 18 / 16, 64 -> 32 at 4 x 32^3 (512) 55 / 37, 64 -> 64 at 40^3 (600) 78 / 55; for 16 output channels
  // always (32 -> 16 at 128^3 64 / 86).
  if constexpr (CIN % 32 == 0 && (COUT == 32 || COUT == 64)) {
    using T = StreamTile<CIN, COUT>;
    const long long planes =
        (long long)((W + T::XT - 1) / T::XT) * ((H + T::YT - 1) / T::YT) * N * D;
    if (planes >= 512) {
      run(T(), conv_fwd_stream<CIN, COUT, true, UPCAT>, conv_fwd_stream<CIN, COUT, false, UPCAT>, 512,
          2);
      return;
    }
  }
  // planes per block: as many as leave about 2048 blocks (eight per CU), at most 32 (the two halo
  // planes are then 6 % of the planes loaded)
  run(ConvTile<CIN, COUT>(), conv_fwd_mfma<CIN, COUT, true, UPCAT>,
      conv_fwd_mfma<CIN, COUT, false, UPCAT>, 2048, 1);
}

// Supported (Cin, Cout) pairs of the MFMA kernels: the network's layers and their transposes.
bool launch_fwd(int cin, int cout, const void* x, const void* w, const float* b, void* y, int N,
                int D, int H, int W, int relu, hipStream_t s) {
#define FC_CONV_CASE(ci, co) \
  if (cin == ci && cout == co) {                                                     \
    launch_fwd_t<ci, co, false>(x, nullptr, w, b, y, N, D, H, W, relu, s);           \
    return true;                                                                     \
  }
  FC_CONV_CASE(16, 16) FC_CONV_CASE(16, 32) FC_CONV_CASE(32, 32) FC_CONV_CASE(32, 64)
  FC_CONV_CASE(64, 64) FC_CONV_CASE(96, 32) FC_CONV_CASE(48, 16) FC_CONV_CASE(32, 16)
  FC_CONV_CASE(64, 32) FC_CONV_CASE(32, 96) FC_CONV_CASE(16, 48)
#undef FC_CONV_CASE
  return false;
}

bool launch_wgrad(int cin, int cout, const void* x, const void* dy, float* dw, int N, int D,
                  int H, int W, hipStream_t s, const void* skip = nullptr, int ca = 0) {
  bool known = false;  // the network's layers
  for (const auto& p : {std::pair<int, int>{16, 16}, {16, 32}, {32, 32}, {32, 64}, {64, 64},
                        {96, 32}, {48, 16}})
    known = known || (p.first == cin && p.second == cout);
  if (!known) return false;
  WgArgs a;
  a.x = (const uint16_t*)x;
  a.skip = (const uint16_t*)skip;
  a.ca = ca;
  a.dy = (const uint16_t*)dy;
  a.dw = dw;
  a.D = D; a.H = H; a.W = W; a.cin = cin; a.cout = cout;
  a.nseg = (W + kWgSeg - 1) / kWgSeg;
  // about 4096 waves (two rounds of two per SIMD), at least eight rows each: a wave's first two
  // input rows and its share of the final sum are then a small part
  const int combos = cin / 16 * (cout / 16);
  const long long columns = (long long)N * D * a.nseg * combos;
  const int want = (int)std::min<long long>((H + 7) / 8, (4096 + columns - 1) / columns);
  a.yc = (H + want - 1) / want;
  a.nyc = (H + a.yc - 1) / a.yc;
  a.units = (long long)N * D * a.nseg * a.nyc;
  const long long blocks = (a.units + 3) / 4 * combos;
  conv_wgrad_mfma<<<(unsigned)blocks, 256, 0, s>>>(a);
  return true;
}

}  // namespace
}  // namespace fc

using namespace fc;

extern "C" {

int fc_conv3d_fwd_dev(int device, const void* x, const void* w, const float* bias, void* y,
                      int N, int D, int H, int W, int cin, int cout, int relu, void* stream) {
  clear_error();
  FC_CHECK_ARG(x && w && y, "null pointer argument");
  FC_CHECK_ARG(N > 0 && D > 0 && H > 0 && W > 0 && H <= 65535 && (long)N * D <= 65535,
               "bad activation shape");
  int rc = select_device(device);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int tok = prof_begin("conv3d_fwd", s);
  if (cin == 1 && cout == 16) {
    if (relu) launch_one_to_16<false, true>(x, w, bias, y, N, D, H, W, s);
    else launch_one_to_16<false, false>(x, w, bias, y, N, D, H, W, s);
  } else if (cout == 1 && cin == 16) {
    FC_CHECK_ARG(!relu, "the Cout = 1 layer has no activation and writes FP32");
    launch_16_to_one(x, w, bias, (float*)y, N, D, H, W, s);
  } else if (!launch_fwd(cin, cout, x, w, bias, y, N, D, H, W, relu, s)) {
    prof_end(tok, s);
    FC_CHECK_ARG(false, "unsupported channel pair %d -> %d", cin, cout);
  }
  prof_end(tok, s);
  FC_HIP(hipGetLastError());
  return FC_OK;
}

int fc_net_up_cat_conv_dev(int device, const void* a, const void* b, const void* w,
                           const float* bias, void* y, int N, int D, int H, int W, int ca, int cb,
                           int cout, int relu, void* stream) {
  clear_error();
  FC_CHECK_ARG(a && b && w && y, "null pointer argument");
  FC_CHECK_ARG(N > 0 && D > 0 && H > 0 && W > 0 && H <= 65535 && (long)N * D <= 65535,
               "bad activation shape");
  FC_CHECK_ARG(D % 2 == 0 && H % 2 == 0 && W % 2 == 0, "sides must be even");
  FC_CHECK_ARG((long long)H * W * (ca > cb ? ca : cb) < (1ll << 31), "plane too large");
  int rc = select_device(device);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int tok = prof_begin("conv3d_fwd", s);
  if (ca == 64 && cb == 32 && cout == 32) {
    launch_fwd_t<96, 32, true>(a, b, w, bias, y, N, D, H, W, relu, s);
  } else if (ca == 32 && cb == 16 && cout == 16) {
    launch_fwd_t<48, 16, true>(a, b, w, bias, y, N, D, H, W, relu, s);
  } else {
    prof_end(tok, s);
    FC_CHECK_ARG(false, "unsupported channel counts %d + %d -> %d", ca, cb, cout);
  }
  prof_end(tok, s);
  FC_HIP(hipGetLastError());
  return FC_OK;
}

// dx = conv^T(dy): workspace wt (cin*27*cout BF16) receives the flipped transposed weights.
int fc_conv3d_dgrad_dev(int device, const void* dy, const void* w, void* wt, void* dx, int N,
                        int D, int H, int W, int cin, int cout, void* stream) {
  clear_error();
  FC_CHECK_ARG(dy && w && dx, "null pointer argument");
  FC_CHECK_ARG(N > 0 && D > 0 && H > 0 && W > 0 && H <= 65535 && (long)N * D <= 65535,
               "bad activation shape");
  int rc = select_device(device);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int tok = prof_begin("conv3d_dgrad", s);
  if (cout == 1 && cin == 16) {
    launch_one_to_16<true, false>(dy, w, nullptr, dx, N, D, H, W, s);
  } else {
    FC_CHECK_ARG(wt, "null weight workspace");
    const int total = cout * 27 * cin;
    flip_transpose_weights<<<(total + 255) / 256, 256, 0, s>>>((const uint16_t*)w,
                                                              (uint16_t*)wt, cin, cout);
    if (!launch_fwd(cout, cin, dy, wt, nullptr, dx, N, D, H, W, 0, s)) {
      prof_end(tok, s);
      FC_CHECK_ARG(false, "unsupported channel pair %d -> %d", cin, cout);
    }
  }
  prof_end(tok, s);
  FC_HIP(hipGetLastError());
  return FC_OK;
}

// dw (FP32 [cout][27][cin]) += sum over voxels of dy x patch.
int fc_conv3d_wgrad_dev(int device, const void* x, const void* dy, float* dw, int N, int D, int H,
                        int W, int cin, int cout, void* stream) {
  clear_error();
  FC_CHECK_ARG(x && dy && dw, "null pointer argument");
  FC_CHECK_ARG(N > 0 && D > 0 && H > 0 && W > 0, "bad activation shape");
  int rc = select_device(device);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int tok = prof_begin("conv3d_wgrad", s);
  if (cin == 1 && cout == 16) {
    launch_wgrad_narrow<false>(dy, x, dw, N, D, H, W, s);
  } else if (cout == 1 && cin == 16) {
    launch_wgrad_narrow<true>(x, dy, dw, N, D, H, W, s);
  } else if (!launch_wgrad(cin, cout, x, dy, dw, N, D, H, W, s)) {
    prof_end(tok, s);
    FC_CHECK_ARG(false, "unsupported channel pair %d -> %d", cin, cout);
  }
  prof_end(tok, s);
  FC_HIP(hipGetLastError());
  return FC_OK;
}

int fc_net_up_cat_wgrad_dev(int device, const void* a, const void* b, const void* dy, float* dw,
                            int N, int D, int H, int W, int ca, int cb, int cout, void* stream) {
  clear_error();
  FC_CHECK_ARG(a && b && dy && dw, "null pointer argument");
  FC_CHECK_ARG(N > 0 && D > 0 && H > 0 && W > 0, "bad activation shape");
  FC_CHECK_ARG(D % 2 == 0 && H % 2 == 0 && W % 2 == 0, "sides must be even");
  FC_CHECK_ARG((ca == 64 && cb == 32 && cout == 32) || (ca == 32 && cb == 16 && cout == 16),
               "unsupported channel counts %d + %d -> %d", ca, cb, cout);
  int rc = select_device(device);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int tok = prof_begin("conv3d_wgrad", s);
  launch_wgrad(ca + cb, cout, a, dy, dw, N, D, H, W, s, b, ca);
  prof_end(tok, s);
  FC_HIP(hipGetLastError());
  return FC_OK;
}

int fc_mfma_layout_probe(int device, const void* A32, const void* B32, const float* A4,
                         const float* B4, float* D32, float* D4, void* stream) {
  clear_error();
  FC_CHECK_ARG(A32 && B32 && A4 && B4 && D32 && D4, "null pointer argument");
  int rc = select_device(device);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  mfma_probe<<<1, 64, 0, s>>>((const uint16_t*)A32, (const uint16_t*)B32, A4, B4, D32, D4);
  FC_HIP(hipGetLastError());
  return FC_OK;
}

}  // extern "C"
