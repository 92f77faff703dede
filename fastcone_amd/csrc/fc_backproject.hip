// Voxel-driven backprojectors for gfx950: FDK (weight U^2), Katsevich (U^1) and unweighted
// general geometry (mode 0), coneBeamGPU.cu:178-420.
//
//   vol(x) += sum_t norm_t * w_t(x) * B_t(a/c, b/c),   (a, b, c) = M_t (x, 1)
//
// M_t is the view's FP64 3x4 projective matrix (built on the host from the source / detector
// vectors). For the reference's circular/helical geometry a/c and 1/c reproduce
// w = (y cos - x sin) U / pw and U = D / (D + x cos + y sin) of coneBeamGPU.cu:398-399, and the
// mode-0 ray/plane intersection of coneBeamGPU.cu:235-243 in closed form. B_t is the bilinear
// interpolant of window t extended by zeros; the per-view norm multiplies the data at staging,
// as the reference's fillCache does (coneBeamGPU.cu:1081).
//
// Work decomposition: one thread owns a column (x, y) and ZR = 16 consecutive z voxels, held in
// registers over every view ("wavefront-level accumulation over views"); a block owns a
// 16 x 16 x 16 voxel cube. Per view the block stages, in LDS, the detector window that the cube
// projects onto (rows of the raw projection, zero outside the detector), double-buffered: while
// the block accumulates view t from one buffer, the rows of view t+1 are already in flight (FP32
// storage: copied straight into the other buffer, 16 bytes per lane; 16-bit storage: into registers,
// converted and written to the other buffer at the top of the next iteration), so one barrier per
// view suffices and the load latency hides behind the arithmetic. Per view and column the projective
// terms are a few FMAs on the view's table entry (below); when the detector columns do not depend on
// z (untilted detectors) each voxel then costs one FMA for its row and a bilinear interpolation from
// LDS (two ds_read2 pairs, one multiply-add for the address).
//
// View table: every kTab views the block computes, eight threads per view and in FP64, the window of its
// cube — the projective image of a box lies in the box of its eight corners' images, so the corners'
// (u, v) widened by a pixel each side bound every tap — and the view's projective forms relative to
// the window's and the cube's corners, A' = (A - u0 C) / Cm, B' = (B - v0 C) / Cm and q = C / Cm - 1 as
// linear functions of the offset in the cube, Cm being the largest C of its lowest plane. There they
// are small (|A'| < 64, -1 < q <= 0), so rounding them to FP32 moves a tile coordinate by 1.1e-6 pixel
// (rms; FP64 terms rounded to an absolute coordinate 7e-6), and Cm / C = 1 - q / (1 + q) and the weight
// have the error of their last rounding (weight 3.6e-8 of it, rms, as from FP64 terms; the square of an
// FP32 reciprocal of C 1.1e-7). A view whose window does not fit the LDS tile (pixels below about a
// third of a voxel, very short source distances) is gathered from global memory with explicit bounds,
// after the views that fit; a view that misses the detector entirely is skipped.
//
// Small volumes leave compute units idle or the last round of blocks nearly empty: the views are
// then split over several blocks per cube, whose sums go to partial volumes that bp_reduce adds in
// order (launch_backproject).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "fc_device.h"
#include "fc_internal.h"

namespace fc {
namespace {

constexpr int kZR = 16;   // z voxels per thread
constexpr int kBXY = 16;  // 16x16 columns per 256-thread block (8x8 per wave)

constexpr int kTileW = 64;                 // widest staged window
constexpr int kTileH = 48;                 // tallest staged window
// Row pitch of a staged window (floats): fixed, so a bilinear sample's two row pairs are one
// base address with immediate offsets {0, 1, kTileP, kTileP + 1}. 76 = 12 mod 32 banks: timed at
// 512^3 x 720 against pitches 65-80, it leaves the fewest bank conflicts between the lanes' rows
// (65: 51.5 ms, 68: 49.9, 70: 48.6, 72: 48.2, 74-78: 47.7, 80: 48.0). It is also 19 units of 16
// bytes, the load-to-LDS copy's unit per lane.
constexpr uint32_t kTileP = 76;
constexpr uint32_t kUnits = kTileP / 4;    // 16-byte units per row
constexpr int kTileCap = kTileP * kTileH;  // floats per LDS buffer (14.3 KiB)
constexpr int kRowsW = 64 / (int)kUnits;   // rows per wave and copy instruction (57 lanes)
constexpr int kRowsB = 4 * kRowsW;         // and per block
constexpr int kCopies = kTileH / kRowsB;   // copies per thread of the tallest window
static_assert(kTileH % kRowsB == 0, "whole copies");
constexpr uint32_t kWinSkip = 0u;          // window word y: the cube misses the detector
constexpr uint32_t kWinGlobal = 0xffffu;   // window word y low half: gather from global memory
constexpr int kTab = 48;                   // views per table: five blocks fit a CU's LDS

struct BpArgs {
  float* vol;          // accumulated; with nsplit > 1 the partial volumes, one per split, stored
  const void* proj;    // [nviews][nh][nw] in the storage dtype
  const float* norm;   // per-view scale or null
  const double* views;
  double ox, oy, oz;
  int nx, ny, nz;
  int nw, nh, nviews;
  int nbz, nsplit;
};

// One view for one cube: with (dx, dy, dz) a voxel's offset from the cube's first voxel,
// A' = a0 + a1 dx + a2 dy + a3 dz, likewise B' and q; u - u0 = A' / (1 + q), v - v0 = B' / (1 + q). For
// tilted detectors q stands for 1 + q.
struct ViewEntry {
  float a[4], b[4], q[4];
  float s;       // norm times the mode's weight at q = 0
  uint32_t org;  // window origin u0 | v0 << 16 (int16 each)
  uint32_t size; // Wu | Wv << 16, or kWinSkip / kWinGlobal
  uint32_t tilted;  // a3 or c3 nonzero
};

// Entries of the views [t0, t0 + n) for the cube at (x0, y0, z0), eight lanes of a block's threads per
// view: each projects a corner of the cube, and four of them form the constants and slopes.
// Window pixels [u0, u0 + Wu) x [v0, v0 + Wv) with u0 = floor(min u) - 1 and Wu = floor(max u) - u0
// + 3, so every tap (iu, iu + 1) of a voxel in the cube lies at least one pixel inside; likewise v.
template <int MODE>
__device__ __forceinline__ void view_table(const BpArgs& a, ViewEntry* tab, int t0, int n, int x0,
                                           int y0, int z0) {
  int c = threadIdx.x & 7;
  asm volatile("" : "+v"(c), "+s"(x0), "+s"(y0), "+s"(z0));  // nothing of this stays in registers
  const double X0 = x0 + a.ox, Y0 = y0 + a.oy, Z0 = z0 + a.oz;
  const double ex = min(kBXY - 1, a.nx - 1 - x0), ey = min(kBXY - 1, a.ny - 1 - y0),
               ez = min(kZR - 1, a.nz - 1 - z0);
#pragma unroll 1
  for (int i = threadIdx.x >> 3; i < n; i += 32) {
    const double* M = a.views + (size_t)(t0 + i) * FC_VIEW_DOUBLES + 12;
    // the matrix is reread where it is used: held in registers, it would spill the block's accumulators
    auto form = [&](int r, double x, double y, double z) {
      asm volatile("" : "+v"(M));
      return M[4 * r] * x + M[4 * r + 1] * y + M[4 * r + 2] * z + M[4 * r + 3];
    };
    const double X = X0 + (c & 1 ? ex : 0.0), Y = Y0 + (c & 2 ? ey : 0.0), Z = Z0 + (c & 4 ? ez : 0.0);
    const double C = form(2, X, Y, Z), rc = 1.0 / C;
    int ok = C > 0.0;
    // least and greatest whole pixel of the corners in one direction; ok: within the integers' reach
    // and, if the detector's n pixels are nowhere near, hit = false
    bool hit = true;
    int lo[2], hi[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      double least = form(d, X, Y, Z) * rc, most = least;
#pragma unroll
      for (int m = 1; m < 8; m <<= 1) {
        least = fmin(least, __shfl_xor(least, m));
        most = fmax(most, __shfl_xor(most, m));
      }
      ok &= least > -1e6 && most < 1e6;
      hit = hit && !(most <= -1.0 || least >= (double)(d ? a.nh : a.nw));
      lo[d] = (int)floor(fmax(least, -1e6));
      hi[d] = (int)floor(fmin(most, 1e6));
    }
#pragma unroll
    for (int m = 1; m < 8; m <<= 1) ok &= __shfl_xor(ok, m);
    uint32_t org = 0u, size = kWinGlobal;
    int u0 = 0, v0 = 0;
    if (ok && !hit) {
      size = kWinSkip;  // zero-extended data: every sample of the cube is 0
    } else if (ok) {
      u0 = lo[0] - 1;
      v0 = lo[1] - 1;
      const int Wu = hi[0] - u0 + 3, Wv = hi[1] - v0 + 3;
      if (Wu <= kTileW && Wv <= kTileH && u0 >= -32768 && u0 <= 32767 && v0 >= -32768 && v0 <= 32767) {
        org = ((uint32_t)u0 & 0xffffu) | ((uint32_t)v0 << 16);
        size = (uint32_t)Wu | ((uint32_t)Wv << 16);
      }
    }
    asm volatile("" : "+v"(M));
    const bool tilted = M[2] != 0.0 || M[10] != 0.0;
    const double C0 = form(2, X0, Y0, Z0);
    const double Cm = C0 + fmax(M[8], 0.0) * ex + fmax(M[9], 0.0) * ey, rm = 1.0 / Cm;
    ViewEntry& e = tab[i];
    if (c < 4) {
      const double fa = c ? M[c - 1] : form(0, X0, Y0, Z0), fb = c ? M[c + 3] : form(1, X0, Y0, Z0),
                   fc = c ? M[c + 7] : C0;
      e.a[c] = (float)((fa - u0 * fc) * rm);
      e.b[c] = (float)((fb - v0 * fc) * rm);
      e.q[c] = (float)((c || tilted ? fc : C0 - Cm) * rm);
    } else if (c == 4) {
      const double s = a.norm ? a.norm[t0 + i] : 1.0f;
      e.s = (float)(MODE == FC_BP_FDK ? s * rm * rm : MODE == FC_BP_KATSEVICH ? s * rm : s);
      e.org = org;
      e.size = size;
      e.tilted = tilted;
    }
  }
}

// Zero-extended bilinear samples of one view straight from global memory, for windows that do not fit
// the LDS tile: acc[k] += the weighted sample at (af + k da, bf + k db) / (cf + k dc). kG samples'
// loads are in flight; taps off the detector load the nearest pixel on it and count as zero, so no
// load waits for a branch. Bound by the loads (four of an element per sample and lane). 256^3 voxels,
// 720 views of 768^2 pixels of 0.375 voxel (94 % of the cubes' views), FP32 / BF16: 24.9 / 24.6 ms;
// with branches around the loads 24.8 / 36.9 for sixteen samples in flight and 32.8 / 49.9 for one,
// in the loop over the views, where more registers are not to be had. In the kernel's second pass
// over the views four groups of four fit beside the sums.
template <int DT, int MODE>
__device__ __forceinline__ void global_samples(float* acc, const BpArgs& a, size_t vbase, float af,
                                               float bf, float cf, float da, float db, float dc,
                                               float s) {
  constexpr int kG = 4;
#pragma unroll
  for (int k0 = 0; k0 < kZR; k0 += kG) {
    // one group's positions, loads and sums at a time in registers
    asm volatile("" : "+v"(af), "+v"(bf), "+v"(cf));
    float p[kG][4], au[kG], av[kG], wt[kG];
#pragma unroll
    for (int g = 0; g < kG; ++g) {
      const float kf = (float)(k0 + g);
      const float rc = 1.0f / fmaf(kf, dc, cf);
      const float u = fmaf(kf, da, af) * rc, v = fmaf(kf, db, bf) * rc;
      wt[g] = s;
      if constexpr (MODE == FC_BP_FDK) wt[g] = s * rc * rc;
      if constexpr (MODE == FC_BP_KATSEVICH) wt[g] = s * rc;
      const bool on = u > -1.0f && u < (float)a.nw && v > -1.0f && v < (float)a.nh;
      // off the detector u and v may be anything, infinite or NaN on the source's plane: bounded
      // before they become integers
      const float fu = fminf(fmaxf(floorf(u), -1.0f), (float)a.nw);
      const float fv = fminf(fmaxf(floorf(v), -1.0f), (float)a.nh);
      au[g] = u - fu, av[g] = v - fv;
      const int iu = (int)fu, iv = (int)fv;
      const int c0 = min(max(iu, 0), a.nw - 1), c1 = min(iu + 1, a.nw - 1);
      const size_t r0 = vbase + (size_t)min(max(iv, 0), a.nh - 1) * a.nw;
      const size_t r1 = vbase + (size_t)min(iv + 1, a.nh - 1) * a.nw;
      const bool x0 = on && iu >= 0, x1 = on && iu + 1 < a.nw, y0 = iv >= 0, y1 = iv + 1 < a.nh;
      p[g][0] = load_elem<DT>(a.proj, r0 + c0);
      p[g][1] = load_elem<DT>(a.proj, r0 + c1);
      p[g][2] = load_elem<DT>(a.proj, r1 + c0);
      p[g][3] = load_elem<DT>(a.proj, r1 + c1);
      p[g][0] = x0 && y0 ? p[g][0] : 0.0f;
      p[g][1] = x1 && y0 ? p[g][1] : 0.0f;
      p[g][2] = x0 && y1 ? p[g][2] : 0.0f;
      p[g][3] = x1 && y1 ? p[g][3] : 0.0f;
      if (!on) au[g] = av[g] = 0.0f;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < kG; ++g)
      acc[k0 + g] = fmaf(wt[g], lerp(lerp(p[g][0], p[g][1], au[g]), lerp(p[g][2], p[g][3], au[g]), av[g]),
                         acc[k0 + g]);
#pragma unroll
    for (int g = 0; g < kG; ++g) asm volatile("" : "+v"(acc[k0 + g]));
  }
}

// The views of [tbeg, tend) whose windows do not fit the LDS tile, for a whole block, after the others.
template <int DT, int MODE>
__device__ __forceinline__ void gather_views(float* acc, const BpArgs& a, ViewEntry* tab, int tbeg,
                                             int tend, int x, int y, int z0, int bx0, int by0) {
  const double X = (double)x + a.ox, Y = (double)y + a.oy, Z0 = (double)z0 + a.oz;
  for (int tb = tbeg; tb < tend; tb += kTab) {
    const int n = min(kTab, tend - tb);
    __syncthreads();  // the previous table is no longer read
    view_table<MODE>(a, tab, tb, n, bx0, by0, z0);
    __syncthreads();
    for (int i = 0; i < n; ++i) {
      if ((__builtin_amdgcn_readfirstlane(tab[i].size) & 0xffffu) != kWinGlobal) continue;
      const int t = tb + i;
      const double* M = a.views + (size_t)t * FC_VIEW_DOUBLES + 12;
      global_samples<DT, MODE>(acc, a, (size_t)t * a.nh * a.nw,
                               (float)(M[0] * X + M[1] * Y + M[2] * Z0 + M[3]),
                               (float)(M[4] * X + M[5] * Y + M[6] * Z0 + M[7]),
                               (float)(M[8] * X + M[9] * Y + M[10] * Z0 + M[11]), (float)M[2],
                               (float)M[6], (float)M[10], a.norm ? a.norm[t] : 1.0f);
    }
  }
}

// Clamp to [lo, hi], one instruction; NaN maps to lo (the median of a NaN and two numbers is the
// smaller number).
__device__ __forceinline__ float clampf(float v, float lo, float hi) {
  return __builtin_amdgcn_fmed3f(v, lo, hi);
}

// LDS byte address of a pointer into a __shared__ array.
__device__ __forceinline__ uint32_t lds_address(const void* p) { return (uint32_t)(size_t)p; }

// Bilinear sample of an LDS window (row pitch kTileP) at row coordinate v >= 0 and fraction au of
// the column at LDS byte address `col` (row 0).
__device__ __forceinline__ float tile_bilinear(uint32_t col, float au, float v) {
  typedef __attribute__((address_space(3))) const float* lds_p;
  const float av = __builtin_amdgcn_fractf(v);
  const lds_p p = (lds_p)mad_u24((uint32_t)(int)v, 4u * kTileP, col);
  return lerp(lerp(p[0], p[1], au), lerp(p[kTileP], p[kTileP + 1], au), av);
}

// acc[k] += wt times the bilinear sample at row vb + kz[k] dv of the column at LDS byte address `col`.
// Two samples' reads are issued before the previous two are used.
__device__ __forceinline__ void column_samples(float* acc, const float* kz, uint32_t col, float au,
                                               float vb, float dv, float wt) {
  typedef __attribute__((address_space(3))) const float* lds_p;
  constexpr int kG = 2;
  float p[2][kG][4], av[2][kG];
  auto read = [&](int g) {
#pragma unroll
    for (int q = 0; q < kG; ++q) {
      const float v = fmaf(kz[g * kG + q], dv, vb);
      av[g & 1][q] = __builtin_amdgcn_fractf(v);
      const lds_p a = (lds_p)mad_u24((uint32_t)(int)v, 4u * kTileP, col);
      p[g & 1][q][0] = a[0];
      p[g & 1][q][1] = a[1];
      p[g & 1][q][2] = a[kTileP];
      p[g & 1][q][3] = a[kTileP + 1];
    }
  };
  read(0);
#pragma unroll
  for (int g = 0; g < kZR / kG; ++g) {
    if (g + 1 < kZR / kG) read(g + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < kG; ++q) {
      const float* r = p[g & 1][q];
      acc[g * kG + q] = fmaf(wt, lerp(lerp(r[0], r[1], au), lerp(r[2], r[3], au), av[g & 1][q]),
                             acc[g * kG + q]);
    }
  }
}

// The same for a tilted detector: column, row and weight by voxel, from the view's forms at the
// column's first voxel.
template <int MODE>
__device__ __forceinline__ void tilted_samples(float* acc, const float* kz, uint32_t T0, float A,
                                               float B, float C, const ViewEntry& E) {
#pragma unroll
  for (int k = 0; k < kZR; ++k) {
    if (k % 2 == 0) __builtin_amdgcn_sched_barrier(0);  // two samples at a time in registers
    const float rc = __builtin_amdgcn_rcpf(fmaf(kz[k], E.q[3], C));  // 1 ulp, as the positions
    const float u = fmaf(kz[k], E.a[3], A) * rc, v = fmaf(kz[k], E.b[3], B) * rc;
    float wt = E.s;
    if constexpr (MODE == FC_BP_FDK) wt = E.s * rc * rc;
    if constexpr (MODE == FC_BP_KATSEVICH) wt = E.s * rc;
    acc[k] = fmaf(wt, tile_bilinear(T0 + 4u * (uint32_t)(int)u, __builtin_amdgcn_fractf(u), v), acc[k]);
  }
}

typedef uint32_t fc_u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));

// Bound by VALU issue (1.02 instructions per CU clock, 14.1 per voxel-view at 512^3 x 720) with the LDS
// busy 72 % of the time; five blocks per CU for FP32 storage (96 registers, of which two to four and one
// scalar one spill, outside the samples), four for 16-bit storage (113), which at five spills and is 1 to
// 6 % slower. Against per-view FP64 terms by column and dword copies row by row (17.5 instructions, 49 %):
// 512^3 x 720 FP32 39.2 -> 36.9 ms, 256^3 x 360 BF16 2.85 -> 2.72 ms, 150 x 333 x 290 x 275 tilted FP16 2.84 ->
// 2.66 ms. Keeping two samples' reads ahead (column_samples) is part of that: with four ahead the
// registers allow only four blocks (38.0 against 37.0 ms).
template <int DT, int MODE>
__global__ __launch_bounds__(256, DT == FC_F32 ? 5 : 4) void bp_kernel(BpArgs a) {
  __shared__ __align__(16) float tile[2][kTileCap];
  __shared__ __align__(16) ViewEntry tab[kTab + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  const int ix = (wave & 1) * 8 + (lane & 7), iy = (wave >> 1) * 8 + (lane >> 3);
  const int bx0 = blockIdx.x * kBXY, by0 = blockIdx.y * kBXY;
  const int split = blockIdx.z / a.nbz, z0 = (int)(blockIdx.z - split * a.nbz) * kZR;
  const int x = bx0 + ix, y = by0 + iy;
  // Columns and voxels beyond the volume (partial cubes) repeat its last ones, so that every sample's
  // taps lie >= 1 pixel inside the window; their sums are not stored. kz in scalar registers.
  const float dx = (float)min(ix, a.nx - 1 - bx0), dy = (float)min(iy, a.ny - 1 - by0);
  const uint32_t last = __builtin_amdgcn_readfirstlane(__float_as_uint((float)(a.nz - 1 - z0)));
  float kz[kZR];
  kz[0] = 0.0f;
#pragma unroll
  for (int k = 1; k < kZR; ++k) {
    // the smaller of two non-negative floats
    kz[k] = __uint_as_float(
        __builtin_amdgcn_readfirstlane(min(__builtin_bit_cast(uint32_t, (float)k), last)));
  }
  const int tbeg = (int)((long long)a.nviews * split / a.nsplit);
  const int tend = (int)((long long)a.nviews * (split + 1) / a.nsplit);
  float acc[kZR];
#pragma unroll
  for (int k = 0; k < kZR; ++k) acc[k] = 0.0f;

  // A window is copied in units of four pixels, kUnits per row: lane l of a wave takes unit l mod
  // kUnits of row kRowsW wave + l / kUnits + kRowsB i, so a wave's units are consecutive in LDS.
  // Units past the window's last column (rounded up) are left out; they are never read.
  constexpr uint32_t kSize = DT == FC_F32 ? 4u : 2u;  // bytes per pixel
  const uint32_t lrow = (uint32_t)lane / kUnits;
  const uint32_t col = lane < kRowsW * (int)kUnits ? 4u * ((uint32_t)lane - lrow * kUnits) : 0xffffu;
  const uint32_t off = (lrow * (uint32_t)a.nw + col) * kSize;
  // whole units of the window lie on the detector
  auto whole = [&](int u0, int v0, uint32_t Wu, uint32_t Wv) {
    return u0 >= 0 && u0 + (int)((Wu + 3u) & ~3u) <= a.nw && v0 >= 0 && v0 + (int)Wv <= a.nh;
  };
  // FP32 storage: global memory -> LDS buffer
  auto issue_lds = [&](int t, uint32_t org, uint32_t size, uint32_t buf) {
    const uint32_t Wu = size & 0xffffu, Wv = size >> 16;
    if (Wu == kWinSkip || Wu == kWinGlobal) return;
    const int u0 = (int)(int16_t)(org & 0xffffu), v0 = (int)(int16_t)(org >> 16);
    // the window's first pixel (it may lie before the detector, but only pixels on it are loaded)
    const float* win = static_cast<const float*>(a.proj) + ((long long)t * a.nh + v0) * a.nw + u0;
    if (whole(u0, v0, Wu, Wv)) {
      const int rows = (int)Wv - kRowsW * wv;  // of this wave's copies
      if (col < Wu) {
#pragma unroll
        for (int i = 0; i < kCopies; ++i)
          if (kRowsB * i < rows && (int)lrow < rows - kRowsB * i)
            copy_units_to_lds(win + (long long)(kRowsW * wv + kRowsB * i) * a.nw, off,
                              buf + 4u * kTileP * (uint32_t)(kRowsW * wv + kRowsB * i));
      }
      return;
    }
    // a window over the detector's edge, row by row: row wv + 4 q, column = lane; pixels outside the
    // detector are stored as zero by the lanes themselves
    const int pu = u0 + lane;
    const bool colok = pu >= 0 && pu < a.nw;
    if ((uint32_t)lane < Wu) {
      for (uint32_t r = (uint32_t)wv; r < Wv; r += 4u) {
        const uint32_t dst = buf + 4u * kTileP * r;
        if (colok && (uint32_t)(v0 + (int)r) < (uint32_t)a.nh) {
          copy_dword_to_lds(win + (long long)r * a.nw, 4u * (uint32_t)lane, dst);
        } else {
          typedef __attribute__((address_space(3))) float* lds_p;
          *(lds_p)(dst + 4u * (uint32_t)lane) = 0.0f;
        }
      }
    }
  };
  // 16-bit storage: registers hold the raw bits of a unit (converting at commit keeps the loads in
  // flight). A unit over the detector's edge is loaded from the nearest place on it and shifted into
  // place at commit; zero bits are +0 in every storage format.
  uint2 pre[kCopies];
  auto issue = [&](int t, uint32_t org, uint32_t size) {
    const uint32_t Wu = size & 0xffffu, Wv = size >> 16;
    if (Wu == kWinSkip || Wu == kWinGlobal) return;
    const int u0 = (int)(int16_t)(org & 0xffffu), v0 = (int)(int16_t)(org >> 16);
    const int rows = (int)Wv - kRowsW * wv;
    const int vlo = min(max(v0, 0), a.nh - 1);
    const uint16_t* base = static_cast<const uint16_t*>(a.proj) + ((long long)t * a.nh + vlo) * a.nw;
    const int cs = min(max(u0 + (int)col, 0), max(a.nw - 4, 0));
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
      if (kRowsB * i < rows && (int)lrow < rows - kRowsB * i && col < Wu) {
        const int r = min(max(v0 + kRowsW * wv + kRowsB * i + (int)lrow, vlo), a.nh - 1) - vlo;
        const uint16_t* p = base + (uint32_t)(r * a.nw + cs);
        if (a.nw >= 4) {
          const fc_u32x2_a2 q = *reinterpret_cast<const fc_u32x2_a2*>(p);
          pre[i] = make_uint2(q.x, q.y);
        } else {  // rows of one to three pixels, zeros after them
          const uint32_t h1 = a.nw > 1 ? p[1] : 0u, h2 = a.nw > 2 ? p[2] : 0u;
          pre[i] = make_uint2((uint32_t)p[0] | h1 << 16, h2);
        }
      }
    }
  };
  auto commit = [&](float* T, uint32_t org, uint32_t size) {
    const uint32_t Wu = size & 0xffffu, Wv = size >> 16;
    if (Wu == kWinSkip || Wu == kWinGlobal) return;
    const int u0 = (int)(int16_t)(org & 0xffffu), v0 = (int)(int16_t)(org >> 16);
    const int rows = (int)Wv - kRowsW * wv;
    const bool all = whole(u0, v0, Wu, Wv);
#pragma unroll
    for (int i = 0; i < kCopies; ++i)
      if (kRowsB * i < rows && (int)lrow < rows - kRowsB * i && col < Wu) {
        const int r = kRowsW * wv + kRowsB * i + (int)lrow;
        uint2 q = pre[i];
        if (!all) {
          // pixel k of the unit is pixel k + d of what was loaded
          const int d = u0 + (int)col - min(max(u0 + (int)col, 0), max(a.nw - 4, 0));
          unsigned long long b = (unsigned long long)q.y << 32 | q.x;
          b = d >= 0 ? b >> (16 * min(d, 3)) : b << (16 * min(-d, 3));
          if (d <= -4 || d >= 4 || (uint32_t)(v0 + r) >= (uint32_t)a.nh) b = 0ull;
          q = make_uint2((uint32_t)b, (uint32_t)(b >> 32));
        }
        *reinterpret_cast<float4*>(T + kTileP * (uint32_t)r + col) =
            make_float4(bits_to_f32<DT>(q.x & 0xffffu), bits_to_f32<DT>(q.x >> 16),
                        bits_to_f32<DT>(q.y & 0xffffu), bits_to_f32<DT>(q.y >> 16));
      }
  };

  bool gather = false;  // uniform: some views' windows do not fit
  for (int tb = tbeg; tb < tend; tb += kTab) {
    const int n = min(kTab, tend - tb);
    __syncthreads();  // the previous table is no longer read
    // one entry more than the table's views: the next view's window
    view_table<MODE>(a, tab, tb, min(n + 1, tend - tb), bx0, by0, z0);
    __syncthreads();
    if (tb == tbeg) {
      const uint32_t org = __builtin_amdgcn_readfirstlane(tab[0].org),
                     size = __builtin_amdgcn_readfirstlane(tab[0].size);
      if constexpr (DT == FC_F32) issue_lds(tb, org, size, lds_address(tile[0]));
      else issue(tb, org, size);
    }
    for (int i = 0; i < n; ++i) {
      const int t = tb + i;
      float* T = tile[(t - tbeg) & 1];
      const bool more = t + 1 < tend;
      // the entries first (they do not depend on the barrier: a wave that finishes view t - 1 early
      // waits for them while the others still compute)
      const ViewEntry E = tab[i];
      const ViewEntry* next = tab + (more ? i + 1 : i);
      const uint32_t norg = __builtin_amdgcn_readfirstlane(next->org),
                     nsize = __builtin_amdgcn_readfirstlane(next->size);
      const uint32_t org = __builtin_amdgcn_readfirstlane(E.org),
                     size = __builtin_amdgcn_readfirstlane(E.size);
      if constexpr (DT == FC_F32) {
        // this wave's copies of view t have landed; the barrier then covers every wave's
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      } else {
        // the other buffer's readers (view t-1) all passed the previous barrier before this write
        commit(T, org, size);
      }
      __syncthreads();
      // the next view's rows are in flight while view t is accumulated; the other buffer's readers
      // (view t-1) all passed the barrier above
      if (more) {
        if constexpr (DT == FC_F32) issue_lds(t + 1, norg, nsize, lds_address(tile[(t + 1 - tbeg) & 1]));
        else issue(t + 1, norg, nsize);
      }
      const uint32_t Wu = size & 0xffffu, Wv = size >> 16;
      if (Wu == kWinSkip) continue;  // uniform: the cube misses the detector in this view
      if (Wu == kWinGlobal) {  // gathered after the views whose windows fit
        gather = true;
        continue;
      }
      const uint32_t T0 = lds_address(T);
      const float A = fmaf(dx, E.a[1], fmaf(dy, E.a[2], E.a[0]));
      const float B = fmaf(dx, E.b[1], fmaf(dy, E.b[2], E.b[0]));
      const float q = fmaf(dx, E.q[1], fmaf(dy, E.q[2], E.q[0]));
      if (__builtin_amdgcn_readfirstlane(E.tilted) == 0u) {
        // Columns independent of z: u and the weight are per column, the row is linear in z.
        const float p = -q * __builtin_amdgcn_rcpf(1.0f + q), rc = 1.0f + p;  // Cm / C
        const float u = A * rc, vb = B * rc, dv = E.b[3] * rc;
        float wt = E.s;
        if constexpr (MODE == FC_BP_FDK) wt = fmaf(E.s, p * (p + 2.0f), E.s);
        if constexpr (MODE == FC_BP_KATSEVICH) wt = fmaf(E.s, p, E.s);
        const uint32_t col0 = T0 + 4u * (uint32_t)(int)u;
        const float au = __builtin_amdgcn_fractf(u);
        column_samples(acc, kz, col0, au, vb, dv, wt);
      } else {
        tilted_samples<MODE>(acc, kz, T0, A, B, q, E);
      }
    }
  }
  if (gather) gather_views<DT, MODE>(acc, a, tab, tbeg, tend, x, y, z0, bx0, by0);
  if (x < a.nx && y < a.ny) {
    const size_t plane = (size_t)a.nx * a.ny;
    float* o = a.vol + (a.nsplit > 1 ? (size_t)split * plane * a.nz : 0) + (size_t)y * a.nx + x;
#pragma unroll
    for (int k = 0; k < kZR; ++k) {
      const int z = z0 + k;
      if (z >= a.nz) break;
      if (a.nsplit > 1) o[(size_t)z * plane] = acc[k];
      else o[(size_t)z * plane] += acc[k];
    }
  }
}

// vol += sum over the splits' partial volumes, in order.
__global__ __launch_bounds__(256) void bp_reduce(const float* __restrict__ part, int nsplit,
                                                 size_t n, float* __restrict__ vol) {
  const size_t stride = (size_t)gridDim.x * 256;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
    float s = part[i];
    for (int k = 1; k < nsplit; ++k) s += part[(size_t)k * n + i];
    vol[i] += s;
  }
}

// Gather-roofline microbenchmark for the backprojector: bilinear samples from one staged 64 x 48
// LDS window per block at pseudo-random positions (same tile_bilinear as bp_kernel).
__global__ __launch_bounds__(256) void gather_bench_bp(const float* __restrict__ src, int pitch,
                                                       int nsamp, float* __restrict__ sink) {
  __shared__ float T[kTileCap];
  const float* g = src + (size_t)(blockIdx.x % 64) * 48 * pitch;
  for (int e = threadIdx.x; e < kTileCap; e += 256)
    T[e] = g[(e / kTileP) * pitch + min(e % kTileP, (uint32_t)kTileW - 1u)];
  __syncthreads();
  uint32_t s = 0x9e3779b9u * (blockIdx.x * 256 + threadIdx.x + 1);
  const float su = 62.0f / 16777216.0f, sv = 46.0f / 16777216.0f;
  float acc = 0.0f;
  for (int k = 0; k < nsamp; ++k) {
    s = s * 1664525u + 1013904223u;
    const float u = (float)(s >> 8) * su;
    s = s * 1664525u + 1013904223u;
    const float v = (float)(s >> 8) * sv;
    acc = fmaf(1.0001f, tile_bilinear(lds_address(T + (int)u), __builtin_amdgcn_fractf(u), v), acc);
  }
  if (acc == 12345.678f) sink[0] = acc;
}

// Ray-coherent ceiling for the backprojector: bp_kernel's fast-path inner loop for blocks inside
// the volume (per column one u and weight per view, 16 z voxels whose rows advance by dv:
// bilinear sample from the LDS window, weighted accumulate) over one resident 64 x 48 window per
// block, with the backprojector's lane layout and view-to-view drift. No per-view projective
// set-up, no window staging and no barriers, so it bounds the voxel-view rate of the LDS gather
// itself. Bounds: u <= 2 + 10.5 + 4.5 + 0.35 < 62, v <= 2 + 3 + 1.5 + 0.35 + 15 * 1.3 < 46.
__global__ __launch_bounds__(256) void gather_bench_bp_ray(const float* __restrict__ src,
                                                           int pitch, int nviews,
                                                           float* __restrict__ sink) {
  __shared__ float T[kTileCap];
  const float* g = src + (size_t)(blockIdx.x % 64) * 48 * pitch;
  for (int e = threadIdx.x; e < kTileCap; e += 256)
    T[e] = g[(e / kTileP) * pitch + min(e % kTileP, (uint32_t)kTileW - 1u)];
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float xl = (float)((wave & 1) * 8 + (lane & 7)), yl = (float)((wave >> 1) * 8 + (lane >> 3));
  float acc[kZR];
#pragma unroll
  for (int k = 0; k < kZR; ++k) acc[k] = 0.0f;
#pragma unroll 1
  for (int t = 0; t < nviews; ++t) {
    const float tt = (float)(t & 7);
    const float u = clampf(2.0f + 0.7f * xl + 0.3f * yl + 0.05f * tt, 0.0f, 62.0f);
    const float vb = 2.0f + 0.2f * xl + 0.1f * yl + 0.05f * tt;
    const float wt = 1.0f + 0.001f * tt;
    const uint32_t col0 = lds_address(T + (int)u);
    const float au = __builtin_amdgcn_fractf(u);
#pragma unroll
    for (int k = 0; k < kZR; ++k) {
      acc[k] = fmaf(wt, tile_bilinear(col0, au, fmaf((float)k, 1.3f, vb)), acc[k]);
    }
  }
  float sum = 0.0f;
#pragma unroll
  for (int k = 0; k < kZR; ++k) sum += acc[k];
  if (sum == 12345.678f) sink[0] = sum;
}

template <int DT>
int dispatch_bp(const BpArgs& a, int mode, dim3 grid, hipStream_t s) {
  if (mode == FC_BP_UNWEIGHTED) bp_kernel<DT, FC_BP_UNWEIGHTED><<<grid, 256, 0, s>>>(a);
  else if (mode == FC_BP_KATSEVICH) bp_kernel<DT, FC_BP_KATSEVICH><<<grid, 256, 0, s>>>(a);
  else bp_kernel<DT, FC_BP_FDK><<<grid, 256, 0, s>>>(a);
  FC_HIP(hipGetLastError());
  return FC_OK;
}

}  // namespace

// Splits of the views. Blocks run in rounds of five per CU (1280): fewer cubes than that leave CUs
// idle, and a few rounds waste much of the last one. A split costs its partial volume's write and
// read, so it needs enough views. Timed (us, 1 split / 2 / the number chosen): 64^3 x 60 views 81 / 47 / 26
// (12 splits), 96^3 x 120 152 / 99 / 73 (11), 128^3 x 180 247 / 188 / 193 (5), 150 x 200 x 210 x 200 658 / 619 /
// 598 (3), 256^3 x 360 2319 / 2339 / 2317 (3), 240 x 300^2 x 360 3148 / 3093 / 3070 (3); at 320 x 400^2 x 200
// (12500 cubes) 3768 / 3933.
int bp_splits(long long nblocks, int nviews) {
  if (nblocks < 1280) return (int)std::max(1LL, std::min<long long>(2560 / nblocks, nviews / 5));
  return nblocks < 8192 && nviews >= 128 ? 3 : 1;
}

int launch_backproject(int device, float* vol, const int vs[3], const double origin[3],
                       const void* proj, int dt, const int ps[3], const double* views,
                       const float* norm, int mode, hipStream_t stream) {
  const int nw = ps[0], nh = ps[1], nv = ps[2];
  if (nv == 0 || vs[0] == 0 || vs[1] == 0 || vs[2] == 0) return FC_OK;
  const int nbx = (vs[0] + kBXY - 1) / kBXY, nby = (vs[1] + kBXY - 1) / kBXY,
            nbz = (vs[2] + kZR - 1) / kZR;
  FC_CHECK_ARG(nby <= 65535 && nbz <= 65535, "volume too large for the grid");
  const size_t n = (size_t)vs[0] * vs[1] * vs[2];
  BpArgs a;
  a.vol = vol;
  a.proj = proj;
  a.norm = norm;
  a.views = views;
  a.ox = origin[0]; a.oy = origin[1]; a.oz = origin[2];
  a.nx = vs[0]; a.ny = vs[1]; a.nz = vs[2];
  a.nw = nw; a.nh = nh; a.nviews = nv;
  a.nbz = nbz;
  a.nsplit = std::min(bp_splits((long long)nbx * nby * nbz, nv), 65535 / nbz);
  void* ws = nullptr;
  if (a.nsplit > 1) {
    int rc = acquire_ws(device, SLOT_QUAD, (size_t)a.nsplit * n * sizeof(float), stream, &ws);
    if (rc == FC_ERR_MEMORY) {  // no room for the partial volumes: one block per cube
      clear_error();
      a.nsplit = 1;
    } else if (rc) {
      return rc;
    } else {
      a.vol = static_cast<float*>(ws);
    }
  }
  const dim3 grid(nbx, nby, nbz * a.nsplit);
  int tok = prof_begin("backproject", stream);
  int r2;
  if (dt == FC_F32) r2 = dispatch_bp<FC_F32>(a, mode, grid, stream);
  else if (dt == FC_BF16) r2 = dispatch_bp<FC_BF16>(a, mode, grid, stream);
  else r2 = dispatch_bp<FC_F16>(a, mode, grid, stream);
  if (a.nsplit > 1) {
    bp_reduce<<<(unsigned)std::min<size_t>((n + 255) / 256, 4096), 256, 0, stream>>>(
        a.vol, a.nsplit, n, vol);
  }
  prof_end(tok, stream);
  if (r2) return r2;
  FC_HIP(hipGetLastError());
  return a.nsplit > 1 ? release_ws(device, SLOT_QUAD, stream) : FC_OK;
}

int launch_gather_bench_bp(int device, int dt, int ray, double* samples_per_s) {
  (void)device;
  (void)dt;  // LDS windows hold FP32 whatever the storage type; only the staging converts
  const int pitch = 1024, rows = 64 * 48;
  std::vector<float> host((size_t)pitch * rows);
  for (size_t q = 0; q < host.size(); ++q) host[q] = (float)((q * 2654435761u) % 1000) * 1e-3f;
  float* src = nullptr;
  float* sink = nullptr;
  FC_HIP(hipMalloc(&src, host.size() * sizeof(float)));
  FC_HIP(hipMalloc(&sink, sizeof(float)));
  FC_HIP(hipMemcpy(src, host.data(), host.size() * sizeof(float), hipMemcpyHostToDevice));
  hipEvent_t e0, e1;
  FC_HIP(hipEventCreate(&e0));
  FC_HIP(hipEventCreate(&e1));
  const int blocks = 256 * 16, nsamp = 4096;
  double best = 0.0;
  for (int rep = 0; rep < 3; ++rep) {
    FC_HIP(hipEventRecord(e0, nullptr));
    if (ray) gather_bench_bp_ray<<<blocks, 256>>>(src, pitch, nsamp / kZR, sink);
    else gather_bench_bp<<<blocks, 256>>>(src, pitch, nsamp, sink);
    FC_HIP(hipEventRecord(e1, nullptr));
    FC_HIP(hipEventSynchronize(e1));
    float ms = 0.f;
    FC_HIP(hipEventElapsedTime(&ms, e0, e1));
    double rate = (double)blocks * 256.0 * nsamp / (ms * 1e-3);
    if (rep > 0 && rate > best) best = rate;
  }
  FC_HIP(hipEventDestroy(e0));
  FC_HIP(hipEventDestroy(e1));
  FC_HIP(hipFree(src));
  FC_HIP(hipFree(sink));
  *samples_per_s = best;
  return FC_OK;
}

}  // namespace fc
