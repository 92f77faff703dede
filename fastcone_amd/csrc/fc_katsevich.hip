// Katsevich helical reconstruction on a cylindrical (source-centred) detector, for gfx950.
//
// The reference only backprojects with a U^1 weight (coneBeamGPU.cu:258-338) and leaves the
// derivative and kappa-line filtering to the caller; it cannot represent a curved detector. This
// file implements the whole exact algorithm (Katsevich 2002, in the native curved-detector form of
// Noo, Pack & Heuscher 2003, Phys. Med. Biol. 48:3787):
//
//   g1 = [G(k+1, g + dl) - G(k-1, g - dl)] / (2 dl)        derivative at a fixed ray direction
//   g2 = g1 SDD / sqrt(SDD^2 + w^2)                         cone-angle weight
//   g3(psi_m) = g2 at w = w_k(g, psi_m)                      forward height rebinning (kappa lines)
//   g4 = sum_{n odd} 2/(pi n) (n dg / sin(n dg)) g3[j - n]   Hilbert transform, kernel 1/(pi sin)
//   g5(w) = g4 at the psi with w_k(g, psi) = w               backward height rebinning
//   f(x) += dl/(2 pi) sum_k g5(k, g*, w*) / v*   over views where x projects into the
//           Tam-Danielsson window (the PI interval of x)
//
// Helix: a(l) = (R cos l, R sin l, zs0 + hp (l - l0)), l_k = l0 + k dl. Detector: column j at fan
// angle g = (j - col_c) dg from e_v = -(cos l, sin l, 0) towards e_u = (-sin l, cos l, 0), row i
// at height w = (i - row_c) drow, SDD from the source. w_k(g, psi) = (SDD hp / R)(psi cos g +
// psi cot psi sin g), psi_m uniform on [-(pi/2 + am), pi/2 + am], am = largest |fan angle|.
//
// Layout: every stage is a dense [view][row][column] FP32 array in HBM (c2: 0.57 GB per stage,
// 1.1 GB for the kappa-line stages); the backprojector reads g5 as pairs of a value and the step to
// the next column's, with a border of zeros (kat_stage). The Hilbert stage is the FFT row filter of fc_filter.hip (one convolution
// per kappa line), the other filter stages are elementwise gathers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "fc_device.h"
#include "fc_internal.h"

namespace fc {
namespace {

struct KatGeom {
  double l0, dl, zs0, hp, R, SDD, dg, drow, col_c, row_c, pmax, dpsi;
  int nw, nh, nv, npsi;
};

__device__ __forceinline__ double kappa_w(const KatGeom& g, double gam, double psi) {
  double pc = fabs(psi) < 1e-12 ? 1.0 : psi / tan(psi);
  return g.SDD * g.hp / g.R * (psi * cos(gam) + pc * sin(gam));
}

// Tables: fwd[m][j] = detector row coordinate of kappa line m at column j;
// bwd[i][j] = (m + t) with w_k(g_j, psi_m..m+1) bracketing row i's height, or -1 outside;
// cone[i] = the cone-angle weight of row i.
__global__ __launch_bounds__(64) void kat_tables(KatGeom g, float* __restrict__ fwd,
                                                 float* __restrict__ bwd,
                                                 float* __restrict__ cone) {
  const int j = blockIdx.y * 64 + threadIdx.x;
  if (j >= g.nw) return;
  const double gam = ((double)j - g.col_c) * g.dg;
  const int m = blockIdx.x;
  if (m < g.npsi) {
    fwd[(size_t)m * g.nw + j] = (float)(kappa_w(g, gam, -g.pmax + m * g.dpsi) / g.drow + g.row_c);
    return;
  }
  const int i = m - g.npsi;
  const double w = ((double)i - g.row_c) * g.drow;
  if (j == 0) cone[i] = (float)(g.SDD / sqrt(g.SDD * g.SDD + w * w));
  float r = -1.0f;
  if (w >= kappa_w(g, gam, -g.pmax) && w <= kappa_w(g, gam, g.pmax)) {
    int lo = 0, hi = g.npsi - 1;  // w_k is increasing in psi for every detector column
    while (hi - lo > 1) {
      int mid = (lo + hi) / 2;
      if (kappa_w(g, gam, -g.pmax + mid * g.dpsi) <= w) lo = mid; else hi = mid;
    }
    double wl = kappa_w(g, gam, -g.pmax + lo * g.dpsi);
    double wh = kappa_w(g, gam, -g.pmax + hi * g.dpsi);
    r = (float)((double)lo + (w - wl) / (wh - wl));
  }
  bwd[(size_t)i * g.nw + j] = r;
}

// g3[k][m][j] = g2[k][row(m, j)][j], linear in the row, zero outside, with g2 = cone weight x
// fixed-direction derivative. A thread walks kRebinLines kappa lines down its column: their rows rise
// with m, so it keeps the two rows of g2 that it interpolates and evaluates the next one when a line
// passes it. Bound by memory (the projections, and 1.1 GB of g3 for 4320 views of 64 x 512):
// 0.92 ms; the derivative and the rebinning in two passes took 0.72 and 0.99 ms.
constexpr int kRebinLines = 48;
template <int DT>
__global__ __launch_bounds__(256) void kat_rebin(const void* __restrict__ proj, KatGeom g,
                                                 const float* __restrict__ fwd,
                                                 const float* __restrict__ cone,
                                                 float* __restrict__ g3) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  const int ma = blockIdx.y * kRebinLines, mb = min(ma + kRebinLines, g.npsi), k = blockIdx.z;
  if (j >= g.nw) return;
  const bool inner = k > 0 && k < g.nv - 1;  // the first and the last view have no derivative
  const float shift = (float)(g.dl / g.dg), scale = (float)(0.5 / g.dl);
  auto val = [&](int kk, int i, float c) {
    float fc = floorf(c);
    int j0 = (int)fc;
    float t = c - fc, s = 0.0f;
    size_t rb = ((size_t)kk * g.nh + i) * g.nw;
    if (j0 >= 0 && j0 < g.nw) s += (1.0f - t) * load_elem<DT>(proj, rb + j0);
    if (j0 + 1 >= 0 && j0 + 1 < g.nw) s += t * load_elem<DT>(proj, rb + j0 + 1);
    return s;
  };
  auto g2 = [&](int i) {
    if (!inner || i < 0 || i >= g.nh) return 0.0f;
    float d = (val(k + 1, i, (float)j + shift) - val(k - 1, i, (float)j - shift)) * scale;
    return d * cone[i];
  };
  int have = -3;  // rows `have` and `have` + 1 are in v0 and v1
  float v0 = 0.0f, v1 = 0.0f;
  for (int m = ma; m < mb; ++m) {
    const float r = fwd[(size_t)m * g.nw + j], fr = floorf(r);
    // rows further out than -2 and nh are zero as these
    const int i0 = min(max((int)fr, -2), g.nh);
    if (i0 != have) {
      v0 = i0 == have + 1 ? v1 : g2(i0);
      v1 = g2(i0 + 1);
      have = i0;
    }
    const float t = r - fr;
    float s = 0.0f;
    if (i0 >= 0 && i0 < g.nh) s += (1.0f - t) * v0;
    if (i0 + 1 >= 0 && i0 + 1 < g.nh) s += t * v1;
    g3[((size_t)k * g.npsi + m) * g.nw + j] = s;
  }
}

// The Hilbert transform of each kappa line, g4[j] = sum_{n odd} h[n] g3[j - n] with
// h[n] = 2/(pi n) * n dg / sin(n dg), is the FFT row filter's FC_FILTER_HILBERT kernel.
constexpr int kMaxCols = 2048;  // detector columns (FFT length <= 4096 in the Hilbert stage)

// g5[k][i][j] = g4 interpolated between the kappa lines bracketing row i at column j, staged for the
// backprojection: element (r, c) of a view is the pixel p = g5(r - 1, c - 1) and the step to the next
// column's, (p, g5(r - 1, c) - p); pixels off the detector are zero. A wave owns 63 columns and
// kStageRows rows: a lane interpolates its own column's pixel and takes the next column's from its
// neighbour. g5 itself is written only if the caller wants it.
// Bound by memory (2.3 GB read and written for 4320 views of 64 x 512): 0.7 ms; the interpolation and
// the staging of 16-byte quads in kernels of their own took 0.4 and 1.1 ms.
constexpr int kStageRows = 22;
__host__ __device__ constexpr int stage_pitch(int nw) { return (nw + 3) & ~1; }  // 16-byte rows
__global__ __launch_bounds__(256) void kat_stage(const float* __restrict__ g4, KatGeom g,
                                                 const float* __restrict__ bwd,
                                                 float2* __restrict__ pairs,
                                                 float* __restrict__ g5) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int pitch = stage_pitch(g.nw), rows = g.nh + 3;
  const int c = (blockIdx.x * 4 + wave) * 63 + lane, j = c - 1;  // element and pixel column
  const int ra = blockIdx.y * kStageRows, rb = min(ra + kStageRows, rows), k = blockIdx.z;
  const bool col = j >= 0 && j < g.nw;
  const float* line = g4 + (size_t)k * g.npsi * g.nw + j;
  for (int r = ra; r < rb; ++r) {
    const int i = r - 1;
    float p = 0.0f;
    if (col && i >= 0 && i < g.nh) {
      const float b = bwd[(size_t)i * g.nw + j];
      if (b >= 0.0f) {
        const int m0 = min((int)b, g.npsi - 2);
        const float t = b - (float)m0;
        p = (1.0f - t) * line[(size_t)m0 * g.nw] + t * line[(size_t)(m0 + 1) * g.nw];
      }
      if (g5 && lane < 63) g5[((size_t)k * g.nh + i) * g.nw + j] = p;
    }
    const float d = __shfl_down(p, 1, 64) - p;
    if (lane < 63 && c < pitch) pairs[((size_t)k * rows + r) * pitch + c] = make_float2(p, d);
  }
}

// PI-window backprojection. A block owns 16 x 16 columns (8 x 8 per wave, a thread per column) and
// SLABS * kZR consecutive z; per view and column: v* = R - x cos l - y sin l, g* = atan(u* / v*), the
// column coordinate and the Tam-Danielsson row bounds; per voxel: the row (linear in z), the window
// test, one bilinear sample. Views go by in chunks of kViews: a thread per view bounds what the
// block's columns need of it (KatEntry) and the views that no voxel sees through its window drop out;
// the others' detector windows are copied to LDS one view ahead.
constexpr int kZR = 8;
constexpr int kViews = 128;
constexpr int kWinW = 40;                 // window columns
constexpr uint32_t kWinB = kWinW * 8;     // bytes per window row: 16 banks on from the row above
constexpr int win_rows(int slabs) { return 6 + 10 * slabs; }
struct KatBpArgs {
  float* vol;
  const float2* pairs;   // staged g5: (nh + 3) x stage_pitch(nw) per view
  const float4* vtab;    // per view: cos l, sin l, source z, 0
  KatGeom g;
  float ox, oy, oz;
  int nx, ny, nz;
  double zmax;  // largest |z - zs| a voxel can have inside the window (voxels)
};
// A view as a block sees it: every sample's column coordinate lies in [ulo, uhi] and its row in
// [vlo, vhi]; those of the detector elements from (row, col) on, `units` 16-byte units long.
struct KatEntry {
  float cosl, sinl, zs;
  int k;
  float ulo, uhi, vlo, vhi;
  int row, col, units, lds;  // lds: the window fits the LDS buffers
};

__global__ __launch_bounds__(256) void kat_view_table(KatGeom g, float4* __restrict__ vt) {
  int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= g.nv) return;
  double l = g.l0 + k * g.dl;
  vt[k] = make_float4((float)cos(l), (float)sin(l), (float)(g.zs0 + k * g.dl * g.hp), 0.0f);
}

// 1 / b, a / b and the square root of x in 3, 3 more and 8 instructions (the operators' 10, 10 and 14
// also scale against overflow and underflow of their intermediate values, which no volume and helix of
// finite voxel coordinates gets near). That one Newton step rounds correctly is a property of this
// GPU's v_rcp_f32 and v_rsq_f32, not of any 1-ulp start: compared on gfx950, the results equal the
// operators' for all 2^23 mantissas b, all floats x in [1, 4) and 2^30 random pairs (a, b).
__device__ __forceinline__ float recip(float b) {
  const float y = __builtin_amdgcn_rcpf(b);
  return fmaf(fmaf(-b, y, 1.0f), y, y);
}
__device__ __forceinline__ float quotient(float a, float b, float recip_b) {
  const float q = a * recip_b;
  return fmaf(fmaf(-b, q, a), recip_b, q);
}
__device__ __forceinline__ float square_root(float x) {
  const float y = __builtin_amdgcn_rsqf(x);
  float s = x * y, h = 0.5f * y;
  const float r = fmaf(-h, s, 0.5f);
  s = fmaf(s, r, s);
  h = fmaf(h, r, h);
  return fmaf(fmaf(-s, s, x), h, s);
}
__device__ __forceinline__ int floor_int(float x) {
  int i;
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(i) : "v"(x));
  return i;
}

// Bounds of what the columns within `rad` of (X, Y), z in [z0, z1], need of view k; false if none of
// their voxels projects into its window. Margins of 0.05 element (and 1e-5 of the row) cover the
// rounding of this bound and of the samples' own coordinates.
__device__ __forceinline__ bool kat_entry(const KatBpArgs& a, int k, float X, float Y, float rad,
                                          float z0, float z1, int max_rows, KatEntry& e) {
  const KatGeom& g = a.g;
  const float4 vt = a.vtab[k];
  e.cosl = vt.x, e.sinl = vt.y, e.zs = vt.z, e.k = k;
  const float vs = (float)g.R - X * vt.x - Y * vt.y, us = Y * vt.x - X * vt.y;
  const float dist = sqrtf(vs * vs + us * us), dg = (float)g.dg;
  e.ulo = -1.0f, e.uhi = (float)g.nw, e.vlo = -1.0f, e.vhi = (float)g.nh;
  e.row = e.col = e.units = e.lds = 0;
  if (!(dist > 1.05f * rad)) return true;  // next to the source: no bound
  const float gam = atan2f(us, vs), half = rad / sqrtf((dist - rad) * (dist + rad));  // >= asin
  const float ga = gam - half, gb = gam + half;
  // (pi/2 - g) / cos g falls with g: the window's ends are largest at the tile's ends
  const float sd = (float)(g.SDD / g.drow), ch = (float)(g.SDD * g.hp / g.R / g.drow);
  const float rowc = (float)g.row_c, hpi = 1.57079632679489662f;
  float lo = z0 - vt.z, hi = z1 - vt.z;
  lo = sd * lo / (lo < 0.0f ? dist - rad : dist + rad);
  hi = sd * hi / (hi > 0.0f ? dist - rad : dist + rad);
  if (ga > -1.5f) hi = fminf(hi, ch * (hpi - ga) / cosf(fminf(ga, 1.5f)));
  if (gb < 1.5f) lo = fmaxf(lo, -ch * (hpi + gb) / cosf(fmaxf(gb, -1.5f)));
  lo -= 0.05f + 1e-5f * fabsf(lo), hi += 0.05f + 1e-5f * fabsf(hi);
  if (lo > hi) return false;
  e.vlo = fminf(fmaxf(lo + rowc, -1.0f), e.vhi);
  e.vhi = fminf(fmaxf(hi + rowc, -1.0f), e.vhi);
  const float cc = (float)g.col_c;
  e.ulo = fminf(fmaxf(ga / dg + cc - 0.05f, -1.0f), e.uhi);
  e.uhi = fminf(fmaxf(gb / dg + cc + 0.05f, -1.0f), e.uhi);
  e.row = (int)floorf(e.vlo) + 1;
  e.col = ((int)floorf(e.ulo) + 1) & ~1;
  const int rows = (int)floorf(e.vhi) + 3 - e.row;
  e.lds = rows <= max_rows && (int)floorf(e.uhi) + 1 - e.col < kWinW;
  e.units = rows * (kWinW / 2);
  return true;
}

// kZR voxels of a column at rows rr = (q + qa) dr + r0: acc[q] += wgt * sample if rbot <= rr <= rtop. The
// sample is bilinear between the elements at `at` + row * pitch and the next row's, `at` standing for
// row 0 of the column, an LDS or a global address. [lo, hi] is the window within the copied rows.
typedef float f2 __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(3))) f2* lds_f2;
template <bool LDS, class P>
__device__ __forceinline__ void kat_samples(float* acc, P at, uint32_t pitch, float au, float dr,
                                            float r0, int qa, float lo, float hi, float wgt) {
  constexpr int B = 4;  // samples in flight
#pragma unroll
  for (int q0 = 0; q0 < kZR; q0 += B) {
    f2 p[B], n[B];
    float av[B], w[B];
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const float rr = fmaf((float)(qa + q0 + q), dr, r0);
      const float v = __builtin_amdgcn_fmed3f(rr, lo, hi);
      w[q] = v == rr ? wgt : 0.0f;
      av[q] = __builtin_amdgcn_fractf(v);
      const int row = floor_int(v);
      if constexpr (LDS) {
        const lds_f2 src = (lds_f2)(size_t)mad_i24(row, (int)kWinB, at);
        p[q] = src[0], n[q] = src[kWinW];
      } else {
        const char* src = at + (long long)row * pitch;
        p[q] = *reinterpret_cast<const f2*>(src), n[q] = *reinterpret_cast<const f2*>(src + pitch);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const float top = fmaf(au, p[q].y, p[q].x), bot = fmaf(au, n[q].y, n[q].x);
      acc[q0 + q] = fmaf(w[q], lerp(top, bot, av[q]), acc[q0 + q]);
    }
  }
}

// Bound by VALU issue: about 65 instructions per view and column (division, atan, square root) and
// 12.5 per sample, of which the helix's geometry makes a fifth miss their own window in a group of
// eight; the LDS reads (16 bytes per sample, without conflicts) take half of that time. 512 x 512 x
// 256 voxels, 4320 views of 64 x 512: 15.2 ms against 38.9 ms for gathering 16-byte quads of every
// visited view from global memory (20 L1 accesses per wave and sample: L1-bound at best, 21.6 ms, once
// the views outside the window were skipped).
// Views whose window does not fit the buffers are gathered from global memory, slabs outside the
// window left out, four samples in flight. 256 x 256 x 128 voxels of twice the size on the same
// detector (89 % of the blocks' views), whole reconstruction: 9.7 ms, of 128 x 64 x 64 of four times the
// size 5.2; one sample in flight and every slab 20.4 and 6.7, the quads' gather 12.6 and 9.9 ms.
template <int SLABS>
__global__ __launch_bounds__(256, 4) void kat_bp_kernel(KatBpArgs a) {
  constexpr int NZ = SLABS * kZR, ROWS = win_rows(SLABS), SLOTS = (ROWS * kWinW / 2 + 255) / 256;
  __shared__ float4 win[2][ROWS * kWinW / 2];
  __shared__ KatEntry table[kViews];
  __shared__ int count[kViews / 64];
  const KatGeom& g = a.g;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // columns beyond the volume repeat its last ones
  const int xb = blockIdx.x * 16, yb = blockIdx.y * 16;
  const int x = xb + (wave & 1) * 8 + (lane & 7), y = yb + (wave >> 1) * 8 + (lane >> 3);
  const float X = (float)min(x, a.nx - 1) + a.ox, Y = (float)min(y, a.ny - 1) + a.oy;
  const float hx = 0.5f * (float)(min(xb + 15, a.nx - 1) - xb);
  const float hy = 0.5f * (float)(min(yb + 15, a.ny - 1) - yb);
  const float Xc = (float)xb + a.ox + hx, Yc = (float)yb + a.oy + hy;
  const float rad = 1.001f * sqrtf(hx * hx + hy * hy) + 0.01f;
  const int pitch = stage_pitch(g.nw);
  const uint32_t pitchB = (uint32_t)pitch * 8u;
  const size_t viewB = (size_t)(g.nh + 3) * pitchB;
  const char* pairs = reinterpret_cast<const char*>(a.pairs);
  const uint32_t win0 = (uint32_t)(size_t)(lds_f2)&win[0][0];
  uint32_t off[SLOTS];  // bytes from the window's first element to this thread's units
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    const uint32_t unit = threadIdx.x + 256u * i;
    off[i] = unit / (kWinW / 2) * pitchB + unit % (kWinW / 2) * 16u;
  }
  const float Rf = (float)g.R, inv_dg = (float)(1.0 / g.dg), colc = (float)g.col_c;
  const float rowc = (float)g.row_c;
  const float sdd_drow = (float)(g.SDD / g.drow);
  const float c0r = (float)(g.SDD * g.hp / g.R / g.drow);
  const float hpi = 1.57079632679489662f;
  const double dz = g.hp * g.dl;
  for (int z0 = blockIdx.z * NZ; z0 < a.nz; z0 += gridDim.z * NZ) {
    // views whose source height lies within zmax of the block's z range (block-uniform)
    int klo = (int)floor(((double)z0 + a.oz - a.zmax - g.zs0) / dz) - 1;
    int khi = (int)ceil(((double)z0 + a.oz + NZ - 1 + a.zmax - g.zs0) / dz) + 1;
    klo = max(klo, 0);
    khi = min(khi, g.nv - 1);
    float acc[NZ];
#pragma unroll
    for (int q = 0; q < NZ; ++q) acc[q] = 0.0f;
    for (int kc = klo; kc <= khi; kc += kViews) {
      __syncthreads();  // the previous chunk's table and windows are no longer read
      KatEntry e;
      bool used = false;
      const int k = kc + (int)threadIdx.x;
      if (threadIdx.x < kViews && k <= khi)
        used = kat_entry(a, k, Xc, Yc, rad, (float)z0 + a.oz, (float)(z0 + NZ - 1) + a.oz, ROWS, e);
      const unsigned long long mask = __ballot(used);
      if (lane == 0 && wave < kViews / 64) count[wave] = __popcll(mask);
      __syncthreads();
      int first = 0, n = 0;
#pragma unroll
      for (int i = 0; i < kViews / 64; ++i) {
        if (i < wave) first += count[i];
        n += count[i];
      }
      if (used) table[first + __popcll(mask & ((1ull << lane) - 1))] = e;
      __syncthreads();
      n = __builtin_amdgcn_readfirstlane(n);
      auto copy = [&](int i) {
        const int units = __builtin_amdgcn_readfirstlane(table[i].lds ? table[i].units : 0);
        const char* src = pairs + (size_t)__builtin_amdgcn_readfirstlane(table[i].k) * viewB +
                          (size_t)__builtin_amdgcn_readfirstlane(table[i].row) * pitchB +
                          (size_t)__builtin_amdgcn_readfirstlane(table[i].col) * 8u;
        const uint32_t dst = win0 + (i & 1) * (uint32_t)sizeof(win[0]);
#pragma unroll
        for (int s = 0; s < SLOTS; ++s)
          if ((int)threadIdx.x + 256 * s < units)
            copy_units_to_lds(src, off[s], dst + 16u * (256u * s + 64u * wave));
      };
      if (n > 0) copy(0);
      for (int i = 0; i < n; ++i) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();  // view i is in LDS, and nobody reads view i - 1's buffer any more
        if (i + 1 < n) copy(i + 1);
        const KatEntry t = table[i];
        const float vs = fmaf(-X, t.cosl, fmaf(-Y, t.sinl, Rf));  // R - x cos l - y sin l
        const float us = fmaf(-X, t.sinl, Y * t.cosl);            // -x sin l + y cos l
        const float wgt = recip(vs);
        const float tg = quotient(us, vs, wgt);
        const float gam = atanf(tg);
        const float sec = square_root(fmaf(tg, tg, 1.0f));  // 1 / cos g
        // w* / drow = SDD (z - zs) cos g / (v* drow): the row is linear in the voxel index
        const float vsec = vs * sec, dr = quotient(sdd_drow, vsec, recip(vsec));
        const float rtop = fmaf(c0r * (hpi - gam), sec, rowc);
        const float rbot = fmaf(-c0r * (hpi + gam), sec, rowc);
        const float u = __builtin_amdgcn_fmed3f(fmaf(gam, inv_dg, colc), t.ulo, t.uhi);
        const float au = u - floorf(u);
        const int iu = floor_int(u) + 1;
        // the window within [vlo, vhi]: in-window rows lie strictly inside these
        const float lo = __builtin_amdgcn_fmed3f(rbot, t.vlo, t.vhi);
        const float hi = __builtin_amdgcn_fmed3f(rtop, t.vlo, t.vhi);
        const uint32_t at = win0 + (i & 1) * (uint32_t)sizeof(win[0]) +
                            (uint32_t)((iu - t.col) * 8 + (1 - t.row) * (int)kWinB);
        // the rows of a slab count from the sixteenth voxel below it, whatever the slabs
        auto row0 = [&](int zs, int& qa) {
          qa = SLABS > 1 ? (zs - z0) & 15 : zs & 15;
          return fmaf((float)(zs - qa) + a.oz - t.zs, dr, rowc);
        };
        int qa;
        const bool big = !__builtin_amdgcn_readfirstlane(t.lds);
#pragma unroll
        for (int s = 0; s < SLABS; ++s) {
          const float r0 = row0(z0 + s * kZR, qa);
          const float ra = fmaf((float)qa, dr, r0), rb = fmaf((float)(qa + kZR - 1), dr, r0);
          if (big || !__any(ra <= rtop && rb >= rbot)) continue;  // the rows rise with z
          kat_samples<true>(acc + s * kZR, at, 0, au, dr, r0, qa, lo, hi, wgt);
        }
        if (big) {  // windows wider than the LDS buffers: columns finer than about half a voxel
          const char* src = pairs + (size_t)t.k * viewB + pitchB + (size_t)(uint32_t)iu * 8u;
#pragma unroll
          for (int s = 0; s < SLABS; ++s) {
            const float r0 = row0(z0 + s * kZR, qa);
            const float ra = fmaf((float)qa, dr, r0), rb = fmaf((float)(qa + kZR - 1), dr, r0);
            if (!__any(ra <= rtop && rb >= rbot)) continue;
            kat_samples<false>(acc + s * kZR, src, pitchB, au, dr, r0, qa, lo, hi, wgt);
          }
        }
      }
    }
    if (x < a.nx && y < a.ny) {
      const float s = (float)(g.dl / (2.0 * M_PI));
#pragma unroll
      for (int q = 0; q < NZ; ++q) {
        const int z = z0 + q;
        if (z < a.nz) a.vol[((size_t)z * a.ny + y) * a.nx + x] += s * acc[q];
      }
    }
  }
}

}  // namespace
}  // namespace fc

using namespace fc;

extern "C" int fc_katsevich_dev(int device, const void* proj, int proj_dtype, int nw, int nh,
                                int nviews, double l0, double dl, double zs0, double hp, double R,
                                double SDD, double dgamma, double drow, double col_c,
                                double row_c, int npsi, float* vol, const int vol_shape[3],
                                const double origin[3], float* g5_out, void* stream_) {
  clear_error();
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  FC_CHECK_ARG(dtype_ok(proj_dtype), "unknown projection dtype %d", proj_dtype);
  FC_CHECK_ARG(nw > 1 && nw <= kMaxCols && nh > 1 && nh <= 65535 && nviews >= 3 &&
                   nviews <= 65535,
               "detector %d x %d / %d views out of range", nw, nh, nviews);
  FC_CHECK_ARG(npsi >= 3 && npsi <= 65535, "npsi must be in [3, 65535]");
  FC_CHECK_ARG(std::isfinite(R) && R > 0 && std::isfinite(SDD) && SDD > R, "need 0 < R < SDD");
  FC_CHECK_ARG(dl > 0 && hp > 0 && dgamma > 0 && drow > 0 && std::isfinite(l0) &&
                   std::isfinite(zs0) && std::isfinite(col_c) && std::isfinite(row_c),
               "bad helix / detector parameters");
  FC_CHECK_ARG(proj && vol && vol_shape && origin, "null pointer argument");
  FC_CHECK_ARG(vol_shape[0] > 0 && vol_shape[1] > 0 && vol_shape[2] > 0, "empty volume");
  const double am = fmax(fabs(0 - col_c), fabs(nw - 1 - col_c)) * dgamma;
  FC_CHECK_ARG(am < 1.2, "fan angle too large");
  // every voxel of the block must lie inside the helix cylinder
  double r2 = 0.0;
  for (int ax = 0; ax < 2; ++ax) {
    double lo = origin[ax], hi = origin[ax] + vol_shape[ax] - 1;
    double m = fmax(fabs(lo), fabs(hi));
    r2 += m * m;
  }
  const double rmax = sqrt(r2);
  FC_CHECK_ARG(rmax < 0.99 * R, "volume block reaches the source path");
  int rc = select_device(device);
  if (rc) return rc;

  KatGeom g;
  g.l0 = l0; g.dl = dl; g.zs0 = zs0; g.hp = hp; g.R = R; g.SDD = SDD; g.dg = dgamma;
  g.drow = drow; g.col_c = col_c; g.row_c = row_c;
  g.pmax = M_PI / 2 + am;
  g.dpsi = 2 * g.pmax / (npsi - 1);
  g.nw = nw; g.nh = nh; g.nv = nviews; g.npsi = npsi;

  const size_t plane = (size_t)nh * nw, kplane = (size_t)npsi * nw;
  void *A = nullptr, *T = nullptr;  // A: g3, filtered in place to g4
  const size_t lines = (size_t)nviews * kplane * sizeof(float);
  if ((rc = acquire_ws(device, SLOT_KAT, lines, stream, &A))) return rc;
  const size_t tab = (kplane + plane + (size_t)nh + 4 * (size_t)nviews + 4) * sizeof(float);
  if ((rc = acquire_ws(device, SLOT_KAT_TAB, tab, stream, &T))) return rc;
  void* ftab = nullptr;
  if ((rc = acquire_ws(device, SLOT_FILTER, filter_table_bytes(nw), stream, &ftab))) return rc;
  float* fwd = static_cast<float*>(T);
  float* bwd = fwd + kplane;
  float* cone = bwd + plane;
  float4* vtab = reinterpret_cast<float4*>(fwd + ((kplane + plane + nh + 3) & ~(size_t)3));

  int tok = prof_begin("katsevich_filter", stream);
  kat_tables<<<dim3(npsi + nh, (nw + 63) / 64), 64, 0, stream>>>(g, fwd, bwd, cone);
  float* g4 = static_cast<float*>(A);
  const dim3 rg((nw + 255) / 256, (npsi + kRebinLines - 1) / kRebinLines, nviews);
  if (proj_dtype == FC_F32) kat_rebin<FC_F32><<<rg, 256, 0, stream>>>(proj, g, fwd, cone, g4);
  else if (proj_dtype == FC_BF16) kat_rebin<FC_BF16><<<rg, 256, 0, stream>>>(proj, g, fwd, cone, g4);
  else kat_rebin<FC_F16><<<rg, 256, 0, stream>>>(proj, g, fwd, cone, g4);
  // Hilbert transform along every kappa line: FFT convolution with the curved-detector kernel
  if ((rc = launch_row_filter(g4, FC_F32, g4, FC_F32, nw, npsi, (long long)npsi * nviews, nullptr,
                              FC_FILTER_HILBERT, dgamma, ftab, stream)))
    return rc;
  // g5, staged in element pairs for the backprojection over the PI windows; its last window row may
  // be copied kWinW elements beyond the end
  FC_CHECK_ARG(nh + 2 <= 65535, "projection stack too large for the staging grid");
  void* Q = nullptr;
  const int pitch = stage_pitch(nw);
  const size_t qbytes = ((size_t)pitch * (nh + 3) * nviews + kWinW) * sizeof(float2);
  if ((rc = acquire_ws(device, SLOT_QUAD, qbytes, stream, &Q))) return rc;
  kat_stage<<<dim3((pitch + 251) / 252, (nh + 3 + kStageRows - 1) / kStageRows, nviews), 256, 0,
              stream>>>(g4, g, bwd, static_cast<float2*>(Q), g5_out);
  prof_end(tok, stream);
  FC_HIP(hipGetLastError());
  KatBpArgs a;
  a.vol = vol;
  a.pairs = static_cast<const float2*>(Q);
  a.vtab = vtab;
  a.g = g;
  a.ox = (float)origin[0]; a.oy = (float)origin[1]; a.oz = (float)origin[2];
  kat_view_table<<<(nviews + 255) / 256, 256, 0, stream>>>(g, vtab);
  a.nx = vol_shape[0]; a.ny = vol_shape[1]; a.nz = vol_shape[2];
  // |z - zs| <= (hp/R) (pi/2 + am) / cos^2(am) * v*,  v* <= R + rmax
  a.zmax = hp / R * (M_PI / 2 + am) / (cos(am) * cos(am)) * (R + rmax) + 2.0 * drow;
  FC_CHECK_ARG((a.ny + 15) / 16 <= 65535 && (a.nz + 15) / 16 <= 65535,
               "volume too large for the grid");
  const auto slabs = [&](int n) { return (a.nz + n * kZR - 1) / (n * kZR); };
  dim3 grid((a.nx + 15) / 16, (a.ny + 15) / 16, slabs(4));
  // Four slabs per block share a view's bounds and per-column terms; one slab gives four times the
  // blocks, each with fewer views. The line lies where four still fill the chip (4 against 1, ms:
  // 20 blocks 1.03 / 0.43, 144: 1.59 / 0.87, 544: 4.00 / 3.81, 816: 2.42 / 2.60, 1800: 7.0 / 7.8).
  const bool tall = (size_t)grid.x * grid.y * grid.z >= 768;
  if (!tall) grid.z = std::min(slabs(1), 65535);
  tok = prof_begin("katsevich_bp", stream);
  if (tall) kat_bp_kernel<4><<<grid, 256, 0, stream>>>(a);
  else kat_bp_kernel<1><<<grid, 256, 0, stream>>>(a);
  prof_end(tok, stream);
  FC_HIP(hipGetLastError());
  if ((rc = release_ws(device, SLOT_QUAD, stream))) return rc;
  if ((rc = release_ws(device, SLOT_KAT, stream))) return rc;
  if ((rc = release_ws(device, SLOT_FILTER, stream))) return rc;
  return release_ws(device, SLOT_KAT_TAB, stream);
}
