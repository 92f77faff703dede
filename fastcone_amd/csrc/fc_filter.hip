// Row filters for gfx950: every detector row (or kappa line) convolved with a fixed real kernel,
//
//   out[r, j] = sum_{m=0}^{nw-1} kern[j - m] * wgt(r, m) * in[r, m],     j in [0, nw),
//
// with kern supported on [-(nw-1), nw-1]. Two kernels are built in:
//   * RAMP — the FDK ramp of fastcone.py:272-292: a row zero-padded to n = 2 nw (data at [0, nw)),
//     its rfft multiplied by H[k] = pi k / n (k = 1..nw), H[0] = pi / (8 n), irfft, crop [0, nw).
//     That operator is the convolution with kern[d] = irfft(H)[d mod n] for |d| < nw, times a
//     caller scale (1/pw turns the reference's cycles-per-pixel ramp into physical units). With
//     view records, wgt is the FDK cosine pre-weight: the cosine of the angle between the pixel's
//     ray and the detector normal (physical units; fastcone.py:260-267 uses pixel units);
//   * HILBERT — the curved-detector kappa-line Hilbert kernel of the Katsevich filter:
//     kern[d] = 2 / (pi d) * (d dg / sin(d dg)) for odd d, 0 for even d.
//
// Method. The linear convolution equals a circular one of any length L >= 2 nw - 1, so each row
// is zero-padded to L = 2^p (64 <= L <= 8192), and two rows share one complex transform (row a in
// the real part, row b in the imaginary part: the kernel is real, so the two convolutions do not
// mix). L / 16 threads transform a pair of rows, sixteen elements each in registers: the forward
// transform is decimated in frequency, radix 16 and a last radix of 2 to 16, and leaves the spectrum
// in digit-reversed order in registers; there it is multiplied by DFT_L(kern) / L (loaded in that
// order) and conjugated; that DFT is real (RAMP) or imaginary (HILBERT: then row a goes in as the
// imaginary and row b as the real part, which turns the factor i into one sign of the output), so
// the product is two multiplications; the same stages transposed, in reverse order, transform it back to natural
// order (ifft(X) = conj(fft(conj(X))) / L): the result's real part is row a, minus its imaginary part
// row b (HILBERT: plus). A stage writes to LDS exactly the elements it read, so one barrier per exchange suffices and
// none separates two pairs. DFT_L(kern) is evaluated on the device in FP64 from the closed-form taps
// (not from the length-2nw bins, which zero padding to L would not reproduce), and rounded to FP32;
// so are the twiddles exp(-2 pi i m / L). Both rows of a pair are read completely before either is
// written, so the filter may run in place.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>

#include "fc_device.h"
#include "fc_internal.h"

namespace fc {
namespace {

__device__ __forceinline__ float2 cadd(float2 a, float2 b) {
  return make_float2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ float2 csub(float2 a, float2 b) {
  return make_float2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 mul_mi(float2 a) { return make_float2(a.y, -a.x); }  // a * -i

// In-register forward DFTs of 2, 4 and 8 points (kernel e^{-2 pi i n k / R}).
template <int R>
__device__ __forceinline__ void dft(float2* v);

template <>
__device__ __forceinline__ void dft<2>(float2* v) {
  const float2 a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}

template <>
__device__ __forceinline__ void dft<4>(float2* v) {
  const float2 t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
  const float2 t2 = cadd(v[1], v[3]), t3 = mul_mi(csub(v[1], v[3]));
  v[0] = cadd(t0, t2);
  v[2] = csub(t0, t2);
  v[1] = cadd(t1, t3);
  v[3] = csub(t1, t3);
}

template <>
__device__ __forceinline__ void dft<8>(float2* v) {
  float2 e[4] = {v[0], v[2], v[4], v[6]};
  float2 o[4] = {v[1], v[3], v[5], v[7]};
  dft<4>(e);
  dft<4>(o);
  const float c = 0.70710678118654752f;
  o[1] = make_float2(c * (o[1].x + o[1].y), c * (o[1].y - o[1].x));     // * e^{-i pi/4}
  o[2] = mul_mi(o[2]);                                                  // * e^{-i pi/2}
  o[3] = make_float2(c * (o[3].y - o[3].x), -c * (o[3].x + o[3].y));    // * e^{-3 i pi/4}
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[k] = cadd(e[k], o[k]);
    v[k + 4] = csub(e[k], o[k]);
  }
}

// v W16 and v W16^3, W16 = cos - i sin of pi/8. cos is applied as 1 - 0.076..: rounded to FP32 by
// itself it is 3.1e-8 too small, an error that all the transform's stages would share.
__device__ __forceinline__ float2 rot16(float2 v) {
  const float d = 0.07612046748871326f, s = 0.38268343236508977f;
  return make_float2(fmaf(-d, v.x, fmaf(s, v.y, v.x)), fmaf(-d, v.y, fmaf(-s, v.x, v.y)));
}
__device__ __forceinline__ float2 rot16_3(float2 v) {
  const float d = 0.07612046748871326f, s = 0.38268343236508977f;
  return make_float2(fmaf(-d, v.y, fmaf(s, v.x, v.y)), fmaf(d, v.x, fmaf(s, v.y, -v.x)));
}

// c + a b and c - a b
__device__ __forceinline__ float2 cfma(float2 a, float2 b, float2 c) {
  return make_float2(fmaf(a.x, b.x, fmaf(-a.y, b.y, c.x)), fmaf(a.x, b.y, fmaf(a.y, b.x, c.y)));
}
__device__ __forceinline__ float2 cfms(float2 a, float2 b, float2 c) {
  return make_float2(fmaf(-a.x, b.x, fmaf(a.y, b.y, c.x)), fmaf(-a.x, b.y, fmaf(-a.y, b.x, c.y)));
}

// dft<16> of v[0], w[0] v[1], .., w[14] v[15] (w null: of v itself). Half of the twiddles are
// factors of the first butterflies' FMAs: as many instructions, one rounding less. HALF: v[8..15]
// are zeros.
template <bool HALF = false>
__device__ __forceinline__ void dft16(float2* v, const float2* w) {
  // 4 x 4: columns n1 + 4 n2 over n2, twiddles W16^(n1 k2), rows over n1; X[4 k1 + k2]
  const float r = 0.70710678118654752f;
  float2 t[4][4];
#pragma unroll
  for (int n1 = 0; n1 < 4; ++n1) {
    if (w) {
      const float2 p0 = n1 ? cmul(w[n1 - 1], v[n1]) : v[0], p1 = cmul(w[n1 + 3], v[n1 + 4]);
      const float2 t0 = cfma(w[n1 + 7], v[n1 + 8], p0), t1 = cfms(w[n1 + 7], v[n1 + 8], p0);
      const float2 t2 = cfma(w[n1 + 11], v[n1 + 12], p1),
                   t3 = mul_mi(cfms(w[n1 + 11], v[n1 + 12], p1));
      t[n1][0] = cadd(t0, t2);
      t[n1][2] = csub(t0, t2);
      t[n1][1] = cadd(t1, t3);
      t[n1][3] = csub(t1, t3);
    } else if (HALF) {
      const float2 p1 = mul_mi(v[n1 + 4]);
      t[n1][0] = cadd(v[n1], v[n1 + 4]);
      t[n1][2] = csub(v[n1], v[n1 + 4]);
      t[n1][1] = cadd(v[n1], p1);
      t[n1][3] = csub(v[n1], p1);
    } else {
#pragma unroll
      for (int n2 = 0; n2 < 4; ++n2) t[n1][n2] = v[n1 + 4 * n2];
      dft<4>(t[n1]);
    }
  }
  t[1][1] = rot16(t[1][1]);
  t[1][2] = make_float2(r * (t[1][2].x + t[1][2].y), r * (t[1][2].y - t[1][2].x));
  t[1][3] = rot16_3(t[1][3]);
  t[2][1] = make_float2(r * (t[2][1].x + t[2][1].y), r * (t[2][1].y - t[2][1].x));
  t[2][2] = mul_mi(t[2][2]);
  t[2][3] = make_float2(r * (t[2][3].y - t[2][3].x), -r * (t[2][3].x + t[2][3].y));
  t[3][1] = rot16_3(t[3][1]);
  t[3][2] = make_float2(r * (t[3][2].y - t[3][2].x), -r * (t[3][2].x + t[3][2].y));
  t[3][3] = rot16(t[3][3]);  // times -W16: the sign is in its use
  t[3][3] = make_float2(-t[3][3].x, -t[3][3].y);
#pragma unroll
  for (int k2 = 0; k2 < 4; ++k2) {
    float2 u[4] = {t[0][k2], t[1][k2], t[2][k2], t[3][k2]};
    dft<4>(u);
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) v[4 * k1 + k2] = u[k1];
  }
}

template <>
__device__ __forceinline__ void dft<16>(float2* v) {
  dft16(v, nullptr);
}

// Length-L transforms by L / 16 threads, sixteen elements each (file header). A stage works on
// sub-blocks of M elements: thread `tid` has elements j + r M / 16 of sub-block tid / (M / 16), with
// j = tid mod M / 16; the last one (M < 16, or M = 16) has 16 / M whole sub-blocks, tid + b L / 16.
constexpr int kE = 16;

template <int L, int M>
__device__ __forceinline__ constexpr int element(int tid, int r) {
  if constexpr (M >= kE) {
    constexpr int S = M / kE;
    return tid / S * M + tid % S + r * S;
  } else {
    return (tid + r / M * (L / kE)) * M + r % M;
  }
}

// LDS slot of an element: one float2 of padding after every 16, so that a stage's reads and writes
// (strides of a power of two) use all banks. element(tid, 0) and element(0, r) share no carry into
// bit 4, so slot(element(tid, r)) is the sum of their slots and r costs no address arithmetic.
__device__ __forceinline__ constexpr int slot(int i) { return i + (i >> 4); }

template <int L, int M>
__device__ __forceinline__ void put(float2* buf, const float2* v, int tid) {
  float2* b = buf + slot(element<L, M>(tid, 0));
#pragma unroll
  for (int r = 0; r < kE; ++r) b[slot(element<L, M>(0, r))] = v[r];
}
template <int L, int M>
__device__ __forceinline__ void get(float2* v, const float2* buf, int tid) {
  const float2* b = buf + slot(element<L, M>(tid, 0));
#pragma unroll
  for (int r = 0; r < kE; ++r) v[r] = b[slot(element<L, M>(0, r))];
}

// Twiddles of the stage with sub-blocks of M elements.
template <int L, int M>
__device__ __forceinline__ void stage_twiddles(float2* t, const float2* __restrict__ tw, int tid) {
  if constexpr (M > kE) {
    const int j = tid % (M / kE);
#pragma unroll
    for (int q = 1; q < kE; ++q) t[q - 1] = tw[j * q * (L / M)];
  }
}

// Those of the first stage are in registers (t0); the others are loaded where they are used, from a
// few distinct addresses per wave.
template <int L, int M>
__device__ __forceinline__ void twiddles(float2* t, const float2* t0, const float2* __restrict__ tw,
                                         int tid) {
  if constexpr (M == L) {
#pragma unroll
    for (int q = 0; q < kE - 1; ++q) t[q] = t0[q];
  } else {
    asm volatile("" : "+v"(tid));  // not kept in registers from pair to pair
    stage_twiddles<L, M>(t, tw, tid);
  }
}

// Sub-block length of the last stage.
constexpr int last_block(int M) { return M > kE ? last_block(M / kE) : M; }

// Forward stages from sub-blocks of M elements down: v ends as the spectrum in the last stage's
// elements.
template <int L, int M>
__device__ __forceinline__ void fft_down(float2* v, float2* buf, const float2* t0,
                                         const float2* __restrict__ tw, int tid) {
  if constexpr (M > kE) {
    dft16<M == L>(v, nullptr);  // rows fill at most half of the length
    float2 t[kE - 1];
    twiddles<L, M>(t, t0, tw, tid);
#pragma unroll
    for (int q = 1; q < kE; ++q) v[q] = cmul(v[q], t[q - 1]);
    put<L, M>(buf, v, tid);
    __syncthreads();
    get<L, M / kE>(v, buf, tid);
    fft_down<L, M / kE>(v, buf, t0, tw, tid);
  } else {
#pragma unroll
    for (int g = 0; g < kE / M; ++g) dft<M>(v + g * M);
  }
}

// The same stages transposed, from the last one up to sub-blocks of M elements: v ends as the
// transform's natural order, elements j + r L / 16.
template <int L, int M>
__device__ __forceinline__ void fft_up(float2* v, float2* buf, const float2* t0,
                                       const float2* __restrict__ tw, int tid) {
  if constexpr (M > kE) {
    fft_up<L, M / kE>(v, buf, t0, tw, tid);
    put<L, M / kE>(buf, v, tid);
    __syncthreads();
    get<L, M>(v, buf, tid);
    float2 t[kE - 1];
    twiddles<L, M>(t, t0, tw, tid);
    dft16(v, t);
  } else {
#pragma unroll
    for (int g = 0; g < kE / M; ++g) dft<M>(v + g * M);
  }
}

// Frequency of element p after fft_down: the digits of p (radix 16 from the top, the last one the
// remaining radix) in reverse order.
template <int L>
__device__ __forceinline__ int frequency(int p) {
  int k = 0, mul = 1, size = L;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    if (size > 1) {
      const int radix = size < kE ? size : kE, sub = size / radix;
      k += p / sub * mul;
      p %= sub;
      mul *= radix;
      size = sub;
    }
  }
  return k;
}

struct FiltArgs {
  const void* in;
  void* out;
  const double* views;  // flat-detector view records for the cosine weight, or null
  const float2* tw;     // L twiddles
  const float* mult;    // L multipliers: DFT_L(kern) / L, or its imaginary part (hilbert)
  bool hilbert;         // DFT_L(kern) is imaginary (else real)
  long long nrows;
  int nw, nh;
  int in_dt, out_dt;
};

// fn called with the storage type dt as a constant, once for all of a thread's elements.
template <class F>
__device__ __forceinline__ void by_type(int dt, F&& fn) {
  if (dt == FC_F32) fn(std::integral_constant<int, FC_F32>());
  else if (dt == FC_BF16) fn(std::integral_constant<int, FC_BF16>());
  else fn(std::integral_constant<int, FC_F16>());
}

template <int DT>
__device__ __forceinline__ void store_elem(void* p, size_t i, float v) {
  if constexpr (DT == FC_F32) static_cast<float*>(p)[i] = v;
  else if constexpr (DT == FC_BF16) static_cast<uint16_t*>(p)[i] = f32_to_bf16_bits(v);
  else static_cast<uint16_t*>(p)[i] = f32_to_f16_bits(v);
}

// Cosine pre-weight of a row: pixel j sits at b + j u (relative to the source, FP64); its weight is
// dperp / |b + j u|, dperp the source's distance from the detector plane. |b + j u|^2 is kept as a
// polynomial in j.
struct RowWeight {
  double c0, c1, c2;
  float dperp;
};

__device__ __forceinline__ RowWeight row_weight(const FiltArgs& a, long long r) {
  const long long t = r / a.nh;
  const double i = (double)(r - t * a.nh);
  const double* V = a.views + (size_t)t * FC_VIEW_DOUBLES;
  const double r0x = V[3] - V[0], r0y = V[4] - V[1], r0z = V[5] - V[2];
  const double bx = r0x + i * V[9], by = r0y + i * V[10], bz = r0z + i * V[11];
  const double ux = V[6], uy = V[7], uz = V[8];
  const double nx = V[7] * V[11] - V[8] * V[10], ny = V[8] * V[9] - V[6] * V[11],
               nz = V[6] * V[10] - V[7] * V[9];
  const double nn = sqrt(nx * nx + ny * ny + nz * nz);
  RowWeight w;
  w.c0 = bx * bx + by * by + bz * bz;
  w.c1 = 2.0 * (bx * ux + by * uy + bz * uz);
  w.c2 = ux * ux + uy * uy + uz * uz;
  // only flat-detector records carry the plane geometry this weight needs
  w.dperp = V[24] == (double)FC_DET_FLAT ? (float)(fabs(r0x * nx + r0y * ny + r0z * nz) / nn)
                                         : __builtin_nanf("");
  return w;
}

__device__ __forceinline__ float weight_at(const RowWeight& w, int j) {
  const double jd = (double)j;
  return w.dperp * __builtin_amdgcn_rsqf((float)fma(jd, fma(jd, w.c2, w.c1), w.c0));
}

// Element r of a thread lies within the row whatever its length: L / 4 < nw for all L but the
// smallest, which also serves shorter rows.
template <int L>
__device__ __forceinline__ constexpr bool in_row(int r) {
  return L > 64 && r < kE / 4;
}

// Threads per block: one pair, or the pairs of one wave.
constexpr int filt_threads(int L) { return L / kE > 64 ? L / kE : 64; }

// Per pair and wave (2048 points, cosine weights): about 1600 VALU and 72 double LDS instructions
// against 32 to 48 memory ones. Three waves per SIMD hide the exchanges' and loads' latency best
// (166 registers, two spilled at 512 and 8192 points; 3.46 GB of FP32 rows of 768 columns, in ms: two waves 2.27, three 2.14, three with
// the loads issued after the round begins 2.18); about 60 % VALU busy, 1.6 TB/s. The radix-8
// Stockham stages with every exchange, load and the spectrum product through LDS that this replaces
// took 3.82 ms; rows of 384 columns 0.56 -> 0.29, 3000 columns 1.36 -> 0.67, and 200000 rows of 31
// columns 0.29 -> 0.028 (one pair per block left most threads idle there).
// Relative error against FP64 (white rows of 31 to 3000 columns): 0.83e-7 to 1.23e-7, before
// 0.87e-7 to 1.26e-7.
constexpr int kWaves = 3;  // per SIMD

template <int LOG2L>
__global__ __launch_bounds__((filt_threads(1 << LOG2L)), kWaves) void row_filter_kernel(FiltArgs a) {
  constexpr int L = 1 << LOG2L, T = L / kE, NT = filt_threads(L), P = NT / T;
  constexpr int H = kE / 2;  // a row has at most L / 2 values: elements r < 8 of the first stage
  __shared__ float2 lds[P][L + L / 16];
  __shared__ RowWeight wt[2][2 * P];  // both rows of each pair, for this round and the next
  const int tid = P == 1 ? threadIdx.x : threadIdx.x % T, sub = P == 1 ? 0 : threadIdx.x / T;
  float2* buf = lds[sub];
  float h[kE];
  float2 t0[kE - 1];
  constexpr int ML = last_block(L);
#pragma unroll
  for (int r = 0; r < kE; ++r) h[r] = a.mult[frequency<L>(element<L, ML>(tid, r))];
  stage_twiddles<L, L>(t0, a.tw, tid);
  const long long npairs = (a.nrows + 1) / 2, step = (long long)gridDim.x * P;
  // weights of round p0's rows, into half s
  auto weights = [&](long long p0, int s) {
    if (a.views && threadIdx.x < 2 * P) {
      const long long r = 2 * p0 + threadIdx.x;
      if (r < a.nrows) wt[s][threadIdx.x] = row_weight(a, r);
    }
  };
  // The pair's rows; columns and rows that do not exist hold some other element's value.
  float f0[H], f1[H];
  auto fetch = [&](long long pair) {
    const long long r0 = std::min(2 * pair, a.nrows - 1), r1 = std::min(r0 + 1, a.nrows - 1);
    const long long x = a.hilbert ? r1 : r0, y = a.hilbert ? r0 : r1;
    by_type(a.in_dt, [&](auto dt) {
      constexpr int B = dt() == FC_F32 ? 4 : 2;
      const char* px = static_cast<const char*>(a.in) + (size_t)x * (size_t)a.nw * B;
      const char* py = static_cast<const char*>(a.in) + (size_t)y * (size_t)a.nw * B;
#pragma unroll
      for (int r = 0; r < H; ++r) {
        const unsigned m = in_row<L>(r) ? tid + r * T : std::min(tid + r * T, a.nw - 1);
        f0[r] = load_elem<dt()>(px + m * B, 0);
        f1[r] = load_elem<dt()>(py + m * B, 0);
      }
    });
  };
  long long p0 = (long long)blockIdx.x * P;
  weights(p0, 0);
  fetch(p0 + sub);
  __syncthreads();
  int s = 0;
  for (; p0 < npairs; p0 += step, s ^= 1) {
    const long long r0 = 2 * (p0 + sub);
    float2 v[kE];
    int lt = tid;
    asm volatile("" : "+v"(lt));  // the FP64 columns are not kept in registers from pair to pair
    if (a.views) {
      const RowWeight w0 = wt[s][2 * sub + a.hilbert], w1 = wt[s][2 * sub + 1 - a.hilbert];
#pragma unroll
      for (int r = 0; r < H; ++r) {
        f0[r] *= weight_at(w0, lt + r * T);
        f1[r] *= weight_at(w1, lt + r * T);
      }
    }
    const bool two = r0 + 1 < a.nrows;
    if (!two) {
#pragma unroll
      for (int r = 0; r < H; ++r) (a.hilbert ? f0[r] : f1[r]) = 0.0f;
    }
#pragma unroll
    for (int r = 0; r < H; ++r) {
      const bool in = in_row<L>(r) || lt + r * T < a.nw;
      v[r] = make_float2(in ? f0[r] : 0.0f, in ? f1[r] : 0.0f);
    }
    if (p0 + step < npairs) {
      weights(p0 + step, s ^ 1);  // read after the exchanges' barriers
      fetch(p0 + step + sub);
    }
    fft_down<L, L>(v, buf, t0, a.tw, tid);
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      v[r] = make_float2(h[r] * v[r].x, -h[r] * v[r].y);
    }
    fft_up<L, L>(v, buf, t0, a.tw, tid);
    if (r0 < a.nrows) {
      const float sign1 = a.hilbert ? 1.0f : -1.0f;
      by_type(a.out_dt, [&](auto dt) {
        constexpr int B = dt() == FC_F32 ? 4 : 2;
        char* q0 = static_cast<char*>(a.out) + (size_t)r0 * (size_t)a.nw * B;
        char* q1 = q0 + (size_t)a.nw * B;
#pragma unroll
        for (int r = 0; r < H; ++r) {
          const unsigned j = tid + r * T;
          if (in_row<L>(r) || (int)j < a.nw) {
            store_elem<dt()>(q0 + j * B, 0, v[r].x);
            if (two) store_elem<dt()>(q1 + j * B, 0, sign1 * v[r].y);
          }
        }
      });
    }
  }
}

// ---- tables (FP64) ---------------------------------------------------------------------------

// Tap kern[d], d in [0, nw); kern[-d] = kern[d] (ramp) or -kern[d] (Hilbert). Ramp: irfft of H over
// n = 2 nw bins, (1/n) [H0 + 2 sum_{k=1}^{nw-1} H_k cos(2 pi k d / n) + H_nw cos(pi d)] with
// H_k = c k, H0 = c / 8, c = pi / n. The sum has a closed form: with t = pi d / nw,
// sum k cos(k t) = -nw / 2 for even d > 0 and nw / 2 - 1 / (2 sin^2(t / 2)) for odd d.
__device__ __forceinline__ double filt_tap(int kind, double p0, int nw, int d) {
  if (kind == FC_FILTER_RAMP) {
    const double n = 2.0 * (double)nw, c = M_PI / n;
    double v = 0.125 * c;
    if (d == 0) {
      v += c * (double)nw * (double)nw;
    } else if (d & 1) {
      const double s = sinpi((double)d / n);
      v -= c / (s * s);
    }
    return p0 * v / n;
  }
  if (!(d & 1)) return 0.0;
  const double x = (double)d * p0;
  return 2.0 / (M_PI * (double)d) * (x / sin(x));
}

// cos(2 pi m / L) from the table of its first quarter, q[j] = cos(2 pi j / L), j in [0, L/4].
__device__ __forceinline__ double cos_table(const double* q, int L, int m) {
  m &= L - 1;
  if (m > L / 2) m = L - m;
  return m > L / 4 ? -q[L / 2 - m] : q[m];
}

// Twiddles tw[m] = e^{-2 pi i m / L} and multipliers mult[k] = (1/L) sum_d kern[d] e^{-2 pi i k d / L}
// in FP64, rounded to FP32. Every block holds the taps and a quarter wave of the length-L cosine in
// LDS; a wave owns a bin k <= L/2 (its lanes share the taps' sum, k d mod L being an exact mask) and
// writes it and its conjugate at L - k.
// Bound by latency: a few FP64 transcendentals per thread, then one LDS gather and FMA per term. The
// three kernels this replaces evaluated a sum of nw cosines per tap and 2 nw - 1 FP64 sine/cosine
// pairs with a 64-bit remainder per bin, one thread each: 108 us at nw = 96 (L = 256) and 850 us at
// nw = 768 (L = 2048) against 4.2 and 6.1 us
// for this one.
__global__ __launch_bounds__(256) void filt_tables(int kind, double p0, int nw, int L,
                                                   float2* __restrict__ tw,
                                                   float* __restrict__ mult) {
  extern __shared__ double lds_tab[];
  double* quarter = lds_tab;               // L/4 + 1
  double* taps = lds_tab + L / 4 + 1;      // nw
  for (int j = threadIdx.x; j <= L / 4; j += 256) quarter[j] = cospi(2.0 * (double)j / (double)L);
  for (int d = threadIdx.x; d < nw; d += 256) taps[d] = filt_tap(kind, p0, nw, d);
  __syncthreads();
  for (int m = blockIdx.x * 256 + threadIdx.x; m < L; m += gridDim.x * 256)
    tw[m] = make_float2((float)cos_table(quarter, L, m), (float)-cos_table(quarter, L, m - L / 4));
  const int lane = threadIdx.x & 63;
  const int shift = kind == FC_FILTER_RAMP ? 0 : L / 4;  // sum of cosines or of sines
  for (int k = blockIdx.x * 4 + (threadIdx.x >> 6); k <= L / 2; k += gridDim.x * 4) {
    double s = 0.0;
    for (int d = 1 + lane; d < nw; d += 64)
      s = fma(taps[d], cos_table(quarter, L, k * d - shift), s);
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) {
      const bool ramp = kind == FC_FILTER_RAMP;
      const float v = (float)((ramp ? taps[0] + 2.0 * s : -2.0 * s) / L);
      mult[k] = v;
      if (k > 0 && k < L / 2) mult[L - k] = ramp ? v : -v;
    }
  }
}

int filter_log2(int nw) {
  int p = 6;
  while ((1 << p) < 2 * nw - 1) ++p;
  return p;
}

inline constexpr size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Tables of the widest supported row (FC_FILTER_MAX_COLS columns, FFT length 8192): twiddles and
// multipliers (8192 float2 and floats). Every row filter needs at most this.
constexpr size_t table_bytes(size_t L) {
  return align256(L * sizeof(float2)) + align256(L * sizeof(float));
}
constexpr size_t kMaxTableBytes = table_bytes(8192);

// Device-resident tables for fc_fdk_filter_noalloc_dev (one copy per GPU, held until the process
// ends). In host code the name is only a stand-in: the device address comes from
// hipGetSymbolAddress, once per device.
static __device__ __align__(256) unsigned char scratch[kMaxTableBytes];

template <int LOG2L>
void launch_rows(const FiltArgs& a, hipStream_t s) {
  constexpr int NT = filt_threads(1 << LOG2L), P = NT / ((1 << LOG2L) / kE);
  const long long rounds = ((a.nrows + 1) / 2 + P - 1) / P;
  // the blocks that are resident at once: each loads its multipliers and twiddles once
  const int blocks = (int)std::min(rounds, 256LL * (4 * kWaves / (NT / 64)));
  row_filter_kernel<LOG2L><<<blocks, NT, 0, s>>>(a);
}

std::mutex g_scratch_mutex;
void* g_scratch_ptr[64] = {nullptr};

// The calling thread's current device's address of `scratch`, looked up on first use.
int scratch_address(int device, void** out) {
  FC_CHECK_ARG(device >= 0 && device < 64, "device id %d too large", device);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[device]) {
    void* p = nullptr;
    FC_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[device] = p;
  }
  *out = g_scratch_ptr[device];
  return FC_OK;
}

}  // namespace

size_t filter_table_bytes(int nw) {
  return table_bytes((size_t)1 << filter_log2(nw));
}

int launch_row_filter(const void* in, int in_dt, void* out, int out_dt, int nw, int nh,
                      long long nrows, const double* views, int kind, double p0, void* tables,
                      hipStream_t stream) {
  FC_CHECK_ARG(nw >= 1 && nw <= FC_FILTER_MAX_COLS, "row length %d out of [1, %d]", nw,
               FC_FILTER_MAX_COLS);
  FC_CHECK_ARG(nh >= 1, "rows per view must be positive");
  if (nrows == 0) return FC_OK;
  const int p = filter_log2(nw);
  const int L = 1 << p;
  char* base = static_cast<char*>(tables);
  float2* tw = reinterpret_cast<float2*>(base);
  float* mult = reinterpret_cast<float*>(base + align256((size_t)L * sizeof(float2)));
  // one bin per wave up to L = 2048, at most a block per CU (its LDS holds up to 49 KB of tables)
  const int tblocks = std::min(256, (L / 2 + 4) / 4);
  filt_tables<<<tblocks, 256, (L / 4 + 1 + (size_t)nw) * sizeof(double), stream>>>(kind, p0, nw, L,
                                                                                   tw, mult);
  FiltArgs a;
  a.in = in;
  a.out = out;
  a.views = views;
  a.tw = tw;
  a.mult = mult;
  a.hilbert = kind == FC_FILTER_HILBERT;
  a.nrows = nrows;
  a.nw = nw;
  a.nh = nh;
  a.in_dt = in_dt;
  a.out_dt = out_dt;
  switch (p) {
    case 6: launch_rows<6>(a, stream); break;
    case 7: launch_rows<7>(a, stream); break;
    case 8: launch_rows<8>(a, stream); break;
    case 9: launch_rows<9>(a, stream); break;
    case 10: launch_rows<10>(a, stream); break;
    case 11: launch_rows<11>(a, stream); break;
    case 12: launch_rows<12>(a, stream); break;
    default: launch_rows<13>(a, stream); break;
  }
  FC_HIP(hipGetLastError());
  return FC_OK;
}

}  // namespace fc

using namespace fc;

extern "C" {

int fc_fdk_filter_dev(int device, const void* proj, int proj_dtype, void* out, int out_dtype,
                      const int proj_shape[3], const double* views, double ramp_scale,
                      void* stream) {
  clear_error();
  FC_CHECK_ARG(proj_shape, "null shape");
  const int nw = proj_shape[0], nh = proj_shape[1], nv = proj_shape[2];
  FC_CHECK_ARG(nw >= 1 && nw <= FC_FILTER_MAX_COLS, "detector width %d out of [1, %d]", nw,
               FC_FILTER_MAX_COLS);
  FC_CHECK_ARG(nh >= 1 && nv >= 0, "projection shape invalid (%d,%d,%d)", nw, nh, nv);
  FC_CHECK_ARG(dtype_ok(proj_dtype) && dtype_ok(out_dtype), "unknown dtype");
  FC_CHECK_ARG(std::isfinite(ramp_scale), "ramp scale not finite");
  FC_CHECK_ARG(nv == 0 || (proj && out), "null pointer argument");
  int rc = select_device(device);
  if (rc) return rc;
  if (nv == 0) return FC_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  void* tables = nullptr;
  if ((rc = acquire_ws(device, SLOT_FILTER, filter_table_bytes(nw), s, &tables))) return rc;
  int tok = prof_begin("fdk_filter", s);
  rc = launch_row_filter(proj, proj_dtype, out, out_dtype, nw, nh, (long long)nh * nv, views,
                         FC_FILTER_RAMP, ramp_scale, tables, s);
  prof_end(tok, s);
  if (rc) return rc;
  return release_ws(device, SLOT_FILTER, s);
}

// The same filter with no device allocation: its tables live in the file-scope `scratch` array
// (kMaxTableBytes, enough for FC_FILTER_MAX_COLS columns) instead of a library workspace. No
// counterpart in the reference.
int fc_fdk_filter_noalloc_dev(int device, const void* proj, int proj_dtype, void* out,
                              int out_dtype, const int proj_shape[3], const double* views,
                              double ramp_scale, void* stream) {
  clear_error();
  FC_CHECK_ARG(proj_shape, "null shape");
  const int nw = proj_shape[0], nh = proj_shape[1], nv = proj_shape[2];
  FC_CHECK_ARG(nw >= 1 && nw <= FC_FILTER_MAX_COLS,
               "detector width %d out of [1, %d] (the no-allocation tables hold %zu bytes)", nw,
               FC_FILTER_MAX_COLS, kMaxTableBytes);
  FC_CHECK_ARG(filter_table_bytes(nw) <= kMaxTableBytes, "filter tables exceed the scratch array");
  FC_CHECK_ARG(nh >= 1 && nv >= 0, "projection shape invalid (%d,%d,%d)", nw, nh, nv);
  FC_CHECK_ARG(dtype_ok(proj_dtype) && dtype_ok(out_dtype), "unknown dtype");
  FC_CHECK_ARG(std::isfinite(ramp_scale), "ramp scale not finite");
  FC_CHECK_ARG(nv == 0 || (proj && out), "null pointer argument");
  int rc = select_device(device);
  if (rc) return rc;
  void* tables = nullptr;
  if ((rc = scratch_address(device, &tables))) return rc;
  if (nv == 0) return FC_OK;
  // every table entry the filter reads is rewritten by this call's table kernels (same stream)
  return launch_row_filter(proj, proj_dtype, out, out_dtype, nw, nh, (long long)nh * nv, views,
                           FC_FILTER_RAMP, ramp_scale, tables, static_cast<hipStream_t>(stream));
}

}  // extern "C"
