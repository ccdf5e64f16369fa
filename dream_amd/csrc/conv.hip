// conv.hip -- batched linear convolution (fftconv_p, sum_fftconv) on gfx950.
//
// Reference: FFTConvP::run (extra_src/fftconv_p.cc:154-403, per column
// fftconv, extra_src/fftconv.cc:32-106) and sum_fftconv (add_fftconv,
// extra_src/fftconv.cc:119-209; extra_src/oct_sum_fftconv.cc).  Both are
// linear convolutions computed by the reference through zero-padded FFTs of
// length M_A + M_B - 1; the result is the same sum
//     y[k] = sum_l sum_i b_l[i] a_l[k - i],   k = 0 .. M_A + M_B - 2,
// taken directly in the data type for short filters, through transforms for
// long ones (the FFT path below).
//
// Mapping of the direct sum.  One work-group per (output column, tile of kTile outputs).  The
// filter b is consumed in chunks of kChunk taps; for each chunk the taps and
// the window of a they meet are staged in LDS, and each thread accumulates
// kR outputs spaced kThreads apart, so consecutive lanes read consecutive
// LDS words (no bank conflicts) and the taps are broadcast.

#include "conv.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>
#include <vector>

namespace dream {

namespace {

constexpr int kThreads = 256;
constexpr int kR = 4;
constexpr int kTile = kThreads * kR;      // outputs per work-group
constexpr int kChunk = 256;               // taps staged per step

template <typename T>
__global__ void __launch_bounds__(kThreads)
conv_sum_kernel(T *__restrict__ Y, const T *__restrict__ A, int64_t MA, int64_t L,
                int64_t a_col, int64_t a_layer, const T *__restrict__ B, int64_t MB,
                int64_t b_col, int64_t b_layer, int mode)
{
  __shared__ T sb[kChunk];
  __shared__ T sa[kTile + kChunk];
  const int64_t n = blockIdx.y;
  const int64_t k0 = (int64_t) blockIdx.x * kTile;
  const int64_t MY = MA + MB - 1;
  const int t = threadIdx.x;
  T acc[kR];
#pragma unroll
  for (int r = 0; r < kR; r++) acc[r] = T(0);

  // Taps i that meet an output of this tile: k - i in [0, MA).
  const int64_t i_lo = std::max<int64_t>(0, k0 - MA + 1);
  const int64_t i_hi = std::min<int64_t>(MB - 1, k0 + kTile - 1);
  for (int64_t l = 0; l < L; l++) {
    const T *a = A + l * a_layer + n * a_col;
    const T *b = B + l * b_layer + n * b_col;
    for (int64_t i0 = i_lo; i0 <= i_hi; i0 += kChunk) {
      __syncthreads();                            // the previous chunk is consumed
      for (int q = t; q < kChunk; q += kThreads) {
        const int64_t i = i0 + q;
        sb[q] = i <= i_hi ? b[i] : T(0);
      }
      // a window: j = k - i for k in [k0, k0 + kTile), i in [i0, i0 + kChunk).
      const int64_t j0 = k0 - i0 - (kChunk - 1);
      for (int q = t; q < kTile + kChunk - 1; q += kThreads) {
        const int64_t j = j0 + q;
        sa[q] = (j >= 0 && j < MA) ? a[j] : T(0);
      }
      __syncthreads();
      const int cnt = (int) std::min<int64_t>(kChunk, i_hi - i0 + 1);
      // Output k0 + r*kThreads + t reads sa[r*kThreads + t - ii + kChunk - 1].
      const int base = t + kChunk - 1;
      int ii = 0;
      for (; ii + 4 <= cnt; ii += 4) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const T bv = sb[ii + u];
#pragma unroll
          for (int r = 0; r < kR; r++) acc[r] += bv * sa[r * kThreads + base - (ii + u)];
        }
      }
      for (; ii < cnt; ii++) {
        const T bv = sb[ii];
#pragma unroll
        for (int r = 0; r < kR; r++) acc[r] += bv * sa[r * kThreads + base - ii];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kR; r++) {
    const int64_t k = k0 + (int64_t) r * kThreads + t;
    if (k >= MY) continue;
    T *y = Y + n * MY + k;
    if (mode == CONV_SUM) *y += acc[r];
    else if (mode == CONV_NEG) *y -= acc[r];
    else *y = acc[r];
  }
}

// ------------------------------------------------------------------ FFT path
//
// For long filters the same sums go through FFTs of a power-of-two length
// N >= M_A + M_B - 1 (zero padding makes the cyclic convolution linear, as
// in the reference's zero-padded FFTs).  Column 2p of the output is the real
// part, 2p+1 the imaginary part of one complex transform.
//
// A transform lives in the registers of N/16 threads, 16 points each: passes
// of radix 16 (the last one 2, 4, 8 or 16), LDS only to exchange the points
// between passes.  Forward transforms are decimation in frequency (natural
// order in, digit-reversed out), the product is formed in that order, the
// inverse is decimation in time: no reordering passes.  What bounds it: the
// butterflies' FP64/FP32 instructions, about 45 per point and transform at N =
// 4096 (FP32: the VALU busy 55 %), then the exchanges (4 per column pair, 2 N
// complex each).  Radix-2 passes in LDS took 12 reads and writes of the array
// per transform instead of 2 and were bound by them: a call of 4096 x 2000 by
// 300 taps FP32 went from 158 to 36 us, 1024 x 2000 by 2000 taps FP64 from 77
// to 20 us.
//
// LDS positions are padded by one point in 16, which spreads the strided
// accesses of every pass over the banks (without, the last pass's stride of
// 16 points meets one bank pair in 16 lanes).
//
// One filter shared by the columns: every work-group transforms it itself,
// keeps its spectrum in registers and serves several column pairs.  With
// layers the spectra come from fft_filter_kernel and the products add in the
// frequency domain before one inverse transform.  Per-column filters are
// transformed two at a time and separated by conjugate symmetry, as are the
// two data columns then: C = A1 B1 + i A2 B2.  Twiddles come from a host
// table (correctly rounded cos and sin) laid out as the passes read them.
// Reading 6 of a pass's 15 factors and multiplying out the rest was no faster
// (41 against 39 us) and raised the FP32 error from 1.9e-7 to 2.2e-7.

template <typename T>
struct Cx {
  T x, y;
};
template <typename T>
__device__ __forceinline__ Cx<T> operator+(Cx<T> a, Cx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ Cx<T> operator-(Cx<T> a, Cx<T> b) { return {a.x - b.x, a.y - b.y}; }

__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }

// a * b, or a * conj(b).
template <bool CONJ, typename T>
__device__ __forceinline__ Cx<T> cmul(Cx<T> a, Cx<T> b)
{
  if (CONJ) return {fma_t(a.x, b.x, a.y * b.y), fma_t(a.y, b.x, -(a.x * b.y))};
  return {fma_t(a.x, b.x, -(a.y * b.y)), fma_t(a.x, b.y, a.y * b.x)};
}

// a * exp(-i pi/2) (forward) or a * exp(i pi/2) (inverse).
template <bool INV, typename T>
__device__ __forceinline__ Cx<T> quarter(Cx<T> a)
{
  if (INV) return {-a.y, a.x};
  return {a.y, -a.x};
}

template <bool INV, typename T>
__device__ __forceinline__ void dft4(Cx<T> &a, Cx<T> &b, Cx<T> &c, Cx<T> &d)
{
  const Cx<T> t0 = a + c, t1 = a - c, t2 = b + d, t3 = quarter<INV>(b - d);
  a = t0 + t2;
  b = t1 + t3;
  c = t0 - t2;
  d = t1 - t3;
}

// In-place transforms of R points in natural order.
template <int R, bool INV, typename T>
__device__ __forceinline__ void dft(Cx<T> *x)
{
  constexpr T h = (T) 0.70710678118654752440;
  if constexpr (R == 2) {
    const Cx<T> t = x[0] - x[1];
    x[0] = x[0] + x[1];
    x[1] = t;
  } else if constexpr (R == 4) {
    dft4<INV>(x[0], x[1], x[2], x[3]);
  } else if constexpr (R == 8) {
    Cx<T> e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
    dft4<INV>(e[0], e[1], e[2], e[3]);
    dft4<INV>(o[0], o[1], o[2], o[3]);
    o[1] = cmul<INV>(o[1], Cx<T>{h, -h});
    o[2] = quarter<INV>(o[2]);
    o[3] = cmul<INV>(o[3], Cx<T>{-h, -h});
#pragma unroll
    for (int k = 0; k < 4; k++) {
      x[k] = e[k] + o[k];
      x[k + 4] = e[k] - o[k];
    }
  } else {
    static_assert(R == 16, "radix");
    // n = j + 4 n1, k = q + 4 p: four transforms over n1, the factors
    // exp(-2 pi i j q/16), four over j.
    constexpr T c = (T) 0.92387953251128675613, s = (T) 0.38268343236508977173;
#pragma unroll
    for (int j = 0; j < 4; j++) dft4<INV>(x[j], x[j + 4], x[j + 8], x[j + 12]);
    x[5] = cmul<INV>(x[5], Cx<T>{c, -s});
    x[9] = cmul<INV>(x[9], Cx<T>{h, -h});
    x[13] = cmul<INV>(x[13], Cx<T>{s, -c});
    x[6] = cmul<INV>(x[6], Cx<T>{h, -h});
    x[10] = quarter<INV>(x[10]);
    x[14] = cmul<INV>(x[14], Cx<T>{-h, -h});
    x[7] = cmul<INV>(x[7], Cx<T>{s, -c});
    x[11] = cmul<INV>(x[11], Cx<T>{-h, -h});
    x[15] = cmul<INV>(x[15], Cx<T>{-c, s});
    Cx<T> y[16];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      dft4<INV>(x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]);
#pragma unroll
      for (int p = 0; p < 4; p++) y[q + 4 * p] = x[4 * q + p];
    }
#pragma unroll
    for (int k = 0; k < 16; k++) x[k] = y[k];
  }
}

// Transforms of length N = 2^LG on N/16 threads, thread t's 16 points in
// registers.  Pass P works on blocks of M = N/16^P points: slot m of thread t
// is position blk M + s + (M/16) m (t = blk M/16 + s), the last pass's slots
// are the positions 16 t + m.
template <typename T, int LG>
struct Fft {
  static constexpr int N = 1 << LG, NT = N / 16, LAST = (LG - 1) / 4;
  static constexpr size_t kLds = (size_t) (N + N / 16) * sizeof(Cx<T>);

  template <int P>
  static __device__ __forceinline__ int pos(int t, int m)
  {
    constexpr int M = N >> (4 * P);
    if constexpr (M <= 16) {
      return 16 * t + m;
    } else {
      constexpr int SL = M / 16;
      return (t / SL) * M + t % SL + SL * m;
    }
  }
  // LDS index of a position, and of pass P's slots: a base per thread plus a
  // constant per slot.
  static __device__ __forceinline__ int pad(int p) { return p + (p >> 4); }
  template <int P>
  static __device__ __forceinline__ int pad_base(int t)
  {
    constexpr int M = N >> (4 * P);
    if constexpr (M <= 16) return 17 * t;
    else if constexpr (M >= 256) return pad(pos<P>(t, 0));
    else return pos<P>(t, 0) + t / (M / 16) * (M / 16);
  }
  template <int P>
  static constexpr int pad_slot(int m)
  {
    constexpr int M = N >> (4 * P);
    return M <= 16 ? m : M / 16 * m + (M / 16 * m >> 4);
  }

  // The factors of passes 0 .. LAST - 1, each 15 rows (r = 1 .. 15) of M/16:
  // neighbouring threads read neighbouring factors.
  static constexpr int tw_at(int P)
  {
    int n = 0;
    for (int q = 0; q < P; q++) n += 15 * ((N >> (4 * q)) / 16);
    return n;
  }
  static constexpr int kTw = tw_at(LAST);

  // The frequency held at a position after the forward passes, and back.
  static __device__ __forceinline__ int freq(int p)
  {
    int k = 0;
#pragma unroll
    for (int d = 0; d <= LAST; d++) {
      const int sh = LG - 4 * (d + 1);
      k |= (sh >= 0 ? (p >> sh) & 15 : p & ((1 << (sh + 4)) - 1)) << (4 * d);
    }
    return k;
  }
  static __device__ __forceinline__ int place(int k)
  {
    int p = 0;
#pragma unroll
    for (int d = 0; d <= LAST; d++) {
      const int sh = LG - 4 * (d + 1);
      p |= sh >= 0 ? ((k >> (4 * d)) & 15) << sh : (k >> (4 * d)) & ((1 << (sh + 4)) - 1);
    }
    return p;
  }

  // From pass FROM's slots to pass TO's.
  template <int FROM, int TO>
  static __device__ __forceinline__ void exchange(Cx<T> (&x)[16], Cx<T> *lds, int t)
  {
    __syncthreads();                            // earlier reads are done
    Cx<T> *w = lds + pad_base<FROM>(t);
#pragma unroll
    for (int m = 0; m < 16; m++) w[pad_slot<FROM>(m)] = x[m];
    __syncthreads();
    const Cx<T> *r = lds + pad_base<TO>(t);
#pragma unroll
    for (int m = 0; m < 16; m++) x[m] = r[pad_slot<TO>(m)];
  }

  // Slot r times exp(-+2 pi i s r/M).
  template <int P, bool INV>
  static __device__ __forceinline__ void twiddle(Cx<T> (&x)[16], const Cx<T> *__restrict__ tw, int t)
  {
    constexpr int M = N >> (4 * P), SL = M / 16;
    // The factors are read anew each time: kept over a work-group's column
    // pairs they would take 12 points' registers per pass.
    asm volatile("" : "+v"(t));
    const int s = t % SL;
    Cx<T> w[16];
#pragma unroll
    for (int r = 1; r < 16; r++) w[r] = tw[tw_at(P) + (r - 1) * SL + s];
#pragma unroll
    for (int r = 1; r < 16; r++) x[r] = cmul<INV>(x[r], w[r]);
  }

  template <int P, bool INV>
  static __device__ __forceinline__ void butterflies(Cx<T> (&x)[16])
  {
    constexpr int M = N >> (4 * P), R = M < 16 ? M : 16;
#pragma unroll
    for (int g = 0; g < 16; g += R) dft<R, INV>(x + g);
  }

  // Natural order in (pass 0's slots), digit-reversed out (the last pass's).
  template <int P = 0>
  static __device__ __forceinline__ void forward(Cx<T> (&x)[16], Cx<T> *lds,
                                                 const Cx<T> *__restrict__ tw, int t)
  {
    butterflies<P, false>(x);
    if constexpr (P < LAST) {
      twiddle<P, false>(x, tw, t);
      exchange<P, P + 1>(x, lds, t);
      forward<P + 1>(x, lds, tw, t);
    }
  }

  // Back, without the factor 1/N.
  template <int P = LAST>
  static __device__ __forceinline__ void inverse(Cx<T> (&x)[16], Cx<T> *lds,
                                                 const Cx<T> *__restrict__ tw, int t)
  {
    if constexpr (P < LAST) twiddle<P, true>(x, tw, t);
    butterflies<P, true>(x);
    if constexpr (P > 0) {
      exchange<P, P - 1>(x, lds, t);
      inverse<P - 1>(x, lds, tw, t);
    }
  }

  // Two real columns (b: may be null) of length len, zero-padded.
  static __device__ __forceinline__ void load(Cx<T> (&x)[16], const T *__restrict__ a,
                                              const T *__restrict__ b, int64_t len, int t)
  {
#pragma unroll
    for (int m = 0; m < 16; m++) {
      const int64_t k = pos<0>(t, m);
      x[m].x = k < len ? a[k] : T(0);
      x[m].y = b && k < len ? b[k] : T(0);
    }
  }
};

// Spectra of the layers' shared filters over N, in slot order:
// F[l][m][t], slot m of thread t.
template <typename T, int LG>
__global__ void __launch_bounds__((1 << LG) / 16)
fft_filter_kernel(const T *__restrict__ B, int64_t MB, int64_t b_layer,
                  const Cx<T> *__restrict__ tw, Cx<T> *__restrict__ F)
{
  using X = Fft<T, LG>;
  extern __shared__ __align__(16) unsigned char smem[];
  const int t = (int) threadIdx.x;
  Cx<T> x[16];
  X::load(x, B + (int64_t) blockIdx.x * b_layer, nullptr, MB, t);
  X::forward(x, reinterpret_cast<Cx<T> *>(smem), tw, t);
  const T inv = T(1) / T(X::N);
  Cx<T> *f = F + (int64_t) blockIdx.x * X::N + t;
#pragma unroll
  for (int m = 0; m < 16; m++) f[m * X::NT] = {x[m].x * inv, x[m].y * inv};
}

// How the filters are given: one for all columns (one layer), one per layer
// (spectra F), one per column.
enum { FFT_ONE = 0, FFT_LAYERS = 1, FFT_COLUMNS = 2 };

// Waves per SIMD: with one filter as many work-groups of 2^12 points as LDS
// holds (four FP32, two FP64), the registers held to that; half of it with
// layers or per-column filters, which keep a sum or a second spectrum.
template <typename T, int KIND = FFT_ONE>
constexpr int kFftWaves = (sizeof(T) == 4 ? 4 : 2) / (KIND == FFT_ONE ? 1 : 2);

// Pairs of output columns (2p, 2p + 1), p = blockIdx.x, + gridDim.x, ...
template <typename T, int LG, int KIND>
__global__ void __launch_bounds__((1 << LG) / 16)
__attribute__((amdgpu_waves_per_eu(kFftWaves<T, KIND>)))
conv_fft_kernel(T *__restrict__ Y, const T *__restrict__ A, int64_t MA, int64_t N, int64_t L,
                int64_t a_col, int64_t a_layer, const T *__restrict__ B, int64_t MB,
                int64_t b_col, int64_t b_layer, int mode, const Cx<T> *__restrict__ tw,
                const Cx<T> *__restrict__ F)
{
  using X = Fft<T, LG>;
  extern __shared__ __align__(16) unsigned char smem[];
  Cx<T> *lds = reinterpret_cast<Cx<T> *>(smem);
  const int t = (int) threadIdx.x;
  const T inv = T(1) / T(X::N);
  const int64_t MY = MA + MB - 1;
  Cx<T> f[16];
  if constexpr (KIND == FFT_ONE) {
    X::load(f, B, nullptr, MB, t);
    X::forward(f, lds, tw, t);
#pragma unroll
    for (int m = 0; m < 16; m++) f[m] = {f[m].x * inv, f[m].y * inv};
  }
  for (int64_t p = blockIdx.x; 2 * p < N; p += gridDim.x) {
    const int64_t n1 = 2 * p, n2 = n1 + 1;
    const bool has2 = n2 < N;
    Cx<T> x[16], sum[16];
    for (int64_t l = 0; l < (KIND == FFT_ONE ? 1 : L); l++) {
      const T *a1 = A + l * a_layer + n1 * a_col;
      X::load(x, a1, has2 ? a1 + a_col : nullptr, MA, t);
      X::forward(x, lds, tw, t);
      if constexpr (KIND == FFT_ONE) {
        // One real filter for both columns: (A1 + i A2) B = A1 B + i A2 B.
#pragma unroll
        for (int m = 0; m < 16; m++) x[m] = cmul<false>(x[m], f[m]);
      } else if constexpr (KIND == FFT_LAYERS) {
        const Cx<T> *fl = F + l * X::N + t;
#pragma unroll
        for (int m = 0; m < 16; m++) x[m] = cmul<false>(x[m], fl[m * X::NT]);
      } else {
        // Spectra W of the two filters in f; both spectra at -k through LDS.
        // A1[k] = (X[k] + conj X[-k])/2, A2[k] = (X[k] - conj X[-k])/(2i).
        const T *b1 = B + l * b_layer + n1 * b_col;
        Cx<T> *xs = lds + (X::N + X::N / 16);
        X::load(f, b1, has2 ? b1 + b_col : nullptr, MB, t);
        X::forward(f, lds, tw, t);
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 16; m++) {
          lds[X::template pad_base<X::LAST>(t) + m] = f[m];
          xs[X::template pad_base<X::LAST>(t) + m] = x[m];
        }
        __syncthreads();
        const T q = T(0.25) * inv;
#pragma unroll
        for (int m = 0; m < 16; m++) {
          const int k = X::freq(X::template pos<X::LAST>(t, m));
          const int at = X::pad(X::place((X::N - k) & (X::N - 1)));
          const Cx<T> u = xs[at], v = lds[at];
          const Cx<T> A1 = {x[m].x + u.x, x[m].y - u.y}, A2 = {x[m].y + u.y, u.x - x[m].x};
          const Cx<T> B1 = {f[m].x + v.x, f[m].y - v.y}, B2 = {f[m].y + v.y, v.x - f[m].x};
          const Cx<T> c1 = cmul<false>(A1, B1), c2 = cmul<false>(A2, B2);
          x[m] = {(c1.x - c2.y) * q, (c1.y + c2.x) * q};
        }
      }
      if constexpr (KIND != FFT_ONE) {
#pragma unroll
        for (int m = 0; m < 16; m++) sum[m] = l ? sum[m] + x[m] : x[m];
      }
    }
    if constexpr (KIND != FFT_ONE) {
#pragma unroll
      for (int m = 0; m < 16; m++) x[m] = sum[m];
    }
    X::inverse(x, lds, tw, t);
    T *y1 = Y + n1 * MY;
    auto put = [&](T *y, T v) {
      if (mode == CONV_SUM) *y += v;
      else if (mode == CONV_NEG) *y -= v;
      else *y = v;
    };
#pragma unroll
    for (int m = 0; m < 16; m++) {
      const int64_t k = X::template pos<0>(t, m);
      if (k < MY) {
        put(y1 + k, x[m].x);
        if (has2) put(y1 + MY + k, x[m].y);
      }
    }
  }
}

int max_lds_bytes()
{
  static int bytes = 0;
  if (!bytes) {
    int dev = 0, v = 0;
    DREAM_HIP_CHECK(hipGetDevice(&dev));
    DREAM_HIP_CHECK(hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    bytes = v > 0 ? v : 65536;
  }
  return bytes;
}

// Transform lengths: 2^10 .. 2^14 FP32, .. 2^13 FP64, half the longest with
// layers, a quarter with filters per column; shorter outputs are padded to
// 2^10, longer ones summed directly.  (These limits -- one, two or three arrays
// of points in 160 KiB -- are the radix-2 kernels' of before; the sums and second
// spectra are in registers now, so longer transforms would fit, but a call's
// rounding would change with its route.)  The rule and the launches share
// them, so what is chosen is built.
constexpr int kMinLog = 10;
template <typename T>
constexpr int kMaxLog = sizeof(T) == 4 ? 14 : 13;
template <typename T>
constexpr bool fft_length(int lg, int kind)
{
  return lg >= kMinLog && lg <= kMaxLog<T> && ((size_t) (kind + 1) << lg) * sizeof(Cx<T>) <= 160 * 1024;
}
// LDS a transform's work-group asks for: an array of points, two with filters
// per column, each padded by one point in 16.
template <typename T>
size_t fft_lds(int lg, int kind)
{
  const size_t points = (size_t) 1 << lg;
  return (kind == FFT_COLUMNS ? 2 : 1) * (points + points / 16) * sizeof(Cx<T>);
}

// DREAM_HIP_CONV = direct | fft forces a path (for comparisons and tests);
// otherwise the FFT path is taken when its length is built and the direct sum
// would cost more than four times its arithmetic.  Returns log2 of the
// transform's length, 0 for the direct sum.  The ratio was set for radix-2
// passes through LDS and kept: the transforms are about four times faster now,
// but a transform's rounding errors are relative to the column's largest
// sample, the direct sum's to each output's own terms, so moving the line
// would change the results of calls on it.
template <typename T>
int fft_log_if_chosen(int64_t MA, int64_t MB, int64_t L, bool per_col)
{
  const char *e = std::getenv("DREAM_HIP_CONV");
  const bool force_direct = e && std::strcmp(e, "direct") == 0;
  const bool force_fft = e && std::strcmp(e, "fft") == 0;
  if (force_direct) return 0;
  const int64_t MY = MA + MB - 1;
  int bits = 1;
  while ((1ll << bits) < MY) bits++;
  const int64_t NF = 1ll << bits;
  const int lg = std::max(bits, kMinLog), kind = per_col ? FFT_COLUMNS : (L > 1 ? FFT_LAYERS : FFT_ONE);
  if (!fft_length<T>(lg, kind) || fft_lds<T>(lg, kind) > (size_t) max_lds_bytes()) return 0;
  if (force_fft) return lg;
  // Per column: direct 2 MA MB L flops; FFT (two columns per transform)
  // about 5 NF log2 NF per transform, (L + 1) transforms per pair (2 L + 1
  // with per-column filters).
  const double direct = 2.0 * (double) MA * (double) MB * (double) L;
  const double fft = 5.0 * (double) NF * bits * (per_col ? 2 * L + 1 : L + 1) / 2.0;
  return direct > 4.0 * fft ? lg : 0;
}

// Device table of the passes' factors exp(-2 pi i s r/M) (Fft::tw_at), per
// (device, N, type), built once and kept for the life of the process.
template <typename T, int LG>
const Cx<T> *twiddles()
{
  using X = Fft<T, LG>;
  constexpr int N = X::N;
  static std::mutex mu;
  static std::map<std::pair<int, int>, void *> cache;
  int dev = 0;
  DREAM_HIP_CHECK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  void *&p = cache[{dev, N}];
  if (!p) {
    std::vector<Cx<T>> h((size_t) X::kTw);
    for (int P = 0; P < X::LAST; P++) {
      const int M = N >> (4 * P), SL = M / 16;
      for (int r = 1; r < 16; r++)
        for (int j = 0; j < SL; j++) {
          const double ang = -2.0 * M_PI * (double) (j * r) / (double) M;
          h[(size_t) (X::tw_at(P) + (r - 1) * SL + j)] = {(T) std::cos(ang), (T) std::sin(ang)};
        }
    }
    void *d = nullptr;
    DREAM_HIP_CHECK(device_malloc(&d, h.size() * sizeof(Cx<T>)));
    DREAM_HIP_CHECK(hipMemcpy(d, h.data(), h.size() * sizeof(Cx<T>), hipMemcpyHostToDevice));
    p = d;
  }
  return static_cast<const Cx<T> *>(p);
}

int cu_count()
{
  static int cus = 0;
  if (!cus) {
    int dev = 0;
    DREAM_HIP_CHECK(hipGetDevice(&dev));
    DREAM_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    if (cus <= 0) cus = 256;
  }
  return cus;
}

template <typename T, int LG>
void launch_conv_fft(T *Y, const T *A, int64_t MA, int64_t N, int64_t L, int64_t a_col,
                     int64_t a_layer, const T *B, int64_t MB, int64_t b_col, int64_t b_layer,
                     int mode, hipStream_t s)
{
  using X = Fft<T, LG>;
  const Cx<T> *tw = twiddles<T, LG>();
  const int64_t pairs = (N + 1) / 2;
  const dim3 block(X::NT);
  if (b_col != 0) {
    if constexpr (fft_length<T>(LG, FFT_COLUMNS)) {
      hipLaunchKernelGGL((conv_fft_kernel<T, LG, FFT_COLUMNS>), dim3((unsigned) pairs), block,
                         2 * X::kLds, s, Y, A, MA, N, L, a_col, a_layer, B, MB, b_col, b_layer,
                         mode, tw, (const Cx<T> *) nullptr);
      DREAM_HIP_CHECK(hipGetLastError());
      return;
    }
    throw Error(DREAM_HIP_ERUNTIME, "conv: no transform of this length for filters per column");
  }
  if (L == 1) {
    // As many work-groups as the device holds at once, with an equal number
    // of column pairs each: the filter is transformed once per work-group.
    const int64_t held = cu_count() * std::max<int64_t>(1, std::min<int64_t>(160 * 1024 / X::kLds, 256 * kFftWaves<T> / X::NT));
    const int64_t rounds = (pairs + held - 1) / held;
    hipLaunchKernelGGL((conv_fft_kernel<T, LG, FFT_ONE>), dim3((unsigned) ((pairs + rounds - 1) / rounds)),
                       block, X::kLds, s, Y, A, MA, N, L, a_col, a_layer, B, MB, b_col, b_layer,
                       mode, tw, (const Cx<T> *) nullptr);
    DREAM_HIP_CHECK(hipGetLastError());
    return;
  }
  if constexpr (fft_length<T>(LG, FFT_LAYERS)) {
    // The layers' filter spectra, stream-ordered scratch.
    Cx<T> *F = nullptr;
    const size_t bytes = (size_t) L * X::N * sizeof(Cx<T>);
    hipError_t got = hipMallocAsync((void **) &F, bytes, s);
    if (got == hipErrorOutOfMemory && device_make_room()) {
      (void) hipGetLastError();
      got = hipMallocAsync((void **) &F, bytes, s);
    }
    DREAM_HIP_CHECK(got);
    hipLaunchKernelGGL((fft_filter_kernel<T, LG>), dim3((unsigned) L), block, X::kLds, s, B, MB,
                       b_layer, tw, F);
    hipLaunchKernelGGL((conv_fft_kernel<T, LG, FFT_LAYERS>), dim3((unsigned) pairs), block, X::kLds,
                       s, Y, A, MA, N, L, a_col, a_layer, B, MB, b_col, b_layer, mode, tw,
                       (const Cx<T> *) F);
    const hipError_t e = hipGetLastError();
    (void) hipFreeAsync(F, s);
    DREAM_HIP_CHECK(e);
    return;
  }
  throw Error(DREAM_HIP_ERUNTIME, "conv: no transform of this length for layers");
}

} // namespace

template <typename T>
void launch_conv_sum(T *Y, const T *A, int64_t MA, int64_t N, int64_t L, int64_t a_col,
                     int64_t a_layer, const T *B, int64_t MB, int64_t b_col, int64_t b_layer,
                     int mode, hipStream_t s)
{
  require(MA >= 1 && MB >= 1 && N >= 0 && L >= 1, "conv: need M_A, M_B, L >= 1 and N >= 0");
  require(mode == CONV_EQU || mode == CONV_SUM || mode == CONV_NEG, "conv: unknown mode");
  if (N == 0) return;
  require(N < (1ll << 31), "conv: too many columns");
  const int lg = fft_log_if_chosen<T>(MA, MB, L, b_col != 0);
  auto fft = [&](auto log) {
    launch_conv_fft<T, decltype(log)::value>(Y, A, MA, N, L, a_col, a_layer, B, MB, b_col, b_layer,
                                             mode, s);
  };
  switch (lg) {
  case 0: break;
  case 10: fft(std::integral_constant<int, 10>{}); return;
  case 11: fft(std::integral_constant<int, 11>{}); return;
  case 12: fft(std::integral_constant<int, 12>{}); return;
  case 13: fft(std::integral_constant<int, 13>{}); return;
  default: fft(std::integral_constant<int, kMaxLog<T>>{}); return;
  }
  const int64_t MY = MA + MB - 1;
  const int64_t tiles = (MY + kTile - 1) / kTile;
  require(tiles < (1ll << 31), "conv: output too long");
  hipLaunchKernelGGL(conv_sum_kernel<T>, dim3((unsigned) tiles, (unsigned) N), dim3(kThreads), 0,
                     s, Y, A, MA, L, a_col, a_layer, B, MB, b_col, b_layer, mode);
  DREAM_HIP_CHECK(hipGetLastError());
}

template void launch_conv_sum<double>(double *, const double *, int64_t, int64_t, int64_t,
                                      int64_t, int64_t, const double *, int64_t, int64_t,
                                      int64_t, int, hipStream_t);
template void launch_conv_sum<float>(float *, const float *, int64_t, int64_t, int64_t, int64_t,
                                     int64_t, const float *, int64_t, int64_t, int64_t, int,
                                     hipStream_t);

} // namespace dream
