// att.hip -- SIR with frequency-dependent attenuation (alpha > 0) on gfx950.
//
// Reference: Attenuation::att (src/attenuation.cc:72-140), called from the
// DR sums for every in-range contribution (e.g. src/dreamrect.cc:341-395).
// Each contribution of amplitude ai, distance r and sample it adds ai times
// the inverse real FFT (length nt, divided by nt) of the lossy Green's
// function spectrum
//     X[0] = 1,  X[k] = exp(-r a w_k/(2 pi)) exp(i(-w_k r a b_k/pi^2 - t w_k)),
//     w_k = k (2 pi/nt) Fs,  b_k = log(1/(a1 w_k)),  a1 = dt 0.95/pi,  t = it dt
// (r, dt in SI units; a = alpha/(8.686 10^4) in Np/(m Hz)), k = 1 .. nt/2.
//
// The transform is linear, so the sum over contributions is taken in the
// frequency domain.  With gamma_k = a w_k (1/(2 pi) + i b_k/pi^2) a
// contribution is ai exp(-r gamma_k) exp(-2 pi i k it/nt), and the r of one
// element's contributions in one sample lie within cp dt/2 of the sample's
// distance r0 = cp (it dt + d).  So they are first summed as moments,
//     M_p = sum ai x^p,  x = (r - r0)/h,  h = cp dt/2,  p = 0 .. P-1,
// and each (element, sample) cell adds to the spectrum
//     exp(-r0 gamma_k) exp(-2 pi i k it/nt) sum_p M_p (-gamma_k h)^p / p!.
// |gamma_k h| <= rho = 0.2575 a cp for every k (0.022 at 5 dB/(cm MHz) and
// 1500 m/s, whatever dt is), so that P = 8 terms leave less than 2^-54 of
// the cell's sum up to rho = 0.03, and 12 terms up to 0.2; stronger
// attenuation cuts each sample into q sub-cells of rho/q <= 0.2.
//
// One work-group per (point, chunk of contributions, block of bins) walks
// the chunk's elements: geometry, index and amplitude as the DR sums compute
// them, moments added into an LDS window of the samples that the element's
// bounding box reaches, then every thread adds the window's cells to the
// bins it owns.  A table of exp(-cp dt it gamma_k) exp(-2 pi i k it/nt) per
// (it, k) leaves one complex exponential per (point, element, bin); without
// the table (below) a cell evaluates its own.  Chunks write their spectra
// side by side and the second kernel adds them, then turns each point's
// spectrum into its nt samples by the direct complex-to-real sum (the
// imaginary parts of X[0] and X[nt/2] drop out, as in FFTW's c2r transform).
//
// The exponentials of every (contribution, bin) pair were the whole cost of
// the direct sum: 64 points x 16 elements x 3600 sub-elements at nt = 400
// took 3950 us for 7.4e8 of them; the moments take 43 us (147 with an LDS
// atomic per contribution instead of the lanes' runs), the grid tables 6 and
// the transform 12, and the call went from 4060 to 124 us.  What bounds it
// now is the call on the host (its set-up, one upload, one read-back); on the
// device the geometry and the moments' LDS atomics, with 1.5 waves per SIMD.
// A work-group holds at most kBinBlock bins; longer responses split each
// point's bins over several work-groups (any nt).

#include "sir.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <string>
#include <unordered_map>

namespace dream {

namespace {

constexpr int kThreads = 256;
constexpr int kCells = 256;      // moment cells of one LDS window
constexpr double kBoundScale = 0x1p-36;

typedef const __attribute__((address_space(1))) double gdouble;

// What depends on (nt, dt, cp) only: gamma_k, the transform's twiddles and
// (table) the per-sample factors.  Problems of a call share it when equal.
struct AttGrid {
  int64_t nt;
  double dt_s, alpha, step;     // step = cp dt in m
  double2 *gam;                 // K: gamma_k [1/m]
  double2 *tw;                  // nt: cos(2 pi m/nt), sin(2 pi m/nt)
  double2 *table;               // nt x K or null
};

// One problem on the device.
struct AttDev {
  const double *Ro;  int64_t No;
  const double *delay;  int32_t delay_multi;  int32_t L;
  const double *sub;    // 3 x S: sub-element x | y | z offset (rz = z - zoff)
  int64_t S;            // sub-elements per element
  const double *el;     // 6 x L: gx gy gz foc steer ((w v) ds)
  int64_t nt;
  double cp, dt, inv_dt, c1, amp;
  double lo[3], hi[3];  // bounding box of the sub-element offsets
  AttGrid grid;
  double gmax;          // bound of |gamma_k|
  double2 *spec;        // No x chunks x K
  void *h;  int32_t out_f64;  int32_t chunks;
  int32_t bin_blocks;   // the K bins in blocks of kBinBlock, one work-group each
  int32_t q;            // sub-cells per sample
  int32_t empty, pad;   // no sub-elements: zeros
  Status *status;
  int64_t item_begin;
  int64_t out_begin;    // first work-group of the complex-to-real kernel
};

// Spectrum bins one work-group accumulates in LDS (two FP64 accumulators
// each, beside the moments): nt up to 2 (kBinBlock - 1) in one block, longer
// ones over several.
constexpr int64_t kBinBlock = 2304;

// Largest per-sample table (nt <= 2047): it stays in the L2 caches.
constexpr int64_t kTableBytes = 32ll << 20;

__device__ __forceinline__ unsigned wave_sum_u(unsigned v)
{
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// exp(-r gamma) exp(-2 pi i m/nt).
__device__ __forceinline__ double2 lossy_phase(double r, double2 g, double m, double inv_nt)
{
  double sn, cs;
  sincos(__builtin_fma(r, g.y, (2.0 * M_PI) * (m * inv_nt)), &sn, &cs);
  const double x = exp(-r * g.x);
  return {x * cs, -(x * sn)};
}

// gamma_k, twiddles and table of one grid (blockIdx.y), and the status words
// zeroed.  w_k and b_k by the reference's expressions (src/attenuation.cc:84-110).
__global__ void __launch_bounds__(kThreads)
att_grid_kernel(const AttGrid *__restrict__ grids, Status *st, int n_st)
{
  const AttGrid G = grids[blockIdx.y];
  const int64_t K = G.nt / 2 + 1;
  const int64_t n = G.table ? G.nt * K : std::max(K, G.nt);
  const double Fs = 1 / G.dt_s, dw = 2.0 * M_PI / (double) G.nt, a1 = G.dt_s * 0.95 / M_PI;
  const double inv_nt = 1.0 / (double) G.nt;
  for (int64_t i = (int64_t) blockIdx.x * kThreads + threadIdx.x; i < n;
       i += (int64_t) gridDim.x * kThreads) {
    const int64_t it = i / K, k = i - it * K;
    double2 g = {0.0, 0.0};
    if (k > 0) {
      const double w = ((double) k * dw) * Fs, b = log(1.0 / (a1 * w));
      g.x = G.alpha * w / (2.0 * M_PI);
      g.y = w * G.alpha / (M_PI * M_PI) * b;
    }
    if (it == 0) G.gam[k] = g;
    if (G.table)
      G.table[i] = lossy_phase((double) it * G.step, g, (double) ((k * it) % G.nt), inv_nt);
    if (i < G.nt) {
      double sn, cs;
      sincospi(2.0 * (double) i * inv_nt, &sn, &cs);
      G.tw[i] = {cs, sn};
    }
  }
  if (blockIdx.y == 0)
    for (int64_t i = (int64_t) blockIdx.x * kThreads + threadIdx.x; i < n_st;
         i += (int64_t) gridDim.x * kThreads) {
      st[i].any_oob = 0u;
      st[i].last_elem_oob = 0u;
      st[i].oob = 0ull;
    }
}

// Range of (c - p)^2 over p in [lo, hi].
__device__ __forceinline__ void square_range(double c, double lo, double hi, double &mn, double &mx)
{
  const double a = c - lo, b = c - hi;
  const double m = __builtin_fmin(__builtin_fabs(a), __builtin_fabs(b));
  mn += (a >= 0.0 && b <= 0.0) ? 0.0 : m * m;
  mx += __builtin_fmax(a * a, b * b);
}

// Spectrum bins [k0, k1) of one (point, chunk): sum over the chunk's
// contributions of ai * X[k].  A work item is (point, chunk, bin block).
template <int P>
__global__ void __launch_bounds__(kThreads)
att_spectrum_kernel(const AttDev *__restrict__ probs, int n_probs)
{
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double mom[P][kCells];
  const int64_t item = blockIdx.x;
  int pi = 0;
  {
    int hi = n_probs - 1;
    while (pi < hi) {
      const int mid = (pi + hi + 1) >> 1;
      if (probs[mid].item_begin <= item) pi = mid; else hi = mid - 1;
    }
  }
  const AttDev &A = probs[pi];
  const int64_t local = item - A.item_begin;
  const int64_t per_point = (int64_t) A.chunks * A.bin_blocks;
  const int64_t n = local / per_point;
  const int64_t rest = local - n * per_point;
  const int c = (int) (rest / A.bin_blocks);
  const int bb = (int) (rest - (int64_t) c * A.bin_blocks);
  const int64_t K = A.nt / 2 + 1;
  const int64_t k0 = (int64_t) bb * kBinBlock, k1 = std::min<int64_t>(K, k0 + kBinBlock);
  const int nk = (int) (k1 - k0);
  const int64_t total = (int64_t) A.L * A.S;
  const int64_t c0 = (int64_t) c * total / A.chunks, c1 = (int64_t) (c + 1) * total / A.chunks;

  double2 *acc = reinterpret_cast<double2 *>(smem);         // nk
  for (int k = threadIdx.x; k < nk; k += kThreads) acc[k] = {0.0, 0.0};

  gdouble *Ro = (gdouble *) A.Ro;
  const double xo = Ro[n], yo = Ro[n + A.No], zo = Ro[n + 2 * A.No];
  const double dlay = A.delay_multi ? ((gdouble *) A.delay)[n] : ((gdouble *) A.delay)[0];
  gdouble *el = (gdouble *) A.el;
  gdouble *sub = (gdouble *) A.sub;
  const double2 *gam = A.grid.gam;
  const double2 *table = A.grid.table;
  const int L = A.L;
  const int64_t S = A.S;
  const int q = A.q;
  const double qd = (double) q, inv_q = 1.0 / qd, inv_nt = 1.0 / (double) A.nt;
  const double ntd = (double) A.nt;
  const double step = A.grid.step;              // m per sample
  const double h = 0.5 * step * inv_q;
  unsigned oob = 0;
  bool oob_last = false;

  for (int64_t f0 = c0; f0 < c1;) {
    // The part [s0, s1) of element e that lies in the chunk.
    const int e = (int) (f0 / S);
    const int64_t s0 = f0 - (int64_t) e * S, s1 = std::min<int64_t>(S, s0 + (c1 - f0));
    f0 += s1 - s0;
    const double xe = xo - el[e], ye = yo - el[L + e], ze = zo - el[2 * L + e];
    const double d = (dlay - el[3 * L + e]) - el[4 * L + e];
    const double c2 = d * A.inv_dt;
    const double lim = 0.5 - kBoundScale * (ntd + 2.0 + __builtin_fabs(c2));
    const double num = el[5 * L + e] * A.amp;
    // Samples the element can reach: distances to the box of its
    // sub-elements, two samples of margin, inside [0, nt).
    double mn = 0.0, mx = 0.0;
    square_range(xe, A.lo[0], A.hi[0], mn, mx);
    square_range(ye, A.lo[1], A.hi[1], mn, mx);
    square_range(ze, A.lo[2], A.hi[2], mn, mx);
    // (A negative speed turns the range round.)
    const double ua = __builtin_sqrt(mn) * A.c1 - c2, ub = __builtin_sqrt(mx) * A.c1 - c2;
    const double ulo = __builtin_fmin(ua, ub) - 2.0, uhi = __builtin_fmax(ua, ub) + 2.0;
    const int64_t lo = ulo > 0.0 ? (int64_t) __builtin_fmin(ulo, ntd) : 0;
    const int64_t hi = uhi < ntd - 1.0 ? (int64_t) __builtin_fmax(uhi, -1.0) : A.nt - 1;
    const bool use_table = table && q == 1 && __builtin_fabs(d * (A.cp * 1e-6)) * A.gmax <= 300.0;
    const int width = kCells / q;
    int64_t w0 = lo;
    bool first = true;
    do {
      const int ns = (int) std::max<int64_t>(0, std::min<int64_t>(width, hi - w0 + 1));
      const int cells = ns * q;
      __syncthreads();                          // the last window is consumed
      for (int i = threadIdx.x; i < P * kCells; i += kThreads) (&mom[0][0])[i] = 0.0;
      // A lane's sub-elements are neighbours (run_order), so it keeps its
      // cell's moments in registers and adds them when the cell changes.
      int cur = -1;
      double run[P];
#pragma unroll
      for (int p = 0; p < P; p++) run[p] = 0.0;
      auto flush = [&]() {
        if (cur >= 0) {
#pragma unroll
          for (int p = 0; p < P; p++)
            __hip_atomic_fetch_add(&mom[p][cur], run[p], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        }
      };
      for (int64_t s = s0 + threadIdx.x; s < s1; s += kThreads) {
        const double rx = xe - sub[s], ry = ye - sub[S + s], rz = ze - sub[2 * S + s];
        const double sq = (rx * rx + ry * ry) + rz * rz;
        double r, rinv;
        sqrt_rsqrt<2>(sq, r, rinv);
        double u = __builtin_fma(r, A.c1, -c2);
        double ru = __builtin_rint(u);
        if (!(__builtin_fabs(u - ru) <= lim)) {   // not certified, 0 or not finite
          const double re = __builtin_sqrt(sq);
          u = ((re * 1000.0) / A.cp - d) / A.dt;
          ru = __builtin_rint(u);
          rinv = 1.0 / re;
        }
        if (ru >= 0.0 && ru < ntd) {
          int cell = (int) (ru - (double) w0);
          double x = u - ru;
          if (q > 1) {
            const double v = (x + 0.5) * qd;
            const double sc = __builtin_fmin(__builtin_fmax(__builtin_floor(v), 0.0), qd - 1.0);
            cell = cell * q + (int) sc;
            x = v - sc - 0.5;
          }
          x += x;
          if ((unsigned) cell < (unsigned) cells) {
            const bool same = cell == cur;
            if (!same) flush();
            cur = cell;
            double m = num * rinv;
#pragma unroll
            for (int p = 0; p < P; p++) {
              run[p] = same ? run[p] + m : m;
              m *= x;
            }
          }
        } else if (first) {
          oob++;
          oob_last |= (e == L - 1);
        }
      }
      flush();
      __syncthreads();
      for (int kk = threadIdx.x; kk < nk; kk += kThreads) {
        const int64_t k = k0 + kk;
        const double2 g = gam[k];
        double cr[P], ci[P];
        cr[0] = 1.0;
        ci[0] = 0.0;
#pragma unroll
        for (int p = 1; p < P; p++) {
          const double hp = -h / (double) p;
          cr[p] = (cr[p - 1] * g.x - ci[p - 1] * g.y) * hp;
          ci[p] = (cr[p - 1] * g.y + ci[p - 1] * g.x) * hp;
        }
        double sr = 0.0, si = 0.0;
        auto add = [&](int cell, double2 t) {
          double pr = mom[0][cell], pim = 0.0;
#pragma unroll
          for (int p = 1; p < P; p++) {
            const double m = mom[p][cell];
            pr = __builtin_fma(cr[p], m, pr);
            pim = __builtin_fma(ci[p], m, pim);
          }
          sr += pr * t.x - pim * t.y;
          si += pr * t.y + pim * t.x;
        };
        if (use_table) {
          // Four cells' factors in flight together; cells past the window
          // hold zero moments.
          for (int cell = 0; cell < cells; cell += 4) {
            double2 t[4];
#pragma unroll
            for (int i = 0; i < 4; i++)
              t[i] = table[std::min<int64_t>(w0 + cell + i, A.nt - 1) * K + k];
#pragma unroll
            for (int i = 0; i < 4; i++) add(cell + i, t[i]);
          }
          const double2 f = lossy_phase(d * (A.cp * 1e-6), g, 0.0, inv_nt);
          acc[kk].x += sr * f.x - si * f.y;
          acc[kk].y += sr * f.y + si * f.x;
        } else {
          for (int cell = 0; cell < cells; cell++) {
            if (mom[0][cell] == 0.0) continue;
            const int64_t it = w0 + cell / q;
            const double off = ((double) (cell % q) + 0.5) * inv_q - 0.5;
            const double r0 = (((double) it + off) * A.dt + d) * (A.cp * 1e-6);
            add(cell, lossy_phase(r0, g, (double) ((k * it) % A.nt), inv_nt));
          }
          acc[kk].x += sr;
          acc[kk].y += si;
        }
      }
      w0 += width;
      first = false;
    } while (w0 <= hi);
  }
  double2 *spec = A.spec + (n * A.chunks + c) * K;
  for (int k = threadIdx.x; k < nk; k += kThreads) spec[k0 + k] = acc[k];
  // Every bin block sees the same contributions: the first one counts them.
  const unsigned wsum = bb == 0 ? wave_sum_u(oob) : 0u;
  const bool any_last = __any(oob_last);
  if ((threadIdx.x & 63) == 0 && wsum) {
    atomicOr(&A.status->any_oob, 1u);
    if (any_last) atomicOr(&A.status->last_elem_oob, 1u);
    atomicAdd(&A.status->oob, (unsigned long long) wsum);
  }
}

// Samples of one point from its spectrum (the sum of its chunks' spectra):
// the complex-to-real inverse DFT
//   x[j] = (X0 + 2 sum_{k=1}^{kmax} (Re X_k cos(2 pi jk/n) - Im X_k sin(2 pi jk/n))
//          + [n even] Re X_{n/2} (-1)^j) / n.
// One work-group per (point, kOut samples): its four waves share the
// samples and take every fourth bin, so a call of few points still spreads
// over the device (64 points x 400 samples: 63 us with one work-group per
// point and a serial chain of nt/2 terms per thread).
constexpr int kOut = 64;
constexpr int kSpecTile = 1024;

__global__ void __launch_bounds__(kThreads)
att_c2r_kernel(const AttDev *__restrict__ probs, int n_probs)
{
  __shared__ double2 X[kSpecTile];
  __shared__ double part[kThreads / kOut][kOut];
  const int64_t g = blockIdx.x;
  int lo = 0, hi = n_probs - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (probs[mid].out_begin <= g) lo = mid; else hi = mid - 1;
  }
  const AttDev &A = probs[lo];
  const int64_t nt = A.nt, K = nt / 2 + 1;
  const int64_t blocks = (nt + kOut - 1) / kOut;
  const int64_t n = (g - A.out_begin) / blocks;
  const int lane = (int) threadIdx.x % kOut, w = (int) threadIdx.x / kOut;
  const int64_t j = (g - A.out_begin - n * blocks) * kOut + lane;
  const int64_t jm = std::min<int64_t>(j, nt - 1);
  const bool even = nt % 2 == 0;
  const double2 *spec = A.spec + n * A.chunks * K;
  const double2 *tw = A.grid.tw;
  constexpr int kWays = kThreads / kOut;
  const int64_t stride = (kWays * jm) % nt;
  double s = 0.0;
  for (int64_t t0 = 0; t0 < K; t0 += kSpecTile) {
    const int nt_k = (int) std::min<int64_t>(kSpecTile, K - t0);
    __syncthreads();
    for (int k = threadIdx.x; k < nt_k; k += kThreads) {
      double2 v = {0.0, 0.0};
      if (!A.empty)
#pragma unroll 4
        for (int c = 0; c < A.chunks; c++) {
          const double2 p = spec[c * K + t0 + k];
          v.x += p.x;
          v.y += p.y;
        }
      // Every bin but 0 and nt/2 stands for its conjugate too.
      const bool once = t0 + k == 0 || (even && t0 + k == nt / 2);
      X[k] = once ? double2{v.x, 0.0} : double2{2.0 * v.x, 2.0 * v.y};
    }
    __syncthreads();
    int64_t m = ((t0 + w) * jm) % nt;
#pragma unroll 4
    for (int k = w; k < nt_k; k += kWays) {
      const double2 t = tw[m], v = X[k];
      s += v.x * t.x - v.y * t.y;
      m += stride;
      if (m >= nt) m -= nt;
    }
  }
  part[w][lane] = s;
  __syncthreads();
  if (w == 0 && j < nt) {
    for (int i = 1; i < kWays; i++) s += part[i][lane];
    const double x = s / (double) nt;
    if (A.out_f64) reinterpret_cast<double *>(A.h)[n * nt + j] = x;
    else reinterpret_cast<float *>(A.h)[n * nt + j] = (float) x;
  }
}

// Sub-element offsets of one element.  Rectangles and cylinders list their
// columns (y inner): along y, across the array's plane, the sample changes
// more slowly than along x, where the elements are spread.
void sub_elements(const SirProblem &p, std::vector<double> &x, std::vector<double> &y,
                  std::vector<double> &z)
{
  x.clear(); y.clear(); z.clear();
  if (p.shape == SIR_CIRC) {
    std::vector<double> ys, x0, cnt;
    disc_rows(p.R, p.dx, p.dy, ys, x0, cnt);
    for (size_t r = 0; r < ys.size(); r++) {
      double xs = x0[r];
      for (int64_t i = 0; i < (int64_t) cnt[r]; i++) {
        x.push_back(xs);
        y.push_back(ys[r]);
        z.push_back(0.0);
        xs += p.dx;
      }
    }
    return;
  }
  std::vector<double> xs = subgrid(p.a, p.dx), ys, zr;
  if (p.shape == SIR_CYLIND) {
    cylinder_rows(p.b, p.R, p.dy, ys, zr);
  } else {
    ys = subgrid(p.b, p.dy);
    zr.assign(ys.size(), 0.0);
  }
  x.reserve(xs.size() * ys.size());
  y.reserve(xs.size() * ys.size());
  z.reserve(xs.size() * ys.size());
  for (double v : xs)
    for (size_t r = 0; r < ys.size(); r++) {
      x.push_back(v);
      y.push_back(ys[r]);
      z.push_back(zr[r]);
    }
}

// The list in the order in which lane t of kThreads, which takes entries t, t +
// kThreads, ..., walks a run of neighbours.  Written in sequence (the 256 runs
// read side by side stay in the cache): 40000 entries scattered to their places
// took 260 us, twice the rest of such a call.
void run_order(const std::vector<double> &v, double *out)
{
  const size_t S = v.size(), full = S / kThreads, more = S % kThreads;
  for (size_t i = 0, at = 0; at < S; i++)
    for (size_t t = 0; t < (size_t) kThreads && at < S; t++, at++)
      out[at] = v[t * full + std::min(t, more) + i];
}

} // namespace

void run_sir_att(const std::vector<SirProblem> &problems, double alpha_db, int out_dtype,
                 hipStream_t s, int32_t *codes, int64_t *oobs)
{
  require(out_dtype == DREAM_HIP_F64 || out_dtype == DREAM_HIP_F32,
          "SIR: output precision must be DREAM_HIP_F64 or DREAM_HIP_F32");
  const size_t P = problems.size();
  if (P == 0) return;
  int dev = 0, cus = 256;
  DREAM_HIP_CHECK(hipGetDevice(&dev));
  DREAM_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const int64_t target = 4 * (int64_t) std::max(cus, 1);
  const double alpha = alpha_db / (8.686 * 10000.0);

  // Terms and sub-cells by the largest rho of the call (see the file comment).
  double rho = 0.0;
  for (const SirProblem &p : problems) rho = std::max(rho, 0.2575 * alpha * std::fabs(p.cp));
  const int terms = rho <= 0.03 ? 8 : 12;
  const int q = rho <= 0.2 ? 1 : (rho < 0.2 * kCells ? (int) std::ceil(rho / 0.2) : kCells);

  std::vector<double> tables;
  std::vector<AttDev> dev_p(P);
  std::vector<AttGrid> grids;
  std::unordered_map<std::string, size_t> known;        // grids by their bytes
  std::vector<int64_t> cells;                   // per grid: (point, element) pairs it serves
  std::vector<size_t> off_sub(P), off_el(P), grid_of(P);
  std::vector<int64_t> spec_off(P);
  int64_t spec_total = 0, outs = 0, items = 0, max_K = 1;
  for (size_t i = 0; i < P; i++) {
    const SirProblem &p = problems[i];
    const int64_t L = (int64_t) (p.G.size() / 3);
    require(L >= 1 && p.nt >= 1 && p.No >= 0, "SIR: need elements, nt >= 1 and No >= 0");
    require(p.dx > 0 && p.dy > 0 && p.dt > 0, "SIR: dx, dy and dt must be positive");
    require(p.No == 0 || (p.Ro && p.delay && p.h), "SIR: null Ro, delay or h");
    std::vector<double> x, y, z;
    sub_elements(p, x, y, z);
    const int64_t S = (int64_t) x.size();
    AttDev &d = dev_p[i];
    std::memset(&d, 0, sizeof d);
    off_sub[i] = tables.size();
    const std::vector<double> *xyz[3] = {&x, &y, &z};
    tables.resize(tables.size() + 3 * x.size());
    for (size_t a = 0; a < 3; a++) {
      run_order(*xyz[a], tables.data() + off_sub[i] + a * x.size());
      if (S) d.lo[a] = d.hi[a] = xyz[a]->front();
      for (double v : *xyz[a]) {
        d.lo[a] = v < d.lo[a] ? v : d.lo[a];
        d.hi[a] = v > d.hi[a] ? v : d.hi[a];
      }
    }
    std::vector<double> el = element_table(p);
    off_el[i] = tables.size();
    tables.insert(tables.end(), el.begin(), el.end());
    const int64_t nt = p.nt, K = nt / 2 + 1;
    d.Ro = p.Ro;  d.No = p.No;
    d.delay = p.delay;  d.delay_multi = p.delay_type != 0;
    d.L = (int32_t) L;  d.S = S;
    d.nt = nt;  d.cp = p.cp;  d.dt = p.dt;
    d.inv_dt = 1.0 / p.dt;
    d.c1 = 1000.0 / (p.cp * p.dt);
    d.amp = 1000.0 / (2.0 * M_PI * p.dt);
    d.q = q;
    d.empty = S == 0;
    d.h = p.h;  d.out_f64 = out_dtype == DREAM_HIP_F64;
    AttGrid g;
    std::memset(&g, 0, sizeof g);
    g.nt = nt;
    g.dt_s = p.dt * 1.0e-6;
    g.alpha = alpha;
    g.step = p.cp * g.dt_s;
    d.gmax = 0.515 * alpha / g.dt_s;
    const size_t gi = known.try_emplace(std::string((const char *) &g, sizeof g), grids.size()).first->second;
    if (gi == grids.size()) {
      grids.push_back(g);
      cells.push_back(0);
    }
    grid_of[i] = gi;
    cells[gi] += p.No * L;
    const int64_t total = L * S;
    int64_t chunks = 1;
    if (p.No > 0 && p.No < target) chunks = (target + p.No - 1) / p.No;
    chunks = std::max<int64_t>(1, std::min<int64_t>(chunks, (total + kThreads - 1) / kThreads));
    // Whole elements per chunk where the array has enough of them: a chunk
    // that ends inside an element transforms that element's cells twice.
    if (chunks <= L) chunks = L / (L / chunks);
    // The chunks' spectra are kept apart: at most 256 MiB of them in the call.
    chunks = std::max<int64_t>(1, std::min<int64_t>(chunks, (256ll << 20) / 16 / (int64_t) P / K / std::max<int64_t>(p.No, 1)));
    d.chunks = (int32_t) chunks;
    d.bin_blocks = (int32_t) ((K + kBinBlock - 1) / kBinBlock);
    d.item_begin = items;
    items += (S > 0) ? p.No * chunks * d.bin_blocks : 0;
    spec_off[i] = spec_total;
    spec_total += p.No * chunks * K;
    d.out_begin = outs;
    outs += p.No * ((nt + kOut - 1) / kOut);
    max_K = std::max<int64_t>(max_K, std::min<int64_t>(K, kBinBlock));
  }
  require(items < (1ll << 31), "SIR with attenuation: too many work items");
  require(outs < (1ll << 31), "SIR with attenuation: too many points");
  const size_t lds = (size_t) max_K * sizeof(double2);

  // One block of device memory: grids, problems, tables (copied in), then
  // status, grid tables and spectra.
  size_t bytes = 0;
  auto take = [&](size_t n) {
    const size_t at = bytes;
    bytes += (n + 255) & ~(size_t) 255;
    return at;
  };
  const size_t o_grids = take(grids.size() * sizeof(AttGrid));
  const size_t o_probs = take(P * sizeof(AttDev));
  const size_t o_tables = take(tables.size() * sizeof(double));
  const size_t copied = bytes;
  const size_t o_status = take(P * sizeof(Status));
  std::vector<size_t> o_gam, o_tw, o_table;
  std::vector<bool> has_table;
  int64_t grid_work = 1, table_total = 0;
  for (size_t k = 0; k < grids.size(); k++) {
    const int64_t nt = grids[k].nt, K = nt / 2 + 1;
    // The table pays when the (point, element) pairs that read it, about 16
    // samples each, are more than its nt rows, and is not used with sub-cells.
    // All tables of a call take 8 times kTableBytes at the most.
    const int64_t table = nt * K * (int64_t) sizeof(double2);
    const bool t = q == 1 && grids[k].step > 0.0 && table <= kTableBytes && cells[k] * 16 >= nt &&
                   table_total + table <= 8 * kTableBytes;
    if (t) table_total += table;
    has_table.push_back(t);
    o_gam.push_back(take((size_t) K * sizeof(double2)));
    o_tw.push_back(take((size_t) nt * sizeof(double2)));
    o_table.push_back(t ? take((size_t) (nt * K) * sizeof(double2)) : 0);
    grid_work = std::max(grid_work, t ? nt * K : nt);
  }
  const size_t o_spec = take((size_t) spec_total * sizeof(double2));
  // Small tables go up with the descriptors, large ones from where they are: a
  // copy more takes 20 us, so at 86 kB one copy 154 against 174 us a call, at 240
  // kB 214 against 238, at 540 kB the same, above that apart is faster.
  const size_t table_bytes = tables.size() * sizeof(double);
  const bool apart = table_bytes > ((size_t) 1 << 18);
  std::vector<char> host(apart ? o_tables : copied);
  std::vector<Status> st(P);
  ScratchHold scratch(SCRATCH_ATT);
  char *base = (char *) scratch.get(bytes);
  scratch.pending(s);
  Status *d_status = (Status *) (base + o_status);
  for (size_t k = 0; k < grids.size(); k++) {
    grids[k].gam = (double2 *) (base + o_gam[k]);
    grids[k].tw = (double2 *) (base + o_tw[k]);
    if (has_table[k]) grids[k].table = (double2 *) (base + o_table[k]);
  }
  for (size_t i = 0; i < P; i++) {
    AttDev &d = dev_p[i];
    d.sub = (const double *) (base + o_tables) + off_sub[i];
    d.el = (const double *) (base + o_tables) + off_el[i];
    d.grid = grids[grid_of[i]];
    d.spec = (double2 *) (base + o_spec) + spec_off[i];
    d.status = d_status + i;
  }
  std::memcpy(host.data() + o_grids, grids.data(), grids.size() * sizeof(AttGrid));
  std::memcpy(host.data() + o_probs, dev_p.data(), P * sizeof(AttDev));
  if (apart)
    DREAM_HIP_CHECK(hipMemcpyAsync(base + o_tables, tables.data(), table_bytes,
                                   hipMemcpyHostToDevice, s));
  else if (table_bytes)
    std::memcpy(host.data() + o_tables, tables.data(), table_bytes);
  DREAM_HIP_CHECK(hipMemcpyAsync(base, host.data(), host.size(), hipMemcpyHostToDevice, s));
  const AttGrid *d_grids = (const AttGrid *) (base + o_grids);
  const AttDev *d_probs = (const AttDev *) (base + o_probs);
  // In launches of up to 32768 grids (HIP states 65535 as the y extent's limit).
  for (size_t k = 0; k < grids.size(); k += 32768) {
    const size_t n = std::min<size_t>(grids.size() - k, 32768);
    hipLaunchKernelGGL(att_grid_kernel,
                       dim3((unsigned) std::min<int64_t>((grid_work + kThreads - 1) / kThreads, 4096),
                            (unsigned) n),
                       dim3(kThreads), 0, s, d_grids + k, d_status, k == 0 ? (int) P : 0);
    DREAM_HIP_CHECK(hipGetLastError());
  }
  if (items > 0) {
    if (terms == 8)
      hipLaunchKernelGGL(att_spectrum_kernel<8>, dim3((unsigned) items), dim3(kThreads), lds, s,
                         d_probs, (int) P);
    else
      hipLaunchKernelGGL(att_spectrum_kernel<12>, dim3((unsigned) items), dim3(kThreads), lds, s,
                         d_probs, (int) P);
    DREAM_HIP_CHECK(hipGetLastError());
  }
  if (outs > 0) {
    hipLaunchKernelGGL(att_c2r_kernel, dim3((unsigned) outs), dim3(kThreads), 0, s, d_probs,
                       (int) P);
    DREAM_HIP_CHECK(hipGetLastError());
  }
  DREAM_HIP_CHECK(hipMemcpyAsync(st.data(), d_status, P * sizeof(Status),
                                 hipMemcpyDeviceToHost, s));
  DREAM_HIP_CHECK(hipStreamSynchronize(s));
  scratch.settled();
  for (size_t i = 0; i < P; i++) {
    const int lv = problems[i].err_level;
    int code = E_NONE;
    if (lv == L_STOP || lv == L_PSTOP) {
      if (st[i].any_oob) code = E_OOB;
    } else if (st[i].last_elem_oob) {
      code = level_code(lv);
    }
    if (codes) codes[i] = code;
    if (oobs) oobs[i] = (int64_t) st[i].oob;
  }
}

} // namespace dream
