// sir_runs.hpp -- one line of equally spaced sub-elements, run by run.
//
// Along a line the coordinate offset is v_k = v0 - k dv and the distance
// r_k = sqrt(v_k^2 + w); on each side of the foot of the perpendicular r
// rises outwards, so the sub-elements of one sample bin are one run of
// consecutive steps.  Instead of evaluating every sub-element's index,
// walk_half solves for the step at which r crosses the bin's upper edge, and
// sums 1/r over the run in closed form: with c the run's middle, n its
// length and x the offset from it,
//   1/r(c + x) = 1/r_c sum_j (-x/r_c)^j P_j(v_c/r_c)     (Legendre),
// whose odd terms cancel over the run and whose even ones need only the
// moments of 0 .. n-1.  Runs are cut at n dv <= r/36 (r/20 for an FP32
// output), where the terms to P6 (P4) leave at most 2e-16 |P8| (2e-10) of
// the sum, below the rounding of the sums themselves; at r/30 (7e-16) some
// drawn workloads were 5 % further from their 64-bit values, at r/41 the
// annular one takes 6 % longer.
//
// A bin edge that falls so close to a sub-element that the estimate could
// round differently from the exact index sequence ends the walk there:
// walk_line has the rest of the half stepped by exact indices (about one line in 10^4;
// keeping the exact sequence out of the loop keeps its registers out).  With
// B the certification bound in samples, u = c1 r - c2 the index before
// rounding, T the edge and vb > 0 the offset there, sub-element k is
// certified when
//   |u_k - T| = c1 |v_k^2 - vb^2| / (r_k + R) >= c1 dv |k - k*| vb / (2.2 R)
// is at least B (r_k + R <= 2.2 R as w >= (8 dv)^2), k* the crossing.
#pragma once

#include <algorithm>
#include <cmath>
#include <vector>

#if defined(__HIP_DEVICE_COMPILE__)
#define DREAM_RUNS_FN __device__ __forceinline__
#elif defined(__HIPCC__)
#define DREAM_RUNS_FN __host__ __device__ inline
#else
#define DREAM_RUNS_FN inline
#endif

namespace dream {

DREAM_RUNS_FN double runs_rsq(double s)
{
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rsq(s);
#else
  return (double) (float) (1.0 / std::sqrt(s));
#endif
}

// sqrt(s), s > 0, to 2^-46.
DREAM_RUNS_FN double runs_sqrt(double s)
{
  const double y = runs_rsq(s), g = s * y;
  return __builtin_fma(0.5 * g, __builtin_fma(-g, y, 1.0), g);
}

// One line: v_k = v0 - k dv for 0 <= k < n, w the sum of the other two
// squares, u = c1 r - c2, ic1 = 1/c1, bound the certification margin; and
// what runs_ready derives from them.
struct RunLine {
  double v0, dv, inv_dv, w, c1, ic1, c2, bound;
  double dev = 0.0;   // the positions' largest deviation from v0 - k dv
  double roff;    // the upper edge of bin b is b ic1 + roff
  double tol;     // step j is certified when |j - j*| vb >= tol
  int foot;       // first sub-element past the foot, within [0, n]
  int cap;        // a run's longest length
};

// Whether walk_half holds on this line (n sub-elements): positive spacing,
// at most four bins per step, w clear of the spacing, the bin width and (FP64
// output) the deviation, and bins that fit an int.  False for NaN.
template <bool REFINE>
DREAM_RUNS_FN bool runs_ready(RunLine &l, int n)
{
  const double va = __builtin_fabs(l.v0), vz = __builtin_fabs(__builtin_fma(-(double) n, l.dv, l.v0));
  const double vm = va > vz ? va : vz;
  const double r = runs_sqrt(__builtin_fma(vm, vm, l.w));        // the line's longest distance
  const double f = __builtin_ceil(l.v0 * l.inv_dv);
  l.foot = f > 0.0 ? (f < (double) n ? (int) f : n) : 0;
  l.roff = (l.c2 + 0.5) * l.ic1;
  l.tol = 2.2 * l.bound * l.ic1 * l.inv_dv * r;
  const double m = l.w * runs_rsq(l.w) * l.inv_dv * (REFINE ? 1.0 / 36.0 : 1.0 / 20.0);
  l.cap = m > 1.0 ? (int) (m < 1e6 ? m : 1e6) : 1;
  const double near = REFINE ? 0x1p46 * l.dev : 0.0;
  return l.dv > 0.0 && l.c1 * l.dv <= 4.0 && l.w >= 64.0 * (l.dv * l.dv) && l.w >= near * near &&
         l.w >= 4.0 * (l.ic1 * l.ic1) && l.w < 1e200 &&
         l.c1 * r + __builtin_fabs(l.c2) < 0x1p30 && r * l.inv_dv < 0x1p30;
}

// About how many iterations walk_half takes a step, for a line whose squared
// distance from the point is w and whose sub-elements lie `along` from the
// foot on average, s bins a step at the most, cap_per_mm w^0.5 the longest run: a
// run ends with its bin or at its longest (one sub-element at the least).
// The larger of the two rates and half the smaller.
DREAM_RUNS_FN float runs_per_step(float along, float w, float s, float cap_per_mm)
{
#if defined(__HIP_DEVICE_COMPILE__)
  const float q = __builtin_amdgcn_rsqf(w), qa = __builtin_amdgcn_rsqf(w + along * along);
#else
  const float q = 1.0f / std::sqrt(w), qa = 1.0f / std::sqrt(w + along * along);
#endif
  const float bins = along * qa * s;
  const float cuts = 1.0f / __builtin_fmaxf(1.0f, __builtin_floorf(w * q * cap_per_mm));
  return __builtin_fmaxf(bins, cuts) + 0.5f * __builtin_fminf(bins, cuts);
}

// The two halves of sub-elements [k0, k1): half 0 starts at the first one
// past the foot and goes up, half 1 starts before it and goes down.  Sets
// the half's length and returns its first sub-element; step j of it is
// sub-element first + j (first - j).
DREAM_RUNS_FN int half_of(const RunLine &l, int half, int k0, int k1, int &len)
{
  const int kc = l.foot < k0 ? k0 : l.foot > k1 ? k1 : l.foot;
  len = half ? kc - k0 : k1 - kc;
  return half ? kc - 1 : kc;
}

// Walks one half (first and len as half_of gives them) outwards:
// emit(bin, n, sum) for each run (n may be 0), sum being the run's sum of
// 1/r.  Returns the number of steps walked: len, or up to where an index is
// not certified.  It ends: an iteration that takes no step raises the bin,
// and with it the crossing (bins fit 30 bits, so r rises every time), until
// the crossing passes a step or is not certified (NaN included).
template <bool REFINE, typename Emit>
DREAM_RUNS_FN int walk_half(const RunLine &l, int half, int first, int len, Emit emit)
{
  if (len <= 0) return 0;
  const double ac = __builtin_fma((double) first, l.dv, -l.v0);
  const double a0 = half ? -ac : ac;                  // offset of step 0, >= 0
  const double us = __builtin_fma(runs_sqrt(__builtin_fma(a0, a0, l.w)), l.c1, -l.c2);
  const double bs = __builtin_rint(us);
  if (!(__builtin_fabs(us - bs) <= 0.5 - l.bound)) return 0;
  int b = (int) bs;
  const double as = __builtin_fma(-a0, l.inv_dv, 1.0), am = a0 - 0.5 * l.dv;
  const double half_dv = 0.5 * l.dv, half_inv = 0.5 * l.inv_dv;
  // t and p below in units that leave the products' leading factors 1.
  constexpr double kT = 0x1.0cfeeb28b9fabp+2;         // 74.25^(1/3)
  const double wt = kT * l.w, p1 = l.dv * l.dv * (1.0 / 12.0);
  int j = 0;
  bool sure;
  do {
    const double r = __builtin_fma((double) b, l.ic1, l.roff), rr = __builtin_fma(r, r, -l.w);
    const double yr = runs_rsq(rr), g = rr * yr;
    const double js1 = __builtin_fma(g, __builtin_fma(__builtin_fma(-g, yr, 1.0), half_inv, l.inv_dv), as);
    sure = __builtin_fabs(js1 - __builtin_rint(js1)) * g >= l.tol;   // j* + 1
    const int je = sure ? (int) js1 : j;
    const int lim = j + l.cap < len ? j + l.cap : len;
    const int jt = je > j ? je : j, jn = jt < lim ? jt : lim;
    const int n = jn - j;
    // The run's middle, its 1/r to 2^-69 (2^-46), t = kT w/r^2, p =
    // (dv/r)^2/12 and d = p (n^2 - 1).
    const double vm = __builtin_fma((double) (j + jn), half_dv, am);
    const double s = __builtin_fma(vm, vm, l.w);
    const double y = runs_rsq(s), e = __builtin_fma(-(s * y), y, 1.0);
    const double q = __builtin_fma(y * e, REFINE ? __builtin_fma(0.375, e, 0.5) : 0.5, y);
    const double nd = (double) n;
    const double z = q * q, t = wt * z, p = p1 * z;
    const double d = __builtin_fma(nd * nd, p, -p), h = __builtin_fma(-2.0, p, d);
    // P2k(v/r), in factors of t = kT (1 - (v/r)^2), times the run's mean
    // 2k-th power of offset / r^2k, over d.
    double c = __builtin_fma(-1.5 / kT, t, 1.0);
    constexpr double k4 = 4.375 / (kT * kT);
    c = __builtin_fma((t - kT * 0x1.c4d1c42d7271dp-1) * (t - kT * 0x1.08a59c3764410p-2),
                      __builtin_fma(1.8 * k4, h, 1.2 * k4 * p), c);
    if (REFINE)
      c = __builtin_fma((kT * 0x1.e2d8e04e1dfa8p-1 - t) * (kT * 0x1.20279a611af21p-1 - t) *
                            (kT * 0x1.0b43e6b779650p-3 - t),
                        __builtin_fma(0.75 * h, h, p * p), c);
    const double nq = nd * q;
    emit(b, n, __builtin_fma(nq * d, c, nq));
    b += sure && je <= lim ? 1 : 0;
    j = jn;
  } while (sure && j < len);
  return j;
}

// Sub-elements [k0, k1) of a usable line: emit as walk_half's, and step(lo,
// hi) for the stretch of a half that no run certifies, at most two of them,
// each to be walked upwards (a disc's position is accumulated from its row's
// start, so that one by one and downwards they would cost their square).
template <bool REFINE, typename Emit, typename Step>
DREAM_RUNS_FN void walk_line(const RunLine &l, int k0, int k1, Emit emit, Step step)
{
#pragma clang loop unroll(disable)
  for (int half = 0; half < 2; half++) {
    int len;
    const int first = half_of(l, half, k0, k1, len);
    const int m = walk_half<REFINE>(l, half, first, len, emit);
    if (m < len) step(half ? first - len + 1 : first + m, half ? first - m + 1 : first + len);
  }
}

// ------------------------------------------------------------------ host

// The fit of positions y (rising by about d): y[0] + k dv, and the largest
// deviation from it.
inline void line_fit(const std::vector<double> &y, double d, double &dv, double &dev)
{
  const size_t n = y.size();
  dv = n > 1 ? (y[n - 1] - y[0]) / (double) (n - 1) : d;
  dev = 0.0;
  for (size_t k = 0; k < n; k++) dev = std::max(dev, std::fabs(y[k] - (y[0] + (double) k * dv)));
}

// Mean step of each disc row's accumulated x walk (from x0 < 0 to near -x0),
// to a few 1e-14 of the disc's size; returns the rows' largest deviation from
// their mean steps.
inline double disc_row_steps(double R, double dx, const std::vector<double> &x0,
                             const std::vector<double> &count, std::vector<double> &step)
{
  // Within one binade of |x| the accumulated walk advances by a constant
  // step, dx rounded to the binade's spacing: a row's mean step is dx plus
  // those deviations over the lengths the row spends in each binade.
  double lo[16], dev[16];
  int n = 0;
  for (double b = std::ldexp(1.0, std::ilogb(R)); b > 4.0 * dx && n < 16; b *= 0.5, n++) {
    lo[n] = b;
    dev[n] = 2.0 * ((1.5 * b + dx) - 1.5 * b - dx) / dx;
  }
  step.clear();
  double worst = 0.0;
  for (size_t r = 0; r < x0.size(); r++) {
    const double half = std::fabs(x0[r]);
    double drift = 0.0;
    for (int k = 0; k < n; k++)
      if (half > lo[k]) drift += (std::min(half, 2.0 * lo[k]) - lo[k]) * dev[k];
    step.push_back(count[r] < 2.0 ? dx : dx + drift / (count[r] - 1.0));
    // The walk strays from the mean step most where it leaves a binade, on
    // either side of the middle alike.
    double at = 0.0;
    for (int k = 0; k < n; k++)
      if (half > lo[k]) {
        at += 0.5 * (std::min(half, 2.0 * lo[k]) - lo[k]) * dev[k];
        worst = std::max(worst, std::fabs(at - 0.5 * drift * (half - lo[k]) / half));
      }
  }
  // The roundings of the steps that cross binades, of the ends and of the
  // mean step itself.
  return R > 0.0 ? worst + std::ldexp(1.0, std::ilogb(R) - 50) : 0.0;
}

} // namespace dream
