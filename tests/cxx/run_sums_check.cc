// Sums of 1/r of the run walk (sir_runs.hpp) against long double.
//   run_sums_check equal SEED LINES: lines whose positions are v0 - k dv.
//     Prints usable lines, worst relative error of a bin's sum (REFINE), the
//     same without, and the largest share left to step of the kinds of lines.
//   run_sums_check row SIZE STEP NEAR: the rows of a flat rectangle's column
//     of SIZE mm, accumulated as the package does.
//   run_sums_check disc RADIUS STEP NEAR: a disc's rows.
//     Points NEAR mm and more away.  Print lines walked, lines left to step,
//     worst error (REFINE), largest deviation from the fit and its bound.
//   run_sums_check rest SEED LINES: disc rows with a sub-element on a rounding
//     boundary.  Prints lines, sub-elements left to step, the most position
//     updates that these take (in lengths of the row), and sub-elements not
//     walked exactly once.
//   run_sums_check price SEED LINES: prints lines and the least and largest
//     ratio of a line's iterations to runs_per_step's.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <random>

#include "sir_runs.hpp"

using dream::RunLine;

static std::mt19937_64 gen;
static double uni(double a, double b) { return std::uniform_real_distribution<double>(a, b)(gen); }

static void grid_of(RunLine &l, double cp, double dt, double d, double nt)
{
  l.c1 = 1000.0 / (cp * dt);
  l.ic1 = 1.0 / l.c1;
  l.c2 = d / dt;
  l.bound = 0x1p-36 * (nt + 2.0 + std::fabs(l.c2));
}

// Worst relative error of a whole line's bins; steps not walked are counted.
template <bool REFINE, typename Offset>
static double line_error(const RunLine &l, int n, Offset offset, long &stepped)
{
  std::map<int, std::pair<long double, long double>> bins;
  for (int half = 0; half < 2; half++) {
    int len, at = 0;
    const int first = dream::half_of(l, half, 0, n, len);
    at = dream::walk_half<REFINE>(l, half, first, len, [&](int b, int c, double v) {
      auto &s = bins[b];
      s.first += v;
      for (int j = 0; j < c; j++, at++) {
        const long double x = offset(half ? first - at : first + at);
        s.second += 1.0L / sqrtl(x * x + (long double) l.w);
      }
    });
    stepped += len - at;
  }
  double worst = 0.0;
  for (auto &b : bins)
    if (b.second.second > 0.0L)
      worst = std::fmax(worst, (double) fabsl(b.second.first / b.second.second - 1.0L));
  return worst;
}

static int equal(int lines)
{
  long usable = 0, elems[4] = {}, stepped[4] = {}, rest = 0;
  double worst = 0.0, worst32 = 0.0;
  for (int q = 0; q < lines; q++) {
    const int kind = q % 4, n = 1 + (int) uni(0.0, kind == 3 ? 3000.0 : 330.0);
    RunLine l;
    l.dv = kind == 0 ? 0.05 : uni(0.01, 0.2);
    l.inv_dv = 1.0 / l.dv;
    const double mid = 0.5 * (n - 1) * l.dv;
    // kind 1: the foot in the middle; 2: at an end or past it; else anywhere.
    l.v0 = kind == 1 ? mid : kind == 2 ? (q & 4 ? -1.0 : 2.0) * mid + uni(0.0, 1.0) : mid + uni(-20.0, 20.0);
    const double ra = uni(-8.0, 8.0), rb = uni(0.5, 80.0);
    l.w = ra * ra + rb * rb;
    grid_of(l, uni(900.0, 1700.0), uni(0.01, q % 8 < 4 ? 0.3 : 0.06), uni(0.0, 60.0), 100.0 + uni(0.0, 2000.0));
    auto offset = [&](int k) { return (long double) l.v0 - (long double) k * (long double) l.dv; };
    if (!dream::runs_ready<true>(l, n)) continue;
    usable++;
    elems[kind] += n;
    worst = std::fmax(worst, line_error<true>(l, n, offset, stepped[kind]));
    dream::runs_ready<false>(l, n);
    worst32 = std::fmax(worst32, line_error<false>(l, n, offset, rest));
  }
  double share = 0.0;
  for (int k = 0; k < 4; k++) share = std::fmax(share, (double) stepped[k] / (double) elems[k]);
  std::printf("%ld %.3e %.3e %.3e\n", usable, worst, worst32, share);
  return 0;
}

// A row's accumulated positions.
static std::vector<double> accumulate(double x, double dx, int n)
{
  std::vector<double> p((size_t) n);
  for (int k = 0; k < n; k++, x += dx) p[(size_t) k] = x;
  return p;
}

static int aperture(bool disc, double size, double step, double near)
{
  std::vector<double> x0, count, mean;
  double dv = 0.0, dev = 0.0, seen = 0.0, worst = 0.0;
  if (disc) {
    for (int r = 0; r < 24; r++) {
      const double y = (r + 0.37) / 24.0 * size, h = std::sqrt(size * size - y * y);
      const double first = -h + step / 2.0;
      int n = 0;
      for (double x = first; x <= h; x += step) n++;
      x0.push_back(first);
      count.push_back(n);
    }
    dev = dream::disc_row_steps(size, step, x0, count, mean);
  } else {
    x0.push_back(-size / 2.0 + step / 2.0);
    int n = 0;
    for (double x = x0[0]; x <= size / 2.0; x += step) n++;
    count.push_back(n);
    dream::line_fit(accumulate(x0[0], step, n), step, dv, dev);
    mean.push_back(dv);
  }
  long fit = 0, left = 0, stepped = 0;
  for (size_t r = 0; r < x0.size(); r++) {
    const int n = (int) count[r];
    if (n < 1) continue;
    const std::vector<double> p = accumulate(x0[r], step, n);
    for (int k = 0; k < n; k++)
      seen = std::fmax(seen, (double) fabsl((long double) p[(size_t) k] -
                                            ((long double) x0[r] + (long double) k * (long double) mean[r])));
    for (int q = 0; q < (disc ? 4 : 96); q++) {
      const double xo = uni(-0.6, 0.6) * size, z = near * std::exp(uni(0.0, 3.0));
      RunLine l;
      l.v0 = xo - x0[r];
      l.dv = mean[r];
      l.inv_dv = 1.0 / l.dv;
      l.w = z * z;
      l.dev = dev;
      const double dt = std::fmax(0.02, 1.1 * step / 6.0);   // at most four bins a step
      grid_of(l, 1500.0, dt, z / 1.5, 8000.0);
      if (!dream::runs_ready<true>(l, n)) { left++; continue; }
      fit++;
      worst = std::fmax(worst, line_error<true>(l, n, [&](int k) {
        return (long double) xo - (long double) p[(size_t) k];
      }, stepped));
    }
  }
  std::printf("%ld %ld %.3e %.3e %.3e\n", fit, left, worst, seen, dev);
  return 0;
}

static int rest(int lines)
{
  double most = 0.0;
  long wrong = 0, used = 0, left = 0;
  for (int q = 0; q < lines; q++) {
    const int n = 200 + (int) uni(0.0, 4000.0), tie = (int) uni(0.0, n);
    RunLine l;
    l.dv = 0.02;
    l.inv_dv = 50.0;
    l.v0 = uni(-0.2, 1.2) * n * l.dv;
    const double z = uni(4.0, 40.0), vt = l.v0 - tie * l.dv, dt = uni(0.02, 0.1);
    const double t = std::sqrt(z * z + vt * vt) * 1000.0 / 1500.0;
    l.w = z * z;
    grid_of(l, 1500.0, dt, t - (std::floor(t / dt) + 0.5) * dt, 2000.0);
    if (!dream::runs_ready<true>(l, n)) continue;
    used++;
    // In parts, as the kernel walks them.
    const int parts = 1 + q % 5;
    for (int p = 0; p < parts; p++) {
      const int k0 = n * p / parts, k1 = n * (p + 1) / parts;
      long updates = 0, walked = 0;
      std::vector<int> seen((size_t) n, 0);
      dream::walk_line<true>(l, k0, k1, [&](int, int c, double) { walked += c; },
                             [&](int lo, int hi) {
        updates += hi;                       // from the row's start, then along
        left += hi - lo;
        for (; lo < hi; lo++) seen[(size_t) lo]++;
      });
      for (int k = 0; k < n; k++) {
        walked += seen[(size_t) k];
        wrong += seen[(size_t) k] > (k >= k0 && k < k1 ? 1 : 0);
      }
      wrong += std::labs(walked - (k1 - k0));
      most = std::fmax(most, (double) updates / (double) n);
    }
  }
  std::printf("%ld %ld %.3f %ld\n", used, left, most, wrong);
  return 0;
}

static int price(int lines)
{
  double least = 1e9, most = 0.0;
  long used = 0;
  for (int q = 0; q < lines; q++) {
    const int n = 100 + (int) uni(0.0, 400.0);
    RunLine l;
    l.dv = 0.05;
    l.inv_dv = 20.0;
    l.v0 = uni(-0.5, 1.5) * n * l.dv;
    const double z = 0.5 * std::exp(uni(0.0, 4.5));
    l.w = z * z;
    grid_of(l, 1500.0, 0.01 * std::exp(uni(0.0, 3.0)), z / 1.5, 2000.0);
    if (!dream::runs_ready<true>(l, n)) continue;
    long its = 0;
    bool all = true;                       // no doubtful edge
    double along = 0.0;
    for (int k = 0; k < n; k++) along += std::fabs(l.v0 - k * l.dv) / n;
    dream::walk_line<true>(l, 0, n, [&](int, int, double) { its++; }, [&](int, int) { all = false; });
    if (!all) continue;
    used++;
    const double r = (double) its / (n * dream::runs_per_step((float) along, (float) l.w, (float) (l.c1 * l.dv),
                                                              (float) (1.0 / (36.0 * l.dv))));
    least = std::fmin(least, r);
    most = std::fmax(most, r);
  }
  std::printf("%ld %.3f %.3f\n", used, least, most);
  return 0;
}

int main(int argc, char **argv)
{
  if (argc > 3 && std::strcmp(argv[1], "equal") == 0) {
    gen.seed((unsigned) std::atoi(argv[2]));
    return equal(std::atoi(argv[3]));
  }
  if (argc > 3 && std::strcmp(argv[1], "price") == 0) {
    gen.seed((unsigned) std::atoi(argv[2]));
    return price(std::atoi(argv[3]));
  }
  if (argc > 3 && std::strcmp(argv[1], "rest") == 0) {
    gen.seed((unsigned) std::atoi(argv[2]));
    return rest(std::atoi(argv[3]));
  }
  if (argc < 5) return 2;
  gen.seed(1);
  return aperture(std::strcmp(argv[1], "disc") == 0, std::atof(argv[2]), std::atof(argv[3]), std::atof(argv[4]));
}
