// Walks random lines of sub-elements run by run (sir_runs.hpp) and one by
// one, and compares bins, counts and sums.  argv: seed, lines.  Prints
//   lines, usable lines, moved sub-elements, share left to step, worst relative
//   error of a bin's sum (REFINE), the same without, runs per sub-element
// The exact index is the reference's sequence in IEEE double.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>
#include <vector>

#include "sir_runs.hpp"

static int sat(double x)
{
  if (x != x) return -1;
  return x > 2147483647.0 ? 2147483647 : x < -2147483648.0 ? -2147483647 - 1 : (int) x;
}

int main(int argc, char **argv)
{
  std::mt19937_64 gen((unsigned) std::atoi(argv[1]));
  const int lines = std::atoi(argv[2]);
  auto uni = [&](double a, double b) { return std::uniform_real_distribution<double>(a, b)(gen); };
  long usable = 0, moved = 0, runs = 0, elems = 0, stepped = 0;
  double worst = 0.0, worst32 = 0.0;
  for (int q = 0; q < lines; q++) {
    const int kind = q % 6;
    // Positions as the package accumulates them; on a grid of 1/64 mm with
    // whole speeds and intervals of 1/8 us (kinds 4, 5) ties are common.
    const bool grid = kind >= 4;
    const double dx = grid ? 0.0625 : (kind == 0 ? 0.05 : uni(0.01, 0.2));
    const double cp = grid ? 1000.0 : uni(900.0, 1700.0), dt = grid ? 0.125 : uni(0.01, q % 2 ? 0.3 : 0.06);
    const int n = 1 + (int) uni(0.0, 330.0), nt = 100 + (int) uni(0, 2000);
    std::vector<double> pos((size_t) n);
    double s = -n * dx / 2.0 + dx / 2.0;
    if (grid) s = std::floor(s * 64) / 64;
    for (int k = 0; k < n; k++, s += dx) pos[(size_t) k] = s;
    auto snap = [&](double v) { return grid ? std::rint(v * 64.0) / 64.0 : v; };
    const double vo = snap(kind == 1 ? 0.0 : kind == 2 ? pos[(size_t) (n / 2)] : uni(-20, 20));
    const double ra = snap(kind == 5 ? 0.0 : uni(-8, 8)), rb = snap(uni(0.5, 80.0));
    double d = grid ? std::rint(uni(0, 60) * 8) / 16.0 : uni(0.0, 60.0);
    const double c1 = 1000.0 / (cp * dt), c2s = 1.0 / dt;
    if (kind == 3) {      // one sub-element exactly on a rounding boundary
      const double p = pos[(size_t) (n / 3)];
      const double t = std::sqrt((ra * ra + (vo - p) * (vo - p)) + rb * rb) * 1000.0 / cp;
      d = t - (std::floor(t / dt) + 0.5) * dt;
    }
    auto index = [&](int k) {
      const double v = vo - pos[(size_t) k];
      const double re = std::sqrt((v * v + ra * ra) + rb * rb);
      return sat(std::rint(((re * 1000.0) / cp - d) / dt));
    };
    dream::RunLine l;
    l.dv = n > 1 ? (pos[(size_t) (n - 1)] - pos[0]) / (n - 1) : dx;
    l.v0 = vo - pos[0];
    l.inv_dv = 1.0 / l.dv;
    l.w = ra * ra + rb * rb;
    l.c1 = c1;
    l.ic1 = 1.0 / c1;
    l.c2 = d * c2s;
    l.bound = 0x1p-36 * (nt + 2.0 + std::fabs(l.c2));
    if (!dream::runs_ready<true>(l, n)) continue;
    usable++;
    std::map<int, std::pair<int, long double>> want;
    for (int k = 0; k < n; k++) {
      const long double v = (long double) vo - pos[(size_t) k];
      auto &c = want[index(k)];
      c.first++;
      c.second += 1.0L / sqrtl(v * v + (long double) ra * ra + (long double) rb * rb);
    }
    // In segments, as the kernel walks them.
    const int segs = 1 + q % 3;
    for (int refine = 0; refine < 2; refine++) {
      if (refine) dream::runs_ready<true>(l, n);
      else dream::runs_ready<false>(l, n);
      std::map<int, std::pair<int, double>> got;
      auto emit = [&](int b, int c, double v) {
        if (c > 0) {
          got[b].first += c;
          got[b].second += v;
        }
        runs++;
      };
      for (int g = 0; g < segs; g++) {
        const int k0 = n * g / segs, k1 = n * (g + 1) / segs;
        if (k0 >= k1) continue;
        for (int half = 0; half < 2; half++) {
          int len;
          const int first = dream::half_of(l, half, k0, k1, len);
          int j = refine ? dream::walk_half<true>(l, half, first, len, emit)
                         : dream::walk_half<false>(l, half, first, len, emit);
          stepped += len - j;
          for (; j < len; j++) {
            const int k = half ? first - j : first + j;
            const double v = vo - pos[(size_t) k];
            got[index(k)].first++;
            got[index(k)].second += 1.0 / std::sqrt(v * v + l.w);
          }
        }
      }
      elems += n;
      for (auto &x : want) {
        auto &g = got[x.first];
        moved += std::abs(g.first - x.second.first);
        if (g.first != x.second.first) continue;
        const double e = (double) fabsl((g.second - x.second.second) / x.second.second);
        (refine ? worst : worst32) = std::fmax(refine ? worst : worst32, e);
      }
      for (auto &x : got) if (!want.count(x.first)) moved += x.second.first;
    }
  }
  std::printf("%d %ld %ld %.4f %.3e %.3e %.4f\n", lines, usable, moved,
              (double) stepped / (double) elems, worst, worst32, (double) runs / (double) elems);
  return 0;
}
