// Root-mean-square errors of the near field's float cos and sin of kappa * r
// over distances and wavenumbers as a near field meets them, against long
// double: dfm::phaseTable (defmm_amd/csrc/phase.hpp) with the table that the
// kernels hold, and polynomials of the phase reduced by pi / 2
// (dfm::sincosRedF), for each wavenumber from the same distances.  First how far
// the table's entries are from cos and sin of their angles.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "../../defmm_amd/csrc/phase.hpp"

struct Entry {
  float x, y, z;
};

int main() {
  std::vector<Entry> tab(dfm::kPhaseN);
  dfm::phaseEntriesF(tab.data());
  double far = 0, shift = 0;
  for (int k = 0; k < dfm::kPhaseN; k++) {
    const long double a =
        2.0L * 3.141592653589793238462643383279502884L * k / dfm::kPhaseN - tab[k].z;
    far = std::max(far, (double)std::max(fabsl(cosl(a) - tab[k].x), fabsl(sinl(a) - tab[k].y)));
    shift = std::max(shift, (double)std::fabs(tab[k].z));
  }
  printf("entries %.4e shift %.4e\n", far, shift);
  std::mt19937_64 g(2025);
  for (double kappa : {1.0, 12.566370614359172, 201.06192982974676, 804.3}) {
    const dfm::PhaseConsts pc = dfm::phaseConstsOf(kappa);
    std::uniform_real_distribution<double> u(std::log(1e-3), std::log(0.2));
    double et = 0, ep = 0;
    const int n = 1000000;
    for (int i = 0; i < n; i++) {
      const double r = std::exp(u(g));
      const long double a = (long double)kappa * (long double)r;
      const long double c = cosl(a), s = sinl(a);
      float ct, st, cp, sp;
      dfm::phaseTable(r, 1.0f, pc, tab.data(), ct, st);
      dfm::sincosRedF(kappa * r, sp, cp);
      auto sq = [&](float co, float si) {
        const double x = (double)(co - c), y = (double)(si - s);
        return x * x + y * y;
      };
      et += sq(ct, st);
      ep += sq(cp, sp);
    }
    printf("kappa %.3e table %.4e polynomials %.4e\n", kappa, std::sqrt(et / n),
           std::sqrt(ep / n));
  }
  return 0;
}
