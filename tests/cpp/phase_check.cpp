// Accuracy of dfm::phaseTable (defmm_amd/csrc/phase.hpp) against long double
// cosl / sinl of kappa * r: prints, for each wavenumber, the largest absolute
// errors of the double and the float values and of the double values formed
// by rounding kappa * r first (dfm::sincosRed).
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "../../defmm_amd/csrc/phase.hpp"

template <typename R>
struct Pair {
  R x, y;
};

int main() {
  std::vector<Pair<double>> td(dfm::kPhaseN);
  std::vector<Pair<float>> tf(dfm::kPhaseN);
  for (int k = 0; k < dfm::kPhaseN; k++) {
    dfm::phaseEntry(k, td[k].x, td[k].y);
    tf[k] = {(float)td[k].x, (float)td[k].y};
  }
  std::mt19937_64 g(4711);
  for (double kappa : {1e-30, 1e-3, 1.0, 12.566370614359172, 201.06192982974676, 804.3, 7.7e4}) {
    const dfm::PhaseConsts pc = dfm::phaseConstsOf(kappa);
    double ed = 0, ef = 0, er = 0;
    auto check = [&](double r) {
      const long double a = (long double)kappa * (long double)r;
      const long double c = cosl(a), s = sinl(a);
      double cd, sd, cr, sr;
      float cf, sf;
      dfm::phaseTable(r, 1.0, pc, td.data(), cd, sd);
      dfm::phaseTable(r, 1.0f, pc, tf.data(), cf, sf);
      dfm::sincosRed(kappa * r, sr, cr);
      ed = std::max(ed, (double)std::max(fabsl(cd - c), fabsl(sd - s)));
      ef = std::max(ef, (double)std::max(fabsl(cf - c), fabsl(sf - s)));
      er = std::max(er, (double)std::max(fabsl(cr - c), fabsl(sr - s)));
    };
    // phases up to 1,000, the points halfway between two table angles, tiny r
    std::uniform_real_distribution<double> u(0.0, 1000.0);
    for (int i = 0; i < 1000000; i++) check(u(g) / kappa);
    for (int k = 0; k < 20000; k++) {
      const double r = (k + 0.5) * pc.h;
      check(r);
      check(std::nextafter(r, 1e300));
      check(std::nextafter(r, 0.0));
      check(k * pc.h);
    }
    for (double x = 1e-200; x < 1.0; x *= 1.7) check(x / std::max(kappa, 1.0));
    check(0.0);
    printf("kappa %.3e double %.3e float %.3e rounded_first %.3e\n", kappa, ed, ef, er);
  }
  // the selection: none, table inside its range, expi outside
  printf("select %d %d %d %d %d %d\n", dfm::phaseOf(0.0, true), dfm::phaseOf(1.0, true),
         dfm::phaseOf(1.0, false), dfm::phaseOf(1e-31, true), dfm::phaseOf(1e-30, true),
         dfm::phaseOf(1.1e30, true));
  return 0;
}
