// dftForward and dftInverse (defmm_amd/csrc/dft.hpp) of every order against
// the direct sums in long double: prints the largest error relative to the
// sum of the inputs' magnitudes.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>

#include "../../defmm_amd/csrc/dft.hpp"

template <typename R>
struct Z {
  R x, y;
};

template <int L, typename R>
double check() {
  constexpr int P = 2 * L - 1;
  const long double tp = 2.0L * 3.141592653589793238462643383279502884L / P;
  R c[L], s[L];
  for (int m = 0; m < L; m++) {
    c[m] = (R)cosl(tp * m);
    s[m] = (R)sinl(tp * m);
  }
  std::mt19937 g(7 + L);
  std::uniform_real_distribution<double> u(-1, 1);
  double worst = 0;
  for (int rep = 0; rep < 200; rep++) {
    Z<R> xf[L], yf[P], xi[P], yi[L];
    long double mf = 0, mi = 0;
    for (auto& v : xf) {
      v = {(R)u(g), (R)u(g)};
      mf += hypotl(v.x, v.y);
    }
    for (auto& v : xi) {
      v = {(R)u(g), (R)u(g)};
      mi += hypotl(v.x, v.y);
    }
    dfm::dftForward<L, R>(xf, yf, c, s);
    dfm::dftInverse<L, R>(xi, yi, c, s);
    for (int k = 0; k < P; k++) {
      long double a = 0, b = 0;
      for (int j = 0; j < L; j++) {
        const long double cc = cosl(tp * (j * k % P)), ss = -sinl(tp * (j * k % P));
        a += cc * xf[j].x - ss * xf[j].y;
        b += cc * xf[j].y + ss * xf[j].x;
      }
      worst = std::max(worst, (double)(hypotl(yf[k].x - a, yf[k].y - b) / mf));
    }
    for (int k = 0; k < L; k++) {
      long double a = 0, b = 0;
      for (int v = 0; v < P; v++) {
        const long double cc = cosl(tp * (v * k % P)), ss = sinl(tp * (v * k % P));
        a += cc * xi[v].x - ss * xi[v].y;
        b += cc * xi[v].y + ss * xi[v].x;
      }
      worst = std::max(worst, (double)(hypotl(yi[k].x - a, yi[k].y - b) / mi));
    }
  }
  return worst;
}

template <int L>
void both() {
  printf("L %d double %.3e float %.3e\n", L, check<L, double>(), check<L, float>());
}

int main() {
  both<2>(); both<3>(); both<4>(); both<5>(); both<6>(); both<7>(); both<8>(); both<9>();
  both<10>();
  return 0;
}
