// A CPU model of L2P's sum over one slot's coefficients in float: the vector
// kernel's nested sums (L terms, then L^2), and the matrix cores' chains of 4
// l2pSlotChain(L) terms (defmm_amd/csrc/leaf_items.hpp), added up.  Prints the
// rms errors against double for random points and coefficients.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "../../defmm_amd/csrc/leaf_items.hpp"

int main() {
  std::mt19937_64 g(5);
  std::normal_distribution<double> nd;
  std::uniform_real_distribution<double> ud(-1, 1);
  for (int L = 2; L <= 10; L++) {
    const int LL = L * L * L, len = 4 * dfm::l2pSlotChain(L);
    double en = 0, ec = 0, ref = 0;
    std::vector<double> xi(L);
    for (int i = 0; i < L; i++) xi[i] = -1 + 2.0 * i / (L - 1);
    std::vector<float> w[3], b(LL);
    for (auto& v : w) v.resize(L);
    for (int it = 0; it < 20000; it++) {
      for (auto& v : w) {
        const double t = ud(g);
        for (int i = 0; i < L; i++) {
          double p = 1;
          for (int j = 0; j < L; j++)
            if (j != i) p *= (t - xi[j]) / (xi[i] - xi[j]);
          v[i] = (float)p;
        }
      }
      for (auto& x : b) x = (float)nd(g);
      double ex = 0;
      float nested = 0, chains = 0;
      for (int a = 0; a < L; a++)
        for (int c = 0; c < L; c++) {
          float s = 0;
          for (int e = 0; e < L; e++) {
            s = fmaf(w[2][e], b[(a * L + c) * L + e], s);
            ex += (double)w[0][a] * w[1][c] * w[2][e] * b[(a * L + c) * L + e];
          }
          const float t = w[0][a] * w[1][c];
          nested = fmaf(t, s, nested);
        }
      for (int i0 = 0; i0 < LL; i0 += len) {
        float s = 0;
        for (int i = i0; i < std::min(LL, i0 + len); i++) {
          const float t = w[0][i / (L * L)] * w[1][(i / L) % L];
          s = fmaf(t * w[2][i % L], b[i], s);
        }
        chains += s;
      }
      en += (nested - ex) * (nested - ex);
      ec += (chains - ex) * (chains - ex);
      ref += ex * ex;
    }
    std::printf("order %d nested %.4e chains %.4e\n", L, std::sqrt(en / ref), std::sqrt(ec / ref));
  }
  return 0;
}
