// Near-field items (defmm_amd/csrc/near_items.hpp) of plans from the host
// builder: the items of both kernels cover every (target, source) pair of
// every leaf once, by a walk of their own, and checkP2PItems accepts them and
// refuses lists with one item changed.
#include <cmath>
#include <cstdio>
#include <random>
#include <string>
#include <vector>

#include "../../defmm_amd/csrc/near_items.hpp"

using namespace dfm;

static std::vector<double> cloud(int n, unsigned seed, bool clustered) {
  std::mt19937_64 g(seed);
  std::normal_distribution<double> nd;
  std::vector<double> p(3 * (size_t)n);
  for (int i = 0; i < n; i++)
    for (int k = 0; k < 3; k++)
      p[3 * (size_t)i + k] = clustered ? (i % 5) * (k + 1) * 0.2 + 0.01 * nd(g) : nd(g);
  return p;
}

int main() {
  struct Case {
    const char* name;
    int ns, nt;  // nt = 0: the targets are the sources
    bool clustered;
    int ncrit;
    double kappa;
  };
  const Case cases[] = {{"uniform", 3000, 0, false, 20, 0.5}, {"few_points", 700, 0, false, 2, 0.5},
                        {"clusters", 4000, 900, true, 60, 2}, {"large_leaves", 9000, 5000, true, 1700, 0}};
  int failed = 0;
  for (const Case& c : cases) {
    const auto src = cloud(c.ns, 3, c.clustered), trg = c.nt ? cloud(c.nt, 4, c.clustered) : src;
    Plan pl;
    std::string msg;
    int rc = buildPlan(pl, src.data(), c.ns, trg.data(), (int64_t)trg.size() / 3, 3, c.ncrit,
                       c.kappa, msg);
    if (rc != OK) {
      std::printf("case %s FAIL build: %s\n", c.name, msg.c_str());
      failed++;
      continue;
    }
    const NearLists lists = nearLists(pl);
    for (int tg : {kP2PTargets, kP2PMfmaTargets}) {
      std::vector<P2PItem> items;
      std::vector<int> beg;
      rc = buildP2PItems(pl, lists, tg, items, beg, msg);
      int wrong = rc != OK;
      for (size_t lf = 0; lf < pl.p2pLeaf.size() && !wrong; lf++) {
        const int n = pl.T.nprt[pl.p2pLeaf[lf]];
        std::vector<int> list;
        for (int r = pl.p2pBeg[lf]; r < pl.p2pBeg[lf + 1]; r++)
          for (int j = pl.p2pSrcB[r]; j < pl.p2pSrcE[r]; j++) list.push_back(j);
        // per target the sources in the order that its items take them
        std::vector<std::vector<int>> got(n);
        for (int k = beg[lf]; k < beg[lf + 1]; k++) {
          const P2PItem& it = items[k];
          int r = it.r, o = it.off;
          for (int s = 0; s < it.cnt; s++, o++) {
            while (o >= pl.p2pSrcE[r] - pl.p2pSrcB[r]) o -= pl.p2pSrcE[r] - pl.p2pSrcB[r], r++;
            for (int t = it.t0; t < it.t0 + it.nt; t++) got.at(t).push_back(pl.p2pSrcB[r] + o);
          }
        }
        for (int t = 0; t < n; t++) wrong += got[t] != list;
      }
      // lists with one item changed
      int missed = 0, tried = 0;
      std::mt19937 g(tg);
      for (int k = 0; k < 400; k++) {
        auto bad = items;
        auto badBeg = beg;
        const size_t i = g() % items.size();
        switch (k % 8) {
          case 0: bad[i].r = pl.p2pBeg[bad[i].leaf + 1]; break;  // the next leaf's list
          case 1: bad[i].off += pl.p2pSrcE[bad[i].r] - pl.p2pSrcB[bad[i].r]; break;
          case 2: bad[i].cnt++; break;
          case 3: bad[i].cnt = 0; break;
          case 4: bad[i].t0++; break;
          case 5: bad[i].nt++; break;
          case 6: bad[i].off--; break;
          case 7:  // an item gone
            bad.erase(bad.begin() + i);
            for (size_t l = 0; l < badBeg.size(); l++) badBeg[l] -= badBeg[l] > (int)i;
            break;
        }
        tried++;
        missed += checkP2PItems(pl, lists, tg, bad, badBeg).empty();
      }
      const bool ok = !wrong && !missed && checkP2PItems(pl, lists, tg, items, beg).empty();
      std::printf("case %s %d %s leaves %zu items %zu wrong %d tried %d missed %d\n", c.name, tg,
                  ok ? "OK" : "FAIL", pl.p2pLeaf.size(), items.size(), wrong, tried, missed);
      failed += !ok;
    }
  }
  return failed ? 1 : 0;
}
