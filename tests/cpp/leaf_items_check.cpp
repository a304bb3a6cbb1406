// P2M work items (defmm_amd/csrc/leaf_items.hpp) of plans from the host
// builder: every item starts at a slot that its leaf has, and the lists of one
// and of 16 right-hand sides each cover every slot of every leaf once.
#include <cmath>
#include <cstdio>
#include <map>
#include <random>
#include <string>
#include <vector>

#include "../../defmm_amd/csrc/leaf_items.hpp"

using namespace dfm;

struct Item {
  int x, y;
};

// n points of the unit sphere; patch: around one pole
static std::vector<double> sphere(int n, unsigned seed, bool patch) {
  std::mt19937_64 g(seed);
  std::normal_distribution<double> nd;
  std::vector<double> p;
  while ((int)p.size() < 3 * n) {
    double v[3], r = 0;
    for (double& x : v) { x = nd(g); r += x * x; }
    r = std::sqrt(r);
    if (patch && v[2] < 0.96 * r) continue;
    for (double x : v) p.push_back(x / r);
  }
  return p;
}

int main() {
  struct Case {
    const char* name;
    int ns, nt;  // nt = 0: the targets are the sources
    int L, ncrit;
    double nlambda;
  };
  const Case cases[] = {
      {"sphere_200", 200, 0, 4, 5, 10},   {"sphere_300", 300, 0, 4, 5, 10},
      {"patch_4000", 4000, 200, 4, 33, 8}, {"patch_40000", 40000, 300, 4, 9, 8},
      {"sphere_6000", 6000, 0, 9, 33, 6}, {"laplace_6000", 6000, 0, 3, 40, 0},
      {"big_leaves", 6000, 0, 4, 200, 1},
  };
  int failed = 0;
  for (const Case& c : cases) {
    const auto src = sphere(c.ns, 11, false), trg = c.nt ? sphere(c.nt, 12, true) : src;
    Plan pl;
    std::string msg;
    const int rc = buildPlan(pl, src.data(), c.ns, trg.data(), (int64_t)trg.size() / 3, c.L, c.ncrit,
                             M_PI * c.nlambda, msg);
    if (rc != OK) {
      std::printf("case %s FAIL build: %s\n", c.name, msg.c_str());
      failed++;
      continue;
    }
    const int pass = c.L >= 9 ? 2 : 4;
    P2MItems<Item> it;
    buildP2MItems(pl, pass, it);
    int beyond = 0, wrong = 0, without = 0;
    // how often a list covers each (leaf, slot)
    std::map<std::pair<int, int>, int> one, many;
    auto add = [&](const std::vector<Item>& list, int width, auto& seen) {
      for (const Item& i : list) {
        const int ns = pl.S.nslot[i.x];
        if (i.y < 0 || i.y >= ns) beyond++;
        for (int k = i.y; k < std::min(i.y + width, ns); k++) seen[{i.x, k}]++;
      }
    };
    add(it.few, pass, one);
    add(it.slots, kSlotCols, one);
    add(it.mfma, kP2MMfmaSlots, many);
    add(it.bigFew, pass, many);
    add(it.bigSlots, kSlotCols, many);
    size_t slots = 0;
    for (int l : pl.p2mCell) {
      const int ns = pl.S.nslot[l];
      if (ns == 0) without++;
      slots += (size_t)ns;
      for (int k = 0; k < ns; k++)
        if (one[{l, k}] != 1 || many[{l, k}] != 1) wrong++;
    }
    if (one.size() != slots || many.size() != slots) wrong++;
    std::printf("case %s %s leaves %zu without %d beyond %d wrong %d few %zu slots %zu mfma %zu big %zu\n",
                c.name, beyond || wrong ? "FAIL" : "OK", pl.p2mCell.size(), without, beyond, wrong,
                it.few.size(), it.slots.size(), it.mfma.size(),
                it.bigFew.size() + it.bigSlots.size());
    if (beyond || wrong) failed++;
  }
  return failed ? 1 : 0;
}
