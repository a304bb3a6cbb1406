// Work items of the near field, built and checked at upload.  Host-only apart
// from the item's layout and free of HIP types, so that a plain C++ program
// can check them.
#pragma once
#include <algorithm>
#include <cstdint>
#include <exception>
#include <string>
#include <thread>
#include <vector>

#include "plan.hpp"
#include "sincos_red.hpp"

namespace dfm {

// Work item: nt targets of one leaf, from t0 (leaf-relative), against cnt
// sources of its list from (range r, offset off).
struct P2PItem {
  int leaf, t0, nt, r, off, cnt;
};
// Targets per item at most: of the kernel with a lane per source, and of the
// matrix cores' (two row blocks of 16).
constexpr int kP2PTargets = 8, kP2PMfmaTargets = 32;
// A leaf's n targets are cut into equal chunks of at most tg; tg itself where
// an item works on whole row blocks of 16.
DFM_HD inline int p2pChunk(int n, int tg) {
  if (tg % 16 == 0) return tg;
  const int chunks = (n + tg - 1) / tg;
  return (n + chunks - 1) / chunks;
}

// Where the ranges stand in their leaves' lists (the sources of the leaf's
// ranges before each), and the lists' lengths.  Filled in parallel over leaves:
// 200,000 points at 64 wavelengths have 3.5 million ranges.
struct NearLists {
  ListVec before;
  std::vector<int> total;
};
inline NearLists nearLists(const Plan& pl) {
  NearLists l;
  const size_t nl = pl.p2pLeaf.size();
  l.before.resize(pl.p2pSrcB.size());
  l.total.assign(nl, 0);
  auto fill = [&](size_t lf0, size_t lf1) {
    for (size_t lf = lf0; lf < lf1; lf++) {
      int n = 0;  // (a list holds a source once, so its length is an int)
      for (int r = pl.p2pBeg[lf]; r < pl.p2pBeg[lf + 1]; r++) {
        l.before[r] = n;
        n += pl.p2pSrcE[r] - pl.p2pSrcB[r];
      }
      l.total[lf] = n;
    }
  };
  const size_t nth = std::max<size_t>(
      1, std::min<size_t>({16, std::thread::hardware_concurrency(), pl.p2pSrcB.size() / 65536}));
  std::vector<std::thread> th;
  th.reserve(nth);
  size_t begun = 1;
  try {
    for (; begun < nth; begun++)
      th.emplace_back(fill, nl * begun / nth, nl * (begun + 1) / nth);
  } catch (const std::exception&) {  // no more threads or memory: the rest here
    fill(nl * begun / nth, nl);
  }
  fill(0, nl / nth);
  for (auto& x : th) x.join();
  return l;
}

// What the kernels take for granted: every item's sources lie inside its
// leaf's list (they walk the ranges from (r, off) without a bound) and its
// targets inside the leaf, and a leaf's items are, run after run of its whole
// list, one per chunk of targets (the reduction counts them so).  Empty, or
// what is wrong.
inline std::string checkP2PItems(const Plan& pl, const NearLists& lists, int tg,
                                 const std::vector<P2PItem>& items, const std::vector<int>& beg) {
  const size_t nl = pl.p2pLeaf.size();
  if (beg.size() != nl + 1 || beg[0] != 0 || beg[nl] != (int)items.size())
    return "internal: P2P item bounds";
  for (size_t lf = 0; lf < nl; lf++) {
    const int n = pl.T.nprt[pl.p2pLeaf[lf]], chunks = (n + tg - 1) / tg;
    const int rb = pl.p2pBeg[lf], re = pl.p2pBeg[lf + 1];
    const int64_t total = lists.total[lf];
    if (beg[lf + 1] < beg[lf] || (total > 0) != (beg[lf + 1] > beg[lf]) ||
        (beg[lf + 1] - beg[lf]) % std::max(1, chunks) != 0)
      return "internal: near-field items do not match the leaf's chunks";
    const int chunk = chunks > 0 ? p2pChunk(n, tg) : 0;
    int64_t pos = 0;  // where the present run starts in the leaf's list
    for (int k = beg[lf]; k < beg[lf + 1]; k++) {
      const P2PItem& it = items[k];
      const int ch = (k - beg[lf]) % chunks;
      if (it.leaf != (int)lf || it.t0 != ch * chunk || it.nt < 1 || it.nt > tg ||
          it.nt != std::min(chunk, n - it.t0) || it.r < rb || it.r >= re || it.cnt < 1)
        return "internal: P2P item out of range";
      if (it.off < 0 || it.off >= pl.p2pSrcE[it.r] - pl.p2pSrcB[it.r] ||
          lists.before[it.r] + it.off != pos || pos + it.cnt > total)
        return "internal: P2P item exceeds its source list";
      if (ch == chunks - 1) pos += it.cnt;
      else if (it.cnt != items[k + 1].cnt) return "internal: P2P item out of range";
    }
    if (pos != total) return "internal: near-field items leave sources out";
  }
  return "";
}

// A leaf's targets in chunks of at most tg (p2pChunk), its source list in
// equal runs (multiples of 64) of at most `budget` sources.  8,192 sources a
// run amortise a wave's start and final sums; where that leaves fewer than
// 16,384 items (16 waves per SIMD's share of the chip are needed to hide
// latency and even out the end) the budget is halved, down to 512.
inline int buildP2PItems(const Plan& pl, const NearLists& lists, int tg,
                         std::vector<P2PItem>& items, std::vector<int>& beg, std::string& msg) {
  const Tree& T = pl.T;
  const size_t nl = pl.p2pLeaf.size();
  auto chunksOf = [&](size_t lf) { return (T.nprt[pl.p2pLeaf[lf]] + tg - 1) / tg; };
  int64_t budget = 8192;
  for (;; budget /= 2) {
    int64_t n = 0;
    for (size_t lf = 0; lf < nl; lf++) n += chunksOf(lf) * ((lists.total[lf] + budget - 1) / budget);
    if (n > INT32_MAX / 2) {
      msg = "near-field work items exceed the launch index range";
      return ERR_ARG;
    }
    if (n >= 16384 || budget <= 512) {
      items.reserve((size_t)n);
      break;
    }
  }
  for (size_t lf = 0; lf < nl; lf++) {
    beg.push_back((int)items.size());
    const int n = T.nprt[pl.p2pLeaf[lf]], chunks = chunksOf(lf);
    const int64_t total = lists.total[lf], runs = (total + budget - 1) / budget;
    if (runs == 0 || chunks == 0) continue;
    const int chunk = p2pChunk(n, tg);
    const int64_t len = ((total + runs - 1) / runs + 63) / 64 * 64;
    const auto first = lists.before.begin() + pl.p2pBeg[lf],
               last = lists.before.begin() + pl.p2pBeg[lf + 1];
    for (int64_t pos = 0; pos < total; pos += len) {
      const int cnt = (int)std::min(len, total - pos);
      // the range that holds source pos of the list
      const auto at = std::upper_bound(first, last, pos) - 1;
      const int r = (int)(at - lists.before.begin()), off = (int)(pos - *at);
      for (int t0 = 0; t0 < n; t0 += chunk)
        items.push_back({(int)lf, t0, std::min(chunk, n - t0), r, off, cnt});
    }
  }
  beg.push_back((int)items.size());
  const std::string bad = checkP2PItems(pl, lists, tg, items, beg);
  if (bad.empty()) return OK;
  msg = bad;
  return ERR_STATE;
}

}  // namespace dfm
