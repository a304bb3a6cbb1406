// How M2L's work groups are dealt to the 8 XCDs.  Free of HIP types, so that a
// plain C++ program can check it.
#pragma once
#include <algorithm>
#include <cstdint>

#include "sincos_red.hpp"

namespace dfm {

// Workgroups are dealt to the 8 XCDs in turn.  The (level, direction, cell)
// group order is cut into segments, each into 8 contiguous parts, one per XCD:
// an XCD's L2 sees the groups that share source rows, and all XCDs read the
// same segment's table rows at a time.  Segments and parts hold equal shares
// of the rows to load (xcdParts), not of the groups.  Block b belongs to XCD
// b mod 8 and takes item b / 8 of that XCD's parts, counted over the segments
// (-1 past the last).
//
// Rows alone do not predict the time (a level's rows may or may not be in the
// caches): with one segment the XCDs ended at 1.00 to 1.39 ms of 1.47
// (100,000-point ellipsoid, order 6), at 1.95 to 2.40 (20,000-point cube,
// order 8) and at 16.6 to 19.3 (1,000,000-point sphere, order 7).  With 8 they
// end within 5% of one another: 1.43 -> 1.31, 2.39 -> 2.20 and 18.9 -> 17.6 ms
// (4: 2.26 and 17.8; 16: 2.29 and 17.9).  Short lists gain nothing and lose
// rows shared across the cuts: 12,682 groups (30,000-point sphere, order 6)
// 1.48 ms in one segment, 1.58 in eight, 5,666 groups 0.22 and 0.26, 7,800
// groups a batch (cube, 16 right-hand sides) 24.1 and 24.4; from 1,024 groups a
// part on the two are level or better.
//
// A launch covers up to kXcdChunks chunks of right-hand sides, chunk after
// chunk; XCD x takes parts (x + chunk) mod 8, so that what still differs
// between the parts evens out, and one chunk's tail overlaps the next's start:
// 16 right-hand sides, ellipsoid 10.5 -> 9.8 ms, cube at order 4 1.28 -> 1.17,
// at order 8 15.9 -> 15.5 (a launch per chunk before).
constexpr int kXcdSegments = 8;       // at most
constexpr int kXcdPartGroups = 1024;  // groups of a part, at least (on average)
constexpr int kXcdChunks = 8;
struct XcdParts {
  int segments, chunks;
  int total[8];                  // groups of part x, all segments
  int at[8 * kXcdSegments + 1];  // first group of part x in segment s: at[8 s + x]
};
// The group of block b and its chunk; -1 for a block past its XCD's last.
DFM_HD inline int partItem(const XcdParts& p, int b, int& chunk) {
  int x = b & 7, i = b >> 3;
  chunk = 0;
  while (i >= p.total[x]) {
    i -= p.total[x];
    x = (x + 1) & 7;
    if (++chunk >= p.chunks) return -1;
  }
  for (int s = 0; s < p.segments; s++) {
    const int a = p.at[8 * s + x], n = p.at[8 * s + x + 1] - a;
    if (i < n) return a + i;
    i -= n;
  }
  return -1;
}

// The parts of ng groups whose costs' running sum is cost[0 .. ng], for
// `chunks` chunks of right-hand sides; grid: 8 times the blocks of the XCD
// with the most.
inline XcdParts xcdParts(const int64_t* cost, int ng, int chunks, int64_t& grid) {
  XcdParts p{};
  p.segments = std::max(1, std::min(kXcdSegments, ng / (8 * kXcdPartGroups)));
  p.chunks = chunks;
  const int n = 8 * p.segments;
  const int64_t c0 = cost[0], total = cost[ng] - c0;
  p.at[0] = 0;
  p.at[n] = ng;
  for (int x = 1; x < n; x++)
    p.at[x] = (int)(std::lower_bound(cost, cost + ng, c0 + total / n * x + total % n * x / n) - cost);
  for (int x = 0; x < n; x++) p.total[x & 7] += p.at[x + 1] - p.at[x];
  grid = 0;
  for (int x = 0; x < 8; x++) {
    int64_t blocks = 0;
    for (int c = 0; c < chunks; c++) blocks += p.total[(x + c) & 7];
    grid = std::max(grid, 8 * blocks);
  }
  return p;
}

}  // namespace dfm
