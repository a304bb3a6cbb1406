// The deal of M2L's groups to the XCDs (defmm_amd/csrc/xcd_parts.hpp): for
// numbers of groups around the lines of the segments, equal, growing and very
// uneven costs and 1 to 8 chunks, the blocks of the grid take every (chunk,
// group) once, and the parts' costs differ by no more than their largest group.
#include <cstdio>
#include <random>
#include <vector>

#include "../../defmm_amd/csrc/xcd_parts.hpp"

using namespace dfm;

int main() {
  std::mt19937 g(7);
  int64_t cases = 0, segments[kXcdSegments + 1] = {};
  for (int ng : {0, 1, 2, 7, 8, 9, 63, 64, 65, 1000, 8191, 8192, 16383, 16384, 16385, 24577, 40000,
                 65535, 65536, 70001})
    for (int kind = 0; kind < 4; kind++)
      for (int chunks = 1; chunks <= kXcdChunks; chunks += ng > 10000 && chunks < 7 ? 3 : 1) {
        std::vector<int64_t> cost(ng + 1, 1000);  // (a batch's sums do not start at 0)
        int64_t most = 0;
        for (int i = 0; i < ng; i++) {
          const int64_t c = kind == 0   ? 5
                            : kind == 1 ? 5 + i % 400
                            : kind == 2 ? (i == ng / 3 ? (int64_t)50 * ng : 4)
                                        : 4 + (int64_t)(g() % 700) * (i < ng / 2);
          most = std::max(most, c);
          cost[i + 1] = cost[i] + c;
        }
        int64_t grid = 0;
        const XcdParts p = xcdParts(cost.data(), ng, chunks, grid);
        segments[p.segments]++;
        cases++;
        std::vector<char> seen((size_t)ng * chunks, 0);
        int64_t found = 0;
        for (int64_t b = 0; b < grid; b++) {
          int chunk = -1;
          const int item = partItem(p, (int)b, chunk);
          if (item < 0) continue;
          if (item >= ng || chunk < 0 || chunk >= chunks || seen[(size_t)chunk * ng + item]++) {
            std::printf("FAIL groups %d kind %d chunks %d block %lld item %d chunk %d\n", ng, kind,
                        chunks, (long long)b, item, chunk);
            return 1;
          }
          found++;
        }
        if (found != (int64_t)ng * chunks || grid % 8 != 0) {
          std::printf("FAIL groups %d kind %d chunks %d: %lld of %lld\n", ng, kind, chunks,
                      (long long)found, (long long)ng * chunks);
          return 1;
        }
        // (a block beyond the grid, as a rounded-up launch has them, takes none)
        for (int64_t b = grid; b < grid + 64; b++) {
          int chunk = -1;
          if (partItem(p, (int)b, chunk) >= 0) {
            std::printf("FAIL block beyond the grid\n");
            return 1;
          }
        }
        const int n = 8 * p.segments;
        for (int x = 0; x < n; x++) {
          const int64_t c = cost[p.at[x + 1]] - cost[p.at[x]], share = (cost[ng] - cost[0]) / n;
          if (p.at[x + 1] < p.at[x] || c > share + most + 1) {
            std::printf("FAIL groups %d kind %d part %d costs %lld of %lld\n", ng, kind, x,
                        (long long)c, (long long)share);
            return 1;
          }
        }
      }
  std::printf("ok %lld cases, of one segment %lld, two %lld, eight %lld\n", (long long)cases,
              (long long)segments[1], (long long)segments[2], (long long)segments[8]);
  return 0;
}
