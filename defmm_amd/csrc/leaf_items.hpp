// Rules and work items of the leaves' operators, used at upload.  Free of HIP
// types, so that a plain C++ program can check them (HIP sources read the
// items as int2).
#pragma once
#include <cstdint>
#include <vector>

#include "plan.hpp"

namespace dfm {

constexpr int kSlotCols = 16;    // slots per matrix-core tile (leaf_slots.hpp)

// P2M of one right-hand side: whether a plan's leaves go to the matrix cores
// (waves: a wave per leaf and kSlotCols slots) or to the vector kernel
// (blocks: a block per leaf and pass of its slots).  A wave takes about two of
// those blocks' time, so leaves of one slot lose (30,000 points, kappa = 0,
// order 8, double: 95 us and 56) and leaves of 5 to 8 break even; from order 5
// on a wave's chain of L^3 / 16 steps also needs enough others beside it (order
// 8, float: 8,000-point ellipsoid, 640 waves, 51 us and 42; 3,000-point sphere,
// 990 waves, 52 and 48; 4,000-point cube, 1,270 waves, 59 and 60;
// 30,000-point ellipsoid, 1,900 waves, 86 and 125; 20,000-point cube, 6,000
// waves, 172 and 250).  The leaves beyond kP2MMfmaPoints points, which 16
// right-hand sides take one by one, have longer sums and gain from fewer (P2M
// of 16, order 6, 100,000-point ellipsoid, 383 such leaves, 954 waves, 1.6 ms
// and 2.2).  One kernel for all of a plan's leaves: a second launch costs more
// than it gains.
inline bool p2mOnColumns(int L, bool large, int64_t waves, int64_t blocks) {
  return (L <= 4 || waves >= (large ? 600 : 1000)) && 2 * waves <= blocks;
}

// L2P of one right-hand side: slots from which the matrix cores are the
// faster.  Plans of fewer than 2,048 leaves take one kernel for all of them
// (small: the mean over the plan's leaves counts), larger plans decide by
// leaf.  Against the vector kernel, float and double, us: order 3, 5,000-point
// cube (28 slots a leaf) 16 and 13, 29 and 15, 60,000-point sphere (178) 167
// and 158, 410 and 250; order 4, 5,000-point cube 16 and 18, 29 and 21,
// 4,000-point cube (36) 16 and 21, 18 and 25; order 5, 30,000-point ellipsoid
// (17) 36 and 46, 76 and 58; order 8, 8,000-point ellipsoid (4) 57 and 37, 72
// and 56, 5,000-point cube 74 and 88, 84 and 140, 20,000-point cube (81) 226
// and 420, 308 and 690.  The vector kernel's staging does not fit its LDS well
// at order 9 in float and 10 in double (8,000-point ellipsoid 57 and 94, 196
// and 312).
inline int l2pSlotsMin(int L, int realBytes, bool small) {
  const bool f = realBytes == 4;
  constexpr int never = INT32_MAX;
  if (L == 2) return f ? 24 : small ? 48 : never;
  if (L == 3) return f && small ? 48 : never;
  if (L == (f ? 9 : 10)) return 3;
  if (!small) return 24;
  if (L == 4) return f ? 24 : 32;
  return f || L >= 7 ? 12 : L == 6 ? 24 : 32;
}

// Matrix-core steps (of 4 weight indices) of k_l2p_slots whose sum is added to
// the slot's: one chain of L^3 terms is less exact than the vector kernel's
// nested sums of L and L^2 (float, random coefficients, order 8: 4.0e-7 and
// 1.6e-7, in chains of 16 terms 1.3e-7; order 4: 1.5e-7 and 8.6e-8, in chains
// of 8 terms 8.4e-8).  Far field of 40,000 points on a sphere at 24
// wavelengths, float, order 6: relative error 5.2e-7 with one chain, 4.6e-7
// with these, 4.8e-7 with the vector kernel.
constexpr int l2pSlotChain(int L) { return L <= 4 ? 2 : 4; }

// P2M for 16 right-hand sides: slots per block, points of a leaf at most
constexpr int kP2MMfmaSlots = 32, kP2MMfmaPoints = 64;

// (leaf cell, first slot) items: by kSlotCols slots on the matrix cores (slots)
// or by the vector kernel's `pass` slots (few); for 16 right-hand sides at a
// time the leaves of up to kP2MMfmaPoints points by kP2MMfmaSlots (mfma), the
// larger ones right-hand side by right-hand side (bigSlots or bigFew).  A leaf
// without slots (neither its cell nor an ancestor takes part in M2L) has no
// expansions to write and makes no item.
template <typename I2>
struct P2MItems {
  std::vector<I2> few, slots, mfma, bigFew, bigSlots;
};
template <typename I2>
void buildP2MItems(const Plan& pl, int pass, P2MItems<I2>& out) {
  auto one = [&](bool all, std::vector<I2>& slots, std::vector<I2>& few) {
    auto takes = [&](int c) { return all || pl.S.nprt[c] > kP2MMfmaPoints; };
    int64_t waves = 0, blocks = 0;
    for (int c : pl.p2mCell)
      if (takes(c)) {
        waves += (pl.S.nslot[c] + kSlotCols - 1) / kSlotCols;
        blocks += (pl.S.nslot[c] + pass - 1) / pass;
      }
    const bool cols = p2mOnColumns(pl.L, !all, waves, blocks);
    for (int c : pl.p2mCell)
      if (takes(c))
        for (int k0 = 0; k0 < pl.S.nslot[c]; k0 += cols ? kSlotCols : pass)
          (cols ? slots : few).push_back(I2{c, k0});
  };
  one(true, out.slots, out.few);
  one(false, out.bigSlots, out.bigFew);
  for (int c : pl.p2mCell)
    if (pl.S.nprt[c] <= kP2MMfmaPoints)
      for (int k0 = 0; k0 < pl.S.nslot[c]; k0 += kP2MMfmaSlots) out.mfma.push_back(I2{c, k0});
}

}  // namespace dfm
