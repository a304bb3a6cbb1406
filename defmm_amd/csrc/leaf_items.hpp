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
// (blocks: a block per leaf and pass of its slots).  One kernel for all of a
// plan's leaves: a second launch costs more than it gains.
//
// Up to order 3 the matrix cores are the faster ones also for leaves of one
// slot (12,000-point sphere, kappa = 0, order 2, double, 12 us and 19;
// 30,000-point ellipsoid, 1.1 slots a leaf, order 3, float, 18 and 28), at order
// 4 for all but those.  From order 5 on a wave's chain of L^3 / 16 steps takes
// about two of the blocks' time and needs enough others beside it (double,
// 30,000-point cube, 1,420 waves, order 5, 70 us and 44, order 8, 204 and 175;
// 30,000-point ellipsoid, 1,900 waves, order 8, float, 86 and 125; 20,000-point
// cube, 6,000 waves, 172 and 250).  Of 700 plans in each type (four geometries,
// 3,000 to 60,000 points, 0 to 14 wavelengths, orders 2 to 10) the kernel taken
// is 1% slower than the better one in the mean.  The leaves beyond
// kP2MMfmaPoints points (large), which 16 right-hand sides take one by one,
// have longer sums and gain from fewer (P2M of 16, order 6, 100,000-point
// ellipsoid, 383 such leaves, 954 waves, 1.6 ms and 2.2).
inline bool p2mOnColumns(int L, bool large, int64_t waves, int64_t blocks) {
  if (L <= 3) return true;
  if (L == 4) return 20 * blocks >= 21 * waves;
  return waves >= (large ? 600 : 1500) && 2 * waves <= blocks;
}

// L2P of one right-hand side: slots from which the matrix cores are the
// faster.  Plans of fewer than 2,048 leaves take one kernel for all of them
// (the mean over the plan's leaves counts), larger plans decide by leaf.
//
// Below 300 leaves, about a block a CU, a launch takes as long as its longest
// leaf, which the vector kernel goes through 4 or 8 slots at a time and the
// matrix cores 64: the vector kernel is the faster one only for leaves of one
// or two slots (kappa = 0), at order 3 in double up to 20.  Matrix cores and
// vector kernel, us, 4,978 to 5,000 points in 125 to 202 leaves: order 4, 9 slots
// a leaf, double 13 and 19, float 11 and 15; order 6, 22 slots, 26 and 68, 17
// and 42; order 8, 9 slots, 36 and 78, 31 and 64; order 4, one slot, 9 and 7.
// From there on, double and float: order 4, 8,000-point sphere (17) 26 and 20,
// 12,000-point sphere (18), float, 15 and 18; order 5, 12,000-point sphere (18)
// 40 and 34, 30,000-point ellipsoid (9), float, 27 and 43; order 6,
// 30,000-point sphere (16) 90 and 107, 8,000 points in clusters (8), float, 34
// and 24; order 8, 12,000 points in clusters (9) 103 and 85, 66 and 51, ellipsoid
// (10) 80 and 93.  The vector kernel's staging does not fit its LDS well at
// order 9 in float and 10 in double.
//
// Of 540 plans each in double and float (four geometries, 3,000 to 30,000
// points, 0 to 14 wavelengths, orders 2 to 10) 95% take the faster kernel or
// one within 5% of it.
inline int l2pSlotsMin(int L, int realBytes, size_t leaves) {
  const bool f = realBytes == 4;
  constexpr int never = INT32_MAX;
  if (leaves < 300) {
    if (f) return L == 9 ? 1 : 5;
    return L == 3 ? 21 : L == 10 ? 2 : 5;
  }
  if (leaves < 2048) {
    constexpr int dbl[11] = {0, 0, 36, never, 20, 20, 16, 6, 10, 9, 3};
    constexpr int flt[11] = {0, 0, 9, 20, 9, 6, 9, 9, 10, 2, 9};
    return f ? flt[L] : dbl[L];
  }
  if (L == 2) return f ? 24 : never;
  if (L == 3) return never;
  return L == (f ? 9 : 10) ? 3 : 24;
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
