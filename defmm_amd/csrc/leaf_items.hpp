// Rules and work items of the leaves' operators, used at upload.  Free of HIP
// types, so that a plain C++ program can check them (HIP sources read the
// items as int2).
#pragma once
#include <algorithm>
#include <vector>

#include "plan.hpp"

namespace dfm {

constexpr int kSlotCols = 16;    // slots per matrix-core tile (leaf_slots.hpp)
// Leaves with fewer slots stay on the vector units, whose work does not round
// slots up to 16: L2P of a million points at 16 wavelengths, 17 slots a leaf,
// takes 1.5 ms with a line at 24 and 2.3 with one at 6 (order 7, float), at 50
// slots a leaf (41,334 points, order 6, double) 0.28 against 0.49; P2M, whose
// vector kernel is further behind, gains from 6 slots on (1.19 -> 0.91 ms).
// Plans of few leaves leave SIMDs idle on either path, so rounding up costs
// nothing there, splitting a leaf's slots over blocks pays (510 leaves, order
// 10: L2P 0.61 -> 0.42 ms with the line at 6), and one kernel does for all.
inline int p2mSlotsMin(size_t leaves) { return leaves < 2048 ? 1 : 6; }
inline int l2pSlotsMin(size_t leaves) { return leaves < 2048 ? 1 : 24; }

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

// (leaf cell, first slot) items: leaves of several slots by kSlotCols on the
// matrix cores (slots), the others by the vector kernel's `pass` slots (few);
// for 16 right-hand sides at a time the leaves of up to kP2MMfmaPoints points
// by kP2MMfmaSlots (mfma), the larger ones right-hand side by right-hand side
// (bigSlots, bigFew).  A leaf without slots (neither its cell nor an ancestor
// takes part in M2L) has no expansions to write and makes no item.
template <typename I2>
struct P2MItems {
  std::vector<I2> few, slots, mfma, bigFew, bigSlots;
};
template <typename I2>
void buildP2MItems(const Plan& pl, int pass, P2MItems<I2>& out) {
  const int slotsMin = p2mSlotsMin(pl.p2mCell.size());
  for (int c : pl.p2mCell) {
    const int ns = pl.S.nslot[c];
    if (ns == 0) continue;
    const bool small = pl.S.nprt[c] <= kP2MMfmaPoints, cols = ns >= slotsMin;
    auto& one = cols ? out.slots : out.few;
    auto& big = cols ? out.bigSlots : out.bigFew;
    for (int k0 = 0; k0 < ns; k0 += cols ? kSlotCols : pass) {
      one.push_back(I2{c, k0});
      if (!small) big.push_back(I2{c, k0});
    }
    if (small)
      for (int k0 = 0; k0 < ns; k0 += kP2MMfmaSlots) out.mfma.push_back(I2{c, k0});
  }
}

}  // namespace dfm
