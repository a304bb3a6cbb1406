// P2M and L2P of one right-hand side on the matrix cores, for leaves with
// several direction slots (reference include/operators/P2M.hpp:113-136,
// L2P.hpp:121-173):
//   M_s[I] = conj(sig2_s[I]) sum_j S_I(y_j) W_s[j],  W_s[j] = q_j exp(-i kappa d_s.(y_j - c))
//   p_i   += sum_s exp(i kappa d_s.(x_i - c)) sum_I S_I(x_i) (sig2_s[I] L_s[I])
// The Lagrange weights S are real and the same for all of a leaf's slots, so
// both are products of a real matrix with 16 slots' complex columns (L2P) or
// rows (P2M): V_MFMA_F64_16X16X4_F64 or V_MFMA_F32_16X16X4_F32, one each for
// the real and the imaginary part.  Operand layouts (A 16 x 4, B 4 x 16, D 16 x 16): lane
// l holds A[l % 16][l / 16] and B[l / 16][l % 16]; D column l % 16, and row
// 4 (l / 16) + v (float) or 4 v + l / 16 (double) in register v.
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "leaf_items.hpp"

namespace dfm {

constexpr int kL2PSlots = 128;   // slots per block of k_l2p_slots

typedef double mfma_v4d __attribute__((ext_vector_type(4)));
template <typename R>
struct Mfma16;
template <>
struct Mfma16<float> {
  typedef mfma_v4f V;
  static __device__ __forceinline__ V mac(float a, float b, V c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int quad, int v) { return 4 * quad + v; }
};
template <>
struct Mfma16<double> {
  typedef mfma_v4d V;
  static __device__ __forceinline__ V mac(double a, double b, V c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int quad, int v) { return 4 * v + quad; }
};

// 1D Lagrange weights of up to NP points of a cell: Wt[3][NP][L], zero
// beyond n, and the offsets rel[3][NP] from its centre.
template <typename R, int L, int NP>
__device__ __forceinline__ void stageWeights(R (&Wt)[3][NP][L], double (&rel)[3][NP],
                                             const double* __restrict__ px,
                                             const double* __restrict__ py,
                                             const double* __restrict__ pz, int p0, int n,
                                             const double* ctr, double rad, const OpConsts<R>& oc,
                                             int tid, int threads) {
  for (int x = tid; x < 3 * NP; x += threads) {
    const int k = x / NP, i = x - k * NP;
    double r = 0.;
    if (i < n) r = (k == 0 ? px : k == 1 ? py : pz)[p0 + i] - ctr[k];
    rel[k][i] = r;
    R t[LMAX];
    lagrangeAll<R>((R)(r / rad), L, oc.xi, oc.iden, t);
#pragma unroll
    for (int a = 0; a < L; a++) Wt[k][i][a] = i < n ? t[a] : (R)0;
  }
}

// P2M.  A wave per (leaf, 16 slots).  The leaf's points are taken 64 at a
// time: a lane forms the charges W of its slot at 16 of them (A operands: slots
// x points, kept in registers) and every 16 columns of L^3 run ceil(n / 4)
// steps (B operands: the products of three weights).  Lane l ends with weight
// index 16 m + l % 16 of four slots, so a store covers whole lines of 16
// values.  Points beyond the first 64 add to the expansions that the wave
// itself has written.
//
// Bound by writing the expansions (20,000 points, order 8, double: 0.8 GB,
// 0.17 ms at the copy rate) and the latency of a wave's short chains.  Against
// a thread per grid point over all points with weights and charges from LDS
// (k_p2m): there 0.56 -> 0.29 ms, order 4 92 -> 52 us, 200,000-point sphere at
// 64 wavelengths, order 5, 3.7 -> 2.5 ms (double), 2.2 -> 1.3 ms (float).  With
// the operands the other way round (slots as columns: 8 bytes of every 32 a
// store in float) 60,000 points, order 7, float, took 1.45 ms where this takes
// 0.74 and k_p2m 1.19.
template <typename R, int L>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void k_p2m_slots(
    const int2* __restrict__ items, DevCells S, DevLevels lv, const double* __restrict__ px,
    const double* __restrict__ py, const double* __restrict__ pz,
    const typename C2T<R>::T* __restrict__ q, const double* __restrict__ dirs,
    const typename C2T<R>::T* __restrict__ sig2, OpConsts<R> oc, double kappa,
    typename C2T<R>::T* __restrict__ M, int nItems) {
  typedef typename C2T<R>::T R2;
  typedef Mfma16<R> X;
  constexpr int LL = L * L * L, MT = (LL + 15) / 16, NP = 64, KS = NP / 4;
  __shared__ R Wt[3][NP][L];
  __shared__ double rel[3][NP];
  const int item = (int)(blockIdx.y * gridDim.x + blockIdx.x);
  if (item >= nItems) return;
  const int2 it = items[item];
  const int c = it.x, k0 = it.y;
  const int lvl = S.lvl[c], pb = S.pbeg[c], n = S.nprt[c], s0 = S.slot0[c], ns = S.nslot[c];
  if (k0 >= ns) return;  // (ns - 1 below is one of the leaf's slots)
  const double ctr[3] = {S.ctr[3 * c], S.ctr[3 * c + 1], S.ctr[3 * c + 2]}, rad = S.rad[c];
  const int hf = lv.isHF[lvl], doff = lv.dirOff[lvl], srow = lv.sigRow0[lvl];
  const int lane = threadIdx.x;
  const int lr = lane & 15, quad = lane >> 4;
  // this lane's slot as an operand, and the directions of the four slots that
  // it stores
  const int d = hf ? S.slotDir[s0 + min(k0 + lr, ns - 1)] : 0;
  int dirOf[4];
#pragma unroll
  for (int v = 0; v < 4; v++)
    dirOf[v] = hf ? S.slotDir[s0 + min(k0 + X::row(quad, v), ns - 1)] : 0;
  double dx = 0., dy = 0., dz = 0.;
  if (hf) {
    dx = dirs[3 * (doff + d)];
    dy = dirs[3 * (doff + d) + 1];
    dz = dirs[3 * (doff + d) + 2];
  }
  for (int j0 = 0; j0 < n; j0 += NP) {
    const int cn = min(NP, n - j0);
    if (j0 > 0) __syncthreads();
    stageWeights<R, L, NP>(Wt, rel, px, py, pz, pb + j0, cn, ctr, rad, oc, lane, 64);
    __syncthreads();
    const int ksn = (cn + 3) / 4;
    R br[KS], bi[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      br[ks] = bi[ks] = 0;
      const int j = 4 * ks + quad;
      if (ks < ksn && j < cn) {
        R2 v = q[pb + j0 + j];
        if (hf) {
          R cs, sn;
          expi(-kappa * (dx * rel[0][j] + dy * rel[1][j] + dz * rel[2][j]), cs, sn);
          v = cmul(v, c2<R>(cs, sn));
        }
        br[ks] = v.x;
        bi[ks] = v.y;
      }
    }
    // (not unrolled: the operands of several row blocks would not fit the
    // registers beside the slot's charges)
#pragma unroll 1
    for (int mt = 0; mt < MT; mt++) {
      const int I = min(16 * mt + lr, LL - 1);  // (columns beyond LL are not stored)
      const int a0 = I / (L * L), a1 = (I / L) % L, a2 = I % L;
      // (in float the epilogue's operands are loaded ahead of the steps; in
      // double they would not fit the registers)
      constexpr bool kAhead = sizeof(R) == 4;
      auto phase = [&](int v) { return sig2[(size_t)(srow + dirOf[v]) * LL + I]; };
      auto out = [&](int v) { return M + (size_t)(s0 + k0) * LL + X::row(quad, v) * LL + I; };
      R2 sg[kAhead ? 4 : 1], old[kAhead ? 4 : 1];
      if constexpr (kAhead)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          if (hf) sg[v] = phase(v);
          if (j0 > 0 && k0 + X::row(quad, v) < ns) old[v] = *out(v);
        }
      typename X::V dre = {0, 0, 0, 0}, dim = {0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        if (ks >= ksn) break;
        const int j = 4 * ks + quad;
        const R a = Wt[0][j][a0] * Wt[1][j][a1] * Wt[2][j][a2];
        dre = X::mac(br[ks], a, dre);
        dim = X::mac(bi[ks], a, dim);
      }
      if (16 * mt + lr < LL) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
          if (k0 + X::row(quad, v) < ns) {
            R2 val = c2<R>(dre[v], dim[v]);
            R2* o = out(v);
            if (hf) {
              if constexpr (kAhead) val = cmulc(val, sg[v]);
              else val = cmulc(val, phase(v));
            }
            if (j0 > 0) {
              R2 was;
              if constexpr (kAhead) was = old[v];
              else was = *o;
              val.x += was.x;
              val.y += was.y;
            }
            *o = val;
          }
        }
      }
    }
  }
}

// Points per tile of k_l2p_slots: 32 where their S (points x L^3, without
// padding) fits 64 KB (double up to order 6, float up to 8), else 16 whatever
// they take: with padding 70, 95 and 132 KB in double at orders 8, 9 and 10, so
// that one block fits a CU at the last two.
template <typename R, int L>
constexpr int l2pSlotTile() {
  return L * L * L * 32 * (int)sizeof(R) <= 65536 ? 32 : 16;
}
inline int l2pSlotTileAt(int L, int realBytes) {
  return L * L * L * 32 * realBytes <= 65536 ? 32 : 16;
}
// Elements from one point's row of S to the next: 4 beyond a multiple of the
// 256 bytes of the LDS banks, so that the 16 rows x 4 columns of an A operand
// fall into different banks.
template <typename R, int L>
constexpr int l2pSlotStride() {
  constexpr int w = 256 / (int)sizeof(R);
  return (L * L * L + 4 + w - 1) / w * w + 4;
}
// Work item: target leaf, first point and number of points of the tile, slot
// range, and where its sums go: out < 0 adds them to p (the only item of its
// points), else to partial[out * 32 ...].
struct L2PItem {
  int leaf, i0, nt, k0, k1, out;
};

// L2P.  A block of 4 waves per item; S is formed once, wave w takes the slots
// k0 + 16 w, + 64, ...: ceil(L^3 / 4) steps whose B operands (4 consecutive
// coefficients of 16 slots times their phase rows) are loaded kU steps at a
// time, then the 16 x 16 sums times the points' phases.  At the end the
// columns are added within the wave, the waves in order.
//
// Bound by reading the expansions (as much as P2M writes) and by the loads'
// latency.  Against lanes per point reading the slots' rows from LDS (k_l2p),
// a block per leaf whatever its number of slots: 20,000 points order 8 0.75 ->
// 0.31 ms (double), 0.44 -> 0.22 ms (float), 200,000-point sphere order 5 3.7
// -> 2.3 ms (double).  Adding the chains up (l2pSlotChain) costs 5% at orders
// 5 and 6 (41,334 points, double, 0.30 -> 0.32 ms) and nothing at 7 and 8.
template <typename R, int L>
__global__ __launch_bounds__(256) void k_l2p_slots(
    const L2PItem* __restrict__ items, DevCells T, DevLevels lv, const double* __restrict__ px,
    const double* __restrict__ py, const double* __restrict__ pz,
    const double* __restrict__ dirs, const typename C2T<R>::T* __restrict__ sig2,
    const typename C2T<R>::T* __restrict__ Lst, OpConsts<R> oc, double kappa,
    typename C2T<R>::T* __restrict__ p, typename C2T<R>::T* __restrict__ partial, int nItems) {
  typedef typename C2T<R>::T R2;
  typedef Mfma16<R> X;
  constexpr int LL = L * L * L, KS = (LL + 3) / 4, TP = l2pSlotTile<R, L>(), NB = TP / 16;
  constexpr int ST = l2pSlotStride<R, L>(), kU = sizeof(R) == 8 ? 4 : 8;
  constexpr int kB = l2pSlotChain(L);
  static_assert(kU % kB == 0, "chains end with a batch of loads");
  static_assert(ST >= 4 * KS, "rows of S hold the last step's padding");
  static_assert(TP * ((ST + 3 * L) * sizeof(R) + 3 * 8 + 4 * 2 * sizeof(R)) <= 160 * 1024, "LDS");
  __shared__ R Sm[TP][ST];
  __shared__ R Wt[3][TP][L];
  __shared__ double rel[3][TP];
  __shared__ R2 red[4][TP];
  const int item = (int)(blockIdx.y * gridDim.x + blockIdx.x);
  if (item >= nItems) return;
  const L2PItem it = items[item];
  const int c = it.leaf;
  const int lvl = T.lvl[c], pb = T.pbeg[c] + it.i0, s0 = T.slot0[c];
  const double ctr[3] = {T.ctr[3 * c], T.ctr[3 * c + 1], T.ctr[3 * c + 2]}, rad = T.rad[c];
  const int hf = lv.isHF[lvl], doff = lv.dirOff[lvl], srow = lv.sigRow0[lvl];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  stageWeights<R, L, TP>(Wt, rel, px, py, pz, pb, it.nt, ctr, rad, oc, tid, 256);
  __syncthreads();
  // a thread per (point, first two indices), L values each
  for (int x = tid; x < TP * L * L; x += 256) {
    const int i = x / (L * L), z = x - i * (L * L);
    const R w01 = Wt[0][i][z / L] * Wt[1][i][z % L];
#pragma unroll
    for (int e = 0; e < L; e++) Sm[i][z * L + e] = w01 * Wt[2][i][e];
  }
  if constexpr (4 * KS > LL)
    if (tid < TP)
#pragma unroll
      for (int I = LL; I < 4 * KS; I++) Sm[tid][I] = (R)0;
  __syncthreads();
  const int lr = lane & 15, quad = lane >> 4;
  R2 pacc[NB][4];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int v = 0; v < 4; v++) pacc[b][v] = c2<R>(0, 0);
  for (int kg = it.k0 + kSlotCols * wave; kg < it.k1; kg += 4 * kSlotCols) {
    const bool col = kg + lr < it.k1;
    const int sl = s0 + min(kg + lr, it.k1 - 1);
    const int d = hf ? T.slotDir[sl] : 0;
    const R2* sg = hf ? sig2 + (size_t)(srow + d) * LL : sig2;
    const R2* Ls = Lst + (size_t)sl * LL;
    typename X::V cre[NB], cim[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
      cre[b] = typename X::V{0, 0, 0, 0};
      cim[b] = typename X::V{0, 0, 0, 0};
    }
    // (not unrolled: the loads of the batches to come would fill the registers)
#pragma unroll 1
    for (int ks0 = 0; ks0 < KS; ks0 += kU) {
      R2 lv2[kU], sv[kU];
#pragma unroll
      for (int u = 0; u < kU; u++) {
        const int kk = min(4 * (ks0 + u) + quad, LL - 1);  // (S is zero beyond LL)
        lv2[u] = Ls[kk];
        if (hf) sv[u] = sg[kk];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u0 = 0; u0 < kU; u0 += kB) {
        if (ks0 + u0 >= KS) break;
        typename X::V tre[NB], tim[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) tre[b] = tim[b] = typename X::V{0, 0, 0, 0};
#pragma unroll
        for (int u = u0; u < u0 + kB; u++) {
          if (ks0 + u >= KS) break;
          const int kk = 4 * (ks0 + u) + quad;
          const R2 bv = hf ? cmul(lv2[u], sv[u]) : lv2[u];
#pragma unroll
          for (int b = 0; b < NB; b++) {
            const R a = Sm[16 * b + lr][kk];
            tre[b] = X::mac(a, bv.x, tre[b]);
            tim[b] = X::mac(a, bv.y, tim[b]);
          }
        }
#pragma unroll
        for (int b = 0; b < NB; b++) {
          cre[b] += tre[b];
          cim[b] += tim[b];
        }
      }
    }
    double dx = 0., dy = 0., dz = 0.;
    if (hf) {
      dx = dirs[3 * (doff + d)];
      dy = dirs[3 * (doff + d) + 1];
      dz = dirs[3 * (doff + d) + 2];
    }
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int i = 16 * b + X::row(quad, v);
        R2 cv = c2<R>(cre[b][v], cim[b][v]);
        if (hf) {
          R cs, sn;
          expi(kappa * (dx * rel[0][i] + dy * rel[1][i] + dz * rel[2][i]), cs, sn);
          cv = cmul(cv, c2<R>(cs, sn));
        }
        if (col) {
          pacc[b][v].x += cv.x;
          pacc[b][v].y += cv.y;
        }
      }
  }
  // the 16 columns of a row lie in the 16 lanes of its quad
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
#pragma unroll
      for (int m = 8; m >= 1; m /= 2) {
        pacc[b][v].x += __shfl_xor(pacc[b][v].x, m);
        pacc[b][v].y += __shfl_xor(pacc[b][v].y, m);
      }
      if (lr == 0) red[wave][16 * b + X::row(quad, v)] = pacc[b][v];
    }
  __syncthreads();
  if (tid < it.nt) {
    R2 t = red[0][tid];
#pragma unroll
    for (int w = 1; w < 4; w++) {
      t.x += red[w][tid].x;
      t.y += red[w][tid].y;
    }
    if (it.out >= 0) {
      partial[(size_t)it.out * 32 + tid] = t;
    } else {
      R2 o = p[pb + tid];
      o.x += t.x;
      o.y += t.y;
      p[pb + tid] = o;
    }
  }
}

// Tiles whose slots several items share: first point, number of points, and
// the items' sums partial[first * 32 ..], added in item order.
struct L2PTile {
  int point, nt, first, count;
};
template <typename R>
__global__ __launch_bounds__(256) void k_l2p_slots_reduce(
    const L2PTile* __restrict__ tiles, const typename C2T<R>::T* __restrict__ partial,
    typename C2T<R>::T* __restrict__ p, int nTiles) {
  typedef typename C2T<R>::T R2;
  const int tile = (int)(blockIdx.y * gridDim.x + blockIdx.x) * 8 + (threadIdx.x >> 5);
  if (tile >= nTiles) return;
  const L2PTile t = tiles[tile];
  const int i = threadIdx.x & 31;
  if (i >= t.nt) return;
  R2 o = p[t.point + i];
  for (int k = 0; k < t.count; k++) {
    const R2 v = partial[(size_t)(t.first + k) * 32 + i];
    o.x += v.x;
    o.y += v.y;
  }
  p[t.point + i] = o;
}

}  // namespace dfm
