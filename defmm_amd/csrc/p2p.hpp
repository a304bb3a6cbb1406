// Near field with a lane per source (1, 2, 3, 4 or 8 right-hand sides).
//
//   p_i += sum_j exp(i kappa r) / (4 pi r) q_j,  r = |x_i - y_j|,
// term 0 when r^2 < 1e-16 (reference include/operators/P2P.hpp:42-79).
//
// with the phase from a table (phase.hpp).
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "phase.hpp"

namespace dfm {

// 1 / r and r of a squared distance; K = 0 where R2 < 1e-16.
// double: the hardware estimate and one third-order step (the estimate's
// relative error e of about 1e-7 or less leaves 5/16 e^3).
__device__ __forceinline__ void invDist(double R2, double& r, double& K) {
  const double y = __builtin_amdgcn_rsq(R2);
  const double g = R2 * y;
  const double e = fma(-g, y, 1.0);
  K = fma(y * e, fma(0.375, e, 0.5), y);
  if (R2 < 1.e-16) K = 0.;
  r = K * R2;
}
// float 1 / r; r to ~1e-14 relative: one Newton step in double
__device__ __forceinline__ void invDist(double R2, double& r, float& K) {
  // (the instruction itself: where it is used R2 >= 1e-16 is no denormal)
  const float y = __builtin_amdgcn_rsqf((float)R2);
  K = (R2 < 1.e-16) ? 0.f : y;
  const double Kd = (double)K, r0 = R2 * Kd;
  r = fma(0.5, Kd * fma(-r0, r0, R2), r0);
}

// Kernel value without the factor 1 / (4 pi), which the caller applies to
// its sums.
template <int Phase, typename R>
__device__ __forceinline__ void p2pValue(double x, double y, double z, const PhaseConsts& pc,
                                         const typename C2T<R>::T* __restrict__ tab, R& co,
                                         R& si) {
  const double R2 = fma(z, z, fma(y, y, x * x));
  double r;
  R K;
  invDist(R2, r, K);
  if constexpr (Phase == kPhaseNone) {
    co = K;
    si = 0;
  } else if constexpr (Phase == kPhaseTable) {
    phaseTable(r, K, pc, tab, co, si);
  } else {
    expi(pc.kappa * r, co, si);
    co *= K;
    si *= K;
  }
}

// Work item of k_p2p_lane: nt <= kP2PTargets targets of one leaf, from t0
// (leaf-relative), against cnt sources of its list from (range r, offset
// off).
constexpr int kP2PTargets = 8;
struct P2PLaneItem {
  int leaf, t0, nt, r, off, cnt;
};

// Sum of v over the wave, N values (a power of two, at most 64) at once: each
// halving step sends half of the values to the other half of the lanes, so N
// values cost N - 1 + log2(64 / N) exchanges.  Afterwards the lane with
// lane % (64 / N) == 0 holds the sum of value waveSumIndex<N>(lane).
template <int N>
__device__ __forceinline__ double waveSum(double (&v)[N], int lane) {
  int m = 32;
#pragma unroll
  for (int h = N / 2; h >= 1; h /= 2, m /= 2) {
    const bool up = (lane & m) != 0;
#pragma unroll
    for (int k = 0; k < N / 2; k++) {
      if (k >= h) break;
      // (kept in registers: a select of two array elements would become an
      // element of a selected index)
      double a = v[k], b = v[k + h];
      asm("" : "+v"(a), "+v"(b));
      const double keep = up ? b : a, send = up ? a : b;
      v[k] = keep + __shfl_xor(send, m);
    }
  }
  double s = v[0];
#pragma unroll
  for (; m >= 1; m /= 2) s += __shfl_xor(s, m);
  return s;
}
template <int N>
__device__ __forceinline__ int waveSumIndex(int lane) {
  return lane / (64 / N);
}

// A wave per item (4 items per block, which share the phase table in LDS).
// Lane l takes the item's sources l, l + 64, ...: the source stays in
// registers for all of the item's targets, whose coordinates are wave-uniform
// (scalar registers), so LDS serves the phase table alone.  The next 64
// sources are loaded while the present ones are evaluated.  Float sums are
// added to double ones every kP2PFlush steps.  At the end the lanes' sums are
// added across the wave in a fixed order and written to
// partial[(item * NR + right-hand side) * kP2PTargets + target].
//
// Bound by the vector units: 44 double instructions and a reciprocal square
// root a pair, at 95% of the measured issue rate.  With a lane per target,
// sources in LDS and polynomials to y^16 over [-pi/4, pi/4] it was 76, and a
// leaf of n points left 64 - n floor(64 / n) lanes idle.  200,000-point
// sphere at 64 wavelengths (8.67e9 pairs): double 23.8 -> 13.2 ms, float
// 14.5 -> 8.6 ms; 4,000-point cube 80 -> 27 us; 150,000-point Laplace
// clusters (no phase) 0.85 -> 0.27 ms; 20,000-point cube, float: 2 right-hand
// sides 0.50 -> 0.31 ms, 3: 0.90 -> 0.34, 4: 0.53 -> 0.40, 8: 0.73 -> 0.74.
// TC targets per sweep of the sources keep the accumulators in registers.
constexpr int kP2PFlush = 16;
template <typename R, int NR>
constexpr int p2pSweep() {
  return NR <= 2 ? kP2PTargets : NR <= 4 ? kP2PTargets / 2 : kP2PTargets / 4;
}
template <typename R, int NR, int Phase>
__global__ __launch_bounds__(256) void k_p2p_lane(
    const P2PLaneItem* __restrict__ items, const int* __restrict__ leafCell,
    const int* __restrict__ tpbeg, const double* __restrict__ tx, const double* __restrict__ ty,
    const double* __restrict__ tz, const double* __restrict__ sx, const double* __restrict__ sy,
    const double* __restrict__ sz, const typename C2T<R>::T* __restrict__ q, size_t qStride,
    const int* __restrict__ rb, const int* __restrict__ re,
    const typename C2T<R>::T* __restrict__ phase, PhaseConsts pc, double2* __restrict__ partial,
    int nItems) {
  typedef typename C2T<R>::T R2;
  constexpr int TC = p2pSweep<R, NR>();
  constexpr bool kFloat = sizeof(R) == 4;
  __shared__ R2 tab[Phase == kPhaseTable ? kPhaseN : 1];
  if constexpr (Phase == kPhaseTable) {
    static_assert(kPhaseN == 256, "one table entry per thread");
    tab[threadIdx.x] = phase[threadIdx.x];
    __syncthreads();
  }
  // addends of the polynomials: an instruction takes one scalar operand
  asm("" : "+v"(pc.s3), "+v"(pc.c4));
  const int lane = threadIdx.x & 63;
  const int item = (int)(blockIdx.y * gridDim.x + blockIdx.x) * 4 +
                   __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (item >= nItems) return;
  const P2PLaneItem it = items[item];
  const int tb = tpbeg[leafCell[it.leaf]] + it.t0;
  for (int t0 = 0; t0 < it.nt; t0 += TC) {
    const int nt = min(TC, it.nt - t0);
    // the sweep's targets as a mask that the compiler cannot relate to one
    // another: with t < nt it nests the targets' bodies, keeps the first half
    // of each in registers until the last and needs 194 of them
    unsigned on = (1u << nt) - 1u;
    double xt[TC], yt[TC], zt[TC];
#pragma unroll
    for (int t = 0; t < TC; t++) {
      const int i = tb + t0 + min(t, nt - 1);
      xt[t] = tx[i];
      yt[t] = ty[i];
      zt[t] = tz[i];
    }
    R ar[TC][NR], ai[TC][NR];
    double dr[TC][NR], di[TC][NR];  // (float sums only)
#pragma unroll
    for (int t = 0; t < TC; t++)
#pragma unroll
      for (int k = 0; k < NR; k++) {
        ar[t][k] = ai[t][k] = 0;
        dr[t][k] = di[t][k] = 0.;
      }
    // this lane's source: offset o of range [b, b + len); a lane past the
    // item's end keeps its last source (or the item's first), without charge
    int rr = it.r, b = rb[rr], len = re[rr] - b, o = it.off, j = b + o;
    auto advance = [&](int pos, int by) {
      if (pos >= it.cnt) return;
      o += by;
      while (o >= len) {
        o -= len;
        rr++;
        b = rb[rr];
        len = re[rr] - b;
      }
      j = b + o;
    };
    double nx, ny, nz;
    R2 nq[NR];
    // (unconditional, so that the wait for it falls in the next step)
    auto load = [&]() {
      nx = sx[j];
      ny = sy[j];
      nz = sz[j];
#pragma unroll
      for (int k = 0; k < NR; k++) nq[k] = q[k * qStride + j];
    };
    advance(lane, lane);
    load();
    for (int pos = 0, step = 0; pos < it.cnt; pos += 64, step++) {
      const bool valid = pos + lane < it.cnt;
      const double xs = nx, ys = ny, zs = nz;
      R2 qs[NR];
#pragma unroll
      for (int k = 0; k < NR; k++) qs[k] = valid ? nq[k] : c2<R>(0, 0);
      advance(pos + 64 + lane, 64);
      load();
      asm volatile("" : "+s"(on));
#pragma unroll
      for (int t = 0; t < TC; t++) {
        if (!((on >> t) & 1u)) continue;
        R co, si;
        p2pValue<Phase, R>(xt[t] - xs, yt[t] - ys, zt[t] - zs, pc, tab, co, si);
#pragma unroll
        for (int k = 0; k < NR; k++) {
          ar[t][k] = fma(co, qs[k].x, ar[t][k]);
          ai[t][k] = fma(co, qs[k].y, ai[t][k]);
          if constexpr (Phase != kPhaseNone) {
            ar[t][k] = fma(-si, qs[k].y, ar[t][k]);
            ai[t][k] = fma(si, qs[k].x, ai[t][k]);
          }
        }
      }
      if constexpr (kFloat) {
        if (step % kP2PFlush == kP2PFlush - 1) {
#pragma unroll
          for (int t = 0; t < TC; t++)
#pragma unroll
            for (int k = 0; k < NR; k++) {
              dr[t][k] += (double)ar[t][k];
              di[t][k] += (double)ai[t][k];
              ar[t][k] = ai[t][k] = 0;
            }
        }
      }
    }
    constexpr double kInv4Pi = 0.079577471545947667884;
#pragma unroll
    for (int k = 0; k < NR; k++) {
      double v[2 * TC];
#pragma unroll
      for (int t = 0; t < TC; t++) {
        v[2 * t] = kFloat ? dr[t][k] + (double)ar[t][k] : (double)ar[t][k];
        v[2 * t + 1] = kFloat ? di[t][k] + (double)ai[t][k] : (double)ai[t][k];
      }
      const double s = waveSum<2 * TC>(v, lane) * kInv4Pi;
      const int id = waveSumIndex<2 * TC>(lane);
      if (lane % (32 / TC) == 0 && id < 2 * nt)
        ((double*)(partial + ((size_t)item * NR + k) * kP2PTargets + t0))[id] = s;
    }
  }
}

// Adds the partial sums of a leaf's items to p: the leaf's targets are cut
// into chunks of `chunk` (the last one smaller), its source list into runs;
// item (run, chunk) of the leaf is itemBeg[leaf] + run * chunks + chunk.
template <typename R, int NR>
__global__ __launch_bounds__(64) void k_p2p_lane_reduce(
    const int* __restrict__ itemBeg, const int* __restrict__ leafCell,
    const int* __restrict__ tpbeg, const int* __restrict__ tnprt,
    const double2* __restrict__ partial, typename C2T<R>::T* __restrict__ p, size_t pStride,
    int nLeaves) {
  typedef typename C2T<R>::T R2;
  const int leaf = (int)(blockIdx.y * gridDim.x + blockIdx.x);
  if (leaf >= nLeaves) return;
  const int c = leafCell[leaf];
  const int pb = tpbeg[c], n = tnprt[c];
  const int ib = itemBeg[leaf], ie = itemBeg[leaf + 1];
  const int chunks = (n + kP2PTargets - 1) / kP2PTargets, chunk = (n + chunks - 1) / chunks;
  for (int i = threadIdx.x; i < n; i += 64) {
    const int ch = i / chunk, t = i - ch * chunk;
    double sr[NR], si[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) sr[r] = si[r] = 0.;
    for (int k = ib + ch; k < ie; k += chunks)
#pragma unroll
      for (int r = 0; r < NR; r++) {
        const double2 v = partial[((size_t)k * NR + r) * kP2PTargets + t];
        sr[r] += v.x;
        si[r] += v.y;
      }
#pragma unroll
    for (int r = 0; r < NR; r++) {
      R2 o = p[r * pStride + pb + i];
      o.x = (R)((double)o.x + sr[r]);
      o.y = (R)((double)o.y + si[r]);
      p[r * pStride + pb + i] = o;
    }
  }
}

}  // namespace dfm
