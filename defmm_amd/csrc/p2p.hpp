// Near field: with a lane per source (1, 2, 3, 4 or 8 right-hand sides), and
// on the matrix cores (16 or 8, float).
//
//   p_i += sum_j exp(i kappa r) / (4 pi r) q_j,  r = |x_i - y_j|,
// term 0 when r^2 < 1e-16 (reference include/operators/P2P.hpp:42-79).
//
// with the phase from a table (phase.hpp).
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "near_items.hpp"
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

// An entry of the phase table: cos and sin, in float with its angle's shift (z)
template <typename R>
struct PhaseT {
  typedef float4 T;
};
template <>
struct PhaseT<double> {
  typedef double2 T;
};

// Kernel value without the factor 1 / (4 pi), which the caller applies to
// its sums.
template <int Phase, typename R>
__device__ __forceinline__ void p2pValue(double x, double y, double z, const PhaseConsts& pc,
                                         const typename PhaseT<R>::T* __restrict__ tab, R& co,
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
// sides 0.50 -> 0.31 ms, 3: 0.90 -> 0.34, 4: 0.53 -> 0.40 (8, where the matrix
// cores are switched off: 0.73 -> 0.74).
// TC targets per sweep of the sources keep the accumulators in registers.
constexpr int kP2PFlush = 16;
template <typename R, int NR>
constexpr int p2pSweep() {
  return NR <= 2 ? kP2PTargets : NR <= 4 ? kP2PTargets / 2 : kP2PTargets / 4;
}
template <typename R, int NR, int Phase>
__global__ __launch_bounds__(256) void k_p2p_lane(
    const P2PItem* __restrict__ items, const int* __restrict__ leafCell,
    const int* __restrict__ tpbeg, const double* __restrict__ tx, const double* __restrict__ ty,
    const double* __restrict__ tz, const double* __restrict__ sx, const double* __restrict__ sy,
    const double* __restrict__ sz, const typename C2T<R>::T* __restrict__ q, size_t qStride,
    const int* __restrict__ rb, const int* __restrict__ re,
    const typename PhaseT<R>::T* __restrict__ phase, PhaseConsts pc, double2* __restrict__ partial,
    int nItems) {
  typedef typename C2T<R>::T R2;
  constexpr int TC = p2pSweep<R, NR>();
  constexpr bool kFloat = sizeof(R) == 4;
  __shared__ typename PhaseT<R>::T tab[Phase == kPhaseTable ? kPhaseN : 1];
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
  const P2PItem it = items[item];
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

// 16 or 8 right-hand sides of the float path on the matrix cores.  An item's
// sums are the product of the kernel matrix G (targets x sources, complex, one
// element per lane and step, phase reduced in double) and the charges Q
// (sources x right-hand sides):
//   P_re += G_re Q_re - G_im Q_im,   P_im += G_re Q_im + G_im Q_re,
// V_MFMA_F32_16X16X4_F32s of 4 sources and 16 targets.  Operands: A (16 x 4)
// lane l holds row l % 16, column l / 16; B (4 x 16) row l / 16, column
// l % 16; D (16 x 16) column l % 16, rows 4 (l / 16) + 0..3.  So lane l
// evaluates G for target l % 16 of a row block and source 4 k + l / 16 of
// step k.  16 right-hand sides take four of them a step (P_re and P_im apart,
// a column each); 8 take two, with the columns of Q_re | Q_im against G_re and
// of -Q_im | Q_re against G_im, so that P_re and P_im are the two halves of
// one result.  Lane l ends with column l % 16 of targets 4 (l / 16) + 0..3.
//
// A wave per item of at most kP2PMfmaTargets targets (two row blocks, which
// share the source operands), 4 items per block with the phase table in LDS.
// The wave stages 16 sources at a time in LDS of its own: lane l loads source
// l % 16 (coordinate l / 16, and right-hand sides l / 16 + 4 u), one step
// ahead; no barrier, so no wave waits for another.  Every 64 sources (8 of them
// with 8 right-hand sides) the sums are added to double ones.
//
// Bound by the SIMD's issue: 64 pairs take the matrix core 128 clocks (16
// right-hand sides; 64 for 8) and the vector unit about 200 (34 instructions,
// 16 of them double), and on this chip the two do not overlap, not even
// between waves (four waves of V_MFMA_F32_16X16X4_F32 and 8 independent v_fma
// each: 74 clocks, 35 and 36 alone).  A block of 4 waves per 64 targets, with
// three barriers per 64 sources and polynomials of kappa r over [-pi/4, pi/4],
// took 5.2 ms where this takes 4.0 (100,000-point ellipsoid at 64 wavelengths,
// Ncrit 97, 16 right-hand sides) and 1.07 for 0.74 (20,000-point cube).
// 8 right-hand sides: 200,000-point sphere at 40 wavelengths 11.9 ms, with a
// lane per source 19.9 (two targets a sweep are too few for each source's
// loads), with a lane per target and polynomials 16.3; 100,000 clustered
// points without phase 0.17, 0.52 and 0.43; 5,000-point cube 0.073, 0.086 and
// 0.111.  That was with sums of 64 sources (128 products in a chain) in float,
// which left errors 1.1 to 2 times those of a lane per source (whole passes,
// 20,000-point cube, order 8: 2.3e-7 and 1.45e-7); with 8 sources a sum it is
// 1.34e-7, for 12.5 ms at the sphere.
constexpr int kP2PMfmaNR = 16;
struct P2PMfmaArgs {
  const P2PItem* items;
  const int *leafCell, *tpbeg;
  const double *tx, *ty, *tz, *sx, *sy, *sz;
  const float2* q;
  size_t qStride;
  const int *rb, *re;
  const float4* phase;
  double2* partial;
  int nItems;
};
// One item of NR right-hand sides with MB row blocks; lc and lq are the wave's
// stage, tab the block's phase table.  lq[source][column]: the charge (16), or
// the operands (Q_re, -Q_im) and (Q_im, Q_re) of columns r and r + 8 (8).
template <int Phase, int NR, int MB>
__device__ __forceinline__ void p2pMfmaItem(const P2PMfmaArgs& A, const PhaseConsts& pc, int item,
                                            const P2PItem& it, const float4* tab,
                                            double (*lc)[16], float2 (*lq)[17]) {
  static_assert(NR == 16 || NR == 8, "columns of the result");
  typedef float v4f __attribute__((ext_vector_type(4)));
  constexpr int kStage = 16;
  const int lane = threadIdx.x & 63, lr = lane & 15, kq = lane >> 4;
  const int tb = A.tpbeg[A.leafCell[it.leaf]] + it.t0;
  // targets past the item's repeat its last; their sums are not written
  double xt[MB], yt[MB], zt[MB];
#pragma unroll
  for (int b = 0; b < MB; b++) {
    const int i = tb + min(16 * b + lr, it.nt - 1);
    xt[b] = A.tx[i];
    yt[b] = A.ty[i];
    zt[b] = A.tz[i];
  }
  v4f dre[MB], dim[MB];  // (dim, ai: of 16 right-hand sides)
  double ar[MB][4], ai[MB][4];
#pragma unroll
  for (int b = 0; b < MB; b++) {
    dre[b] = dim[b] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < 4; v++) ar[b][v] = ai[b][v] = 0.;
  }
  // this lane's source (l % 16 of the stage): offset o of range [b0, b0 +
  // len); past the item's end it keeps its last source (or the item's first),
  // without charge
  int rr = it.r, b0 = A.rb[rr], len = A.re[rr] - b0, o = it.off, j = b0 + o;
  auto advance = [&](int pos, int by) {
    if (pos >= it.cnt) return;
    o += by;
    while (o >= len) {
      o -= len;
      rr++;
      b0 = A.rb[rr];
      len = A.re[rr] - b0;
    }
    j = b0 + o;
  };
  const double* sc = kq == 0 ? A.sx : kq == 1 ? A.sy : A.sz;
  const float2* ql = A.q + (size_t)kq * A.qStride;
  double nc;
  float2 nq[NR / 4];
  auto load = [&]() {
    nc = sc[j];
#pragma unroll
    for (int u = 0; u < NR / 4; u++) nq[u] = ql[4 * u * A.qStride + j];
  };
  auto flush = [&]() {
#pragma unroll
    for (int b = 0; b < MB; b++) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        ar[b][v] += (double)dre[b][v];
        if constexpr (NR == 16) ai[b][v] += (double)dim[b][v];
      }
      dre[b] = dim[b] = v4f{0.f, 0.f, 0.f, 0.f};
    }
  };
  advance(lr, lr);
  load();
  for (int pos = 0; pos < it.cnt; pos += kStage) {
    const bool valid = pos + lr < it.cnt;
    // the wave's LDS accesses are ordered; the fences keep the compiler to it
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (kq < 3) lc[kq][lr] = nc;
#pragma unroll
    for (int u = 0; u < NR / 4; u++) {
      const float2 c = valid ? nq[u] : make_float2(0.f, 0.f);
      if constexpr (NR == 16) {
        lq[lr][kq + 4 * u] = c;
      } else {
        lq[lr][kq + 4 * u] = make_float2(c.x, -c.y);
        lq[lr][kq + 4 * u + 8] = make_float2(c.y, c.x);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    advance(pos + kStage + lr, kStage);
    load();
#pragma unroll
    for (int k = 0; k < kStage / 4; k++) {
      const int s = 4 * k + kq;
      const double xs = lc[0][s], ys = lc[1][s], zs = lc[2][s];
      const float2 ch = lq[s][lr];
      const float im = NR == 16 ? -ch.y : ch.y;
#pragma unroll
      for (int b = 0; b < MB; b++) {
        float co, si;
        p2pValue<Phase, float>(xt[b] - xs, yt[b] - ys, zt[b] - zs, pc, tab, co, si);
        dre[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(co, ch.x, dre[b], 0, 0, 0);
        if constexpr (NR == 16)
          dim[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(co, ch.y, dim[b], 0, 0, 0);
        if constexpr (Phase != kPhaseNone) {
          dre[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(si, im, dre[b], 0, 0, 0);
          if constexpr (NR == 16)
            dim[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(si, ch.x, dim[b], 0, 0, 0);
        }
      }
      if (NR == 8 && k % 2 == 1) flush();
    }
    if (NR == 16 && ((pos & 48) == 48 || pos + kStage >= it.cnt)) flush();
  }
  constexpr double kInv4Pi = 0.079577471545947667884;
#pragma unroll
  for (int b = 0; b < MB; b++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int t = 16 * b + 4 * kq + v;
      if (t >= it.nt) continue;
      double2* o = A.partial + ((size_t)item * NR + lr % NR) * kP2PMfmaTargets + t;
      if constexpr (NR == 16) *o = make_double2(ar[b][v] * kInv4Pi, ai[b][v] * kInv4Pi);
      else ((double*)o)[lr / NR] = ar[b][v] * kInv4Pi;
    }
}
// (at least 4 waves per SIMD: the sums then stay in registers that both kinds
// of instruction take)
template <int Phase, int NR>
__global__ __launch_bounds__(256, 4) void k_p2p_mfma(P2PMfmaArgs A, PhaseConsts pc) {
  __shared__ float4 tab[Phase == kPhaseTable ? kPhaseN : 1];
  __shared__ double lc[4][3][16];
  __shared__ float2 lq[4][16][17];
  if constexpr (Phase == kPhaseTable) {
    static_assert(kPhaseN == 256, "one table entry per thread");
    tab[threadIdx.x] = A.phase[threadIdx.x];
    __syncthreads();
  }
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int item = (int)(blockIdx.y * gridDim.x + blockIdx.x) * 4 + w;
  if (item >= A.nItems) return;
  const P2PItem it = A.items[item];
  if (it.nt > 16) p2pMfmaItem<Phase, NR, 2>(A, pc, item, it, tab, lc[w], lq[w]);
  else p2pMfmaItem<Phase, NR, 1>(A, pc, item, it, tab, lc[w], lq[w]);
}

// Adds the partial sums of a leaf's items to p: the leaf's targets are cut
// into chunks of p2pChunk(n, TG), its source list into runs; item (run,
// chunk) of the leaf is itemBeg[leaf] + run * chunks + chunk, and its sum of
// right-hand side r and target t is partial[(item * NR + r) * TG + t].
template <typename R, int NR, int TG>
__global__ void k_p2p_reduce(
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
  const int chunks = (n + TG - 1) / TG, chunk = p2pChunk(n, TG);
  for (int x = threadIdx.x; x < NR * n; x += blockDim.x) {
    const int r = NR == 1 ? 0 : x / n, i = x - r * n;
    const int ch = i / chunk, t = i - ch * chunk;
    double sr = 0., si = 0.;
    for (int k = ib + ch; k < ie; k += chunks) {
      const double2 v = partial[((size_t)k * NR + r) * TG + t];
      sr += v.x;
      si += v.y;
    }
    R2 o = p[r * pStride + pb + i];
    o.x = (R)((double)o.x + sr);
    o.y = (R)((double)o.y + si);
    p[r * pStride + pb + i] = o;
  }
}

}  // namespace dfm
