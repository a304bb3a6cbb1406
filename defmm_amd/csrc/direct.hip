// FP64 direct sum on the GPU: the check of the reference's CheckFULL
// (include/interface.hpp:178-221) on sampled targets,
//   p_i = sum_j exp(i kappa r_ij) / (4 pi r_ij) q_j,  terms with r_ij^2 < 1e-16 skipped,
// and its variant for callers that cannot allocate device memory.
//
// Few targets against many sources (2,000 sampled targets, 10^6 sources) give
// a one-thread-per-target kernel only a handful of blocks, so the sources are
// split into parts: block (b, k) sums part k of the sources for up to 64
// targets (compensated), writing one partial per (part, target) to a scratch
// buffer; a second kernel adds the partials of each target in part order
// (compensated).  Targets are processed in tiles of kTileTargets, so the
// scratch never exceeds kPartsMax x kTileTargets partials whatever the input
// size; the part count depends only on the number of sources, so both entry
// points return bit-identical results.
#include <hip/hip_runtime.h>

#include <cmath>
#include <mutex>
#include <string>
#include <type_traits>

#include "../../include/defmm_amd.h"
#include "errors.hpp"
#include "p2p.hpp"

namespace dfm {

constexpr int kPartsMax = 64;          // source parts
constexpr int kTileTargets = 4096;     // targets per tile
constexpr int kSourcesPerPart = 256;   // parts = ceil(ns / 256), at most kPartsMax
constexpr int kMaxDevices = 64;

// Scratch of defmm_direct_noalloc: partial sums of one tile, 4 MiB, one
// copy per GPU (held until the process ends).  Host code must not pass the
// array's name to a kernel (it is a host-side stand-in): it uses the device
// address obtained from hipGetSymbolAddress.
static __device__ __align__(256) double2 scratch[kPartsMax * kTileTargets];

static int directParts(int64_t ns) {
  int64_t p = (ns + kSourcesPerPart - 1) / kSourcesPerPart;
  return (int)(p < 1 ? 1 : p > kPartsMax ? kPartsMax : p);
}

// s += v with the compensation c of Kahan's summation.
__device__ __forceinline__ void kahan(double& s, double& c, double v) {
  const double t = v - c, u = s + t;
  c = (u - s) - t;
  s = u;
}

// 2^shift targets per block (at most 64); the block's other threads split the
// staged sources: thread t takes target t mod 2^shift and every
// (256 >> shift)-th source, and the threads' sums are added in order.  The
// kernel value is the near field's (p2p.hpp), r with one more step to half a
// unit in the last place; phases beyond rMax (2^20 radians) take the library's
// sine and cosine.
//
// Bound by the vector units (about 60 double instructions a pair).  Against a
// thread per target over whole parts of 2,048 sources with the library's
// square root, division, sine and cosine: 300,000 sources and 2,000 targets
// 2.58 -> 1.35 ms, 20,000 and 1,000 0.76 -> 0.076 ms, 3,000 and 50 0.53 ->
// 0.028 ms on the device.
template <int Phase>
__global__ __launch_bounds__(256) void k_direct_part(const double* __restrict__ src, int ns,
                                                     const double2* __restrict__ q,
                                                     const double* __restrict__ trg, int nt,
                                                     PhaseConsts pc, double rMax, int chunk,
                                                     int shift, double2* __restrict__ partial) {
  __shared__ double sx[256], sy[256], sz[256];
  __shared__ double2 sq[256];
  __shared__ double2 tab[Phase == kPhaseTable ? kPhaseN : 1];
  const int tid = threadIdx.x;
  if constexpr (Phase == kPhaseTable) {
    static_assert(kPhaseN == 256, "one table entry per thread");
    double c, s;
    sincospi((double)tid * (2.0 / kPhaseN), &s, &c);
    tab[tid] = make_double2(c, s);
  }
  const int nT = 1 << shift, nG = 256 >> shift;
  const int tl = tid & (nT - 1), g = tid >> shift;
  const int i = blockIdx.x * nT + tl;
  const int part = blockIdx.y;
  const int ic = min(i, nt - 1);
  const double xt = trg[3 * (size_t)ic], yt = trg[3 * (size_t)ic + 1], zt = trg[3 * (size_t)ic + 2];
  const int jb = part * chunk;
  const int je = min(ns, jb + chunk);
  double pr = 0., pi = 0., cr = 0., ci = 0.;
  for (int j0 = jb; j0 < je; j0 += 256) {
    const int n = min(256, je - j0);
    __syncthreads();
    if (tid < n) {
      const size_t j = (size_t)j0 + tid;
      sx[tid] = src[3 * j];
      sy[tid] = src[3 * j + 1];
      sz[tid] = src[3 * j + 2];
      sq[tid] = q[j];
    }
    __syncthreads();
    for (int j = g; j < n; j += nG) {
      const double x = xt - sx[j], y = yt - sy[j], z = zt - sz[j];
      const double R2 = x * x + y * y + z * z;
      double r, K, co, si;
      invDist(R2, r, K);
      r = fma(0.5 * K, fma(-r, r, R2), r);
      if constexpr (Phase == kPhaseNone) {
        co = K;
        si = 0.;
      } else {
        if (Phase == kPhaseTable && r <= rMax) {
          phaseTable(r, K, pc, tab, co, si);
        } else {
          sincos(pc.kappa * r, &si, &co);
          co *= K;
          si *= K;
        }
      }
      const double2 qs = sq[j];
      // (a skipped pair has K = 0 and adds nothing, also where its phase is
      // not a number)
      if (K != 0.) {
        kahan(pr, cr, co * qs.x - si * qs.y);
        kahan(pi, ci, co * qs.y + si * qs.x);
      }
    }
  }
  // the groups' sums and what their compensation still holds, in group order
  __syncthreads();
  sq[tid] = make_double2(pr, pi);
  sx[tid] = cr;
  sy[tid] = ci;
  __syncthreads();
  if (g == 0 && i < nt) {
    for (int k = 1; k < nG; k++) {
      const int o = (k << shift) + tl;
      kahan(pr, cr, sq[o].x);
      kahan(pr, cr, -sx[o]);
      kahan(pi, ci, sq[o].y);
      kahan(pi, ci, -sy[o]);
    }
    constexpr double kInv4Pi = 0.079577471545947667884;
    partial[(size_t)part * nt + i] = make_double2((pr - cr) * kInv4Pi, (pi - ci) * kInv4Pi);
  }
}

__global__ __launch_bounds__(256) void k_direct_reduce(const double2* __restrict__ partial,
                                                       int parts, int nt,
                                                       double2* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= nt) return;
  double pr = 0., pi = 0., cr = 0., ci = 0.;
  for (int k = 0; k < parts; k++) {
    const double2 v = partial[(size_t)k * nt + i];
    kahan(pr, cr, v.x);
    kahan(pi, ci, v.y);
  }
  out[i] = make_double2(pr, pi);
}

// Direct sum of device arrays on stream s with a partial-sum buffer of at
// least directParts(ns) * min(nt, kTileTargets) elements.
static int directRun(const double* src, int64_t ns, const double2* q, const double* trg,
                     int64_t nt, double kappa, double2* p, double2* partial, hipStream_t s) {
  const int parts = directParts(ns);
  const int chunk = (int)((ns + parts - 1) / parts);
  const double ka = std::fabs(kappa);
  const int phase = phaseOf(ka, true);
  const PhaseConsts pc = phaseConstsOf(kappa);
  const double rMax = phase == kPhaseTable ? 1048576.0 / ka : 0.;
  for (int64_t t0 = 0; t0 < nt; t0 += kTileTargets) {
    const int n = (int)(nt - t0 < kTileTargets ? nt - t0 : kTileTargets);
    int shift = 6;
    while (shift > 0 && (1 << (shift - 1)) >= n) shift--;
    const unsigned nb = (unsigned)((n + (1 << shift) - 1) >> shift);
    auto go = [&](auto ph) {
      hipLaunchKernelGGL(k_direct_part<decltype(ph)::value>, dim3(nb, (unsigned)parts), dim3(256),
                         0, s, src, (int)ns, q, trg + 3 * t0, n, pc, rMax, chunk, shift, partial);
    };
    if (phase == kPhaseNone) go(std::integral_constant<int, kPhaseNone>());
    else if (phase == kPhaseTable) go(std::integral_constant<int, kPhaseTable>());
    else go(std::integral_constant<int, kPhaseLibrary>());
    hipLaunchKernelGGL(k_direct_reduce, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (const double2*)partial,
                       parts, n, p + t0);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    g_err = std::string("direct sum launch: ") + hipGetErrorString(e);
    return DEFMM_EHIP;
  }
  return DEFMM_OK;
}

// Device address of this GPU's scratch array, looked up once per device.
static int scratchOf(int dev, double2** out) {
  static std::mutex mu;
  static void* addr[kMaxDevices] = {};
  if (dev < 0 || dev >= kMaxDevices) {
    g_err = "device index beyond the scratch table";
    return DEFMM_EARG;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      g_err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
      return DEFMM_EHIP;
    }
    addr[dev] = ptr;
  }
  *out = (double2*)addr[dev];
  return DEFMM_OK;
}

}  // namespace dfm

extern "C" {

int defmm_direct(const double* src_xyz, int64_t n_src, const double* q, const double* trg_xyz,
                 int64_t n_trg, double kappa, double* p) {
  using namespace dfm;
  if (!src_xyz || !q || !trg_xyz || !p || n_src < 1 || n_trg < 1 || n_src > 2147483647 ||
      n_trg > 2147483647) {
    g_err = "invalid argument";
    return DEFMM_EARG;
  }
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) { g_err = "no HIP device"; return DEFMM_ENODEVICE; }
  int rc = DEFMM_OK;
  auto ck = [&](hipError_t e, const char* what) {
    if (e != hipSuccess) (void)hipGetLastError();  // consumed here, not at the next check
    if (e != hipSuccess && rc == DEFMM_OK) {
      g_err = std::string(what) + ": " + hipGetErrorString(e);
      rc = e == hipErrorOutOfMemory ? DEFMM_EMEMORY : DEFMM_EHIP;
    }
  };
  const int64_t tile = n_trg < kTileTargets ? n_trg : kTileTargets;
  // one allocation: charges, potentials, partial sums (16 bytes each), then
  // the points
  const size_t nq = (size_t)n_src, np = (size_t)n_trg, nw = (size_t)directParts(n_src) * tile;
  void* mem = nullptr;
  ck(hipMalloc(&mem, (nq + np + nw) * 16 + (nq + np) * 24), "hipMalloc");
  double2* dq = (double2*)mem;
  double2 *dp = dq + nq, *dw = dp + np;
  double* ds = (double*)(dw + nw);
  double* dt = ds + 3 * nq;
  if (!rc) ck(hipMemcpy(ds, src_xyz, nq * 24, hipMemcpyHostToDevice), "hipMemcpy");
  if (!rc) ck(hipMemcpy(dq, q, nq * 16, hipMemcpyHostToDevice), "hipMemcpy");
  if (!rc) ck(hipMemcpy(dt, trg_xyz, np * 24, hipMemcpyHostToDevice), "hipMemcpy");
  if (!rc) rc = directRun(ds, n_src, dq, dt, n_trg, kappa, dp, dw, 0);
  if (!rc) ck(hipMemcpy(p, dp, np * 16, hipMemcpyDeviceToHost), "hipMemcpy");
  if (mem) (void)hipFree(mem);
  return rc;
}

int defmm_direct_noalloc(const void* src_dev, int64_t n_src, const void* q_dev,
                         const void* trg_dev, int64_t n_trg, double kappa, void* p_dev,
                         void* stream) {
  using namespace dfm;
  if (!src_dev || !q_dev || !trg_dev || !p_dev) {
    g_err = "null argument";
    return DEFMM_EARG;
  }
  if (n_src < 1 || n_trg < 1 || n_src > 2147483647 || n_trg > 2147483647) {
    g_err = "n_src and n_trg must be in 1 .. 2^31-1";
    return DEFMM_EARG;
  }
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    g_err = "hipGetDevice failed";
    return DEFMM_EHIP;
  }
  double2* ws = nullptr;
  int rc = scratchOf(dev, &ws);
  if (rc) return rc;
  return directRun((const double*)src_dev, n_src, (const double2*)q_dev, (const double*)trg_dev,
                   n_trg, kappa, (double2*)p_dev, ws, (hipStream_t)stream);
}

}  // extern "C"
