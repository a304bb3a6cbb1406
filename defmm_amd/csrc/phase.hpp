// cos and sin of kappa * r for the near field, r > 0 a distance, from a table
// of the kPhaseN angles 2 pi k / kPhaseN and short Taylor polynomials of the
// remainder (a table-driven reduction as in P. T. P. Tang, "Table-lookup
// algorithms for elementary functions and their error analysis", 1991).  The
// reduction is done on r itself:
//   n = rint(r kappa N / 2 pi),  y = r - n h,  h = 2 pi / (N kappa),
// so kappa never multiplies r; the polynomials' coefficients carry its powers.
#ifndef DEFMM_PHASE_HPP
#define DEFMM_PHASE_HPP

#include <cmath>
#include <cstring>

#include "sincos_red.hpp"

namespace dfm {

constexpr int kPhaseN = 256;

// Which evaluation of the phase a plan's near field takes (phaseOf): none
// (kappa = 0), the table, or expi() with kappa * r formed first (kappa * r
// beyond 2^20, or a kappa whose powers leave the range of double).
enum { kPhaseNone = 0, kPhaseTable = 1, kPhaseLibrary = 2 };

// Scalars of the table reduction for one wavenumber.
struct PhaseConsts {
  double kappa;
  double inv;        // N kappa / (2 pi)
  double h, hlo;     // 2 pi / (N kappa) = h + hlo
  double s3, s5;     // -kappa^3 / 6, kappa^5 / 120
  double c2, c4, c6; // -kappa^2 / 2, kappa^4 / 24, -kappa^6 / 720
  float kf;          // kappa
};

// The evaluation for a wavenumber, smallArg: kappa times the largest distance
// is at most 2^20 (so that n stays far inside the exact integers).
inline int phaseOf(double kappa, bool smallArg) {
  if (kappa == 0.) return kPhaseNone;
  return smallArg && kappa >= 1e-30 && kappa <= 1e30 ? kPhaseTable : kPhaseLibrary;
}

inline PhaseConsts phaseConstsOf(double kappa) {
  PhaseConsts pc{};
  pc.kappa = kappa;
  if (kappa == 0.) return pc;
  // 2 pi = p1 + p2; the residual of a division is exact under fma
  const double p1 = 6.283185307179586, p2 = 2.4492935982947064e-16;
  pc.h = p1 / kPhaseN / kappa;
  pc.hlo = (fma(-pc.h, kappa, p1 / kPhaseN) + p2 / kPhaseN) / kappa;
  pc.inv = kPhaseN * 0.15915494309189535 * kappa;
  const double k2 = kappa * kappa;
  pc.s3 = -k2 * kappa / 6.;
  pc.s5 = k2 * k2 * kappa / 120.;
  pc.c2 = -k2 / 2.;
  pc.c4 = k2 * k2 / 24.;
  pc.c6 = -k2 * k2 * k2 / 720.;
  pc.kf = (float)kappa;
  return pc;
}

// Entry k of the table, formed in long double.
inline void phaseEntry(int k, double& c, double& s) {
  const long double a = 2.0L * 3.141592653589793238462643383279502884L * k / kPhaseN;
  c = (double)cosl(a);
  s = (double)sinl(a);
}

// The float table's kPhaseN entries: x, y cos and sin of an angle
// 2 pi k / kPhaseN + d, and z = -d, where d is the first of the searched ones
// at which both lie within 2^-29 of a float (accurate tables, as in S. Gal,
// "Computing elementary functions: a new approach for achieving high accuracy
// and good performance", 1986).  An eighth of the circle is searched (0.1 ms),
// the rest mirrored.
constexpr double kPhaseShift = 3e-4;  // |d| at most
template <typename T>
inline void phaseEntriesF(T* tab) {
  constexpr int Q = kPhaseN / 4;
  constexpr double step = 3.1e-7, close = 1.0 / (1 << 29);
  for (int k = 0; k <= Q / 2; k++) {
    const double a = 6.283185307179586 / kPhaseN * k;
    for (int j = 0; j * step / 2 < kPhaseShift; j++) {
      const double d = (j & 1 ? -step : step) * ((j + 1) / 2), c = cos(a + d), s = sin(a + d);
      tab[k].x = (float)c;
      tab[k].y = (float)s;
      tab[k].z = (float)-d;
      if (std::fabs(tab[k].x - c) <= close && std::fabs(tab[k].y - s) <= close) break;
    }
  }
  for (int k = Q / 2 + 1; k < Q; k++) {  // cos(pi / 2 - a) = sin(a)
    const T e = tab[Q - k];
    tab[k].x = e.y;
    tab[k].y = e.x;
    tab[k].z = -e.z;
  }
  for (int k = Q; k < kPhaseN; k++) {  // cos(a + pi / 2) = -sin(a)
    const T e = tab[k - Q];
    tab[k].x = -e.y;
    tab[k].y = e.x;
    tab[k].z = e.z;
  }
}

// n mod kPhaseN of t = n + 1.5 * 2^52 (its low bits)
DFM_HD inline int phaseIndex(double t) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __double2loint(t) & (kPhaseN - 1);
#else
  unsigned long long u;
  std::memcpy(&u, &t, 8);
  return (int)(u & (kPhaseN - 1));
#endif
}

// cos and sin of kappa * r times the factor K.  |y| <= pi / 256: the sine's
// first omitted term kappa^7 y^7 / 7! is below 9e-18 and the cosine's
// kappa^8 y^8 / 8! below 2e-20; the table value and the final sum are each
// rounded once, so the error stays at the 1.4e-16 of sincosRed.
template <typename T2>
DFM_HD inline void phaseTable(double r, double K, const PhaseConsts& pc, const T2* tab, double& co,
                              double& si) {
  const double magic = 6755399441055744.0;  // 1.5 * 2^52: the sum's low bits are rint()
  const double t = fma(r, pc.inv, magic);
  const double n = t - magic;
  const int k = phaseIndex(t);
  double y = fma(-n, pc.h, r);
  y = fma(-n, pc.hlo, y);
  const double z = y * y;
  const double sy = fma(fma(pc.s5, z, pc.s3), z, pc.kappa) * y;
  const double cm = fma(fma(pc.c6, z, pc.c4), z, pc.c2) * z;  // cos - 1
  const T2 e = tab[k];
  co = (e.x + fma(e.x, cm, -e.y * sy)) * K;
  si = (e.y + fma(e.y, cm, e.x * sy)) * K;
}
// An entry's angle as its distance from 2 pi k / kPhaseN, negated; 0 where the
// table holds cos and sin alone.
template <typename T>
DFM_HD inline auto phaseShift(const T& e, int) -> decltype(e.z) {
  return e.z;
}
template <typename T>
DFM_HD inline float phaseShift(const T&, long) {
  return 0.f;
}
// Float values of a double r: the remainder is formed in double, then float,
// the angle y from the entry's.  With 1 - cos y = sin y tan(y / 2), tan(y / 2)
// as y / 2, the last sum alone rounds near 1 (|y| <= pi / 256 + 3e-4: the
// omitted y^5 / 120 and y^4 / 24 are below 3e-12 and 1e-9): rms error 2.1e-8
// at kappa = 201, where polynomials of the phase reduced by pi / 2 have 2.5e-8,
// and 3.6e-8 was that of entries rounded at 2 pi k / kPhaseN with two sums near
// 1, in as many instructions.  Of the float4 entries the kernels read all 16
// bytes: 12 take LDS longer (200,000-point sphere at 40 wavelengths 5.67 and
// 5.75 ms; a table of cos and sin and one of shifts 5.90; without shifts 5.52).
template <typename T>
DFM_HD inline void phaseTable(double r, float K, const PhaseConsts& pc, const T* tab, float& co,
                              float& si) {
  const double magic = 6755399441055744.0;
  const double t = fma(r, pc.inv, magic);
  const double n = t - magic;
  const int k = phaseIndex(t);
  const T e = tab[k];
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : : "v"(e.w));
#endif
  const float y = fmaf((float)fma(-n, pc.h, r), pc.kf, phaseShift(e, 0));
  const float h = 0.5f * y;
  const float sy = fmaf(y * y * -0.16666667f, y, y);
  co = fmaf(-sy, fmaf(e.x, h, e.y), e.x) * K;
  si = fmaf(sy, fmaf(-e.y, h, e.x), e.y) * K;
}

}  // namespace dfm

#endif
