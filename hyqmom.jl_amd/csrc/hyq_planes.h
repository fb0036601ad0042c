// One plane Jacobian of a cell on its own: from the 15 raw moments of its two axes to the
// decision (hyperbolic, complex pair, not finite) and the extreme eigenvalues.
//
// The plane of axes (P, Q) takes only the moments with no exponent on the third axis: the
// Taylor shift along that axis leaves them alone, so shifting the 15 of them along P and Q
// gives the same bits as shifting all 35 (raw_to_central4).  A lane that solves one plane
// therefore holds 15 moments instead of a cell's 35, and a kernel needs one copy of the
// plane solve, which all five planes of a cell share.
#pragma once
#include "hyq_pipeline.h"

namespace hyq {

// position of (i, j), i + j <= 4, in a 2D set of 15 moments
HD constexpr int p2(int i, int j) { return (i + j) * (i + j + 1) / 2 + j; }

// 35-moment index of each set's moments: set 0 the axes (x, y), 1 (x, z), 2 (y, z).
struct SetT {
  int m[3][15];
};
HD constexpr SetT plane_sets() {
  SetT t{};
  for (int s = 0; s < 3; ++s) {
    const int P = s == 2 ? 1 : 0, Q = s == 0 ? 1 : 2;
    for (int i = 0; i <= 4; ++i)
      for (int j = 0; i + j <= 4; ++j) {
        int e[3] = {0, 0, 0};
        e[P] = i;
        e[Q] = j;
        for (int n = 0; n < 35; ++n)
          if (e35().e[n][0] == e[0] && e35().e[n][1] == e[1] && e35().e[n][2] == e[2])
            t.m[s][p2(i, j)] = n;
      }
  }
  return t;
}
// Planes in slot order UV, UW, VU, VW, WU: the set each takes, and whether its flux axis is
// the set's second one.
HD constexpr int plane_set(int q) { return q == kUV || q == kVU ? 0 : (q == kVW ? 2 : 1); }
HD constexpr bool plane_swapped(int q) { return q == kVU || q == kWU; }

// taylor_shift on a 2D set (AX: 0 the first axis, 1 the second).
template <int AX>
HD void taylor_shift2(double* a, double s) {
  double sp[5];
  sp[0] = 1.0;
#pragma unroll
  for (int t = 1; t <= 4; ++t) sp[t] = sp[t - 1] * s;
#pragma unroll
  for (int n = 4; n >= 1; --n) {
#pragma unroll
    for (int j = 0; j <= 4 - n; ++j) {
      double acc = 0.0;
#pragma unroll
      for (int p = 0; p <= n; ++p)
        acc += binom(n, p) * sp[n - p] * a[AX == 0 ? p2(p, j) : p2(j, p)];
      a[AX == 0 ? p2(n, j) : p2(j, n)] = acc;
    }
  }
}

// The plane of a set's raw moments m[15] (m[0] the density), flux along the second axis if
// swapped.
HD Plane plane_of_set(const double* m, bool swapped) {
  double d[15];
  const double r = 1.0 / m[0];
#pragma unroll
  for (int t = 0; t < 15; ++t) d[t] = m[t] * r;
  const double a = d[p2(1, 0)], b = d[p2(0, 1)];
  taylor_shift2<0>(d, -a);
  taylor_shift2<1>(d, -b);
  d[p2(0, 0)] = 1.0;
  d[p2(1, 0)] = 0.0;
  d[p2(0, 1)] = 0.0;
  auto C = [&](int i, int j) { return swapped ? d[p2(j, i)] : d[p2(i, j)]; };
  return plane_of(C(2, 0), C(1, 1), C(0, 2), C(3, 0), C(2, 1), C(1, 2), C(0, 3), C(4, 0), C(3, 1),
                  C(2, 2), C(1, 3), C(0, 4), swapped ? b : a);
}

// What is known of a plane: its state (bits 0-1), the flags its solves set, as the decision
// and as the final values (the speeds after a correction), and the root-polishing
// iterations (bits 16-27).
constexpr uint32_t kPlOpen = 0u, kPlReal = 1u, kPlComplex = 2u, kPlNotFinite = 3u, kPlState = 3u;
constexpr uint32_t kPlFallback = 4u, kPlNoConv = 8u, kPlFallbackFinal = 16u, kPlNoConvFinal = 32u;
constexpr uint32_t kPlNotOkFinal = 64u;
constexpr int kPlIterShift = 16;

// The state of a plane from one solve.  EM 0: the QR.  EM 1 with PAIR = false: the fast
// solve without the 2x2 block test, which leaves some planes open (kPlOpen); with PAIR the
// full decision: block test, then the QR.  fin: the values are wanted even of a complex
// pair (the speeds after a correction), whose real parts the QR then gives.  The same
// solves, flags and values as plane_solve<EM, !fin>.
template <int EM, bool PAIR, bool VALS>
HD uint32_t plane_decide(const Plane& p, float wmin, float wmax, bool fin, double& v0, double& v1) {
  uint32_t info = 0u;
  bool cplx = false;
  v0 = v1 = NAN;
  if (EM == 1) {
    uint32_t fl = 0;
    double a, b;
    const int st = plane_fast_status<PAIR>(p, wmin, wmax, VALS, fl, a, b);
    info = (fl >> 16) << kPlIterShift;
    if (st == kPlaneProven) {
      v0 = a;
      v1 = b;
      return info | kPlReal;
    }
    cplx = st == kPlaneComplex;
    if (cplx && !fin) return info | kPlComplex;
    if (st == kPlaneFull) return info | kPlNotFinite | kPlFallback | kPlFallbackFinal;
    if (!PAIR) return info | kPlOpen;
    info |= cplx ? kPlFallbackFinal : (kPlFallback | kPlFallbackFinal);
  }
  uint32_t fl = 0;
  const EigRes r = plane_eigs(p, fl);
  v0 = r.vmin;
  v1 = r.vmax;
  if (fl & F_NOCONV) info |= cplx ? kPlNoConvFinal : (kPlNoConv | kPlNoConvFinal);
  if (cplx) return info | kPlComplex | (r.ok ? 0u : kPlNotOkFinal);
  return info | (!r.ok ? kPlNotFinite : (r.cplx ? kPlComplex : kPlReal));
}

// The result of a plane's solve as plane_solve returns it: of the decision (the values of a
// complex pair are not defined there) or of the final solve.
HD EigRes plane_result(uint32_t info, double v0, double v1, bool fin) {
  EigRes r;
  const uint32_t st = info & kPlState;
  r.cplx = st == kPlComplex;
  r.ok = st != kPlNotFinite && !(fin && (info & kPlNotOkFinal));
  r.vmin = v0;
  r.vmax = v1;
  return r;
}
HD uint32_t plane_flags(uint32_t fl, uint32_t info, bool fin) {
  if (info & (fin ? kPlFallbackFinal : kPlFallback)) fl |= F_FALLBACK;
  if (info & (fin ? kPlNoConvFinal : kPlNoConv)) fl |= F_NOCONV;
  const uint32_t it = (fl >> 16) + (info >> kPlIterShift);
  return (fl & 0xFFFFu) | ((it < 0xFFFu ? it : 0xFFFu) << 16);
}

}  // namespace hyq
