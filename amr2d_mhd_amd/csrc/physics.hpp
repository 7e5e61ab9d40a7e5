// Pointwise FP64 MHD physics for the stage kernels (device and host).
//
// Every expression keeps the operand order and association of the reference
// implementation (spaceauk/AMR2D_MHD) because the results must be bitwise
// equal to it; the file is compiled with -ffp-contract=off, so no FMA is
// formed.  References are file:line in the reference tree.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

#include "amr_types.hpp"

namespace amr {

// always inlined: a call would move a face's state through scratch memory
#define AMR_INLINE inline __attribute__((always_inline))

constexpr double kEps = 1.0E-15;  // defs.hpp:16

// defs.hpp:110-111 (MIN/MAX macros) and std::min/std::max: they differ on
// signed-zero ties and NaN, and the reference uses each at specific sites.
__host__ __device__ inline double mac_min(double a, double b) { return a < b ? a : b; }
__host__ __device__ inline double mac_max(double a, double b) { return a > b ? a : b; }
__host__ __device__ inline double std_min(double a, double b) { return (b < a) ? b : a; }
__host__ __device__ inline double std_max(double a, double b) { return (a < b) ? b : a; }

// ------------------------------------------------- division, square root
// The stage is bound by the issue and latency of FP64 instructions, and the
// division sequence the compiler emits (two v_div_scale, v_rcp, four Newton
// FMAs, the quotient and its correction, v_div_fmas, v_div_fixup: ~14 issue
// slots) is much of it: 46 divisions and 11 square roots a face.  With FAST
// (device code only) a denominator's reciprocal is refined once and serves
// all of its quotients (4 slots each), and the steps that only rescale
// extreme exponents are left out: they also serialise every division through
// VCC.  The quotient is q = n y corrected by the exact remainder (Markstein,
// IBM J. Res. Dev. 34, 1990) with the same Newton steps as the full sequence,
// so it is the correctly rounded n / d, bit for bit, whenever no intermediate
// leaves the normal range: |d| in [2^-1000, 2^1000], |n| >= 2^-968 and a
// quotient in [2^-1000, 2^1000]; v_div_fixup gives zeros, infinities and NaN
// in n or d their IEEE results.  The callers establish that range from the
// exponents of their inputs (ExpSpan) and otherwise run the FAST = false code.
// The root is the Goldschmidt iteration without the rescaling of arguments
// below 2^-767.  Stage kernel, HLLD + MC, before and with all of stage.hpp's
// changes: 136 blocks 20.5 -> 15.5 us a launch, 340 blocks 32.9 -> 25.7, 757
// blocks 47.3 -> 34.3; WENO5 at 928 blocks 83.6 -> 62.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(AMR_COUNT_OPS)
#define AMR_DEVICE_FP 1
#endif

template <bool FAST>
struct Den {
  double d, y;
};

template <bool FAST>
__host__ __device__ AMR_INLINE Den<FAST> den(double d) {
  Den<FAST> r;
  r.d = d;
  r.y = d;
#ifdef AMR_DEVICE_FP
  if constexpr (FAST) {
    double y = __builtin_amdgcn_rcp(d);
    double e = __builtin_fma(-d, y, 1.);
    y = __builtin_fma(y, e, y);
    e = __builtin_fma(-d, y, 1.);
    r.y = __builtin_fma(y, e, y);
  }
#endif
  return r;
}

// a literal denominator: its correctly rounded reciprocal is formed by the compiler
template <bool FAST>
__host__ __device__ AMR_INLINE Den<FAST> den_literal(double d) {
  Den<FAST> r;
  r.d = d;
  r.y = d;
#ifdef AMR_DEVICE_FP
  if constexpr (FAST) r.y = 1. / d;
#endif
  return r;
}

template <bool FAST>
__host__ __device__ AMR_INLINE double quot(double n, const Den<FAST>& r) {
#ifdef AMR_DEVICE_FP
  if constexpr (FAST) {
    double q = n * r.y;
    const double e = __builtin_fma(-r.d, q, n);
    q = __builtin_fma(e, r.y, q);
    return __builtin_amdgcn_div_fixup(q, r.d, n);
  }
#endif
  return n / r.d;
}

template <bool FAST>
__host__ __device__ AMR_INLINE double root(double x) {
#ifdef AMR_DEVICE_FP
  if constexpr (FAST) {
    const double y = __builtin_amdgcn_rsq(x);
    double s = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, s, 0.5);
    h = __builtin_fma(h, r, h);
    s = __builtin_fma(s, r, s);
    double d = __builtin_fma(-s, s, x);
    s = __builtin_fma(d, h, s);
    d = __builtin_fma(-s, s, x);
    s = __builtin_fma(d, h, s);
    return (x == 0 || x == __builtin_inf()) ? x : s;
  }
#endif
  return sqrt(x);
}

// Range of binary exponents (x = m 2^e, 1/2 <= m < 1) of the values added;
// zeros, infinities and NaN count as exponent 0 (they need no range).
struct ExpSpan {
  int lo = 0, hi = 0;
  __host__ __device__ inline void add(double x) {
#ifdef AMR_DEVICE_FP
    const int e = __builtin_amdgcn_frexp_exp(x);
    lo = e < lo ? e : lo;
    hi = e > hi ? e : hi;
#else
    (void)x;
#endif
  }
  __host__ __device__ inline bool within(int a, int b) const { return lo >= a && hi <= b; }
};
// The ranges.  Far from a disturbance velocities and transverse fields decay
// through 2^-500 (half of a rotor's blocks hold such values), so there is no
// useful lower bound on them; what bounds the quotients is this:
//  - slope ratios divide by difference + 1e-15, which is 0 or above 2^-103, so
//    a tile whose nonzero primitives lie within 2^[-800, 100] has numerators
//    above 2^-853 and ratios within 2^[-955, 204]; WENO's denominators are
//    above 1e-30;
//  - of a face, density and pressure lie within 2^[-60, 60] and velocities and
//    fields below 2^60 (fast_flux).  Quotients whose numerator can underflow
//    are then added to terms above 2^-300, where any value below 2^-400 is
//    absorbed whole (the Alfven parts of the wave speeds, the magnetic energy,
//    the Roe field), or their numerators are checked as they are met (`num`):
//    0 or within 2^[-800, 500].
constexpr int kFaceExp = 60;
constexpr int kPrimLo = -800, kPrimHi = 100;
constexpr int kNumLo = -800, kNumHi = 500;

// conserved -> primitive of one cell (meshblock.cpp:119-179); the caller
// applies the reference's interior p <= 0 check to w[4].  FAST: u[0] within
// 2^[-100, 100], u[1..3] within 2^[-860, 400].
template <bool FAST = false>
__host__ __device__ AMR_INLINE void cons_to_prim(const double* u, double g, double* w) {
  const Den<FAST> r = den<FAST>(u[0]);
  w[0] = u[0];
  w[1] = quot(u[1], r);
  w[2] = quot(u[2], r);
  w[3] = quot(u[3], r);
  double p = (g - 1) * (u[4] - 0.5 * w[0] * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3]));
  w[5] = u[5];
  w[6] = u[6];
  w[7] = u[7];
  w[4] = p - (g - 1) * (0.5 * (u[5] * u[5] + u[6] * u[6] + u[7] * u[7]));
}

// slopelimiter.cpp:6-54
template <bool FAST = false>
__host__ __device__ AMR_INLINE double limiter(int id, double r, double eta) {
  switch (id) {
    case kLim1st: return 0.;
    case kLimNoSL: return r;
    case kLimMinmod: return mac_max(0., mac_min(1., r));
    case kLimVanLeer: return quot(fabs(r) + r, den<FAST>(1. + fabs(r)));
    case kLimSuperbee: {
      double lo = mac_min(2. * r, 1.);
      double hi = mac_min(r, 2.);
      return mac_max(0., mac_max(hi, lo));
    }
    case kLimMC: {
      double c = mac_min(2. * r, 0.5 * (1. + r));
      return mac_max(0., mac_min(c, 2.));
    }
    case kLimKoren: {
      double b = mac_min(quot(1. + 2. * r, den_literal<FAST>(3.)), 2.);
      return mac_max(0., mac_min(2. * r, b));
    }
    case kLimCada: {
      double third = quot(2. + r, den_literal<FAST>(3.));
      double h = mac_max(-0.5 * r, mac_min(mac_min(2. * r, third), 1.6));
      h = mac_max(0., mac_min(third, h));
      if (eta <= 1. - kEps) return third;
      if (eta >= 1. + kEps) return h;
      return 0.5 * ((1. - (eta - 1.) / kEps) * (2. + r) / 3. + (1 + (eta - 1.) / kEps) * h);
    }
    default: return NAN;
  }
}

// misc.cpp:71-79, returns the fast magnetosonic speed along component `norm`
template <bool FAST = false>
__host__ __device__ AMR_INLINE double fast_speed(const double* w, double g, int norm) {
  const Den<FAST> r = den<FAST>(w[0]);
  double ca = root<FAST>(quot(w[5] * w[5] + w[6] * w[6] + w[7] * w[7], r));
  double a = root<FAST>(quot(g * w[4], r));
  double can = root<FAST>(quot(w[norm] * w[norm], r));
  double s0 = (ca * ca) + (a * a);
  double s1 = (ca * ca) - (a * a);
  return root<FAST>(0.5 * (s0 + root<FAST>(s1 * s1 + 4. * (a * a) * ((ca * ca) - (can * can)))));
}

__host__ __device__ inline double sign0(double v) { return v > 0 ? 1. : (v < 0 ? -1. : 0.); }

// conserved state and x-flux of one side (riemannS.cpp:60-108)
struct Side {
  double q[8], F[8], e, H, pt, cf;
};

template <bool FAST = false>
__host__ __device__ AMR_INLINE void side_state(const double* w, double g, Side& s) {
  const Den<FAST> r0 = den<FAST>(w[0]);
  s.cf = fast_speed<FAST>(w, g, 5);
  const double vn = w[1], Bn = w[5];
  const double b2 = w[5] * w[5] + w[6] * w[6] + w[7] * w[7];
  double e = quot(w[4], den<FAST>(w[0] * (g - 1))) + 0.5 * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3]) + quot(0.5 * b2, r0);
  e = e * w[0];
  s.e = e;
  s.H = quot(e + w[4] + 0.5 * b2, r0);
#pragma unroll
  for (int k = 0; k < 8; k++) s.q[k] = w[k];
  s.q[1] = w[0] * w[1];
  s.q[2] = w[0] * w[2];
  s.q[3] = w[0] * w[3];
  s.q[4] = e;
  s.pt = w[4] + 0.5 * b2;
  const double mv = w[0] * vn;
  s.F[0] = mv;
  s.F[1] = mv * w[1] + s.pt - Bn * w[5];
  s.F[2] = mv * w[2] - Bn * w[6];
  s.F[3] = mv * w[3] - Bn * w[7];
  s.F[4] = mv * s.H - Bn * (w[1] * w[5] + w[2] * w[6] + w[3] * w[7]);
  s.F[5] = vn * w[5] - Bn * w[1];
  s.F[6] = vn * w[6] - Bn * w[2];
  s.F[7] = vn * w[7] - Bn * w[3];
}

// Roe-average outer eigenvalues, misc.cpp:95-140 (including the reference's
// sqrt(rhoL + sqrt(rhoR)) normaliser).  Outputs u_roe, lambda_min, lambda_max.
// `num` collects the exponent of u's numerator.
template <bool FAST>
__host__ __device__ AMR_INLINE void roe_bounds(const double* wL, const double* wR, double g, double HL, double HR,
                                               double& u, double& lmin, double& lmax, ExpSpan& num) {
  const double sl = root<FAST>(wL[0]), sr = root<FAST>(wR[0]);
  const Den<FAST> nrm = den<FAST>(root<FAST>(wL[0] + root<FAST>(wR[0])));
  double v[3], B[3];
  if constexpr (FAST) num.add(sl * wL[1] + sr * wR[1]);
#pragma unroll
  for (int i = 0; i < 3; i++) {
    v[i] = quot(sl * wL[i + 1] + sr * wR[i + 1], nrm);
    B[i] = quot(sl * wL[i + 5] + sr * wR[i + 5], nrm);
  }
  const double RT = root<FAST>(quot(wR[0], den<FAST>(wL[0])));
  const Den<FAST> d = den<FAST>(root<FAST>(wR[0] * wL[0]));
  const double d6 = wL[6] - wR[6], d7 = wL[7] - wR[7];
  const double X = quot(0.5 * ((d6 * d6) + (d7 * d7)), den<FAST>(sl + sr));
  const double Y = quot(0.5 * (wL[0] + wR[0]), d);
  const double h = quot(HL + RT * HR, den<FAST>(1 + RT));
  const double vsq = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
  const double btsq = (B[1] * B[1]) + (B[2] * B[2]);
  const double bt2s = (g - 1. - (g - 2) * Y) * btsq;
  const double vax2 = quot(B[0] * B[0], d);
  const double hp = h - (vax2 + quot(btsq, d));
  double a2 = ((g - 1.) * (hp - 0.5 * vsq) - (g - 2.) * X);
  a2 = mac_max(a2, kEps);
  const double ct2 = quot(bt2s, d);
  const double tsum = vax2 + ct2 + a2;
  const double tdif = vax2 + ct2 - a2;
  const double cfast = root<FAST>(0.5 * (tsum + root<FAST>(tdif * tdif + 4. * a2 * ct2)));
  u = v[0];
  lmin = v[0] - cfast;
  lmax = v[0] + cfast;
}

__host__ __device__ AMR_INLINE void roe_bounds(const double* wL, const double* wR, double g, double HL, double HR,
                                               double& u, double& lmin, double& lmax) {
  ExpSpan unused;
  roe_bounds<false>(wL, wR, g, HL, HR, u, lmin, lmax, unused);
}

// riemannS.cpp:58-116
template <bool FAST = false>
__host__ __device__ AMR_INLINE void flux_rusanov(const double* wL, const double* wR, double g, double* f) {
  Side L, R;
  side_state<FAST>(wL, g, L);
  side_state<FAST>(wR, g, R);
  const double s = std_max(L.cf + fabs(wL[1]), R.cf + fabs(wR[1]));
#pragma unroll
  for (int k = 0; k < 8; k++) f[k] = 0.5 * (L.F[k] + R.F[k]) - 0.5 * s * (R.q[k] - L.q[k]);
}

// riemannS.cpp:118-189
template <bool FAST = false>
__host__ __device__ AMR_INLINE bool flux_hlle(const double* wL, const double* wR, double g, double* f) {
  Side L, R;
  side_state<FAST>(wL, g, L);
  side_state<FAST>(wR, g, R);
  double u, lmin, lmax;
  ExpSpan unused, num, dif;
  roe_bounds<FAST>(wL, wR, g, L.H, R.H, u, lmin, lmax, unused);
  const double SL = mac_min(std_min(wL[1] - L.cf, lmin), 0.);
  const double SR = mac_max(std_max(wR[1] + R.cf, lmax), 0.);
  const Den<FAST> ds = den<FAST>(SR - SL);
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const double n = SR * L.F[k] - SL * R.F[k] + SL * SR * (R.q[k] - L.q[k]);
    if constexpr (FAST) num.add(n);
    f[k] = quot(n, ds);
  }
  if constexpr (FAST) dif.add(ds.d);
  return num.within(kNumLo, kNumHi) && dif.within(-150, 150);
}

// riemannS.cpp:192-295 (Linde 1998 alpha heuristic); returns nonzero where the
// reference throws (alpha NaN or SR == SL).  *ok: as flux_hlld.
template <bool FAST = false>
__host__ __device__ AMR_INLINE int flux_hllc(const double* wL, const double* wR, double g, double* f, bool& ok) {
  Side L, R;
  side_state<FAST>(wL, g, L);
  side_state<FAST>(wR, g, R);
  double u, lmin, lmax;
  ExpSpan num, dif;
  roe_bounds<FAST>(wL, wR, g, L.H, R.H, u, lmin, lmax, num);
  const double SL = std_min(wL[1] - L.cf, lmin);
  const double SR = std_max(wR[1] + R.cf, lmax);
  double jump = 0., resid = 0.;
#pragma unroll
  for (int k = 0; k < 8; k++) jump += fabs(R.q[k] - L.q[k]);
#pragma unroll
  for (int k = 0; k < 8; k++) resid += fabs((R.F[k] - L.F[k]) - u * (R.q[k] - L.q[k]));
  const double alpha = mac_max(0., 1. - quot(resid, den<FAST>(jump + kEps)));
  if (alpha > 1 || alpha < 0 || isnan(alpha)) return 1;
  if (SR - SL == 0) return 1;
  const Den<FAST> ds = den<FAST>(SR - SL);
  const double nL = SL * ((1 - alpha) * SR + alpha * u), nR = SR * ((1 - alpha) * SL + alpha * u);
  const double cL = quot(nL, ds), cR = quot(nR, ds);
  if constexpr (FAST) {
    num.add(nL);
    num.add(nR);
    dif.add(ds.d);
    ok = num.within(kNumLo, kNumHi) && dif.within(-150, 150);
  }
  const double aR = quot(SL, ds), aL = quot(SR, ds);
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const double dq = R.q[k] - L.q[k];
    if (SL > 0.) f[k] = L.F[k];
    else if (SL <= 0. && u >= 0.) f[k] = cL * dq - aR * R.F[k] + aL * L.F[k];
    else if (u <= 0. && SR >= 0.) f[k] = cR * dq - aR * R.F[k] + aL * L.F[k];
    else if (SR < 0.) f[k] = R.F[k];
  }
  return 0;
}

__host__ __device__ AMR_INLINE double vdotb(const double* w) {
  double s = 0.;
  s += w[1] * w[5];
  s += w[2] * w[6];
  s += w[3] * w[7];
  return s;
}

// star state of one side, riemannS.cpp:467-497; ws[4] stays 0
__host__ __device__ AMR_INLINE void hlld_star(const double* w, double S, double SM, double pts, double e, double pt,
                                          double* ws, double& es) {
  ws[0] = w[0] * (S - w[1]) / (S - SM);
  ws[1] = SM;
  ws[4] = 0.;
  ws[5] = w[5];
  const double den = w[0] * (S - w[1]) * (S - SM) - (w[5] * w[5]);
  if (den != 0) {
    const double sv = (SM - w[1]) / den;
    ws[2] = w[2] - w[5] * w[6] * sv;
    ws[3] = w[3] - w[5] * w[7] * sv;
    const double sb = (w[0] * ((S - w[1]) * (S - w[1])) - (w[5] * w[5])) / den;
    ws[6] = w[6] * sb;
    ws[7] = w[7] * sb;
  } else {
    ws[2] = w[2];
    ws[3] = w[3];
    ws[6] = 0.;
    ws[7] = 0.;
  }
  es = (((S - w[1]) * e - pt * w[1] + pts * SM + w[5] * (vdotb(w) - vdotb(ws))) / (S - SM));
}

// conserved vector of a star state whose energy is supplied (misc.cpp:82-92 + override)
__host__ __device__ AMR_INLINE void star_cons(const double* w, double e, double* u) {
  u[0] = w[0];
  u[1] = w[0] * w[1];
  u[2] = w[0] * w[2];
  u[3] = w[0] * w[3];
  u[4] = e;
  u[5] = w[5];
  u[6] = w[6];
  u[7] = w[7];
}

// scalars of side_state only (the conserved vector and flux are formed where
// a flux region needs them, with the same expressions)
struct SideScalars {
  double e, H, pt, cf;
};

template <bool FAST = false>
__host__ __device__ AMR_INLINE void side_scalars(const double* w, double g, SideScalars& s) {
  const Den<FAST> r0 = den<FAST>(w[0]);
  s.cf = fast_speed<FAST>(w, g, 5);
  const double b2 = w[5] * w[5] + w[6] * w[6] + w[7] * w[7];
  double e = quot(w[4], den<FAST>(w[0] * (g - 1))) + 0.5 * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3]) + quot(0.5 * b2, r0);
  e = e * w[0];
  s.e = e;
  s.H = quot(e + w[4] + 0.5 * b2, r0);
  s.pt = w[4] + 0.5 * b2;
}

// side_state's x-flux from its scalars
__host__ __device__ AMR_INLINE void side_flux(const double* w, const SideScalars& s, double* F) {
  const double vn = w[1], Bn = w[5];
  const double mv = w[0] * vn;
  F[0] = mv;
  F[1] = mv * w[1] + s.pt - Bn * w[5];
  F[2] = mv * w[2] - Bn * w[6];
  F[3] = mv * w[3] - Bn * w[7];
  F[4] = mv * s.H - Bn * (w[1] * w[5] + w[2] * w[6] + w[3] * w[7]);
  F[5] = vn * w[5] - Bn * w[1];
  F[6] = vn * w[6] - Bn * w[2];
  F[7] = vn * w[7] - Bn * w[3];
}

// riemannS.cpp:397-549 (Miyoshi & Kusano 2005 HLLD).  The flux region is
// decided from the wave speeds and the star densities alone (the first
// component of each star state, riemannS.cpp:467); the star states, the
// double-star state, and the side flux and conserved vectors are formed only
// in the region that uses them -- fewer live registers in the stage kernel,
// the same operations per value.
__host__ __device__ AMR_INLINE void flux_hlld(const double* wL, const double* wR, double g, double* f) {
  SideScalars L, R;
  side_scalars(wL, g, L);
  side_scalars(wR, g, R);
  const double vL = wL[1], vR = wR[1];
  const double cmax = std_max(L.cf, R.cf);
  const double SL = std_min(vL, vR) - cmax;
  const double SR = std_max(vL, vR) + cmax;
  const double den = (SR - vR) * wR[0] - (SL - vL) * wL[0];
  const double SM = ((SR - vR) * wR[0] * vR - (SL - vL) * wL[0] * vL - R.pt + L.pt) / den;
  const double pts = ((SR - vR) * wR[0] * L.pt - (SL - vL) * wL[0] * R.pt +
                      wL[0] * wR[0] * (SR - vR) * (SL - vL) * (vR - vL)) / den;
  const double rhoLs = wL[0] * (SL - wL[1]) / (SL - SM);  // = hlld_star's ws[0]
  const double rhoRs = wR[0] * (SR - wR[1]) / (SR - SM);
  const double rl = sqrt(rhoLs), rr = sqrt(rhoRs);
  const double SLs = SM - fabs(wL[5]) / rl;
  const double SRs = SM + fabs(wR[5]) / rr;
  int region = 0;  // 0: no branch taken (NaN speeds), f keeps its zeros
  if (SL > 0) region = 1;
  else if (SL <= 0. && SLs >= 0.) region = 2;
  else if (SLs <= 0. && SM >= 0.) region = 3;
  else if (SM <= 0. && SRs >= 0.) region = 4;
  else if (SRs <= 0. && SR >= 0.) region = 5;
  else if (SR < 0.) region = 6;
  if (region == 1) {
    side_flux(wL, L, f);
    return;
  }
  if (region == 6) {
    side_flux(wR, R, f);
    return;
  }
  if (region == 0) return;
  double F[8], q[8], qs[8];
  if (region == 2) {
    double wLs[8], eLs;
    hlld_star(wL, SL, SM, pts, L.e, L.pt, wLs, eLs);
    side_flux(wL, L, F);
    star_cons(wL, L.e, q);
    star_cons(wLs, eLs, qs);
#pragma unroll
    for (int k = 0; k < 8; k++) f[k] = F[k] + SL * qs[k] - SL * q[k];
    return;
  }
  if (region == 5) {
    double wRs[8], eRs;
    hlld_star(wR, SR, SM, pts, R.e, R.pt, wRs, eRs);
    side_flux(wR, R, F);
    star_cons(wR, R.e, q);
    star_cons(wRs, eRs, qs);
#pragma unroll
    for (int k = 0; k < 8; k++) f[k] = F[k] + SR * qs[k] - SR * q[k];
    return;
  }
  // regions 3 and 4: the double-star state
  double wLs[8], wRs[8], eLs, eRs;
  hlld_star(wL, SL, SM, pts, L.e, L.pt, wLs, eLs);
  hlld_star(wR, SR, SM, pts, R.e, R.pt, wRs, eRs);
  const double rlr = sqrt(wLs[0] * wRs[0]);
  const double sg = sign0(wL[5]);
  double wss[8], qss[8];
  wss[0] = wLs[0];
  wss[1] = SM;
  wss[2] = (rl * wLs[2] + rr * wRs[2] + (wRs[6] - wLs[6]) * sg) / (rl + rr);
  wss[3] = (rl * wLs[3] + rr * wRs[3] + (wRs[7] - wLs[7]) * sg) / (rl + rr);
  wss[4] = 0.;
  wss[5] = wLs[5];
  wss[6] = (rl * wRs[6] + rr * wLs[6] + rlr * (wRs[2] - wLs[2]) * sg) / (rl + rr);
  wss[7] = (rl * wRs[7] + rr * wLs[7] + rlr * (wRs[3] - wLs[3]) * sg) / (rl + rr);
  const double dss = vdotb(wss);
  if (region == 3) {
    const double eLss = eLs - rl * (vdotb(wLs) - dss) * sg;
    side_flux(wL, L, F);
    star_cons(wL, L.e, q);
    star_cons(wLs, eLs, qs);
    star_cons(wss, eLss, qss);
#pragma unroll
    for (int k = 0; k < 8; k++) f[k] = F[k] + SLs * qss[k] - (SLs - SL) * qs[k] - SL * q[k];
  } else {
    const double eRss = eRs + rr * (vdotb(wRs) - dss) * sign0(wR[5]);
    side_flux(wR, R, F);
    star_cons(wR, R.e, q);
    star_cons(wRs, eRs, qs);
    star_cons(wss, eRss, qss);
#pragma unroll
    for (int k = 0; k < 8; k++) f[k] = F[k] + SRs * qss[k] - (SRs - SR) * qs[k] - SR * q[k];
  }
}

#ifdef AMR_DEVICE_FP
// flux_hlld with FAST quotients on one path: the side whose flux the region
// takes (A: left of the contact in regions 1-3, right in 4-6) is selected per
// lane before the star states are formed, where flux_hlld branches into six
// regions -- a wavefront whose lanes fall into several of them (most do near
// a disturbance, where SM's sign varies) runs the states once, and the star
// energy of the other side is not formed.  The same operations on the same
// operands as flux_hlld for every value used: sums of one term a side are
// taken in (A, B) order, and differences of the sides with their sign moved to
// the factor sg, which is exact but for the sign of a zero difference added
// to -0 (checked below).
//
// Range: with density and pressure in 2^[-60, 60] the wave speeds less the
// velocities are above 2^-62, SM's numerator is 0 or above 2^-254 (a
// difference of total pressures, or of terms above 2^-200) and those of pts
// and the star densities above 2^-300.  What is left is checked on the values
// met: |SM| below 2^100, the star densities within 2^[-200, 200], and the
// numerators that can be as small as a transverse component or cancel to it
// -- w1 and w5 for the star velocity and the Alfven speeds, the star energy
// and the double-star state -- 0 or within 2^[kNumLo, kNumHi].  Returns false
// where a check fails: the caller then takes the plain flux.
__device__ AMR_INLINE bool flux_hlld_fast(const double* wL, const double* wR, double g, double* f) {
  SideScalars L, R;
  side_scalars<true>(wL, g, L);
  side_scalars<true>(wR, g, R);
  const double vL = wL[1], vR = wR[1];
  const double cmax = std_max(L.cf, R.cf);
  const double SL = std_min(vL, vR) - cmax;
  const double SR = std_max(vL, vR) + cmax;
  const Den<true> dm = den<true>((SR - vR) * wR[0] - (SL - vL) * wL[0]);
  const double SM = quot((SR - vR) * wR[0] * vR - (SL - vL) * wL[0] * vL - R.pt + L.pt, dm);
  const double pts = quot((SR - vR) * wR[0] * L.pt - (SL - vL) * wL[0] * R.pt +
                              wL[0] * wR[0] * (SR - vR) * (SL - vL) * (vR - vL),
                          dm);
  const double rhoLs = quot(wL[0] * (SL - vL), den<true>(SL - SM));
  const double rhoRs = quot(wR[0] * (SR - vR), den<true>(SR - SM));
  const double rl = root<true>(rhoLs), rr = root<true>(rhoRs);
  const double SLs = SM - quot(fabs(wL[5]), den<true>(rl));
  const double SRs = SM + quot(fabs(wR[5]), den<true>(rr));
  ExpSpan mid, num, speed;
  mid.add(rhoLs);
  mid.add(rhoRs);
  speed.add(SM);
  num.add(vL);
  num.add(vR);
  num.add(wL[5]);
  num.add(wR[5]);
  bool ok = mid.within(-200, 200) && speed.hi <= 100;
  int region = 0;  // 0: no branch taken (NaN speeds), f keeps its zeros
  if (SL > 0) region = 1;
  else if (SL <= 0. && SLs >= 0.) region = 2;
  else if (SLs <= 0. && SM >= 0.) region = 3;
  else if (SM <= 0. && SRs >= 0.) region = 4;
  else if (SRs <= 0. && SR >= 0.) region = 5;
  else if (SR < 0.) region = 6;
  const bool left = region <= 3, dbl = region == 3 || region == 4;
  double w[8], wb[8];  // states of sides A and B
#pragma unroll
  for (int k = 0; k < 8; k++) {
    w[k] = left ? wL[k] : wR[k];
    wb[k] = left ? wR[k] : wL[k];
  }
  SideScalars A;
  A.e = left ? L.e : R.e;
  A.H = left ? L.H : R.H;
  A.pt = left ? L.pt : R.pt;
  const double S = left ? SL : SR, Sb = left ? SR : SL;
  const double rho = left ? rhoLs : rhoRs;
  const double sgA = sign0(w[5]);
  const double bnL = wL[5], sg = sign0(bnL), rhoss = rhoLs;
  double F[8];
  side_flux(w, A, F);
#pragma unroll
  for (int k = 0; k < 8; k++) f[k] = region ? F[k] : 0.;
  if (region >= 2 && region <= 5) {
    // star state of A (hlld_star)
    double ws[8], es;
    const double Sv = S - w[1];
    ws[0] = rho;
    ws[1] = SM;
    ws[4] = 0.;
    ws[5] = w[5];
    const double dn = w[0] * Sv * (S - SM) - (w[5] * w[5]);
    const Den<true> dd = den<true>(dn);
    const double sv = quot(SM - w[1], dd);
    const double sb = quot(w[0] * (Sv * Sv) - (w[5] * w[5]), dd);
    const bool nz = dn != 0;
    ws[2] = nz ? w[2] - w[5] * w[6] * sv : w[2];
    ws[3] = nz ? w[3] - w[5] * w[7] * sv : w[3];
    ws[6] = nz ? w[6] * sb : 0.;
    ws[7] = nz ? w[7] * sb : 0.;
    const double vbs = vdotb(ws);
    const double n = Sv * A.e - A.pt * w[1] + pts * SM + w[5] * (vdotb(w) - vbs);
    num.add(n);
    es = quot(n, den<true>(S - SM));
    double q[8], qs[8];
    star_cons(w, A.e, q);
    star_cons(ws, es, qs);
    if (!dbl) {
#pragma unroll
      for (int k = 0; k < 8; k++) f[k] = F[k] + S * qs[k] - S * q[k];
    } else {
      // star velocity and field of B, then the double-star state
      double b2, b3, b6, b7;
      {
        const double Svb = Sb - wb[1];
        const double dnb = wb[0] * Svb * (Sb - SM) - (wb[5] * wb[5]);
        const Den<true> ddb = den<true>(dnb);
        const double svb = quot(SM - wb[1], ddb);
        const double sbb = quot(wb[0] * (Svb * Svb) - (wb[5] * wb[5]), ddb);
        const bool nzb = dnb != 0;
        b2 = nzb ? wb[2] - wb[5] * wb[6] * svb : wb[2];
        b3 = nzb ? wb[3] - wb[5] * wb[7] * svb : wb[3];
        b6 = nzb ? wb[6] * sbb : 0.;
        b7 = nzb ? wb[7] * sbb : 0.;
      }
      const double ra = left ? rl : rr, rb = left ? rr : rl;
      const double rlr = root<true>(rhoLs * rhoRs);
      const Den<true> dr = den<true>(rl + rr);
      const double sd = left ? sg : -sg;
      const double t2 = ra * ws[2] + rb * b2, t3 = ra * ws[3] + rb * b3;
      const double t6 = ra * b6 + rb * ws[6], t7 = ra * b7 + rb * ws[7];
      const double n2 = t2 + (b6 - ws[6]) * sd, n3 = t3 + (b7 - ws[7]) * sd;
      const double n6 = t6 + rlr * (b2 - ws[2]) * sd, n7 = t7 + rlr * (b3 - ws[3]) * sd;
      num.add(n2);
      num.add(n3);
      num.add(n6);
      num.add(n7);
      constexpr int kNegZero = 0x20;
      ok = ok && !(__builtin_amdgcn_class(t2, kNegZero) || __builtin_amdgcn_class(t3, kNegZero) ||
                   __builtin_amdgcn_class(t6, kNegZero) || __builtin_amdgcn_class(t7, kNegZero));
      double wss[8], qss[8];
      wss[0] = rhoss;
      wss[1] = SM;
      wss[2] = quot(n2, dr);
      wss[3] = quot(n3, dr);
      wss[4] = 0.;
      wss[5] = bnL;
      wss[6] = quot(n6, dr);
      wss[7] = quot(n7, dr);
      const double ess = es + (left ? -ra : ra) * (vbs - vdotb(wss)) * sgA;
      const double Ss = left ? SLs : SRs;
      star_cons(wss, ess, qss);
#pragma unroll
      for (int k = 0; k < 8; k++) f[k] = F[k] + Ss * qss[k] - (Ss - S) * qs[k] - S * q[k];
    }
  }
  return ok && num.within(kNumLo, kNumHi);
}
#endif

// x-normal flux of the selected solver; a y face is computed by the caller
// with (1,2) and (5,6) exchanged on input and output (riemannS.cpp:12-55).
// Components a solver leaves unset stay 0.  Returns nonzero where the
// reference throws.
// ok turns false where FAST turns out not to apply.
template <bool FAST>
__host__ __device__ AMR_INLINE int solver_flux(int solver, const double* wL, const double* wR, double g, double* f,
                                           bool& ok) {
#pragma unroll
  for (int k = 0; k < 8; k++) f[k] = 0.;
  switch (solver) {
    case kFluxRusanov: flux_rusanov<FAST>(wL, wR, g, f); return 0;
    case kFluxHLLE: ok = flux_hlle<FAST>(wL, wR, g, f); return 0;
    case kFluxHLLC: return flux_hllc<FAST>(wL, wR, g, f, ok);
    case kFluxHLLD:
#ifdef AMR_DEVICE_FP
      if constexpr (FAST) {
        ok = flux_hlld_fast(wL, wR, g, f);
        return 0;
      }
#endif
      flux_hlld(wL, wR, g, f);
      return 0;
    default: return 2;
  }
}

__host__ __device__ AMR_INLINE int normal_flux(int solver, const double* wL, const double* wR, double g, double* f) {
  bool ok = true;
  return solver_flux<false>(solver, wL, wR, g, f, ok);
}

// The FAST flux of a face whose states lie in its range; returns false, with
// f and *st void, for the others: the caller then forms the states again and
// takes normal_flux.  (Not a fallback in here: the 16 states of the face
// would stay in registers through the whole solver.)
#ifndef AMR_COUNT_OPS
__host__ __device__ AMR_INLINE bool fast_flux(int solver, const double* wL, const double* wR, double g, double* f,
                                              int* st) {
  constexpr double kBig = 1152921504606846976., kSmall = 1. / kBig;  // 2^60, 2^-60
  const double lo = fmin(fmin(wL[0], wR[0]), fmin(wL[4], wR[4]));
  double hi = fmax(fmax(wL[0], wR[0]), fmax(wL[4], wR[4]));
#pragma unroll
  for (int k = 1; k < 8; k++)
    if (k != 4) hi = fmax(hi, fmax(fabs(wL[k]), fabs(wR[k])));
  const double g1 = g - 1;
  bool ok = lo >= kSmall && hi <= kBig && g1 >= kSmall && g1 <= kBig;
  if (ok) *st = solver_flux<true>(solver, wL, wR, g, f, ok);
  return ok;
}
#endif

__host__ __device__ AMR_INLINE void swap_xy(double* w) {
  double t = w[1];
  w[1] = w[2];
  w[2] = t;
  t = w[5];
  w[5] = w[6];
  w[6] = t;
}

// WENO5 edge states of one cell from its 5-point stencil
// (WENO2D_primvar.cpp:95-198; beta_1's first term uses w_{i-2} as there).
// left=true: state at i+1/2 (wxL); left=false: state at i-1/2 (wxR).
template <bool FAST = false>
__host__ __device__ AMR_INLINE double weno5_edge(double m2, double m1, double c, double p1, double p2, bool left) {
  const double ew = 1.E-15;
  const Den<FAST> six = den_literal<FAST>(6);
  double t0 = m2 - 2 * m1 + c, u0 = m2 - 4 * m1 + 3 * c;
  double t1 = m2 - 2 * c + p1, u1 = m1 - p1;
  double t2 = c - 2 * p1 + p2, u2 = 3 * c - 4 * p1 + p2;
  const double e0 = ew + ((13. / 12.) * (t0 * t0) + (1. / 4.) * (u0 * u0));
  const double e1 = ew + ((13. / 12.) * (t1 * t1) + (1. / 4.) * (u1 * u1));
  const double e2 = ew + ((13. / 12.) * (t2 * t2) + (1. / 4.) * (u2 * u2));
  const double s0 = e0 * e0, s1 = e1 * e1, s2 = e2 * e2;
  if (!left) {
    const double a0 = quot(1. / 10., den<FAST>(s0)), a1 = quot(6. / 10., den<FAST>(s1)), a2 = quot(3. / 10., den<FAST>(s2));
    const Den<FAST> as = den<FAST>(a0 + a1 + a2);
    return quot(a0, as) * quot(-1 * m2 + 5 * m1 + 2 * c, six) + quot(a1, as) * quot(2 * m1 + 5 * c - p1, six) +
           quot(a2, as) * quot(11 * c - 7 * p1 + 2 * p2, six);
  }
  const double a0 = quot(3. / 10., den<FAST>(s0)), a1 = quot(6. / 10., den<FAST>(s1)), a2 = quot(1. / 10., den<FAST>(s2));
  const Den<FAST> as = den<FAST>(a0 + a1 + a2);
  return quot(a0, as) * quot(2 * m2 - 7 * m1 + 11 * c, six) + quot(a1, as) * quot(-1 * m1 + 5 * c + 2 * p1, six) +
         quot(a2, as) * quot(2 * c + 5 * p1 - p2, six);
}

// WENO3 edge states (WENO2D_primvar.cpp:7-91)
template <bool FAST = false>
__host__ __device__ AMR_INLINE double weno3_edge(double m1, double c, double p1, bool left) {
  const double ew = 1.E-15;
  const double e0 = ew + (c - m1) * (c - m1), e1 = ew + (p1 - c) * (p1 - c);
  const double s0 = e0 * e0, s1 = e1 * e1;
  if (!left) {
    const double a0 = quot(2. / 3., den<FAST>(s0)), a1 = quot(1. / 3., den<FAST>(s1));
    const Den<FAST> as = den<FAST>(a0 + a1);
    return quot(a0, as) * (0.5 * m1 + 0.5 * c) + quot(a1, as) * (1.5 * c - 0.5 * p1);
  }
  const double a0 = quot(1. / 3., den<FAST>(s0)), a1 = quot(2. / 3., den<FAST>(s1));
  const Den<FAST> as = den<FAST>(a0 + a1);
  return quot(a0, as) * (1.5 * c - 0.5 * m1) + quot(a1, as) * (0.5 * p1 + 0.5 * c);
}

// Limited linear edge states of one variable (celledges.cpp:29-64):
// `left` is the state at i+1/2 seen from cell i (slopes d0 = w_i - w_{i-1},
// d1 = w_{i+1} - w_i), `right` the state at i-1/2 seen from cell i.
template <bool FAST = false>
__host__ __device__ AMR_INLINE double muscl_plus(int lim, double w, double d0, double d1, double dxl) {
  const double eta = (lim == kLimCada) ? ((d1 * d1) + (d0 * d0)) / ((1. * dxl) * (1. * dxl)) : 0.;
  const double phi = limiter<FAST>(lim, quot(d1, den<FAST>(d0 + kEps)), eta);
  return w + 0.5 * phi * d0;
}
template <bool FAST = false>
__host__ __device__ AMR_INLINE double muscl_minus(int lim, double w, double d0, double d1, double dxl) {
  const double eta = (lim == kLimCada) ? ((d1 * d1) + (d0 * d0)) / ((1. * dxl) * (1. * dxl)) : 0.;
  const double phi = limiter<FAST>(lim, quot(d0, den<FAST>(d1 + kEps)), eta);
  return w - 0.5 * phi * d1;
}

}  // namespace amr
