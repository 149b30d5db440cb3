// numerics.hpp -- per-cell / per-face arithmetic of the MUSCL-Hancock scheme.
//
// Templated on the arithmetic type T.  With T = double each function evaluates
// the same IEEE operations, in the same order, as the reference's inline
// functions (pkestene/euler2d_kokkos src/HydroBaseFunctor.h), so that the FP64
// path reproduces the reference bit for bit: this file must be compiled without
// FMA contraction (-ffp-contract=off and the pragma below) and without
// fast-math.  Restructurings that keep every FP64 result bit-identical are
// marked where they happen (shared source terms, one star state per HLLC).
// With T = float (the split-precision path) division and square root use the
// hardware reciprocal / square-root instructions (about 1 ulp), which is
// where that path saves most of its instructions.
#pragma once

#include <hip/hip_runtime.h>

#pragma clang fp contract(off)

namespace e2d {

enum { ID = 0, IP = 1, IU = 2, IV = 3 };

// Division, square root, min/max per arithmetic type.
template <class T>
struct Ops;

// mad(a, b, c) = a * b + c: for FP64 the product and the sum are rounded
// separately, exactly as the reference writes the expression (the FP64 path
// must keep every rounding); for FP32 it is one fused multiply-add.  Callers
// pass the operands so that the FP64 form is the reference's own expression
// tree (x - a * b is written mad(-a, b, x): negating a factor is exact).
template <>
struct Ops<double> {
  static __device__ __forceinline__ double div(double a, double b) { return a / b; }
  static __device__ __forceinline__ double mad(double a, double b, double c) { return a * b + c; }
  static __device__ __forceinline__ double sqroot(double x) { return sqrt(x); }
  static __device__ __forceinline__ double mx(double a, double b) { return fmax(a, b); }
  static __device__ __forceinline__ double mn(double a, double b) { return fmin(a, b); }
  static __device__ __forceinline__ double ab(double a) { return fabs(a); }
};

// Square root of x >= smallc^2 for the wave-speed estimates.  The compiler's
// correctly rounded FP64 sqrt first scales x < 2^-767 by 2^256, then runs
// rsq + one Goldschmidt step + two Newton corrections, unscales, and returns
// x itself for +-0 and +inf.  For x in [2^-767, DBL_MAX] the scaling and the
// special cases are identities, so the same core sequence, operation for
// operation, gives the same bits; the host enables it only when smallc^2 (the
// floor of every argument) is >= 2^-220.  +inf gives NaN where sqrt returns inf.
__device__ __forceinline__ double sqrt_core(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y;
  double h = y * 0.5;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  double d = __builtin_fma(-g, g, x);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(d, h, g);
  d = __builtin_fma(-g, g, x);
  g = __builtin_fma(d, h, g);
  return g;
}

template <>
struct Ops<float> {
  static __device__ __forceinline__ float div(float a, float b) {
    return a * __builtin_amdgcn_rcpf(b);
  }
  static __device__ __forceinline__ float mad(float a, float b, float c) {
    return __builtin_fmaf(a, b, c);
  }
  static __device__ __forceinline__ float sqroot(float x) { return __builtin_amdgcn_sqrtf(x); }
  static __device__ __forceinline__ float mx(float a, float b) { return fmaxf(a, b); }
  static __device__ __forceinline__ float mn(float a, float b) { return fminf(a, b); }
  static __device__ __forceinline__ float ab(float a) { return fabsf(a); }
};

// Scheme constants, precomputed on the host in double (entho = 1/(gamma0-1) is
// the same IEEE division the reference performs inside every Riemann call)
// and rounded once for the float path.
template <class T>
struct SchemeT {
  T gamma0, gamma6, smallr, smallc, smallp, smallpp, slope_type, entho;
  T smallc2;    // smallc * smallc
  int riemann;  // 0 approx, 1 hll, 2 hllc (already resolved from honor_riemann)
  // smallr >= 2^-110, smallc 2^-110 .. 2^200, smallp >= 2^-230, gamma0 <= 16, entho <= 2^20,
  // cell sizes of 2^-100 .. 2^100: the sound speeds take the short sqrt and the step's
  // quotients the bounded forms
  int floor_sqrt;
};
using Scheme = SchemeT<double>;

template <class T>
struct Q4T {
  T v[4];
};
using Q4 = Q4T<double>;

// ------------------------------------------------ FP64 quotients sharing d
// The compiler's IEEE FP64 division a / d is div_scale(d), rcp, two Newton
// steps, m = a r, e = a - d m, q = m + e r (div_fmas), div_fixup.  For the
// quotients by one d the reciprocal is formed once, by the same operations,
// and each quotient takes the three steps after it.  The scaling and fix-up
// steps act only where d or 1/d is not normal, where the residual e is
// denormal (a below about 2^-969), or where q is not normal: class tests catch
// each of these, and a wavefront with any such lane takes the IEEE division
// for all of its lanes.  A zero quotient takes the sign of m, as div_fixup
// gives it.  Same bits; 27 instead of 33 VALU instructions for the three
// quotients of prim.  Each fallback is a branch that splits the march's steady
// row; so quotients by one density that a row forms later (the trace's source
// terms, the CFL rate's gamma p / d) join the check of that density's
// conversion instead of adding one.
//
// Bounded kinds (BND).  Where the floors of the deck are not absurdly small
// (SchemeT::floor_sqrt, decided on the host) most of those tests follow from
// ranges that are cheap to check once per cell:
//   d <= 2^80, p <= 2^160, (u^2 + v^2) / 2 <= 2^120, momenta zero or at least
//   2^-801, and the residual of E / d zero or normal.
// Then smallr >= 2^-110 <= d makes d and 1/d normal, and with a residual, a multiple
// of 2^-106 of its numerator, zero or normal the quotients are the IEEE ones.  u and
// v are zero or at least 2^-881 and their differences zero or at least 2^-934, so
// that their halves are exact (a zero residual alone would not bound them: over
// d = 1 every denormal divides exactly).  E / d enters the pressure only;
// p >= smallr smallp >= 2^-340 makes pressure differences zero or at least 2^-393.
// With |dt / dx| <= 2^40 (checked per wavefront) the traced face states stay below
// 2^185 in density, 2^268 in pressure (2^455 once floored, for a large smallp) and
// 2^311 in velocity, and the wave speeds below 2^200; what may still overflow in the
// solvers is named there.  A wavefront with a lane outside these ranges takes the
// IEEE divisions, for a cell out of them in all of its later rows, after the checked
// forms: 1024x1536, 14 rows, 71 us with every wavefront outside, 42.5 with none; 55 with
// a disc of 0.1% of the cells outside.  Floors below the ranges leave the deck to the
// kinds with IEEE divisions: 49.6 us.  The ranges keep both to values that no system
// of units brings about (1e24 in density, 1e48 in pressure, 1e18 in velocity; floors
// under 1e-33).  A branch around the checked forms for wavefronts outside costs all
// others more than it saves: 42.5 -> 43.8 us, 768x384 17.1 -> 19.0.
//
// The march is bound by VALU issue (4 cycles per FP64 instruction, 16 per rcp
// or rsq), so these forms, one wave-speed root per face instead of two, the
// minmod slope without its redundant third limit, one side's energy per HLLC
// face and no branch between its two fluxes count directly: a steady HLLC row
// went from 695 instructions (2900 issue cycles) to 590 (2420).  1024x1536
// blast, 14-row tile: 50.3 -> 44.7 us a step; 8192x8192, 48 rows: HLLC 1874 -> 1579,
// HLL 1701 -> 1510 us.

__device__ __forceinline__ double recip_newton(double d) {
  const double r0 = __builtin_amdgcn_rcp(d);
  const double r1 = __builtin_fma(r0, __builtin_fma(-d, r0, 1.0), r0);
  return __builtin_fma(r1, __builtin_fma(-d, r1, 1.0), r1);
}

constexpr int kClassNormal = (1 << 3) | (1 << 8);
constexpr int kClassZeroOrNormal = kClassNormal | (1 << 5) | (1 << 6);

constexpr double kBndDensity = 0x1p80, kBndPressure = 0x1p160, kBndKinetic = 0x1p120;
constexpr double kBndDtd = 0x1p40;  // |dt / dx|, |dt / dy|
constexpr int kBndMomentumExp = -800;  // frexp exponent: zero (exponent 0) or >= 2^-801

// a / d from r = 1 / d where no step needs scaling and a is not -0
__device__ __forceinline__ double quot_plain(double a, double d, double r) {
  const double m = a * r;
  return __builtin_fma(__builtin_fma(-d, m, a), r, m);
}

// the same with the residual's test: ok is cleared where it is denormal, or
// where a step overflowed or met a NaN
__device__ __forceinline__ double quot_resid(double a, double d, double r, bool &ok) {
  const double m = a * r;
  const double e = __builtin_fma(-d, m, a);
  ok = ok && __builtin_amdgcn_class(e, kClassZeroOrNormal);
  return __builtin_fma(e, r, m);
}

__device__ __forceinline__ double quot_shared(double a, double d, double r, bool &ok) {
  const double m = a * r;
  const double e = __builtin_fma(-d, m, a);
  const double q = __builtin_fma(e, r, m);
  ok = ok && __builtin_amdgcn_class(q, kClassZeroOrNormal) &&
       __builtin_amdgcn_class(e, kClassZeroOrNormal);
  return __builtin_copysign(q, m);
}

// 2^lo <= x < 2^(hi + 1), for positive bounds: one comparison of the high word
__device__ __forceinline__ bool exponent_within(double x, int lo, int hi) {
  const unsigned h = (unsigned)(__double_as_longlong(x) >> 32);
  return h - ((unsigned)(1023 + lo) << 20) < (unsigned)(hi - lo + 1) << 20;
}

// true in every lane when no active lane of the wavefront has !ok
__device__ __forceinline__ bool wave_all(bool ok) {
  return __builtin_amdgcn_ballot_w64(!ok) == 0;
}

// the rest of computePrimitives once the three quotients are formed; returns
// the specific kinetic energy
__device__ __forceinline__ double prim_finish(const SchemeT<double> &s, double d, double ux,
                                              double uy, double e1, Q4T<double> &q) {
  const double eken = 0.5 * (uy * uy + ux * ux);
  const double e = e1 - eken;
  const double p = fmax((s.gamma0 - 1.0) * d * e, d * s.smallp);
  q.v[ID] = d;
  q.v[IP] = p;
  q.v[IU] = ux;
  q.v[IV] = uy;
  return eken;
}

// the cell is outside the ranges of the bounded kinds (a NaN counts as outside)
__device__ __forceinline__ bool out_of_bounds(const Q4T<double> &q) {
  const double eken = 0.5 * (q.v[IV] * q.v[IV] + q.v[IU] * q.v[IU]);
  return !(q.v[ID] <= kBndDensity && q.v[IP] <= kBndPressure && eken <= kBndKinetic);
}

// computePrimitives for FP64 with the three quotients formed from one
// reciprocal and no fallback.  Returns whether this lane's quotients are the
// IEEE ones (BND: and the cell is in the bounded ranges); r is the reciprocal
// and rok whether other quotients by d formed from it can be (d and r normal;
// BND: part of the result instead).  RATE: for the CFL rate, where the sound speed
// covers velocities whose quotients are too small to be exact, so that the momenta
// are not tested (large ones and NaN fail the kinetic energy's bound).
template <bool BND = false, bool RATE = false>
__device__ __forceinline__ bool prim_fp64_shared(const SchemeT<double> &s, double u0, double u1,
                                                 double u2, double u3, Q4T<double> &q, double &r,
                                                 bool &rok) {
  const double d = fmax(u0, s.smallr);
  r = recip_newton(d);
  if constexpr (BND) {
    rok = true;
    bool ok = d <= kBndDensity;
    if constexpr (!RATE)
      ok = ok && min(__builtin_amdgcn_frexp_exp(u2), __builtin_amdgcn_frexp_exp(u3)) >=
                     kBndMomentumExp;
    const double ux = __builtin_copysign(quot_plain(u2, d, r), u2);  // d > 0
    const double uy = __builtin_copysign(quot_plain(u3, d, r), u3);
    const double e1 = quot_resid(u1, d, r, ok);
    const double eken = prim_finish(s, d, ux, uy, e1, q);
    return ok && q.v[IP] <= kBndPressure && eken <= kBndKinetic;
  } else {
    rok = __builtin_amdgcn_class(d, kClassNormal) && __builtin_amdgcn_class(r, kClassNormal);
    bool ok = rok;
    const double ux = quot_shared(u2, d, r, ok);
    const double uy = quot_shared(u3, d, r, ok);
    const double e1 = quot_shared(u1, d, r, ok);
    prim_finish(s, d, ux, uy, e1, q);
    return ok;
  }
}

// computePrimitives for FP64: the shared reciprocal, and the IEEE divisions
// for a wavefront with any lane outside its range
__device__ __forceinline__ void prim_fp64(const SchemeT<double> &s, double u0, double u1,
                                          double u2, double u3, Q4T<double> &q) {
  const double d = fmax(u0, s.smallr);
  const double r = recip_newton(d);
  bool ok = __builtin_amdgcn_class(d, kClassNormal) && __builtin_amdgcn_class(r, kClassNormal);
  double ux = quot_shared(u2, d, r, ok);
  double uy = quot_shared(u3, d, r, ok);
  double e1 = quot_shared(u1, d, r, ok);
  if (!wave_all(ok)) {  // uniform
    ux = u2 / d;
    uy = u3 / d;
    e1 = u1 / d;
  }
  prim_finish(s, d, ux, uy, e1, q);
}

// computePrimitives, HydroBaseFunctor.h:76-102 (the sound speed is returned
// separately because only the dt reduction needs it).  SHARED = false keeps
// the three IEEE divisions for FP64 as well (fewer registers: the split
// step's FP64 fallback for kinetic-dominated cells).
template <class T, bool SHARED = true>
__device__ __forceinline__ void prim_no_c(const SchemeT<T> &s, T u0, T u1, T u2, T u3,
                                          Q4T<T> &q) {
  using O = Ops<T>;
  if constexpr (SHARED && sizeof(T) == sizeof(double)) {
    prim_fp64(s, u0, u1, u2, u3, q);
  } else {
    const T d = O::mx(u0, s.smallr);
    const T ux = O::div(u2, d);
    const T uy = O::div(u3, d);
    const T eken = T(0.5) * O::mad(uy, uy, ux * ux);
    const T e = O::div(u1, d) - eken;
    const T p = O::mx((s.gamma0 - T(1.0)) * d * e, d * s.smallp);
    q.v[ID] = d;
    q.v[IP] = p;
    q.v[IU] = ux;
    q.v[IV] = uy;
  }
}

// Cell sizes for the CFL rate.  When a cell size is an exact power of two its
// reciprocal is exact and x / dx == x * (1/dx) for every x (IEEE division by
// 2^-k is an exact scaling, overflow and NaN included), so the division is
// replaced by a multiplication; other sizes keep the division.
template <class T>
struct RateT {
  T dx, dy, idx, idy;
  int pow2x, pow2y;
};

// ComputeDtFunctor body, HydroRunFunctors.h:53-74: (c+|u|)/dx + (c+|v|)/dy
template <class T>
__device__ __forceinline__ T cfl_rate_q(const SchemeT<T> &s, const Q4T<T> &q, const RateT<T> &r) {
  using O = Ops<T>;
  const T c = O::sqroot(O::div(s.gamma0 * (q.v[IP]), q.v[ID]));
  const T vx = c + O::ab(q.v[IU]);
  const T vy = c + O::ab(q.v[IV]);
  T rx, ry;
  if (r.pow2x)  // uniform
    rx = vx * r.idx;
  else
    rx = O::div(vx, r.dx);
  if (r.pow2y)
    ry = vy * r.idy;
  else
    ry = O::div(vy, r.dy);
  return rx + ry;
}

// The rate's square root of gamma p / d.  p >= d smallp, and under the host's
// floor_sqrt condition (which keeps d smallp normal for every d >= smallr) the
// argument is at least smallp > 2^-231, where the short sequence gives the IEEE
// bits; +inf keeps sqrt's result, and NaN stays NaN.
template <bool FS>
__device__ __forceinline__ double rate_sqrt(double x) {
  if constexpr (FS) {
    constexpr int kClassPosInf = 1 << 9;
    double r = sqrt_core(x);
    // formed in every lane and then selected: a branch around the root would
    // split the march's row for the lanes holding +inf
    asm volatile("" : "+v"(r));
    return __builtin_amdgcn_class(x, kClassPosInf) ? x : r;
  } else {
    return sqrt(x);
  }
}

// cfl_rate_q for FP64 from the conserved state: the quotient gamma p / d
// shares the primitive conversion's reciprocal and its one wave-level check.
// POW2: both cell sizes are known to be powers of two (no test per cell).
template <bool FS, bool POW2 = false>  // FS: also the bounded kinds' conversion
__device__ __forceinline__ double cfl_rate_fp64(const Scheme &s, double u0, double u1, double u2,
                                                double u3, const RateT<double> &rt) {
  Q4 q;
  double r;
  bool rok;
  bool ok = prim_fp64_shared<FS, FS>(s, u0, u1, u2, u3, q, r, rok);
  // bounded: 2^-230 <= smallp <= p / d <= 2^270, nothing to scale
  double x = FS ? quot_plain(s.gamma0 * q.v[IP], q.v[ID], r)
                : quot_shared(s.gamma0 * q.v[IP], q.v[ID], r, rok);
  const bool all = wave_all(ok && rok);
  if (!all) {  // uniform
    prim_no_c<double, false>(s, u0, u1, u2, u3, q);
    x = (s.gamma0 * q.v[IP]) / q.v[ID];
  }
  const double c = rate_sqrt<FS>(x);
  const double vx = c + fabs(q.v[IU]);
  const double vy = c + fabs(q.v[IV]);
  if constexpr (POW2) return vx * rt.idx + vy * rt.idy;
  if constexpr (FS) {
    // The cell sizes' correctly rounded reciprocals are at hand: with them the
    // residual step gives the IEEE quotient (Markstein 1990) wherever nothing
    // leaves the normal range (speeds of 2^-116 .. 2^138 here, cell sizes of 2^-100 ..
    // 2^100 by the host's floor_sqrt condition).  3 instructions instead of 11, one
    // of them a reciprocal, per direction.
    double rx = quot_plain(vx, rt.dx, rt.idx), ry = quot_plain(vy, rt.dy, rt.idy);
    if (!all) {  // uniform
      rx = vx / rt.dx;
      ry = vy / rt.dy;
    }
    return rx + ry;
  }
  double rx, ry;
  if (rt.pow2x)  // uniform
    rx = vx * rt.idx;
  else
    rx = vx / rt.dx;
  if (rt.pow2y)
    ry = vy * rt.idy;
  else
    ry = vy / rt.dy;
  return rx + ry;
}

// neg ? -z : z as one select on the high word (with the operand's negation)
__device__ __forceinline__ double select_neg(bool neg, double z) {
  const long long b = __double_as_longlong(z);
  const float h = __int_as_float((int)(b >> 32));
  const int hi = __float_as_int(neg ? -h : h);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)b);
}
__device__ __forceinline__ float select_neg(bool neg, float z) { return neg ? -z : z; }

// slope_unsplit_hydro_2d_scalar, HydroBaseFunctor.h:419-455 (one direction).
// MINMOD: st == 1, whose products with the one-sided differences are exact
// identities (every value, zeros, infinities and NaN included) and are left out.
template <bool MINMOD = false, class T>
__device__ __forceinline__ T limited_slope(T st, T q, T qplus, T qminus) {
  using O = Ops<T>;
  if constexpr (MINMOD) {
    // The sum of two one-sided differences of one sign is at least twice the
    // smaller, after rounding too, so |dcen| never limits them; and dcen >= 0
    // where qplus >= qminus, except that the smallest denormal difference halves
    // to -0: the FP64 callers keep to values whose differences are zero or larger
    // (in FP32 the sign of that zero slope is the only change).
    const T dl = q - qminus, dr = qplus - q;
    const T z = (dl * dr <= T(0.0)) ? T(0.0) : O::mn(O::ab(dl), O::ab(dr));
    return select_neg(!(qplus >= qminus), z);
  }
  const T dlft = st * (q - qminus);
  const T drgt = st * (qplus - q);
  const T dcen = T(0.5) * (qplus - qminus);
  const T dsgn = (dcen >= T(0.0)) ? T(1.0) : T(-1.0);
  const T slop = O::mn(O::ab(dlft), O::ab(drgt));
  const T dlim = ((dlft * drgt) <= T(0.0)) ? T(0.0) : slop;
  return dsgn * O::mn(dlim, O::ab(dcen));
}

// The limited slopes of the four variables of a cell in one direction, from
// its neighbours qp and qm, for slope_type == 1 (MINMOD) or any other non-zero
// slope_type
template <bool MINMOD, class T>
__device__ __forceinline__ void slopes_dir(T st, const Q4T<T> &q, const Q4T<T> &qp,
                                           const Q4T<T> &qm, Q4T<T> &dq) {
  for (int v = 0; v < 4; v++) dq.v[v] = limited_slope<MINMOD>(st, q.v[v], qp.v[v], qm.v[v]);
}

// Both directions, variable by variable (the order the split step's register
// allocation was tuned with)
template <bool MINMOD, class T>
__device__ __forceinline__ void slopes_xy(T st, const Q4T<T> &q, const Q4T<T> &qpx,
                                          const Q4T<T> &qmx, const Q4T<T> &qpy,
                                          const Q4T<T> &qmy, Q4T<T> &dqX, Q4T<T> &dqY) {
  for (int v = 0; v < 4; v++) {
    dqX.v[v] = limited_slope<MINMOD>(st, q.v[v], qpx.v[v], qmx.v[v]);
    dqY.v[v] = limited_slope<MINMOD>(st, q.v[v], qpy.v[v], qmy.v[v]);
  }
}

// slope_unsplit_hydro_2d, HydroBaseFunctor.h:473-516 for one variable: zero
// slopes when slope_type == 0, limited slopes when 1 (minmod) or 2 (MC)
template <class T>
__device__ __forceinline__ T slope1(const SchemeT<T> &s, T q, T qplus, T qminus) {
  // slope_type is uniform, so this is a scalar branch, not VALU work
  return s.slope_type == T(0.0) ? T(0.0) : limited_slope(s.slope_type, q, qplus, qminus);
}

// Source terms of trace_unsplit_2d_along_dir, HydroBaseFunctor.h:246-249.  They
// do not depend on the face, so one evaluation serves the four faces of a cell.
template <class T>
struct SourcesT {
  T sr0, sp0, su0, sv0;
};
using Sources = SourcesT<double>;

template <class T>
__device__ __forceinline__ SourcesT<T> trace_sources(const SchemeT<T> &s, const Q4T<T> &q,
                                                     const Q4T<T> &dqX, const Q4T<T> &dqY) {
  using O = Ops<T>;
  const T r = q.v[ID], p = q.v[IP], u = q.v[IU], v = q.v[IV];
  SourcesT<T> o;
  // ((-u*a - v*b) - c*d) per source term, with the products fused in FP32
  const T divu = dqX.v[IU] + dqY.v[IV];
  o.sr0 = O::mad(-divu, r, O::mad(-v, dqY.v[ID], -u * dqX.v[ID]));
  o.sp0 = O::mad(-(divu * s.gamma0), p, O::mad(-v, dqY.v[IP], -u * dqX.v[IP]));
  o.su0 = O::mad(-v, dqY.v[IU], -u * dqX.v[IU]) - O::div((dqX.v[IP]), r);
  o.sv0 = O::mad(-v, dqY.v[IV], -u * dqX.v[IV]) - O::div((dqY.v[IP]), r);
  return o;
}

// trace_sources for FP64 with the two pressure-slope quotients formed from the
// reciprocal rinv of the density q.v[ID] that the primitive conversion made
// (rok: d and rinv normal), with no fallback; ok is cleared in a lane whose
// quotients may differ from the IEEE ones (BND: none does where the cells are in
// the bounded ranges).
template <bool BND>
__device__ __forceinline__ Sources trace_sources_shared(const Scheme &s, const Q4 &q,
                                                        const Q4 &dqX, const Q4 &dqY, double rinv,
                                                        bool rok, bool &ok) {
  using O = Ops<double>;
  const double r = q.v[ID], p = q.v[IP], u = q.v[IU], v = q.v[IV];
  Sources o;
  const double divu = dqX.v[IU] + dqY.v[IV];
  o.sr0 = O::mad(-divu, r, O::mad(-v, dqY.v[ID], -u * dqX.v[ID]));
  o.sp0 = O::mad(-(divu * s.gamma0), p, O::mad(-v, dqY.v[IP], -u * dqX.v[IP]));
  double qx, qy;
  if constexpr (BND) {
    qx = __builtin_copysign(quot_plain(dqX.v[IP], r, rinv), dqX.v[IP]);
    qy = __builtin_copysign(quot_plain(dqY.v[IP], r, rinv), dqY.v[IP]);
  } else {
    bool qok = rok;
    qx = quot_shared(dqX.v[IP], r, rinv, qok);
    qy = quot_shared(dqY.v[IP], r, rinv, qok);
    ok = ok && qok;
  }
  o.su0 = O::mad(-v, dqY.v[IU], -u * dqX.v[IU]) - qx;
  o.sv0 = O::mad(-v, dqY.v[IV], -u * dqX.v[IV]) - qy;
  return o;
}

__device__ __forceinline__ double fma_t(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}
__device__ __forceinline__ float fma_t(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}

// Face states of trace_unsplit_2d_along_dir, HydroBaseFunctor.h:251-289.
// plus = false for the XMIN / YMIN faces, true for XMAX / YMAX; dq is the
// slope along the face normal, dtd = dtdx or dtdy.
// HALF: the product of the slope by a half is exact (bounded kinds), so that it
// may be fused with the sum.
template <bool HALF = false, class T>
__device__ __forceinline__ void trace_face(const SchemeT<T> &s, const Q4T<T> &q, const Q4T<T> &dq,
                                           const SourcesT<T> &src, T dtd, bool plus, Q4T<T> &f) {
  using O = Ops<T>;
  // (q +- h*dq) + (src*dtd)*h
  const T h = T(0.5), hs = plus ? h : -h;
  const T t[4] = {src.sr0, src.sp0, src.su0, src.sv0};
  for (int v = 0; v < 4; v++) {
    const T e = HALF ? fma_t(hs, dq.v[v], q.v[v]) : O::mad(hs, dq.v[v], q.v[v]);
    f.v[v] = O::mad(t[v] * dtd, h, e);
  }
  f.v[ID] = O::mx(s.smallr, f.v[ID]);
}

// Largest sound speed of the two states of a face, floored at smallc:
// max(sqrt(max(gamma p / r, smallc^2))) over the two.  A correctly rounded
// square root never decreases where its argument grows, so the root of the
// larger argument is the larger root, bit for bit, and one root serves both
// (the FP32 hardware root was checked to be monotone over every positive float).
// FS: the short root, which would give NaN for the +inf that states outside the bounded
// ranges may bring; the full root there costs every wavefront (768x384 16.9 -> 17.5 us a
// step).  BND: quotients of states in the bounded ranges.
template <bool FS, bool BND, class T>
__device__ __forceinline__ T wave_speed(const SchemeT<T> &s, T pl, T rl, T pr, T rr) {
  using O = Ops<T>;
  if constexpr (BND) {
    const T xl = quot_plain(s.gamma0 * pl, rl, recip_newton(rl));
    const T xr = quot_plain(s.gamma0 * pr, rr, recip_newton(rr));
    return sqrt_core(O::mx(O::mx(xl, xr), s.smallc2));
  } else {
    const T a = O::mx(O::mx(O::div(s.gamma0 * pl, rl), O::div(s.gamma0 * pr, rr)), s.smallc2);
    if constexpr (FS) return a > T(__DBL_MAX__) ? a : sqrt_core(a);
    return O::sqroot(a);
  }
}

// riemann_hllc, HydroBaseFunctor.h:704-809.  `ln`/`tn` are the indices of the
// normal / transverse velocity in the Q4 (IU/IV for x faces, IV/IU for y faces,
// which is the reference's swap before and after the call, :628-632).
// The reference evaluates both star states and then picks one; here the side
// is picked first and its energy, star state and outer state are evaluated
// once with the same expressions, which gives identical bits for the state
// it keeps: the left side where ustar > 0 or SL > 0 (there the reference takes
// the left state itself), the right one elsewhere.
// BND: the two quotients by rcr + rcl share a reciprocal, as do the two by
// Sk - ustar; ok is cleared in a lane where one of them may differ from the
// IEEE quotient.  Of the bounded ranges' consequences these are left to test:
// rcr + rcl (2^-230 .. 2^301) and Sk - ustar (2^-200 at least), and the residuals of
// ustar and etotstar, whose numerators may be tiny.  rcl and rcr are zero or at least
// smallr smallc / 2 >= 2^-221, as is rstar's numerator, and ptotstar's is zero or at
// least 2^-615 (the rounding of its positive part, 2^-221 2^-340).  ustar stays
// below 2^686 and rstar between 2^-907 and 2^698, or zero.  An overflow on the way to
// ustar or ptotstar makes etotstar's numerator, and with it the last residual, NaN
// or infinite.  No numerator is ever -0: each ends in a sum with +0 or with a number
// that is not zero.
template <bool FS = false, bool BND = false, class T>
__device__ __forceinline__ void hllc(const SchemeT<T> &s, const Q4T<T> &ql, const Q4T<T> &qr,
                                     int ln, int tn, T flux[4], bool &ok) {
  using O = Ops<T>;
  const T h = T(0.5);
  // the reference floors the densities at smallr again; trace_face has done it
  const T rl = ql.v[ID], rr = qr.v[ID];
  const T pl = O::mx(ql.v[IP], rl * s.smallp);
  const T pr = O::mx(qr.v[IP], rr * s.smallp);
  const T ul = ql.v[ln], ur = qr.v[ln];

  const T cmax = wave_speed<FS, BND>(s, pl, rl, pr, rr);
  const T SL = O::mn(ul, ur) - cmax;
  const T SR = O::mx(ul, ur) + cmax;

  const T rcl = rl * (ul - SL);
  const T rcr = rr * (SR - ur);
  // separate products: for mirrored states at a reflecting wall they cancel
  // exactly, so ustar and the wall's mass flux are exactly zero
  const T un = rcr * ur + rcl * ul + (pl - pr);
  // the left/right-symmetric sum stays unfused, so that mirrored states give
  // mirrored fluxes in FP32 too
  const T pn = O::mad(rcl * rcr, ul - ur, rcr * pl + rcl * pr);
  const T rc = rcr + rcl;
  T ustar, ptotstar;
  if constexpr (BND) {
    const T r = recip_newton(rc);
    ok = ok && exponent_within(rc, -230, 300);
    ustar = quot_resid(un, rc, r, ok);
    ptotstar = quot_plain(pn, rc, r);
  } else {
    ustar = O::div(un, rc);
    ptotstar = O::div(pn, rc);
  }

  const bool upwind = SL > T(0.0);  // the whole fan moves right
  const bool left = ustar > T(0.0);
  const bool side = left || upwind;
  const T rk = side ? rl : rr;
  const T uk = side ? ul : ur;
  const T pk = side ? pl : pr;
  const T vk = side ? ql.v[tn] : qr.v[tn];
  const T Sk = left ? SL : SR;
  T ek = h * rk * uk * uk;
  ek = O::mad(h * rk * vk, vk, ek);
  ek = O::mad(pk, s.entho, ek);
  T ro = rk, uo = uk, ptoto = pk, etoto = ek;
  // FP32: a branch around the star state; its ends keep the compiler from
  // interleaving the x and y fluxes of a row, which would cost the split step
  // its third wavefront per SIMD (183 registers instead of 167)
  if (sizeof(T) == sizeof(double) || !upwind) {
    const T rn = rk * (Sk - uk);
    const T en = O::mad(ptotstar, ustar, O::mad(-pk, uk, (Sk - uk) * ek));
    const T sd = Sk - ustar;
    T rstar, etotstar;
    if constexpr (BND) {
      const T r = recip_newton(sd);
      ok = ok && O::ab(sd) >= T(0x1p-200);
      rstar = quot_plain(rn, sd, r);
      etotstar = quot_resid(en, sd, r, ok);
    } else {
      rstar = O::div(rn, sd);
      etotstar = O::div(en, sd);
    }
    const bool star = !upwind && (left || SR > T(0.0));
    ro = star ? rstar : rk;
    uo = star ? ustar : uk;
    ptoto = star ? ptotstar : pk;
    etoto = star ? etotstar : ek;
  }
  const T fd = ro * uo;
  flux[ID] = fd;
  flux[ln] = O::mad(ro * uo, uo, ptoto);
  flux[IP] = (etoto + ptoto) * uo;
  flux[tn] = fd * ((fd > T(0.0)) ? ql.v[tn] : qr.v[tn]);
}

// HLL (no reference counterpart; the reference declares the enum only,
// HydroParams.h:49).  Toro 2009, section 10.3, eq. (10.21), with the floors and
// wave speeds of riemann_hllc.  Same expressions as the CPU oracle.  BND: SR - SL
// is at least smallc wherever the middle state is taken, and below 2^313, so its
// reciprocal needs no test.
template <bool FS = false, bool BND = false, class T>
__device__ __forceinline__ void hll(const SchemeT<T> &s, const Q4T<T> &ql, const Q4T<T> &qr,
                                    int ln, int tn, T flux[4]) {
  using O = Ops<T>;
  const T h = T(0.5);
  const T rl = ql.v[ID], rr = qr.v[ID];  // floored by trace_face
  const T pl = O::mx(ql.v[IP], rl * s.smallp);
  const T ul = ql.v[ln], vl = ql.v[tn];
  const T pr = O::mx(qr.v[IP], rr * s.smallp);
  const T ur = qr.v[ln], vr = qr.v[tn];
  const T el = O::mad(pl, s.entho, O::mad(h * rl * vl, vl, h * rl * ul * ul));
  const T er = O::mad(pr, s.entho, O::mad(h * rr * vr, vr, h * rr * ur * ur));
  const T cmax = wave_speed<FS, BND>(s, pl, rl, pr, rr);
  const T SL = O::mn(ul, ur) - cmax;
  const T SR = O::mx(ul, ur) + cmax;
  // variable order of the conserved state: rho, E, normal momentum, transverse momentum
  const T UL[4] = {rl, el, rl * ul, rl * vl};
  const T UR[4] = {rr, er, rr * ur, rr * vr};
  const T FL[4] = {rl * ul, (el + pl) * ul, O::mad(rl * ul, ul, pl), rl * ul * vl};
  const T FR[4] = {rr * ur, (er + pr) * ur, O::mad(rr * ur, ur, pr), rr * ur * vr};
  T f[4];
  if (SL >= T(0.0)) {
    for (int k = 0; k < 4; k++) f[k] = FL[k];
  } else if (SR <= T(0.0)) {
    for (int k = 0; k < 4; k++) f[k] = FR[k];
  } else {
    T inv;
    if constexpr (BND)
      inv = quot_plain(T(1.0), SR - SL, recip_newton(SR - SL));
    else
      inv = O::div(T(1.0), SR - SL);
    // SR*FL - SL*FR with separate products: exactly zero mass flux for
    // mirrored states at a reflecting wall
    for (int k = 0; k < 4; k++)
      f[k] = O::mad(SL * SR, UR[k] - UL[k], SR * FL[k] - SL * FR[k]) * inv;
  }
  flux[ID] = f[0];
  flux[IP] = f[1];
  flux[ln] = f[2];
  flux[tn] = f[3];
}

// riemann_approx + cmpflx, HydroBaseFunctor.h:523-693 (ten Newton iterations at
// most, hard-coded at :592)
template <class T>
__device__ __forceinline__ void approx(const SchemeT<T> &s, const Q4T<T> &qlf, const Q4T<T> &qrf,
                                       int ln, int tn, T flux[4]) {
  using O = Ops<T>;
  const T one = T(1.0), h = T(0.5), zero = T(0.0);
  const T rl = O::mx(qlf.v[ID], s.smallr);
  const T ul = qlf.v[ln];
  const T pl = O::mx(qlf.v[IP], rl * s.smallp);
  const T rr = O::mx(qrf.v[ID], s.smallr);
  const T ur = qrf.v[ln];
  const T pr = O::mx(qrf.v[IP], rr * s.smallp);
  const T cl = s.gamma0 * pl * rl;
  const T cr = s.gamma0 * pr * rr;
  T wl = O::sqroot(cl);
  T wr = O::sqroot(cr);
  T pstar = O::mx(O::div((wr * pl + wl * pr) + wl * wr * (ul - ur), wl + wr), zero);
  T pold = pstar;
  T conv = one;
  for (int iter = 0; (iter < 10) && (conv > T(1e-6)); ++iter) {
    const T wwl = O::sqroot(cl * (one + O::div(s.gamma6 * (pold - pl), pl)));
    const T wwr = O::sqroot(cr * (one + O::div(s.gamma6 * (pold - pr), pr)));
    const T qwl = O::div(T(2.0) * wwl * wwl * wwl, wwl * wwl + cl);
    const T qwr = O::div(T(2.0) * wwr * wwr * wwr, wwr * wwr + cr);
    const T usl = ul - O::div(pold - pl, wwl);
    const T usr = ur + O::div(pold - pr, wwr);
    const T delp = O::mx(O::div(qwr * qwl, qwr + qwl) * (usl - usr), -pold);
    pold = pold + delp;
    conv = O::ab(O::div(delp, pold + s.smallpp));
  }
  pstar = pold;
  wl = O::sqroot(cl * (one + O::div(s.gamma6 * (pstar - pl), pl)));
  wr = O::sqroot(cr * (one + O::div(s.gamma6 * (pstar - pr), pr)));
  const T ustar = h * (ul + O::div(pl - pstar, wl) + ur - O::div(pr - pstar, wr));
  const T sgnm = copysign(one, ustar);
  const bool lft = sgnm > zero;
  const T ro = lft ? rl : rr, uo = lft ? ul : ur, po = lft ? pl : pr, wo = lft ? wl : wr;
  const T co = O::mx(s.smallc, O::sqroot(O::ab(O::div(s.gamma0 * po, ro))));
  const T rstar = O::mx((O::div(ro, one + O::div(ro * (po - pstar), wo * wo))), s.smallr);
  const T cstar = O::mx(s.smallc, O::sqroot(O::ab(O::div(s.gamma0 * pstar, rstar))));
  T spout = co - sgnm * uo;
  T spin = cstar - sgnm * ustar;
  const T ushock = O::div(wo, ro) - sgnm * uo;
  if (pstar >= po) {
    spin = ushock;
    spout = ushock;
  }
  const T scr = O::mx(spout - spin, s.smallc + O::ab(spout + spin));
  T frac = h * (one + O::div(spout + spin, scr));
  if (frac != frac)
    frac = zero;
  else
    frac = frac >= one ? one : frac <= zero ? zero : frac;
  T gd = frac * rstar + (one - frac) * ro;
  T gu = frac * ustar + (one - frac) * uo;
  T gp = frac * pstar + (one - frac) * po;
  if (spout < zero) {
    gd = ro;
    gu = uo;
    gp = po;
  }
  if (spin > zero) {
    gd = rstar;
    gu = ustar;
    gp = pstar;
  }
  const T gv = lft ? qlf.v[tn] : qrf.v[tn];
  // cmpflx, HydroBaseFunctor.h:523-547
  const T fd = gd * gu;
  flux[ID] = fd;
  flux[ln] = fd * gu + gp;
  flux[tn] = fd * gv;
  const T ekin = h * gd * (gu * gu + gv * gv);
  const T etot = gp * s.entho + ekin;
  flux[IP] = gu * (etot + gp);
}

// solver chosen at compile time: RS = 0 approx, 1 hll, 2 hllc
// RS: 0 approx, 1 HLL, 2 HLLC; + kRiemannFloorSqrt: the bounded quotients and the short
// square root in the HLL / HLLC step and in its CFL rate (FP64, where
// SchemeT::floor_sqrt holds)
constexpr int kRiemannFloorSqrt = 8;
// + kMinmodPow2: the march is built for slope_type == 1 (its slopes) and for
// cell sizes that are powers of two (its CFL rate); the host selects such a
// kernel only then
constexpr int kMinmodPow2 = 16;
// + kSlopeMinmod: the march's slopes alone are built for slope_type == 1 (any
// cell sizes)
constexpr int kSlopeMinmod = 32;

// BND: the states are in the bounded ranges; ok is cleared in a lane whose flux
// may not have the IEEE bits
template <int RS, bool BND, class T>
__device__ __forceinline__ void riemann(const SchemeT<T> &s, const Q4T<T> &ql, const Q4T<T> &qr,
                                        int ln, int tn, T flux[4], bool &ok) {
  constexpr int kind = RS & 7;
  constexpr bool fs = (RS & kRiemannFloorSqrt) != 0;
  if constexpr (kind == 2)
    hllc<fs, BND>(s, ql, qr, ln, tn, flux, ok);
  else if constexpr (kind == 1)
    hll<fs, BND>(s, ql, qr, ln, tn, flux);
  else
    approx(s, ql, qr, ln, tn, flux);
}

template <int RS, class T>
__device__ __forceinline__ void riemann(const SchemeT<T> &s, const Q4T<T> &ql, const Q4T<T> &qr,
                                        int ln, int tn, T flux[4]) {
  bool ok = true;
  riemann<RS, false>(s, ql, qr, ln, tn, flux, ok);
}

}  // namespace e2d
