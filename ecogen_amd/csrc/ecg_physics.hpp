// Device physics of the explicit finite-volume step (gfx950).
//
// Face work (EOS evaluations, MUSCL reconstruction, Riemann solvers) is
// templated on the arithmetic type R: double for the plain FP64 path, float
// for the FP32 form.  The cell update (conservative variables, primitive
// rebuild, pressure relaxation, energy correction) is always FP64.  Every
// expression keeps the association order of the reference expression it
// evaluates (built with -ffp-contract=off) so that the FP64 path reproduces the
// reference's CPU arithmetic.
//
// Reference files (paths relative to the reference src/):
//   EOS             Eos/EosSG.cpp:66-257, Eos/EosIG.cpp:64-255
//   HLLC            Models/Euler/ModEuler.cpp:105-221, Models/UEq/ModUEq.cpp:113-268
//   wall            Models/Euler/ModEuler.cpp:368-409, Models/UEq/ModUEq.cpp:452-493
//   cons/prim       Models/Euler/FluxEuler.cpp:113-150, Models/UEq/FluxUEq.cpp:147-207
//   non-conservative Models/UEq/FluxUEq.cpp:224-244, Models/PUEq/FluxPUEq.cpp:44-65
//   scheme corr.    Models/UEq/FluxUEq.cpp:248-269 (VELOCITYEQ only)
//   energy corr.    Models/PUEq/FluxPUEq.cpp:68-116
//   relaxation      Relaxations/RelaxationPInfinite.cpp:43-98, Relaxations/RelaxationP.cpp:43-93
//   limiters        Order2/Limiter*.cpp
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ecg {

enum { M_EULER = 0, M_PUEQ = 1, M_UEQ = 2 };
enum { LIM_NONE = 0, LIM_MINMOD = 1, LIM_VANLEER = 2, LIM_VANALBADA = 3, LIM_SUPERBEE = 4, LIM_MC = 5, LIM_THINC = 6 };
enum { BC_NONREFLECTING = 0, BC_WALL = 1, BC_TANK = 2 };

struct EosDev {
  int sg;          // 1: stiffened gas, 0: ideal gas
  double g;        // gamma
  // An ideal gas is a stiffened gas of pinf = gpinf = 0: adding or subtracting zero
  // changes no pressure, so the formulas of both take one form without a select on sg
  // (the selects cost four instructions per phase of every derived state).
  double pinf;     // SG p_infinity (0 for IG)
  double gm1;      // gamma - 1
  double gpinf;    // gamma * p_infinity
  double eref;
  double mixg;     // gamma*pinf/(gamma-1) (IG: 0)   EosSG.cpp:208-214
  double mixinv;   // 1/(gamma-1)
  double pclamp;   // pressure floor: SG -(1-1e-15)*pinf + 1e-15, IG 1e-8
  // The same constants rounded to float (round to nearest, as a conversion on the
  // device rounds): the FP32 kernels read these instead of converting per use.
  float fg, fpinf, fgm1, fgpinf, feref, fmixinv, fpclamp;
};

// Stagnation tank of an inletTank side (BoundCondInletTank.cpp:37-165) with the
// constants the model's tank solver derives from it (ModUEq.cpp:562-569,
// ModEuler.cpp:474-476), computed on the host: phase densities at (p0, T0), the
// tank's mass fractions and its total enthalpy.
struct TankDev {
  double p0, H0;
  double rhok0[4], Yk0[4];
};

// One warning of RelaxationP::NewtonRaphson (RelaxationP.cpp:62-68): a relaxation
// that spent its 100 Newton iterations with |p*| > 1e-7, appended by the step
// kernels to a bounded per-context log.
struct WarnRec {
  int64_t iteration;   // steps completed before the one that warned
  int64_t cell;
  int stage;           // 0 first-order step, 1 predictor, 2 corrector
  int kind;            // 0: Newton not converged
  double value;        // |f| after the last iteration
};

// Bounds of the phases' volume fractions and densities (verify_correct): a value past
// alo / ahi becomes alo_v / ahi_v, a density below 1e-15 rho_v.  One form for both
// settings of alphaNull: as branches the two forms broke every face's extrapolation into a
// dozen blocks.
struct CellFloors {
  double alo, alo_v, ahi, ahi_v, rho_v;
  float f_alo, f_alo_v, f_ahi, f_ahi_v, f_rho_v, pad;
};

// The three distances of interior face m of an axis with cell size d, cells m | m + 1
// (Element.cpp:77-81, Face.cpp:52-56): which = 0 centre to centre, 1 face to the left
// centre, 2 face to the right centre.  Centres at (i + 0.5) d (MeshCartesian.cpp:178).
// The reference's sqrt(x^2 + 0 + 0) of the coordinate difference is |x| exactly: the
// rounded square's root rounds to |x| unless the square under- or overflows.  The kernels
// evaluate it where an axis has no single value: a table cost a memory latency at every
// slope and two, one after the other, at every face (this and the unconditional reads of the
// second slope: 3D two-phase O2 at 93 x 95 x 91 FP64 442 -> 406 us, 119 x 113 x 117 FP32
// 376 -> 329).
__host__ __device__ inline double face_distance(double d, int m, int which) {
  const double pm = (m + 0.5) * d, pp = (m + 1 + 0.5) * d;
  const double fp = pm + 0.5 * d;
  return fabs((which == 0) ? pm - pp : (which == 1) ? fp - pm : fp - pp);
}

struct Params {
  int nx, ny, nz;
  int64_t ncell;
  int64_t pitch;            // elements between two SoA variables
  double d[3];              // cell sizes
  double coef[3];           // face surface / cell volume per axis
  double lcfl;              // CFL length
  double eps;               // epsilonAlphaNull
  double cfl;
  int alpha_null;
  int relax;                // pressure relaxation active
  int bc[6];
  int lim[4];
  int tiles[3];             // tiles per axis
  EosDev eos[4];
  CellFloors floors;
  // Axes whose three face distances (face_distance) are each one value (the uniform meshes a power-of-two
  // cell count spans exactly): bit a of dist_uniform, the values, and bit a of dcc_pow2 when
  // the cell-to-cell distance is a power of two, so that dividing by it is multiplying by
  // its exact inverse inv_dcc.
  int dist_uniform, dcc_pow2;
  double dcc_c[3], dfl_c[3], dfr_c[3], inv_dcc[3];
  double dwall[3][2];       // first / last cell centre to its boundary face, per axis
  // Float copies (rounded to nearest) of coef, eps, the uniform-axis distances and
  // dwall, for the FP32 kernels.
  float f_coef[3], f_eps, f_dcc_c[3], f_dfl_c[3], f_dfr_c[3], f_inv_dcc[3], f_dwall[3][2];
  double relax_mu;          // > 0: finite-rate pressure relaxation with this rate (VELOCITYEQ)
  int thinc;                // a volume-fraction limiter is THINC (two phases)
  double thinc_cosh, thinc_tanh;   // cosh(1.6), tanh(1.6) of the host's libm
  TankDev tank[6];          // sides whose bc is BC_TANK
  double* tank_buf;         // flux records of the tank faces, TANK_REC doubles each (k_tank)
  int64_t tank_off[6];      // first record of each tank side; faces of a side in plane order
  WarnRec* warn_rec;        // warning log (warn_cap records) and its append counter
  unsigned long long* warn_cnt;
  int64_t warn_cap;
};

// Flux record of one inlet-tank face (alpha, mass, energ per phase up to 4
// phases, momentum in the global frame, mixture energy, sM, uStar).
constexpr int TANK_REC = 3 * 4 + 6;
// Faces of boundary side `side` (0..5 = x-, x+, y-, y+, z-, z+).
inline int64_t tank_faces(const Params& P, int side) {
  const int ax = side >> 1;
  return (ax == 0) ? (int64_t)P.ny * P.nz : (ax == 1) ? (int64_t)P.nx * P.nz : (int64_t)P.nx * P.ny;
}

// Device clock: lagged time step kept on the GPU (Run.cpp:385-498).
struct Clock {
  double t, dt, dt_next, dt_max;
  double t_end;
  int64_t iteration, max_iter;
  int done;
  int fatal;                          // 1: the clock stopped after a step that left an error
  unsigned long long fatal_seen;      // tank_fail + nonfinite over the slots when last checked
};

// Per-step reductions of the step kernels.  Blocks spread their atomics over
// ATOMIC_SLOTS slots, one 128-byte line each (block b uses slot b % ATOMIC_SLOTS),
// so that half a million blocks per launch do not serialise on one line; the
// clock kernel reduces the dtMax slots, the host sums the counters.
constexpr int ATOMIC_SLOTS = 64;
struct Counters {
  unsigned long long newton_fail, newton_iters, relax_calls;
  unsigned long long warm_calls;      // relaxations started from the learned guess
  unsigned long long warm_fallbacks;  // of those, WARM_MAX_IT evaluations short of the tolerance
  double resid_sum;                   // sum over relaxed cells of |f| at exit
  uint64_t dtmax_bits;                // min of the step's dtMax (non-negative doubles order as integers)
  unsigned long long tank_fail;       // inlet-tank Newton solves that spent 50 iterations
  unsigned long long newton_warn;     // of newton_fail, those the reference warns about (|p*| > 1e-7)
  unsigned long long nonfinite;       // cells whose new state holds a non-finite value
  uint64_t pad[6];
};

static_assert(sizeof(Counters) == 128, "one counter slot per 128-byte line");

// std::min / std::max tie semantics.
template <typename R> __device__ __forceinline__ R dmin(R a, R b) { return (b < a) ? b : a; }
template <typename R> __device__ __forceinline__ R dmax(R a, R b) { return (a < b) ? b : a; }
// A parameter in the kernel's arithmetic type: the double, or its float copy.
template <typename R> __device__ __forceinline__ R pv(double d, float f) {
  if constexpr (sizeof(R) == 4) return f; else return d;
}

// Division, square root and power of the face work.  double: the IEEE
// operations (the FP64 path keeps the reference's correctly rounded results).
// float: the hardware reciprocal, square root, log2 and exp2 (about 1 ulp
// each), since the FP32 form's error is set by FP32 storage of the state, not
// by the last bit of these operations.
__device__ __forceinline__ double fdiv(double a, double b) { return a / b; }
__device__ __forceinline__ float fdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ double fsqrt(double x) { return sqrt(x); }
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ double fpow(double x, double y) { return pow(x, y); }
__device__ __forceinline__ float fpow(float x, float y) { return __builtin_amdgcn_exp2f(y * __builtin_amdgcn_logf(x)); }

// The IEEE quotient a / b as the device's division sequence forms it: the
// reciprocal estimate refined by two Newton steps (rcp_ieee), the product, and one
// residual correction (div_ieee).  One rcp_ieee(b) serves every quotient by the
// same b at a product and two FMAs each, instead of the whole sequence per
// quotient, with bit-identical results: the sequence's pre-scaling and fix-up
// act only on operands within a few binades of overflow or underflow and on
// zeros, infinities and NaNs, none of which the face and cell arithmetic divides
// by (multiphase densities and masses are floored, wave-speed differences are nonzero; Euler's
// density is not, and its quotients take the fix-up: derive, build_prim).
__device__ __forceinline__ double rcp_ieee(double b) {
  const double r0 = __builtin_amdgcn_rcp(b);
  const double r1 = fma(r0, fma(-b, r0, 1.), r0);
  return fma(r1, fma(-b, r1, 1.), r1);
}
// rb may also be the correctly rounded 1/b (the host's quotient): the correction
// step then gives the IEEE quotient as well (Markstein), which the quotients by
// gamma - 1 use with the host's 1/(gamma - 1), EosDev::mixinv.
__device__ __forceinline__ double div_ieee(double a, double b, double rb) {
  const double q = a * rb;
  return fma(fma(-b, q, a), rb, q);
}
// A single quotient by the same sequence (no pre-scaling and fix-up steps).
__device__ __forceinline__ double div1(double a, double b) { return div_ieee(a, b, rcp_ieee(b)); }
// The same with the hardware's fix-up, which gives the special values of zero, infinite and NaN
// operands: for the quotients whose operands a broken state reaches (its cells are reported, and
// what it leaves in their neighbours follows the IEEE quotient).
__device__ __forceinline__ double div_special(double a, double b, double rb) {
  return __builtin_amdgcn_div_fixup(div_ieee(a, b, rb), b, a);
}
// Quotients by one divisor.
template <typename R> struct Quot;
template <> struct Quot<double> {
  double b, rb;
  __device__ __forceinline__ explicit Quot(double d) : b(d), rb(rcp_ieee(d)) {}
  __device__ __forceinline__ double operator()(double a) const { return div_special(a, b, rb); }
};
template <> struct Quot<float> {
  float rb;
  __device__ __forceinline__ explicit Quot(float d) : rb(__builtin_amdgcn_rcpf(d)) {}
  __device__ __forceinline__ float operator()(float a) const { return a * rb; }
};
// Quotients by one divisor that may be zero, infinite, NaN or subnormal (Euler densities carry
// no floor): tiny divisors are scaled into the reciprocal's range, exactly, and the hardware's
// fix-up gives the special values.
struct QuotFull {
  double s, b, rb;
  __device__ __forceinline__ explicit QuotFull(double d) : s(fabs(d) < 1.e-290 ? 0x1p512 : 1.), b(d * s), rb(rcp_ieee(b)) {}
  __device__ __forceinline__ double operator()(double a) const {
    return div_special(a, b, rb) * s;
  }
};
// The square root as the device's sequence forms it (reciprocal square-root
// estimate, one Goldschmidt step on the root and its half-reciprocal, two Newton
// corrections), without the sequence's scaling of arguments below 2^-767 and its
// zero / infinity selects: the same bits for the sound speeds' arguments, which
// the pressure and density floors keep far above 2^-767.  The estimate is capped
// so that a zero argument still gives zero.
__device__ __forceinline__ double sqrt_pos(double x) {
  const double g0 = fmin(__builtin_amdgcn_rsq(x), 1.e300);
  double s = x * g0, h = 0.5 * g0;
  const double r = fma(-h, s, 0.5);
  s = fma(s, r, s);
  h = fma(h, r, h);
  double d = fma(-s, s, x);
  s = fma(d, h, s);
  d = fma(-s, s, x);
  return fma(d, h, s);
}
// A quotient of the Riemann solvers: div1 in FP64, the reciprocal estimate in FP32.
__device__ __forceinline__ double qdiv(double a, double b) { return div1(a, b); }
__device__ __forceinline__ float qdiv(float a, float b) { return fdiv(a, b); }

// Correctly rounded exp (round to nearest) for -708 < x < 709.78: x = k ln2 + r
// with ln2 and r in double-double, exp(r) by the nested form
// 1 + r (1 + r/2 (1 + r/3 (...))) in double-double (about 2^-100 relative), then
// one rounding and an exact scaling by 2^k.  The THINC reconstruction uses it so
// that its result does not depend on a math library's last-bit behaviour.
struct DD { double hi, lo; };
__host__ __device__ inline DD dd_fast_two_sum(double a, double b) {
  const double s = a + b;
  return DD{s, b - (s - a)};
}
__host__ __device__ inline DD dd_two_sum(double a, double b) {
  const double s = a + b, bb = s - a;
  return DD{s, (a - (s - bb)) + (b - bb)};
}
__host__ __device__ inline DD dd_mul(DD a, DD b) {
  const double p = a.hi * b.hi;
  double e = fma(a.hi, b.hi, -p);
  e += a.hi * b.lo + a.lo * b.hi;
  return dd_fast_two_sum(p, e);
}
__host__ __device__ inline DD dd_div_int(DD a, double n) {
  const double q1 = a.hi / n;
  const double rem = fma(-q1, n, a.hi);   // exact
  const double q2 = (rem + a.lo) / n;
  return dd_fast_two_sum(q1, q2);
}
__host__ __device__ inline DD dd_add_one(DD a) {
  DD s = dd_two_sum(a.hi, 1.);
  s.lo += a.lo;
  return dd_fast_two_sum(s.hi, s.lo);
}
// exp of a double-double argument z (|z.hi| < 708) as 2^k times a double-double
// (about 2^-100 relative): z = k ln2 + r, exp(r) by the nested series.
__host__ __device__ inline DD exp_dd(DD z, int& k_out) {
  const double LN2_HI = 0x1.62e42fefa39efp-1, LN2_LO = 0x1.abc9e3b39803fp-56;
  const double k = rint(z.hi * 0x1.71547652b82fep0);
  const double p_hi = k * LN2_HI;
  const double p_lo = fma(k, LN2_HI, -p_hi);        // k LN2_HI = p_hi + p_lo exactly
  const DD s = dd_two_sum(z.hi, -p_hi);
  const DD r = dd_fast_two_sum(s.hi, ((s.lo - p_lo) + z.lo) - k * LN2_LO);
  DD acc = DD{1., 0.};
  for (int n = 24; n >= 1; n--) acc = dd_add_one(dd_div_int(dd_mul(r, acc), (double)n));
  k_out = (int)k;
  return acc;
}
__host__ __device__ inline double exp_cr(double x) {
  if (!(x == x)) return x;
  if (x >= 709.79) return 1. / 0.;
  if (x <= -708.) return 0.;
  int k;
  const DD e = exp_dd(DD{x, 0.}, k);
  return ldexp(e.hi, k);
}

// Correctly rounded pow (round to nearest) for a positive finite base and a result
// between 2^-1020 and 2^1020: log x in double-double by one Newton step on exp from
// the library's log (log x = l0 + log(x e^-l0), x e^-l0 = 1 + d with |d| ~ 2^-52),
// t = y log x in double-double, exp(t) in double-double, one rounding.  Other
// arguments take the library's pow.  The relaxation paths whose hard thresholds
// amplify a last-bit difference (the finite-rate relaxation) use it, so that their
// results do not depend on a math library's rounding.
__host__ __device__ inline double pow_cr(double x, double y) {
  if (!(x > 0.) || !(x < 1.e308) || !(fabs(y) < 1.e300)) return pow(x, y);
  if (x == 1. || y == 0.) return 1.;
  const double l0 = log(x);
  int k;
  const DD e = exp_dd(DD{-l0, 0.}, k);                 // exp(-l0) = e 2^k
  const double xs = ldexp(x, k);                        // exact: x 2^k is near 1 / e
  const DD xe = dd_mul(DD{xs, 0.}, e);                  // x exp(-l0) = 1 + d
  DD d = dd_two_sum(xe.hi, -1.);
  d = dd_fast_two_sum(d.hi, d.lo + xe.lo);
  DD L = dd_two_sum(l0, d.hi);                          // log(1 + d) = d - d^2/2 + ...
  L = dd_fast_two_sum(L.hi, L.lo + (d.lo - 0.5 * d.hi * d.hi));
  const DD t = dd_mul(DD{y, 0.}, L);
  if (!(t.hi > -700. && t.hi < 700.)) return pow(x, y);
  int kk;
  const DD r = exp_dd(t, kk);
  return ldexp(r.hi, kk);
}

// Natural logarithm for the FP64 star isentropes outside the full-featured
// kernels: x = m 2^e with m in [1/sqrt(2), sqrt(2)), log m = 2 atanh(u),
// u = (m - 1)/(m + 1), |u| < 0.1716, by the Taylor series of atanh through u^21 (the
// next term is below 2^-60 of the sum), plus e ln 2 with ln 2 split in two doubles
// (the first with 32 significant bits, so that e ln2_hi is exact).  Within 2 ulp of
// the exact logarithm for positive finite x; zero, negative, infinite and NaN
// arguments give what the library's log gives, by selects (no second logarithm in
// the code).
__host__ __device__ inline double log_pos(double x) {
  int e;
  double m = frexp(x, &e);                       // x = m 2^e, m in [0.5, 1)
  if (m < 0.70710678118654752) { m = 2. * m; e -= 1; }
  const double u = (m - 1.) / (m + 1.);           // m - 1 is exact
  const double u2 = u * u;
  double s = 1. / 21.;
  s = fma(s, u2, 1. / 19.);
  s = fma(s, u2, 1. / 17.);
  s = fma(s, u2, 1. / 15.);
  s = fma(s, u2, 1. / 13.);
  s = fma(s, u2, 1. / 11.);
  s = fma(s, u2, 1. / 9.);
  s = fma(s, u2, 1. / 7.);
  s = fma(s, u2, 1. / 5.);
  s = fma(s, u2, 1. / 3.);
  const double t = 2. * u;                         // 2 atanh(u) = t (1 + u2 s)
  const double lm = fma(t * u2, s, t);
  const double de = (double)e;
  const double r = fma(de, 0x1.62e42ff000000p-1, fma(de, -0x1.718432a1b0e26p-35, lm));
  if (!(x > 0.)) return (x == 0.) ? -__builtin_inf() : __builtin_nan("");
  return (x == __builtin_inf()) ? x : r;
}

// ---------------------------------------------------------------------------
// EOS
// ---------------------------------------------------------------------------
template <typename R>
__device__ __forceinline__ R eos_energy(const EosDev& q, R eps, R rho, R p) {
  if constexpr (sizeof(R) == 8) {
    const double rr = dmax<double>(rho, eps);
    return div_ieee(div_ieee(p + q.gpinf, q.gm1, q.mixinv), rr, rcp_ieee(rr)) + q.eref;
  }
  return fdiv(fdiv(p + pv<R>(q.gpinf, q.fgpinf), pv<R>(q.gm1, q.fgm1)), dmax<R>(rho, eps)) + pv<R>(q.eref, q.feref);
}
template <typename R>
__device__ __forceinline__ R eos_pressure(const EosDev& q, R rho, R e) {
  R v = pv<R>(q.gm1, q.fgm1) * rho * (e - pv<R>(q.eref, q.feref));
  return v - pv<R>(q.gpinf, q.fgpinf);
}
template <typename R>
__device__ __forceinline__ R eos_sound(const EosDev& q, R eps, R rho, R p) {
  return fsqrt(fdiv(pv<R>(q.g, q.fg) * (p + pv<R>(q.pinf, q.fpinf)), dmax<R>(rho, eps)));
}

// EosSG/EosIG::computeDensityTimesInterfaceSoundSpeedSquare (EosSG.cpp:115-118, EosIG.cpp:113-116)
__device__ __forceinline__ double eos_rho_ci2(const EosDev& q, double pI, double p) {
  return q.sg ? q.gm1 * pI + p + q.gpinf : q.gm1 * pI + p;
}
// CRPOW: the correctly rounded pow (FP64 kernels of the full-featured instantiation).
template <typename R, bool CRPOW = false>
__device__ __forceinline__ R eos_p_isentropic(const EosDev& q, R eps, R p0, R rho0, R rhof) {
  R base;
  if constexpr (sizeof(R) == 8) {
    const double r0 = dmax<double>(rho0, eps), x = div_ieee(rhof, r0, rcp_ieee(r0));
    base = CRPOW ? pow_cr(x, q.g) : pow(x, q.g);
  } else {
    base = fpow(fdiv(rhof, dmax<R>(rho0, eps)), pv<R>(q.g, q.fg));
  }
  return (p0 + pv<R>(q.pinf, q.fpinf)) * base - pv<R>(q.pinf, q.fpinf);
}
template <typename R>
__device__ __forceinline__ R eos_clamp_p(const EosDev& q, R p) {
  return (p <= pv<R>(q.pclamp, q.fpclamp)) ? pv<R>(q.pclamp, q.fpclamp) : p;
}
// Tools::returnNonZeroValue (Tools.cpp:134-145)
__device__ __forceinline__ double nonzero(double a, double eps) {
  if (a > eps || a < -eps) return a;
  return (double)((0. < a) - (a < 0.)) * eps;
}
// computeDensityPfinal (EosSG.cpp:163-170, EosIG.cpp:161-168); FP64 only (relaxation).
__device__ __forceinline__ double eos_rho_pfinal(const EosDev& q, double eps, double p0, double rho0, double pf) {
  double num = q.g * (pf + q.pinf);
  double denom = num + p0 - pf;
  return div1(rho0 * num, q.sg ? nonzero(denom, eps) : dmax(denom, eps));
}
// Its derivative d rho / d pf.
__device__ __forceinline__ double eos_drhodp_pfinal(const EosDev& q, double eps, double p0, double rho0, double pf) {
  double num = q.g * (pf + q.pinf);
  double denom = num + p0 - pf;
  return div1(rho0 * q.g * (p0 + q.pinf), dmax(denom * denom, eps));
}

// computeDensityHugoniot (EosSG.cpp:152-159, EosIG.cpp:150-157); FP64 only (tank boundary).
__device__ __forceinline__ double eos_rho_hugoniot(const EosDev& q, double eps, double p0, double rho0, double pf) {
  const double P0 = q.sg ? p0 + q.pinf : p0, Pf = q.sg ? pf + q.pinf : pf;
  const double num = (q.g + 1.) * Pf + (q.g - 1.) * P0;
  const double denom = (q.g - 1.) * Pf + (q.g + 1.) * P0;
  return rho0 * num / dmax(denom, eps);
}
// computeDensityIsentropic (EosSG.cpp:143-148, EosIG.cpp:141-146) with d rho / dp.
__device__ __forceinline__ double eos_rho_isentropic(const EosDev& q, double eps, double p0, double rho0, double pf,
                                                     double& drhodp) {
  const double P0 = q.sg ? p0 + q.pinf : p0, Pf = q.sg ? pf + q.pinf : pf;
  const double rhof = rho0 * pow(Pf / dmax(P0, eps), 1. / q.g);
  drhodp = rhof / dmax(q.g * Pf, eps);
  return rhof;
}
// computeEnthalpyIsentropic (EosSG.cpp:174-181, EosIG.cpp:172-179) with d h / dp.
__device__ __forceinline__ double eos_h_isentropic(const EosDev& q, double eps, double p0, double rho0, double pf,
                                                   double& rhof, double& dhdp) {
  double drho;
  rhof = eos_rho_isentropic(q, eps, p0, rho0, pf, drho);
  const double Pf = q.sg ? pf + q.pinf : pf;
  dhdp = q.g / (q.g - 1.) * (rhof - Pf * drho) / dmax(rhof * rhof, eps);
  return q.g * Pf / (q.g - 1.) / dmax(rhof, eps) + q.eref;
}

// ---------------------------------------------------------------------------
// Limiters (Order2/LimiterMinmod.cpp:46-56, LimiterVanLeer.cpp:43-49,
// LimiterVanAlbada.cpp:43-51, LimiterSuperBee.cpp:46-55, LimiterMC.cpp:43-53)
// ---------------------------------------------------------------------------
template <typename R>
__device__ __forceinline__ R limit(int kind, R s1, R s2) {
  R prod = s1 * s2, out = R(0.);
  if (kind == LIM_MINMOD || kind == LIM_THINC) {   // LimiterTHINC::limiteSlope is minmod
    // sign(s1) min(|s1|, |s2|) where s1 s2 > 1e-9: slopes of one sign, so the value
    // is the slope of smaller magnitude (FP32: their median with 0, one v_med3).
    R m;
    if constexpr (sizeof(R) == 4) m = __builtin_amdgcn_fmed3f(s1, s2, 0.f);
    else m = (fabs(s2) < fabs(s1)) ? s2 : s1;
    out = (prod > R(1e-9)) ? m : R(0.);
  } else if (kind == LIM_VANLEER) {
    R sum = s1 + s2;
    // The quotient always, then a select: no mask and branch around every variable's.
    const R q = Quot<R>(sum)(R(2.) * prod);
    out = ((fabs(sum) > R(1e-6)) && (prod > R(1e-6))) ? q : R(0.);
  } else if (kind == LIM_VANALBADA) {
    R sum = s1 + s2;
    const R q = Quot<R>(s1 * s1 + s2 * s2)(prod * sum);
    out = ((fabs(s1) > R(1e-6)) && (fabs(s2) > R(1e-6)) && (fabs(sum) > R(1e-6)) && (prod > R(1e-6))) ? q : R(0.);
  } else if (kind == LIM_SUPERBEE) {
    if (prod > R(1e-6)) out = dmax<R>(dmin<R>(R(2.) * fabs(s1), fabs(s2)), dmin<R>(fabs(s1), R(2.) * fabs(s2)));
    if (s1 < R(0.)) out = -out;
  } else if (kind == LIM_MC) {
    if (prod > R(1e-9)) {
      out = dmin<R>(R(2.) * fabs(s1), R(2.) * fabs(s2));
      out = dmin<R>(out, R(0.5) * (fabs(s1) + fabs(s2)));
    }
    if (s1 < R(0.)) out = -out;
  }
  return out;
}


// THINC volume fraction of a cell at an interface face (CellInterfaceO2Cartesian.cpp:
// 133-149 for the face's left cell, side 0; 165-180 for its right cell, side 1):
// a is the cell's alpha, a_after the alpha beyond its opposite face, a_other the
// alpha across the face.  Returns false where the interface test fails.
__device__ __forceinline__ bool thinc_alpha(const Params& P, int side, double a, double a_after, double a_other,
                                            double& out) {
  const double beta = 1.6, epsI = 1.e-4;
  if (!((a >= epsI) && (a <= 1. - epsI) && ((a_other - a) * (a - a_after) >= 1.e-8))) return false;
  const double hi = (side == 0) ? a_other : a_after, lo = (side == 0) ? a_after : a_other;
  const double sign = (hi - lo > 0.) ? 1. : -1.;
  const double qmin = dmin<double>(hi, lo);
  const double qmax = dmax<double>(hi, lo) - qmin;
  const double C = (a - qmin + 1.e-20) / (qmax + 1.e-20);
  const double B = exp_cr(sign * beta * (2. * C - 1.));
  const double A = (B / P.thinc_cosh - 1.) / P.thinc_tanh;
  double na = (side == 0) ? qmin + 0.5 * qmax * (1. + sign * (P.thinc_tanh + A) / (1. + A * P.thinc_tanh))
                          : qmin + 0.5 * qmax * (1. + sign * A);
  if (na < epsI) na = epsI;
  if (na > 1. - epsI) na = 1. - epsI;
  out = na;
  return true;
}

// ---------------------------------------------------------------------------
// State
// ---------------------------------------------------------------------------
// Persistent primitives plus derived quantities of one cell.  For Euler only
// index 0 of the phase arrays is used (a[0] unused).
template <int N, typename R = double>
struct Cell {
  R a[N], r[N], p[N];
  R e[N], c[N];
  R u[3];
  R rho, pm, em, cF;
  R E;
};

template <int N, typename R = double>
struct Cons {
  R alpha[N], mass[N], energ[N];
  R mom[3];
  R energM;
};

template <int N, typename R = double>
struct Flux {
  Cons<N, R> f;
  R sM, uStar;
};

// Face frames: local (n, t, b) components are a signed permutation of the
// global velocity (MeshCartesian.cpp:282, 315, 348, 387, 411, 440, 482, 511, 535).
enum { FR_XI = 0, FR_YI, FR_ZI, FR_XM, FR_XP, FR_YM, FR_YP, FR_ZM, FR_ZP };
template <int FR> struct Frame;
template <> struct Frame<FR_XI> { static constexpr int i0 = 0, i1 = 1, i2 = 2; static constexpr int s0 = 1, s1 = 1, s2 = 1; };
template <> struct Frame<FR_XP> { static constexpr int i0 = 0, i1 = 1, i2 = 2; static constexpr int s0 = 1, s1 = 1, s2 = 1; };
template <> struct Frame<FR_XM> { static constexpr int i0 = 0, i1 = 1, i2 = 2; static constexpr int s0 = -1, s1 = -1, s2 = 1; };
template <> struct Frame<FR_YI> { static constexpr int i0 = 1, i1 = 0, i2 = 2; static constexpr int s0 = 1, s1 = -1, s2 = 1; };
template <> struct Frame<FR_YP> { static constexpr int i0 = 1, i1 = 0, i2 = 2; static constexpr int s0 = 1, s1 = -1, s2 = 1; };
template <> struct Frame<FR_YM> { static constexpr int i0 = 1, i1 = 0, i2 = 2; static constexpr int s0 = -1, s1 = 1, s2 = 1; };
template <> struct Frame<FR_ZI> { static constexpr int i0 = 2, i1 = 0, i2 = 1; static constexpr int s0 = 1, s1 = 1, s2 = 1; };
template <> struct Frame<FR_ZP> { static constexpr int i0 = 2, i1 = 0, i2 = 1; static constexpr int s0 = 1, s1 = 1, s2 = 1; };
template <> struct Frame<FR_ZM> { static constexpr int i0 = 2, i1 = 0, i2 = 1; static constexpr int s0 = -1, s1 = -1, s2 = 1; };

template <int FR, typename R>
__device__ __forceinline__ void to_local(const R* u, R* l) {
  using F = Frame<FR>;
  l[0] = F::s0 < 0 ? -u[F::i0] : u[F::i0];
  l[1] = F::s1 < 0 ? -u[F::i1] : u[F::i1];
  l[2] = F::s2 < 0 ? -u[F::i2] : u[F::i2];
}
template <int FR, typename R>
__device__ __forceinline__ void to_global(const R* l, R* g) {
  using F = Frame<FR>;
  g[F::i0] = F::s0 < 0 ? -l[0] : l[0];
  g[F::i1] = F::s1 < 0 ? -l[1] : l[1];
  g[F::i2] = F::s2 < 0 ? -l[2] : l[2];
}

template <typename R>
__device__ __forceinline__ R sqn3(const R* u) { return u[0] * u[0] + u[1] * u[1] + u[2] * u[2]; }

// PhaseUEq::extendedCalculusPhase + MixUEq::computeMixtureVariables; Euler:
// PhaseEuler::extendedCalculusPhase (also rebuilds E when rebuildE).
template <int MODEL, int N, typename R>
__device__ __forceinline__ void derive(const Params& P, Cell<N, R>& s, bool rebuildE) {
  const R eps = pv<R>(P.eps, P.f_eps);
  if (MODEL == M_EULER) {
    if constexpr (sizeof(R) == 8) {
      // One reciprocal of the density for the energy and the squared sound speed.  Euler
      // densities and pressures carry no floor: a vacuum's sound speed is infinite, which makes the
      // step's dtMax zero, so the hardware's fix-up gives the quotient by a zero density and the
      // library's root the special values.  (The lean root with a test of its range before the
      // library's: 121 x 119 x 117 first order 96 us a step, this 88; with second-order walls
      // 357 / 343.)  The fix-up's divisor is scaled so that a density whose reciprocal overflows
      // rounds to the zero of its sign (-0 has no sound speed, as in the reference).
      const EosDev& q = P.eos[0];
      const double rr = dmax<double>(s.r[0], eps), ir = rcp_ieee(rr), cn = q.g * (s.p[0] + q.pinf);
      s.e[0] = div_ieee(div_ieee(s.p[0] + q.gpinf, q.gm1, q.mixinv), rr, ir) + q.eref;
      s.c[0] = sqrt(__builtin_amdgcn_div_fixup(div_ieee(cn, rr, ir), rr * 0x1p-51, cn));
    } else {
      s.e[0] = eos_energy<R>(P.eos[0], eps, s.r[0], s.p[0]);
      s.c[0] = eos_sound<R>(P.eos[0], eps, s.r[0], s.p[0]);
    }
    if (rebuildE) s.E = s.e[0] + R(0.5) * sqn3<R>(s.u);
    return;
  }
  if constexpr (sizeof(R) == 4) {
    // FP32 form: one reciprocal per phase density serves its energy and its squared
    // sound speed, one of the mixture density the mass fractions, and only the frozen
    // mixture sound speed takes a square root (the phase sound speeds enter the face
    // solvers only through it).
    R rho = R(0.), pm = R(0.), c2[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
      const EosDev& q = P.eos[k];
      const R ir = __builtin_amdgcn_rcpf(dmax<R>(s.r[k], eps));
      s.e[k] = (s.p[k] + pv<R>(q.gpinf, q.fgpinf)) * pv<R>(q.mixinv, q.fmixinv) * ir + pv<R>(q.eref, q.feref);
      c2[k] = pv<R>(q.g, q.fg) * (s.p[k] + pv<R>(q.pinf, q.fpinf)) * ir;
      rho += s.a[k] * s.r[k];
      pm += s.a[k] * s.p[k];
    }
    const R iden = __builtin_amdgcn_rcpf(dmax<R>(rho, eps));
    R em = R(0.), cf = R(0.);
#pragma unroll
    for (int k = 0; k < N; k++) {
      const R Y = s.a[k] * s.r[k] * iden;
      em += Y * s.e[k];
      cf += Y * c2[k];
    }
    s.rho = rho; s.pm = pm; s.em = em; s.cF = fsqrt(cf);
    return;
  }
  // FP64: the reference's quotients, the phase energy and sound speed sharing one
  // reciprocal of the density and the mass fractions one of the mixture density.
#pragma unroll
  for (int k = 0; k < N; k++) {
    const EosDev& q = P.eos[k];
    const double rr = dmax<double>(s.r[k], eps), ir = rcp_ieee(rr);
    s.e[k] = div_ieee(div_ieee(s.p[k] + q.gpinf, q.gm1, q.mixinv), rr, ir) + q.eref;
    s.c[k] = sqrt_pos(div_ieee(q.g * (s.p[k] + q.pinf), rr, ir));
  }
  double rho = 0., pm = 0.;
#pragma unroll
  for (int k = 0; k < N; k++) { rho += s.a[k] * s.r[k]; pm += s.a[k] * s.p[k]; }
  const double den = dmax<double>(rho, eps), iden = rcp_ieee(den);
  double em = 0., cf = 0.;
#pragma unroll
  for (int k = 0; k < N; k++) {
    const double Y = div_ieee(s.a[k] * s.r[k], den, iden);
    em += Y * s.e[k];
    cf += Y * s.c[k] * s.c[k];
  }
  s.rho = rho; s.pm = pm; s.em = em; s.cF = sqrt_pos(cf);
}

// Mixture density alone (the part of the derived state the cell update and the
// energy correction read), summed in derive's order.
template <int N>
__device__ __forceinline__ void mixture_density(Cell<N>& s) {
  double rho = 0.;
#pragma unroll
  for (int k = 0; k < N; k++) rho += s.a[k] * s.r[k];
  s.rho = rho;
}

// verifyAndCorrectPhase (PhaseUEq.cpp:355-370, PhaseEuler.cpp:395-399)
template <int MODEL, int N, typename R>
__device__ __forceinline__ void verify_correct(const Params& P, Cell<N, R>& s, int k) {
  if (MODEL == M_EULER) {
    if (s.r[0] < R(1.e-10)) s.r[0] = R(1.e-10);
    s.p[0] = eos_clamp_p<R>(P.eos[0], s.p[0]);
    return;
  }
  // With alphaNull: alpha to [0, 1], rho to 1e-15 at least; without: alpha to
  // [1e-14, 1 - 1e-14] where it passes 1e-15 of the ends, rho below 1e-15 to 1e-14.
  const CellFloors& q = P.floors;
  s.a[k] = (s.a[k] < pv<R>(q.alo, q.f_alo)) ? pv<R>(q.alo_v, q.f_alo_v) : s.a[k];
  s.a[k] = (s.a[k] > pv<R>(q.ahi, q.f_ahi)) ? pv<R>(q.ahi_v, q.f_ahi_v) : s.a[k];
  s.r[k] = (s.r[k] < R(1.e-15)) ? pv<R>(q.rho_v, q.f_rho_v) : s.r[k];
  s.p[k] = eos_clamp_p<R>(P.eos[k], s.p[k]);
}

// ---------------------------------------------------------------------------
// Riemann solvers in the face frame; lu = local velocity of each side.
// ---------------------------------------------------------------------------
template <typename R>
__device__ __forceinline__ void cfl_bound(R& dtm, R s, R dx) {
  if (fabs(s) > R(1.e-3)) dtm = dmin<R>(dtm, fdiv(R(1.) * dx, fabs(s)));
}
// The step kernels' form of the same bound.  Every face of a case shares one
// length lcfl, so the reference's dtMax = min over faces of lcfl / |s| (wave
// speeds above 1e-3 in magnitude) is lcfl / max |s|: a correctly rounded quotient
// falls as its divisor grows.  The solvers keep the largest speed; cfl_dt takes
// the quotient once per block.
template <typename R>
__device__ __forceinline__ void cfl_speed(R& smax, R s) {
  if (fabs(s) > R(1.e-3)) smax = dmax<R>(smax, fabs(s));
}
__device__ __forceinline__ double cfl_dt(double lcfl, double smax) {
  return (smax > 0.) ? dmin<double>(1.e10, lcfl / smax) : 1.e10;
}

// ModEuler::solveRiemannIntern
template <int N, typename R>
__device__ __forceinline__ void hllc_euler(const Cell<N, R>& Lc, const R* lu, const R EL, const Cell<N, R>& Rc,
                                           const R* ru, const R ER, R& smax, Flux<N, R>& F) {
  const R uL = lu[0], vL = lu[1], wL = lu[2], pL = Lc.p[0], rhoL = Lc.r[0], cL = Lc.c[0];
  const R uR = ru[0], vR = ru[1], wR = ru[2], pR = Rc.p[0], rhoR = Rc.r[0], cR = Rc.c[0];
  const R sL = dmin<R>(uL - cL, uR - cR);
  const R sR = dmax<R>(uR + cR, uL + cL);
  cfl_speed<R>(smax, sL);
  cfl_speed<R>(smax, sR);
  const R mL = rhoL * (sL - uL), mR = rhoR * (sR - uR);
  R sM = qdiv(pR - pL + mL * uL - mR * uR, mL - mR);
  if (fabs(sM) < R(1.e-8)) sM = R(0.);
  R mass, m0, m1, m2, en;
  if (sL > R(0.)) {
    mass = rhoL * uL; m0 = rhoL * uL * uL + pL; m1 = rhoL * vL * uL; m2 = rhoL * wL * uL; en = (rhoL * EL + pL) * uL;
  } else if (sR < R(0.)) {
    mass = rhoR * uR; m0 = rhoR * uR * uR + pR; m1 = rhoR * vR * uR; m2 = rhoR * wR * uR; en = (rhoR * ER + pR) * uR;
  } else {
    const bool left = (sM >= R(0.));
    const R mS = left ? mL : mR, uS = left ? uL : uR, pS = left ? pL : pR, sS = left ? sL : sR;
    const R ES = left ? EL : ER, vS = left ? vL : vR, wS = left ? wL : wR;
    const R pStar = mS * (sM - uS) + pS;
    const R rhoStar = qdiv(mS, sS - sM);
    const R Estar = ES + (sM - uS) * (sM + qdiv(pS, mS));
    mass = rhoStar * sM; m0 = rhoStar * sM * sM + pStar; m1 = rhoStar * sM * vS; m2 = rhoStar * sM * wS;
    en = (rhoStar * Estar + pStar) * sM;
  }
  F.f.mass[0] = mass; F.f.mom[0] = m0; F.f.mom[1] = m1; F.f.mom[2] = m2; F.f.energM = en;
  F.sM = sM; F.uStar = sM;
}

// ModUEq::solveRiemannIntern
template <int N, typename R, bool CRPOW = false>
__device__ __forceinline__ void hllc_ueq(const Params& P, const Cell<N, R>& Lc, const R* lu, const Cell<N, R>& Rc,
                                         const R* ru, R& smax, Flux<N, R>& F) {
  const R eps = pv<R>(P.eps, P.f_eps);
  const R uL = lu[0], cL = Lc.cF, pL = Lc.pm, rhoL = Lc.rho;
  const R uR = ru[0], cR = Rc.cF, pR = Rc.pm, rhoR = Rc.rho;
  const R sL = dmin<R>(uL - cL, uR - cR);
  const R sR = dmax<R>(uR + cR, uL + cL);
  cfl_speed<R>(smax, sL);
  cfl_speed<R>(smax, sR);
  const R mL = rhoL * (sL - uL), mR = rhoR * (sR - uR);
  R sM = qdiv(pR - pL + mL * uL - mR * uR, mL - mR);
  if (fabs(sM) < R(1.e-8)) sM = R(0.);
  if (sL >= R(0.) || sR <= R(0.)) {
    const bool left = (sL >= R(0.));
    const Cell<N, R>& S = left ? Lc : Rc;
    const R* su = left ? lu : ru;
    const R uS = su[0], rhoS = left ? rhoL : rhoR, pS = left ? pL : pR;
    const R totalEnergy = S.em + R(0.5) * sqn3<R>(su);
#pragma unroll
    for (int k = 0; k < N; k++) {
      F.f.alpha[k] = S.a[k] * sM;
      F.f.mass[k] = S.a[k] * S.r[k] * uS;
      F.f.energ[k] = S.a[k] * S.r[k] * S.e[k] * uS;
    }
    F.f.mom[0] = rhoS * uS * uS + pS;
    F.f.mom[1] = rhoS * su[1] * uS;
    F.f.mom[2] = rhoS * su[2] * uS;
    F.f.energM = (rhoS * totalEnergy + pS) * uS;
    F.uStar = uS;
  } else {
    const bool left = (sM >= R(0.));
    const Cell<N, R>& S = left ? Lc : Rc;
    const R* su = left ? lu : ru;
    const R uS = su[0], pS = left ? pL : pR, mS = left ? mL : mR, sS = left ? sL : sR;
    const R totalEnergy = S.em + R(0.5) * sqn3<R>(su);
    if constexpr (sizeof(R) == 4) {
      // FP32 form: every phase is compressed by the same ratio (s - u) / (s - sM), so
      // one reciprocal and one logarithm serve all star densities and isentropes, and
      // the star energy fluxes need no division.
      const R ratio = (sS - uS) * __builtin_amdgcn_rcpf(sS - sM);
      const R rhoStar = (left ? rhoL : rhoR) * ratio;
      const R EStar = totalEnergy + (sM - uS) * (sM + pS * __builtin_amdgcn_rcpf(mS));
      const R pStar = mS * (sM - uS) + pS;
      const R lr = __builtin_amdgcn_logf(ratio);
#pragma unroll
      for (int k = 0; k < N; k++) {
        const EosDev& q = P.eos[k];
        const R rks = S.r[k] * ratio;
        const R pk0 = S.p[k] + pv<R>(q.pinf, q.fpinf);
        const R pks = pk0 * __builtin_amdgcn_exp2f(pv<R>(q.g, q.fg) * lr) - pv<R>(q.pinf, q.fpinf);
        F.f.alpha[k] = S.a[k] * sM;
        F.f.mass[k] = S.a[k] * rks * sM;
        F.f.energ[k] = S.a[k] * ((pks + pv<R>(q.gpinf, q.fgpinf)) * pv<R>(q.mixinv, q.fmixinv) + rks * pv<R>(q.eref, q.feref)) * sM;
      }
      F.f.mom[0] = rhoStar * sM * sM + pStar;
      F.f.mom[1] = rhoStar * su[1] * sM;
      F.f.mom[2] = rhoStar * su[2] * sM;
      F.f.energM = (rhoStar * EStar + pStar) * sM;
      F.uStar = sM;
      F.sM = sM;
      return;
    }
    // FP64: the star density and the phases' star densities share one reciprocal
    // of sS - sM (the reference's quotients, bit for bit).
    const double dS = sS - sM, idS = rcp_ieee(dS);
    const R rhoStar = div_ieee(mS, dS, idS);
    const R EStar = totalEnergy + (sM - uS) * (sM + div1(pS, mS));
    const R pStar = mS * (sM - uS) + pS;
    // Density ratios of the isentropes.  Every phase is compressed by the same
    // ratio (sS - uS) / dS, so outside the full-featured kernels one logarithm
    // serves all phases: log x_k = log x_0 + log1p(z), z = (x_k - x_0) / x_0, with
    // z at rounding size (its series to second order) unless a phase's density
    // is below eps.
    double rks[N], xk[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
      rks[k] = div_ieee(S.r[k] * (sS - uS), dS, idS);
      const double r0 = dmax<double>(S.r[k], eps);
      xk[k] = div_ieee(rks[k], r0, rcp_ieee(r0));
    }
    const double lx0 = CRPOW ? 0. : log_pos(xk[0]);
#pragma unroll
    for (int k = 0; k < N; k++) {
      const EosDev& q = P.eos[k];
      double base;
      if constexpr (CRPOW) {
        base = pow_cr(xk[k], q.g);
      } else {
        double lxk = lx0;
        if (k > 0) {
          const double z = div1(xk[k] - xk[0], xk[0]);
          lxk = lx0 + z * (1. - 0.5 * z);
          if (!(fabs(z) < 1.e-6)) lxk = log_pos(xk[k]);
        }
        base = exp(q.g * lxk);
      }
      const R pks = (S.p[k] + q.pinf) * base - q.pinf;
      const R rks_k = rks[k];
      const R eks = eos_energy<R>(q, eps, rks_k, pks);
      F.f.alpha[k] = S.a[k] * sM;
      F.f.mass[k] = S.a[k] * rks_k * sM;
      F.f.energ[k] = S.a[k] * rks_k * eks * sM;
    }
    F.f.mom[0] = rhoStar * sM * sM + pStar;
    F.f.mom[1] = rhoStar * su[1] * sM;
    F.f.mom[2] = rhoStar * su[2] * sM;
    F.f.energM = (rhoStar * EStar + pStar) * sM;
    F.uStar = sM;
  }
  F.sM = sM;
}

// Face flux between two derived cells (global-frame velocities), returned in
// the global frame.  EL/ER: total energies the Euler solver uses.
template <int MODEL, int N, int FR, typename R, bool CRPOW = false>
__device__ __forceinline__ void face_flux(const Params& P, const Cell<N, R>& L, R EL, const Cell<N, R>& Rr, R ER,
                                          R& smax, Flux<N, R>& F) {
  R lu[3], ru[3], loc[3];
  to_local<FR, R>(L.u, lu);
  to_local<FR, R>(Rr.u, ru);
  if (MODEL == M_EULER) hllc_euler<N, R>(L, lu, EL, Rr, ru, ER, smax, F);
  else hllc_ueq<N, R, CRPOW>(P, L, lu, Rr, ru, smax, F);
  loc[0] = F.f.mom[0]; loc[1] = F.f.mom[1]; loc[2] = F.f.mom[2];
  to_global<FR, R>(loc, F.f.mom);
}

// Boundary face (BoundCond::solveRiemann, BoundCond.cpp:78-98): the buffer cell
// is the interior cell with its derived state rebuilt (Euler: E rebuilt).
template <int MODEL, int N, int FR, typename R, bool CRPOW = false>
__device__ __forceinline__ void boundary_flux(const Params& P, const Cell<N, R>& B, R EB, int bc, R& smax,
                                              Flux<N, R>& F) {
  if (bc == BC_WALL) {
    R lu[3];
    to_local<FR, R>(B.u, lu);
    const R uL = lu[0];
    const R cL = (MODEL == M_EULER) ? B.c[0] : B.cF;
    const R pL = (MODEL == M_EULER) ? B.p[0] : B.pm;
    const R rhoL = (MODEL == M_EULER) ? B.r[0] : B.rho;
    const R sL = dmin<R>(uL - cL, -uL - cL);
    cfl_speed<R>(smax, sL);
    const R pStar = (MODEL == M_EULER) ? rhoL * uL * (uL - sL) + pL : rhoL * (uL - sL) * uL + pL;
#pragma unroll
    for (int k = 0; k < N; k++) { F.f.alpha[k] = R(0.); F.f.mass[k] = R(0.); F.f.energ[k] = R(0.); }
    R loc[3] = {pStar, R(0.), R(0.)};
    to_global<FR, R>(loc, F.f.mom);
    F.f.energM = R(0.);
    F.sM = R(0.);
    F.uStar = R(0.);
  } else {
    face_flux<MODEL, N, FR, R, CRPOW>(P, B, EB, B, EB, smax, F);
  }
}

// Inlet-tank boundary (ModEuler::solveRiemannInletTank, ModEuler.cpp:413-545;
// ModUEq::solveRiemannInletTank, ModUEq.cpp:496-673, shared by PRESSUREVELOCITYEQ)
// on the derived buffer cell B with face-frame velocity lu (normal out of the
// domain); the flux is returned in the face frame.  FP64 in both arithmetic
// forms: the pressure Newton works to 1e-3 (Euler) / 1e-2 (mixture) in velocity
// and steps p below p0 by 1e-6, which single precision cannot resolve.  Returns
// the Newton iterations of the tank-inflow branch, or -1 once 50 are spent (the
// reference stops with an error there).
template <int MODEL, int N>
__device__ __forceinline__ int tank_flux(const Params& P, const TankDev& T, const Cell<N, double>& B, const double* lu,
                                      double& dtm, Flux<N, double>& F) {
  const double eps = P.eps, p0 = T.p0, lcfl = P.lcfl;
  int iteration = 0;
  if constexpr (MODEL == M_EULER) {
    const EosDev& q = P.eos[0];
    const double uL = lu[0], vL = lu[1], wL = lu[2], pL = B.p[0], rhoL = B.r[0], zL = rhoL * B.c[0];
    double uStar, rhoStar, pStar = p0, vStar, wStar, drho, mL, vmv0;
    double v = 1. / eos_rho_isentropic(q, eps, pL, rhoL, pStar, drho);
    vmv0 = v - 1. / rhoL;
    mL = (fabs(vmv0) > 1e-10) ? sqrt((pL - p0) / vmv0) : zL;
    double sL = uL - mL / rhoL;
    cfl_bound<double>(dtm, sL, lcfl);
    const double u = uL + mL * vmv0;
    if (sL >= 0.) {
      uStar = uL; pStar = pL; rhoStar = rhoL; vStar = vL; wStar = wL;
    } else if (u >= -1e-3) {
      uStar = u; pStar = p0; rhoStar = 1. / v; vStar = vL; wStar = wL;
    } else {
      double p = 0.5 * p0, f = 0., df = 1., uStarR = 0., uStarL = 0.;
      do {
        p -= f / df;
        iteration++;
        if (iteration > 50) return -1;
        p = eos_clamp_p<double>(q, p);
        if (p > p0) p = p0 - 1e-6;
        double dh;
        const double h = eos_h_isentropic(q, eps, p0, T.rhok0[0], p, rhoStar, dh);
        uStarR = -sqrt(2. * (T.H0 - h));
        const double duStarR = -dh / uStarR;
        v = 1.0 / eos_rho_isentropic(q, eps, pL, rhoL, p, drho);
        const double dv = -v * v * drho;
        vmv0 = v - 1. / rhoL;
        double dmL = 0.;
        if (fabs(vmv0) > 1e-10) {
          mL = sqrt((pL - p) / vmv0);
          dmL = 0.5 * (-vmv0 + (p - pL) * dv) / (vmv0 * vmv0) / mL;
        } else {
          mL = zL;
        }
        sL = uL - mL / rhoL;
        cfl_bound<double>(dtm, sL, lcfl);
        uStarL = uL + mL * vmv0;
        const double duStarL = dmL * vmv0 + mL * dv;
        f = uStarR - uStarL;
        df = duStarR - duStarL;
      } while (fabs(f) > 1e-3);
      pStar = p;
      uStar = 0.5 * (uStarL + uStarR);
      vStar = 0.;
      wStar = 0.;
    }
    const double eStar = eos_energy<double>(q, eps, rhoStar, pStar);
    F.f.mass[0] = rhoStar * uStar;
    F.f.mom[0] = rhoStar * uStar * uStar + pStar;
    F.f.mom[1] = rhoStar * uStar * vStar;
    F.f.mom[2] = rhoStar * uStar * wStar;
    F.f.energM = (rhoStar * (eStar + 0.5 * (uStar * uStar + vStar * vStar + wStar * wStar)) + pStar) * uStar;
    F.sM = uStar;
    F.uStar = uStar;
  } else {
    double rks[N], Yks[N];
    const double uL = lu[0], pL = B.pm, rhoL = B.rho;
    // Wood sound speed of the mixture (MixUEq.cpp:152-159)
    double cL = 0.;
#pragma unroll
    for (int k = 0; k < N; k++) cL += B.a[k] / dmax(B.r[k] * B.c[k] * B.c[k], eps);
    cL = 1. / sqrt(rhoL * cL);
    const double zL = rhoL * cL;
    double pStar = p0, vStar = 0., mL, vmv0, uStar, rhoStar, uyStar, uzStar;
#pragma unroll
    for (int k = 0; k < N; k++) {
      rks[k] = eos_rho_hugoniot(P.eos[k], eps, B.p[k], B.r[k], pStar);
      vStar += B.a[k] * B.r[k] / rhoL / dmax(rks[k], eps);
    }
    vmv0 = vStar - 1. / rhoL;
    mL = (fabs(vmv0) > 1e-10) ? sqrt((pL - pStar) / vmv0) : zL;
    double sL = uL - mL / rhoL;
    cfl_bound<double>(dtm, sL, lcfl);
    double sM = uL + mL * vmv0;
    if (sL >= 0.) {
      uStar = uL;
      pStar = pL;
#pragma unroll
      for (int k = 0; k < N; k++) { rks[k] = B.r[k]; Yks[k] = B.a[k] * B.r[k] / rhoL; }
      rhoStar = rhoL;
      uyStar = lu[1];
      uzStar = lu[2];
    } else if (sM >= -1e-3) {
      uStar = sM;
      pStar = p0;
#pragma unroll
      for (int k = 0; k < N; k++) Yks[k] = B.a[k] * B.r[k] / rhoL;
      rhoStar = 1. / vStar;
      uyStar = lu[1];
      uzStar = lu[2];
    } else {
      double p = 0.5 * p0, f = 0., df = 1., uStarR = 0., uStarL = 0.;
      do {
        p -= f / df;
        iteration++;
#pragma unroll
        for (int k = 0; k < N; k++) p = eos_clamp_p<double>(P.eos[k], p);
        if (p > p0) p = p0 - 1e-6;
        if (iteration > 50) return -1;
        // Tank side: isentropes from (p0, rhok0) and H = H0.
        uStarR = T.H0;
        double duStarR = 0.;
#pragma unroll
        for (int k = 0; k < N; k++) {
          double dhk;
          const double hk = eos_h_isentropic(P.eos[k], eps, p0, T.rhok0[k], p, rks[k], dhk);
          uStarR -= T.Yk0[k] * hk;
          duStarR -= T.Yk0[k] * dhk;
        }
        uStarR = -sqrt(2. * uStarR);
        duStarR = duStarR / uStarR;
        // Cell side: isentropes of every phase.
        double vStarL = 0., dvStarL = 0.;
#pragma unroll
        for (int k = 0; k < N; k++) {
          double drhok;
          const double rhok = eos_rho_isentropic(P.eos[k], eps, B.p[k], B.r[k], p, drhok);
          const double YkL = B.a[k] * B.r[k] / rhoL;
          vStarL += YkL / dmax(rhok, eps);
          dvStarL -= YkL / dmax(rhok * rhok, eps) * drhok;
        }
        vmv0 = vStarL - 1. / rhoL;
        double dmL = 0.;
        if (fabs(vmv0) > 1e-10) {
          mL = sqrt((pL - p) / vmv0);
          dmL = 0.5 * (-vmv0 + (p - pL) * dvStarL) / (vmv0 * vmv0) / mL;
        } else {
          mL = zL;
        }
        sL = uL - mL / rhoL;
        cfl_bound<double>(dtm, sL, lcfl);
        uStarL = uL + mL * vmv0;
        const double duStarL = dmL * vmv0 + mL * dvStarL;
        f = uStarR - uStarL;
        df = duStarR - duStarL;
      } while (fabs(f) > 1e-2);
      pStar = p;
      uStar = 0.5 * (uStarL + uStarR);
      rhoStar = 0.;
#pragma unroll
      for (int k = 0; k < N; k++) { Yks[k] = T.Yk0[k]; rhoStar += Yks[k] / dmax(rks[k], eps); }
      rhoStar = 1. / rhoStar;
      uyStar = 0.;
      uzStar = 0.;
      sM = uStar;
    }
    // Flux (ModUEq.cpp:643-665)
    double EStar = 0.5 * (uStar * uStar + uyStar * uyStar + uzStar * uzStar);
#pragma unroll
    for (int k = 0; k < N; k++) {
      const double ek = eos_energy<double>(P.eos[k], eps, rks[k], pStar);
      EStar += Yks[k] * ek;
      const double akStar = Yks[k] * rhoStar / dmax(rks[k], eps);
      F.f.alpha[k] = akStar * sM;
      F.f.mass[k] = akStar * uStar * rks[k];
      F.f.energ[k] = F.f.mass[k] * ek;
    }
    F.f.mom[0] = rhoStar * uStar * uStar + pStar;
    F.f.mom[1] = rhoStar * uStar * uyStar;
    F.f.mom[2] = rhoStar * uStar * uzStar;
    F.f.energM = (rhoStar * EStar + pStar) * uStar;
    F.sM = sM;
    F.uStar = uStar;
  }
  return iteration;
}

// ---------------------------------------------------------------------------
// Accumulation of face contributions into the cell's m_cons buffer.
// FP64: plain double sums in the reference order.  FP32: the float
// contributions summed in double (a conversion and one FP64 addition each, at
// the FP32 rate on CDNA4; the two registers a compensated float pair would
// take, and a sum whose error is far below the contributions' own rounding).
// ---------------------------------------------------------------------------
template <typename R> struct Acc;
template <> struct Acc<double> {
  double v = 0.;
  __device__ __forceinline__ void add(double x) { v += x; }
  __device__ __forceinline__ void sub(double x) { v -= x; }
  __device__ __forceinline__ double value() const { return v; }
};
template <> struct Acc<float> {
  double v = 0.;
  __device__ __forceinline__ void add(float x) { v += (double)x; }
  __device__ __forceinline__ void sub(float x) { v -= (double)x; }
  __device__ __forceinline__ double value() const { return v; }
};

template <int N, typename R>
struct ConsAcc {
  Acc<R> alpha[N], mass[N], energ[N];
  Acc<R> mom[3];
  Acc<R> energM;
};

// CellInterface::addFlux / subtractFlux with the non-conservative terms of the
// cell's time-n phases (FluxUEq.cpp:61-84, 224-244; FluxPUEq.cpp:44-65).
template <int MODEL, int N, int D, typename R>
__device__ __forceinline__ void add_flux(ConsAcc<N, R>& A, const Flux<N, R>& F, R coefA, const R* an, const R* pn) {
  if (MODEL == M_EULER) {
    A.mass[0].add(coefA * F.f.mass[0]);
  } else {
#pragma unroll
    for (int k = 0; k < N; k++) {
      A.alpha[k].add(coefA * F.f.alpha[k]);
      A.mass[k].add(coefA * F.f.mass[k]);
      A.energ[k].add(coefA * F.f.energ[k]);
    }
  }
#pragma unroll
  for (int d = 0; d < D; d++) A.mom[d].add(F.f.mom[d] * coefA);
  A.energM.add(coefA * F.f.energM);
  if (MODEL != M_EULER) {
#pragma unroll
    for (int k = 0; k < N; k++) {
      A.alpha[k].add(-coefA * an[k] * F.sM);
      if (MODEL == M_PUEQ) A.energ[k].add(coefA * an[k] * pn[k] * F.uStar);
    }
  }
}

// FP32 form: the lower face added and the upper face subtracted in one accumulation
// per variable, coefA (F_lower - F_upper) (an absent face is zero).
template <int MODEL, int N, int D>
__device__ __forceinline__ void add_flux_pair(ConsAcc<N, float>& A, const Flux<N, float>& L, const Flux<N, float>& U,
                                              float coefA, const float* an, const float* pn) {
  if (MODEL == M_EULER) {
    A.mass[0].add(coefA * (L.f.mass[0] - U.f.mass[0]));
  } else {
#pragma unroll
    for (int k = 0; k < N; k++) {
      A.alpha[k].add(coefA * (L.f.alpha[k] - U.f.alpha[k]));
      A.mass[k].add(coefA * (L.f.mass[k] - U.f.mass[k]));
      A.energ[k].add(coefA * (L.f.energ[k] - U.f.energ[k]));
    }
  }
#pragma unroll
  for (int d = 0; d < D; d++) A.mom[d].add((L.f.mom[d] - U.f.mom[d]) * coefA);
  A.energM.add(coefA * (L.f.energM - U.f.energM));
  if (MODEL != M_EULER) {
#pragma unroll
    for (int k = 0; k < N; k++) {
      A.alpha[k].add(-coefA * an[k] * (L.sM - U.sM));
      if (MODEL == M_PUEQ) A.energ[k].add(coefA * an[k] * pn[k] * (L.uStar - U.uStar));
    }
  }
}

template <int MODEL, int N, int D, typename R>
__device__ __forceinline__ void sub_flux(ConsAcc<N, R>& A, const Flux<N, R>& F, R coefA, const R* an, const R* pn) {
  if (MODEL == M_EULER) {
    A.mass[0].sub(coefA * F.f.mass[0]);
  } else {
#pragma unroll
    for (int k = 0; k < N; k++) {
      A.alpha[k].sub(coefA * F.f.alpha[k]);
      A.mass[k].sub(coefA * F.f.mass[k]);
      A.energ[k].sub(coefA * F.f.energ[k]);
    }
  }
#pragma unroll
  for (int d = 0; d < D; d++) A.mom[d].sub(F.f.mom[d] * coefA);
  A.energM.sub(coefA * F.f.energM);
  if (MODEL != M_EULER) {
#pragma unroll
    for (int k = 0; k < N; k++) {
      A.alpha[k].sub(-coefA * an[k] * F.sM);
      if (MODEL == M_PUEQ) A.energ[k].sub(coefA * an[k] * pn[k] * F.uStar);
    }
  }
}

// Cell::timeEvolution (Cell.cpp:286-299): A <- scale*sum (+ scheme correction) + U^n, FP64.
template <int MODEL, int N, int D, typename R>
__device__ __forceinline__ void time_evolution(const Params& P, const ConsAcc<N, R>& S, Cons<N>& A,
                                               const Cell<N>& n, double scale) {
  Cons<N> U;
  if (MODEL == M_EULER) {
    U.mass[0] = n.r[0];
    U.mom[0] = n.u[0] * U.mass[0]; U.mom[1] = n.u[1] * U.mass[0]; U.mom[2] = n.u[2] * U.mass[0];
    U.energM = U.mass[0] * n.E;
    A.mass[0] = S.mass[0].value() * scale;
  } else {
#pragma unroll
    for (int k = 0; k < N; k++) {
      U.alpha[k] = n.a[k];
      U.mass[k] = n.a[k] * n.r[k];
      U.energ[k] = n.a[k] * n.r[k] * eos_energy<double>(P.eos[k], P.eps, n.r[k], n.p[k]);
      A.alpha[k] = S.alpha[k].value() * scale;
      A.mass[k] = S.mass[k].value() * scale;
      A.energ[k] = S.energ[k].value() * scale;
    }
    U.mom[0] = n.u[0] * n.rho; U.mom[1] = n.u[1] * n.rho; U.mom[2] = n.u[2] * n.rho;
    U.energM = n.rho * n.E;
  }
#pragma unroll
  for (int d = 0; d < 3; d++) A.mom[d] = (d < D) ? S.mom[d].value() * scale : 0.;
  A.energM = S.energM.value() * scale;
  if (MODEL == M_UEQ) {
    double rhoNp1 = 0., sumD = 0., m[3];
#pragma unroll
    for (int k = 0; k < N; k++) { rhoNp1 += A.mass[k] + U.mass[k]; sumD += A.energ[k]; }
    m[0] = A.mom[0] + U.mom[0]; m[1] = A.mom[1] + U.mom[1]; m[2] = A.mom[2] + U.mom[2];
    const double dRU2 = div1(sqn3<double>(m), rhoNp1) - div1(sqn3<double>(U.mom), n.rho);
    const double err = (A.energM - 0.5 * dRU2) - sumD;
#pragma unroll
    for (int k = 0; k < N; k++) A.energ[k] += n.a[k] * err;
  }
  if (MODEL == M_EULER) {
    A.mass[0] += 1. * U.mass[0];
  } else {
#pragma unroll
    for (int k = 0; k < N; k++) {
      A.alpha[k] += 1. * U.alpha[k]; A.mass[k] += 1. * U.mass[k]; A.energ[k] += 1. * U.energ[k];
    }
  }
  A.mom[0] += U.mom[0] * 1.; A.mom[1] += U.mom[1] * 1.; A.mom[2] += U.mom[2] * 1.;
  A.energM += 1. * U.energM;
}

// Flux::buildPrim (FluxUEq.cpp:161-207, FluxEuler.cpp:124-150); derived rebuilt.  FP64.
template <int MODEL, int N>
__device__ __forceinline__ void build_prim(const Params& P, Cons<N>& A, Cell<N>& s) {
  if (MODEL == M_EULER) {
    const double m = A.mass[0];
    s.r[0] = m;
    // One reciprocal for the four quotients by the density.
    const QuotFull q(m);
    s.u[0] = q(A.mom[0]); s.u[1] = q(A.mom[1]); s.u[2] = q(A.mom[2]);
    s.E = q(A.energM);
    if (fabs(s.u[0]) < 1.e-8) s.u[0] = 0.;
    if (fabs(s.u[1]) < 1.e-8) s.u[1] = 0.;
    if (fabs(s.u[2]) < 1.e-8) s.u[2] = 0.;
    const double e = s.E - 0.5 * sqn3<double>(s.u);
    s.e[0] = e;
    s.p[0] = eos_pressure<double>(P.eos[0], m, e);
    return;
  }
  double un = 0., rhoMel = 0.;
  if (P.eps > 1.e-20) {
#pragma unroll
    for (int k = 0; k < N; k++) {
      if (A.alpha[k] < 0.) A.alpha[k] = 0.;
      if (A.alpha[k] > 1.) A.alpha[k] = 1.;
      un += A.alpha[k];
    }
  } else {
#pragma unroll
    for (int k = 0; k < N; k++) {
      if (A.alpha[k] <= 1.e-15) A.alpha[k] = 1e-15;
      if (A.alpha[k] >= 1. - 1.e-15) A.alpha[k] = 1.0 - 1e-15;
      un += A.alpha[k];
    }
  }
  const double iun = rcp_ieee(un);
#pragma unroll
  for (int k = 0; k < N; k++) A.alpha[k] = div_ieee(A.alpha[k], un, iun);
#pragma unroll
  for (int k = 0; k < N; k++) {
    rhoMel += A.mass[k];
    s.a[k] = A.alpha[k];
    s.r[k] = div1(A.mass[k], dmax(A.alpha[k], P.eps));
    const double ek = div1(A.energ[k], dmax(A.mass[k], P.eps));
    s.p[k] = eos_pressure<double>(P.eos[k], s.r[k], ek);
    verify_correct<MODEL, N, double>(P, s, k);
  }
  const double irm = rcp_ieee(rhoMel);
  s.u[0] = div_ieee(A.mom[0], rhoMel, irm); s.u[1] = div_ieee(A.mom[1], rhoMel, irm);
  s.u[2] = div_ieee(A.mom[2], rhoMel, irm);
  if (fabs(s.u[0]) < 1.e-8) s.u[0] = 0.;
  if (fabs(s.u[1]) < 1.e-8) s.u[1] = 0.;
  if (fabs(s.u[2]) < 1.e-8) s.u[2] = 0.;
  // Of the derived state only the mixture density is read afterwards (energy
  // correction); the rest is rebuilt from the stored primitives when needed.
  mixture_density<N>(s);
  s.E = div_special(A.energM, rhoMel, irm);
}

// alphaNull gate of RelaxationPInfinite::relaxation (RelaxationPInfinite.cpp:51-55):
// no relaxation when a phase fills the cell to within 1e-5.
template <int N>
__device__ __forceinline__ bool relax_gated(const Params& P, const Cell<N>& s) {
  if (P.eps > 1.e-20) {
#pragma unroll
    for (int k = 0; k < N; k++)
      if (s.a[k] > (1. - 1.e-5)) return true;
  }
  return false;
}

// RelaxationP::NewtonRaphson (RelaxationP.cpp:43-70) between two evaluations: the
// iterate, f and f' there, and the evaluations so far.  A procedure from the guess
// g starts at {g, 0, 1, 0}.
struct NewtonState { double p, f, df; int it; };

// Newton evaluations of f = sum_k alpha_k rho_k / rho_k(p) - 1 on the cell's
// pre-relaxation phases (s, unchanged) from st until |f| <= 1e-10 or st.it reaches
// maxit; akS / rkS receive the phases at the last evaluation.
// The first evaluation forms f' only where another iterate follows: nearly every relaxation is
// settled there (1.03 evaluations per relaxation on the 512^3 two-phase case), and the
// derivative is two quotients per phase.  A settled st keeps an unread f'.  With BESIDE the
// evaluations after it form f' beside f, in a copy of their own: a lane behind a shock takes
// tens of them, and its chain is what a small mesh's step waits for.  Two-phase second
// order, us a step with f' on demand throughout / beside: 96^2 69.0 / 65.2, 24^3 76.4 / 72.9;
// the 3D FP64 kernel of the finite-rate relaxation spills 186 / 41 VGPRs and takes 280 / 254
// at 77 x 75 x 73.  The copy costs three-phase (24^3 18.1 / 18.6) and learned kernels
// (2D walls 94 / 96) more than it saves.
template <int N, bool BESIDE = (N == 2)>
__device__ __forceinline__ void newton_resume(const Params& P, const Cell<N>& s, NewtonState& st, double* akS,
                                              double* rkS, int maxit) {
  auto evaluate = [&](bool beside) {
    st.it++;
    st.p -= div1(st.f, st.df);
#pragma unroll
    for (int k = 0; k < N; k++) st.p = eos_clamp_p<double>(P.eos[k], st.p);
    double f = -1., df = 0.;
#pragma unroll
    for (int k = 0; k < N; k++) {
      rkS[k] = eos_rho_pfinal(P.eos[k], P.eps, s.p[k], s.r[k], st.p);
      akS[k] = div1(s.a[k] * s.r[k], rkS[k]);
      f += akS[k];
    }
    st.f = f;
    if (beside || fabs(f) > 1e-10) {
#pragma unroll
      for (int k = 0; k < N; k++) {
        const double drhodp = eos_drhodp_pfinal(P.eos[k], P.eps, s.p[k], s.r[k], st.p);
        df -= div1(s.a[k] * s.r[k] * drhodp, rkS[k] * rkS[k]);
      }
      st.df = df;
    }
  };
  if constexpr (BESIDE) {
    evaluate(false);
    while (fabs(st.f) > 1e-10 && st.it < maxit) evaluate(true);
  } else {
    do evaluate(false);
    while (fabs(st.f) > 1e-10 && st.it < maxit);
  }
}

// Outcome flags of a relaxation's Newton solve: RELAX_FAIL when it spent its 100
// iterations and the cell took the interface pressure; RELAX_WARN when, in
// addition, |p*| > 1e-7, the condition of the reference's warning
// (RelaxationP.cpp:62-68).
constexpr int RELAX_FAIL = 1, RELAX_WARN = 2;
__device__ __forceinline__ int newton_flags(int it, double pStar) {
  return (it >= 100) ? (RELAX_FAIL | ((fabs(pStar) > 1.e-7) ? RELAX_WARN : 0)) : 0;
}

// The end of RelaxationPInfinite::relaxation: a converged Newton (st, with the
// phases akS / rkS of its last evaluation) gives the relaxed phases; one that spent
// the reference's 100 evaluations gives the interface-pressure fallback
// (RelaxationPInfinite.cpp:82-97, RelaxationP.cpp:72-93).  Returns the flags.
template <int N>
__device__ __forceinline__ int relax_end(const Params& P, Cell<N>& s, const NewtonState& st, bool converged,
                                         const double* akS, const double* rkS) {
  if (converged) {
#pragma unroll
    for (int k = 0; k < N; k++) { s.a[k] = akS[k]; s.r[k] = rkS[k]; s.p[k] = st.p; }
    return 0;
  }
  const int flags = newton_flags(st.it, st.p);
  double z[N], pI = 0., sumZk = 0.;
#pragma unroll
  for (int k = 0; k < N; k++) z[k] = s.r[k] * eos_sound<double>(P.eos[k], P.eps, s.r[k], s.p[k]);
#pragma unroll
  for (int k = 0; k < N; k++) {
    sumZk += z[k];
    double sumZj = 0.;
#pragma unroll
    for (int j = 0; j < N; j++)
      if (j != k) sumZj += z[j];
    pI += sumZj * (s.p[k] - 0.);
  }
  pI /= sumZk * (double)(N - 1);
#pragma unroll
  for (int k = 0; k < N; k++) pI = eos_clamp_p<double>(P.eos[k], pI);
#pragma unroll
  for (int k = 0; k < N; k++) {
    const double rho_s = eos_rho_pfinal(P.eos[k], P.eps, s.p[k], s.r[k], pI);
    s.a[k] = s.a[k] * s.r[k] / rho_s;
    s.r[k] = rho_s;
    s.p[k] = pI;
  }
  return flags;
}

// RelaxationPInfinite::relaxation + RelaxationP::NewtonRaphson from a start that
// is either the reference's guess sum alpha_k p_k (maxit 100: the reference
// procedure) or a learned guess (maxit WARM_MAX_IT below 100: when that many
// evaluations do not reach the 1e-10 tolerance, the reference procedure from the
// cold guess p_cold follows and fellback is set).  Returns the total evaluation
// count (0 when gated out); flags receives RELAX_FAIL / RELAX_WARN of the
// reference procedure (a converged learned start has none).  FP64.
template <int N>
__device__ __forceinline__ int relax_start(const Params& P, Cell<N>& s, double pStar, int maxit, double p_cold,
                                           bool& fellback, double& fres, int& flags) {
  fres = 0.;
  flags = 0;
  fellback = false;
  if (relax_gated<N>(P, s)) return 0;
  double akS[N], rkS[N];
  NewtonState st{pStar, 0., 1., 0};
  newton_resume<N>(P, s, st, akS, rkS, maxit);
  int total = st.it;
  bool warm = maxit < 100;
  if (warm && !(fabs(st.f) <= 1e-10)) {
    fellback = true;
    warm = false;
    st = NewtonState{p_cold, 0., 1., 0};
    newton_resume<N>(P, s, st, akS, rkS, 100);
    total += st.it;
  }
  fres = st.f;
  flags = relax_end<N>(P, s, st, warm || st.it < 100, akS, rkS);
  return total;
}

// The reference procedure from the initial guess pStar.
template <int N>
__device__ __forceinline__ int relax_newton(const Params& P, Cell<N>& s, double pStar, double& fres, int& flags) {
  bool fellback;
  return relax_start<N>(P, s, pStar, 100, pStar, fellback, fres, flags);
}

// RelaxationPFinite::relaxation with the Euler variable-step solver
// (RelaxationPFinite.cpp:69-275) over dt: sub-steps of d(alpha_k)/dt = mu Dp_k with
// the phase energies driven by the interface pressure, each sub-step at most half
// the time to the volume-fraction and pressure bounds; once the pressures agree to
// 1e-5 relative (or after 100 sub-steps) the infinite relaxation of the entry state
// finishes.  Returns the sub-steps plus the Newton evaluations.  FP64.
template <int N>
__device__ int relax_finite(const Params& P, Cell<N>& s, double dt, int& flags) {
  const double epsilon = 1.e-15, thrA = 1.e-8, crit = 1.e-5, mu = P.relax_mu;
  flags = 0;
  if (dt < 1.e-20) return 0;
  if (P.eps > 1.e-20) {
#pragma unroll
    for (int k = 0; k < N; k++)
      if (s.a[k] > (1. - thrA)) return 0;
  }
  double ak[N], rk[N], pk[N], e[N], cs[N], dp[N], z[N], rc[N];
  bool anull[N];
#pragma unroll
  for (int k = 0; k < N; k++) {
    ak[k] = s.a[k]; rk[k] = s.r[k]; pk[k] = s.p[k];
    anull[k] = ak[k] < thrA;
    e[k] = eos_energy<double>(P.eos[k], P.eps, s.r[k], s.p[k]);
    cs[k] = eos_sound<double>(P.eos[k], P.eps, s.r[k], s.p[k]);
  }
  // Interface pressure over the phases present (RelaxationP::computeInterfacePressure).
  auto interface_p = [&]() {
    double pI = 0., sumZk = 0.;
#pragma unroll
    for (int k = 0; k < N; k++) z[k] = s.r[k] * cs[k];
#pragma unroll
    for (int k = 0; k < N; k++) {
      if (!anull[k]) {
        sumZk += z[k];
        double sumZj = 0.;
#pragma unroll
        for (int j = 0; j < N; j++)
          if (!anull[j] && j != k) sumZj += z[j];
        pI += sumZj * (s.p[k] - 0.);
      }
    }
    pI /= sumZk * (double)(N - 1);
#pragma unroll
    for (int k = 0; k < N; k++) pI = eos_clamp_p<double>(P.eos[k], pI);
    return pI;
  };
  bool relaxed = true;
  int iter = 0, total = 0;
  double tlocal = 0.;
  while ((dt - tlocal) > 1.e-15) {
    iter++;
    double dtlocal = dt - tlocal;
    double pMix = 0.;
#pragma unroll
    for (int k = 0; k < N; k++) pMix += s.a[k] * s.p[k];
    relaxed = true;
#pragma unroll
    for (int k = 0; k < N; k++)
      if (fabs((s.p[k] - pMix) / s.p[k]) > crit) relaxed = false;
    if (relaxed) break;
#pragma unroll
    for (int k = 0; k < N; k++) {
      dp[k] = 0.;
      if (!anull[k]) {
#pragma unroll
        for (int j = 0; j < N; j++)
          if (!anull[j] && j != k) dp[k] += s.a[j] * (s.p[k] - 0. - s.p[j] + 0.);
        dp[k] *= s.a[k];
      }
    }
    const double pI = interface_p();
    if (mu > 1.e-20) {
      double dtmax = 1.e10;
#pragma unroll
      for (int k = 0; k < N; k++) {
        const double sA = mu * dp[k];
        if (sA > epsilon) dtmax = fmin(dtmax, (1. - s.a[k]) / sA);
        else if (sA < -epsilon) dtmax = fmin(dtmax, -s.a[k] / sA);
      }
#pragma unroll
      for (int k = 0; k < N; k++) rc[k] = eos_rho_ci2(P.eos[k], pI, s.p[k]);
#pragma unroll
      for (int k = 0; k < N; k++) {
        if (s.a[k] > thrA) {
          double sP = -rc[k] * dp[k] / s.a[k];
#pragma unroll
          for (int j = 0; j < N; j++) sP -= (s.p[j] - rc[j]) * dp[j];
          const double dtnew = (pMix - s.p[k]) / mu / sP;
          if (dtnew > 0.) dtmax = fmin(dtmax, dtnew);
        }
      }
      dtmax *= 0.5;
      if (dtmax < dtlocal) dtlocal = dtmax;
    }
#pragma unroll
    for (int k = 0; k < N; k++) {
      if (!anull[k]) {
        const double a0 = s.a[k];
        e[k] = e[k] - dtlocal * mu * pI * dp[k] / dmax<double>(a0 * s.r[k], epsilon);
        s.a[k] = a0 + dtlocal * mu * dp[k];
        s.r[k] = a0 * s.r[k] / dmax<double>(s.a[k], epsilon);
        s.p[k] = eos_pressure<double>(P.eos[k], s.r[k], e[k]);
        verify_correct<M_UEQ, N, double>(P, s, k);
        e[k] = eos_energy<double>(P.eos[k], P.eps, s.r[k], s.p[k]);
        cs[k] = eos_sound<double>(P.eos[k], P.eps, s.r[k], s.p[k]);
      }
    }
    total++;
    tlocal = tlocal + dtlocal;
    if (P.eps > 1.e-20) {
      bool alphaSmall = false;
#pragma unroll
      for (int k = 0; k < N; k++)
        if (s.a[k] > (1. - thrA)) alphaSmall = true;
      if (alphaSmall) break;
    }
    if (iter == 100) {
      relaxed = true;
      break;
    }
  }
  if (relaxed && mu > 1.e-20) {
    double pStar = 0., akS[N], rkS[N];
#pragma unroll
    for (int k = 0; k < N; k++) pStar += ak[k] * pk[k];
    Cell<N> e;   // the entry state, which the Newton relaxes
#pragma unroll
    for (int k = 0; k < N; k++) { e.a[k] = ak[k]; e.r[k] = rk[k]; e.p[k] = pk[k]; }
    NewtonState st{pStar, 0., 1., 0};
    newton_resume<N>(P, e, st, akS, rkS, 100);
    const int it = st.it;
    pStar = st.p;
    total += it;
    flags = newton_flags(it, pStar);
    if (it < 100) {
#pragma unroll
      for (int k = 0; k < N; k++) { s.a[k] = akS[k]; s.r[k] = rkS[k]; s.p[k] = pStar; }
    } else {
      const double pI = interface_p();
#pragma unroll
      for (int k = 0; k < N; k++) s.p[k] = pI;
    }
  }
  return total;
}

template <int N>
__device__ __forceinline__ double relax_guess(const Cell<N>& s) {
  double p = 0.;
#pragma unroll
  for (int k = 0; k < N; k++) p += s.a[k] * s.p[k];
  return p;
}

// Cell::correctionEnergy + FluxPUEq::correctionEnergy (Kapila only), then the
// part of fulfillState that changes stored variables: Euler rebuilds E from (rho,
// p) (PhaseEuler::extendedCalculusPhase).  The multiphase derived quantities are
// not stored and are rebuilt from the primitives by their next reader.  FP64.
template <int MODEL, int N>
__device__ __forceinline__ void correct_and_derive(const Params& P, Cell<N>& s) {
  if (MODEL == M_PUEQ) {
    const double em = s.E - 0.5 * sqn3<double>(s.u);
    double pp = s.rho * em, denom = 0.;
#pragma unroll
    for (int k = 0; k < N; k++) {
      pp -= s.a[k] * (P.eos[k].mixg * (1. - s.r[k] * 0.) + s.r[k] * P.eos[k].eref);
      denom += s.a[k] * P.eos[k].mixinv * (1. - s.r[k] * 0.);
    }
    pp = div_special(pp, denom, rcp_ieee(denom));
#pragma unroll
    for (int k = 0; k < N; k++) {
      s.p[k] = pp;
      verify_correct<MODEL, N, double>(P, s, k);
    }
  }
  if (MODEL == M_EULER) derive<MODEL, N, double>(P, s, true);
}

}  // namespace ecg
