// Kernel templates of the finite-volume step: face-centric tiles.
//
// A 256-thread block owns a tile of cells (256 x 1, 16 x 16, 16 x 4 x 4 or 8 x 8 x 4; small
// meshes take tiles of 64 cells) and
// walks the axes in the reference's face-creation order (X, Y, Z; then the
// boundary faces X-, X+, Y-, Y+, Z-, Z+ of MeshCartesian.cpp:283-557).  For
// each axis it
//   A. (second order) evaluates every face slope the tile needs once into LDS
//      (CellInterfaceO2Cartesian::computeSlopes, CellInterfaceO2Cartesian.cpp:77-99),
//   B. evaluates every interior face flux of the tile once into LDS: MUSCL
//      states (CellO2Cartesian::computeLocalSlopes + extrapolation,
//      CellO2Cartesian.cpp:23-171, CellInterfaceO2Cartesian.cpp:101-202) and the
//      Riemann solver,
//   C. lets each cell add its lower face and subtract its upper face
//      (CellInterface::addFlux / subtractFlux, CellInterface.cpp:267-297).
// Then each thread adds its boundary faces and performs the FP64 cell update,
// primitive rebuild, relaxation and energy correction (Run.cpp:696-716, 771-804;
// CellO2::predictionOrdre2, CellO2.cpp:111-135) and writes the new state.
//
// Second order is two launches: the predictor evaluates fluxes on W^n and writes
// W*; the corrector evaluates them on W* and updates W^n to W^{n+1}.
#pragma once

#include <algorithm>
#include <type_traits>

#include "ecg_kernels.hpp"

namespace ecg {

// Cells per 256-thread tile by dimension and state element size.  3D FP64 tiles
// are 8 x 8 x 4 (fewest halo faces per cell), 3D FP32 tiles 16 x 4 x 4 (longer
// contiguous rows for the narrower rows of floats); both measured faster for
// their form on the 512^3 case.
// Limiter template argument LK of the step kernel: a limiter kind >= 0 fixes every
// limiter of the case at compile time; LK_GENERIC reads the four kinds per face;
// LK_FULL does the same and also builds second-order walls, the THINC
// reconstruction and the finite-rate relaxation (their code costs the other
// instantiations registers).
constexpr int LK_GENERIC = -1;
constexpr int LK_FULL = -2;

// The FP64 kernels of the full-featured instantiation take the correctly rounded
// pow in the star-state isentropes: the finite-rate relaxation's hard thresholds
// would otherwise carry a last-bit difference of the library pow into O(1e-3)
// differences within a dozen steps.
template <typename R, int LK> constexpr bool crpow() { return LK == LK_FULL && sizeof(R) == 8; }

//
// Small meshes in 2D and 3D take tiles of 64 cells (8 x 8 and 4 x 4 x 4), one block's
// waves split over the axes: 128 threads per axis evaluate all its slopes (at most 112),
// then all its fluxes (at most 80), the axes side by side, and the first wave updates the
// cells.  A stage's chain is then one slope, one flux and one update instead of two slopes
// and two fluxes per axis and the update, on four times the blocks (step_small).
//
// The tile shape is named by TK: the element size, plus SMALL_TILE for the small tiles.
constexpr int SMALL_TILE = 64;
constexpr int tile_esize(int tk) { return tk & 63; }
constexpr bool tile_small(int tk) { return tk >= SMALL_TILE; }
template <int D, int TK> struct Tile;
template <int TK> struct Tile<1, TK> { static constexpr int X = 256, Y = 1, Z = 1; };
template <int TK> struct Tile<2, TK> { static constexpr int X = tile_small(TK) ? 8 : 16, Y = X, Z = 1; };
template <> struct Tile<3, 8> { static constexpr int X = 8, Y = 8, Z = 4; };
template <> struct Tile<3, 4> { static constexpr int X = 16, Y = 4, Z = 4; };
template <> struct Tile<3, 8 + SMALL_TILE> { static constexpr int X = 4, Y = 4, Z = 4; };
template <> struct Tile<3, 4 + SMALL_TILE> { static constexpr int X = 4, Y = 4, Z = 4; };
// Cells and threads of a block, and threads that share one axis pass.
template <int TK> constexpr int tile_cells() { return tile_small(TK) ? 64 : 256; }
template <int D, int TK> constexpr int tile_threads() { return tile_small(TK) ? 128 * D : 256; }
template <int TK> constexpr int pass_threads() { return tile_small(TK) ? 128 : 256; }

template <int D, int A, int TK> struct TileAxis {
  static constexpr int T = (A == 0) ? Tile<D, TK>::X : (A == 1) ? Tile<D, TK>::Y : Tile<D, TK>::Z;
  static constexpr int LINES = tile_cells<TK>() / T;
  static constexpr int NSLOPE = (T + 3) * LINES;
  static constexpr int NFACE = (T + 1) * LINES;
};

// LDS bytes one batch of an axis pass may stage (slopes + fluxes); larger
// passes are split into batches of lines so that the resident blocks fit in a
// CU's 160 KB: five blocks of 32 KB, or for the multiphase FP64 kernels, whose
// registers allow three blocks per CU, three of 52 KB (the 8x8 lines of the x
// and y passes then run in one batch).
template <int MODEL, int ES> constexpr int lds_batch_bytes() {
  return (ES == 8 && MODEL != M_EULER) ? 53248 : 32768;
}

// Variables kept per face slope: phase (alpha, rho, p) x N (Euler: rho, p), velocity on the active axes.
template <int MODEL, int N, int D> struct Sizes {
  static constexpr int PV = (MODEL == M_EULER) ? 2 : 3 * N;
  static constexpr int NS = PV + D;
  // flux: alpha, mass, energ per phase (Euler: mass), momentum (D), energy, sM, uStar
  static constexpr int NF = ((MODEL == M_EULER) ? 1 : 3 * N) + D + 1 + 2;
  // Elements staged per line of axis A.
  template <int A, int TK> static constexpr int per_line(bool o2) {
    return (o2 ? (TileAxis<D, A, TK>::T + 3) * NS : 0) + (TileAxis<D, A, TK>::T + 1) * NF;
  }
  // Batches of lines of axis A (the small tiles stage every axis whole).
  template <int A, int TK> static constexpr int batches(bool o2) {
    constexpr int ES = tile_esize(TK);
    int nb = 1;
    while (!tile_small(TK) && nb < TileAxis<D, A, TK>::LINES &&
           per_line<A, TK>(o2) * (TileAxis<D, A, TK>::LINES / nb) * ES > lds_batch_bytes<MODEL, ES>())
      nb *= 2;
    return nb;
  }
  template <int A, int TK> static constexpr int lds_axis(bool o2) {
    return per_line<A, TK>(o2) * (TileAxis<D, A, TK>::LINES / batches<A, TK>(o2));
  }
  static constexpr int cmax(int a, int b) { return a > b ? a : b; }
  template <int TK> static constexpr int lds_elems(bool o2) {
    const int a0 = lds_axis<0, TK>(o2), a1 = D >= 2 ? lds_axis<1, TK>(o2) : 0, a2 = D >= 3 ? lds_axis<2, TK>(o2) : 0;
    return tile_small(TK) ? a0 + a1 + a2 : cmax(a0, cmax(a1, a2));
  }
  // Where axis A's staging starts.
  template <int A, int TK> static constexpr int lds_base(bool o2) {
    return !tile_small(TK) || A == 0 ? 0 : lds_axis<0, TK>(o2) + (A == 2 ? lds_axis<1, TK>(o2) : 0);
  }
};

// Variable v of cell c of a state array (variables pitch cells apart).  OFF32
// (the FP32 step kernels): c counts from the launch's first cell and a launch
// spans at most 4 GiB of a variable (StepLaunchT::cbase), so the byte offset fits
// 32 bits and the access takes the uniform base W + v * pitch plus a per-lane
// 32-bit offset, the scalar-base form of the global memory instructions, with no
// 64-bit address arithmetic per variable.  readfirstlane keeps the base a scalar:
// without it the compiler forms W + offset per lane in 64 bits and adds each
// variable's stride to that.
__device__ __forceinline__ uintptr_t scalar_addr(uintptr_t a) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return ((uintptr_t)hi << 32) | lo;
}
template <bool OFF32, typename S>
__device__ __forceinline__ S ld_var(const S* __restrict__ W, int64_t ld, int v, int64_t c) {
  if constexpr (OFF32) {
    const uintptr_t a = scalar_addr((uintptr_t)(W + v * ld)) + (uint32_t)c * (uint32_t)sizeof(S);
    return *reinterpret_cast<const __attribute__((address_space(1))) S*>(a);
  } else {
    return W[v * ld + c];
  }
}
template <bool OFF32, typename S>
__device__ __forceinline__ void st_var(S* __restrict__ W, int64_t ld, int v, int64_t c, S x) {
  if constexpr (OFF32) {
    const uintptr_t a = scalar_addr((uintptr_t)(W + v * ld)) + (uint32_t)c * (uint32_t)sizeof(S);
    *reinterpret_cast<__attribute__((address_space(1))) S*>(a) = x;
  } else {
    W[v * ld + c] = x;
  }
}
template <typename R> constexpr bool off32() { return sizeof(R) == 4; }

// Persistent variable layout (see include/ecogen_amd.h).
template <int MODEL, int N, int D, bool OFF32 = false, typename S, typename R>
__device__ __forceinline__ void load_prim(const Params& P, const S* __restrict__ W, int64_t c, Cell<N, R>& s) {
  const int64_t ld = P.pitch;
  int v = 0;
  if (MODEL == M_EULER) {
    s.a[0] = R(1.);
    s.r[0] = R(ld_var<OFF32>(W, ld, v++, c));
    s.p[0] = R(ld_var<OFF32>(W, ld, v++, c));
  } else {
#pragma unroll
    for (int k = 0; k < N; k++) {
      s.a[k] = R(ld_var<OFF32>(W, ld, v++, c));
      s.r[k] = R(ld_var<OFF32>(W, ld, v++, c));
      s.p[k] = R(ld_var<OFF32>(W, ld, v++, c));
    }
  }
  s.u[0] = R(ld_var<OFF32>(W, ld, v++, c));
  s.u[1] = (D >= 2) ? R(ld_var<OFF32>(W, ld, v++, c)) : R(0.);
  s.u[2] = (D >= 3) ? R(ld_var<OFF32>(W, ld, v++, c)) : R(0.);
  s.E = R(ld_var<OFF32>(W, ld, v, c));
}

template <int MODEL, int N, int D, bool OFF32 = false, typename S>
__device__ __forceinline__ void store_prim(const Params& P, S* __restrict__ W, int64_t c, const Cell<N>& s) {
  const int64_t ld = P.pitch;
  int v = 0;
  if (MODEL == M_EULER) {
    st_var<OFF32>(W, ld, v++, c, S(s.r[0]));
    st_var<OFF32>(W, ld, v++, c, S(s.p[0]));
  } else {
#pragma unroll
    for (int k = 0; k < N; k++) {
      st_var<OFF32>(W, ld, v++, c, S(s.a[k]));
      st_var<OFF32>(W, ld, v++, c, S(s.r[k]));
      st_var<OFF32>(W, ld, v++, c, S(s.p[k]));
    }
  }
  st_var<OFF32>(W, ld, v++, c, S(s.u[0]));
  if (D >= 2) st_var<OFF32>(W, ld, v++, c, S(s.u[1]));
  if (D >= 3) st_var<OFF32>(W, ld, v++, c, S(s.u[2]));
  st_var<OFF32>(W, ld, v, c, S(s.E));
}

// A stored variable of the new state is NaN or infinite (an invalid state the
// step reports as an error).
template <int MODEL, int N, int D>
__device__ __forceinline__ bool nonfinite_prim(const Cell<N>& s) {
  double acc = s.u[0] * 0.;
  if (D >= 2) acc += s.u[1] * 0.;
  if (D >= 3) acc += s.u[2] * 0.;
  acc += s.E * 0.;
#pragma unroll
  for (int k = 0; k < N; k++) {
    if (MODEL != M_EULER) acc += s.a[k] * 0.;
    acc += s.r[k] * 0. + s.p[k] * 0.;
  }
  return acc != 0.;   // x * 0 is NaN exactly when x is NaN or infinite
}

template <typename R, typename S>
__device__ __forceinline__ R alpha0_at(const S* __restrict__ W, int64_t c) { return R(ld_var<off32<R>()>(W, 0, 0, c)); }

// Cell-to-cell distance of face m of axis AX and the quotient by it: on an axis whose
// distance is one power of two the quotient is the product with its exact inverse
// (the same double); the FP32 form multiplies by the inverse on every uniform axis.
template <typename R, int AX>
struct FaceDist {
  R d, inv;
  bool mul;
  __device__ __forceinline__ FaceDist(const Params& P, int m) {
    const bool uni = (P.dist_uniform >> AX) & 1;
    d = uni ? pv<R>(P.dcc_c[AX], P.f_dcc_c[AX]) : R(face_distance(P.d[AX], m, 0));
    inv = pv<R>(P.inv_dcc[AX], P.f_inv_dcc[AX]);
    mul = (sizeof(R) == 4) ? uni : (((P.dcc_pow2 >> AX) & 1) != 0);
  }
};
template <typename R, int AX>
__device__ __forceinline__ R face_dfl(const Params& P, int m) {
  return ((P.dist_uniform >> AX) & 1) ? pv<R>(P.dfl_c[AX], P.f_dfl_c[AX]) : R(face_distance(P.d[AX], m, 1));
}
template <typename R, int AX>
__device__ __forceinline__ R face_dfr(const Params& P, int m) {
  return ((P.dist_uniform >> AX) & 1) ? pv<R>(P.dfr_c[AX], P.f_dfr_c[AX]) : R(face_distance(P.d[AX], m, 2));
}

// Slope of face (L | L+1): (W_R - W_L) / distance, phase variables then velocity;
// element v at s[v * S].
template <int MODEL, int N, int D, typename R, int AX, int S = 1>
__device__ __forceinline__ void slope_vars(const Cell<N, R>& L, const Cell<N, R>& Rr, const FaceDist<R, AX>& dist,
                                           R* s) {
  int v = 0;
  // One branch for the whole slope (a per-quotient select would evaluate both forms).
  if (dist.mul) {
#pragma unroll
    for (int k = 0; k < N; k++) {
      if (MODEL != M_EULER) s[S * v++] = (Rr.a[k] - L.a[k]) * dist.inv;
      s[S * v++] = (Rr.r[k] - L.r[k]) * dist.inv;
      s[S * v++] = (Rr.p[k] - L.p[k]) * dist.inv;
    }
#pragma unroll
    for (int d = 0; d < D; d++) s[S * v++] = (Rr.u[d] - L.u[d]) * dist.inv;
    return;
  }
  // One reciprocal for every quotient by the distance (FP64: the IEEE quotients bit for
  // bit at three instructions each; the full division sequence took twelve, 9 % of the 2D
  // and 3D two-phase FP64 steps on meshes whose spacing is no power of two).
  const Quot<R> q(dist.d);
#pragma unroll
  for (int k = 0; k < N; k++) {
    if (MODEL != M_EULER) s[S * v++] = q(Rr.a[k] - L.a[k]);
    s[S * v++] = q(Rr.r[k] - L.r[k]);
    s[S * v++] = q(Rr.p[k] - L.p[k]);
  }
#pragma unroll
  for (int d = 0; d < D; d++) s[S * v++] = q(Rr.u[d] - L.u[d]);
}

// Limited slopes of one cell side, kinds known only at run time: one switch for all the
// variables of a kind (lvf the volume fractions, lg the rest).  A switch per variable had
// kept the variables apart and broke every
// face into dozens of blocks (Euler O2 with walls and van Leer, 107 x 109 x 105: 365 -> 326 us).
template <int MODEL, int N, int D, typename R, int S, bool VF>
__device__ __forceinline__ void limit_slopes(int kind, const R* s1, const R* s2, R* out) {
  constexpr int PV = (MODEL == M_EULER) ? 2 : 3 * N;
  auto all = [&](auto k) {
#pragma unroll
    for (int v = 0; v < PV + D; v++)
      if ((MODEL != M_EULER && v < PV && v % 3 == 0) == VF) out[v] = limit<R>(decltype(k)::value, s1[S * v], s2[S * v]);
  };
  switch (kind) {
    case LIM_THINC:   // minmod where the reconstruction itself does not apply
    case LIM_MINMOD: all(std::integral_constant<int, LIM_MINMOD>{}); break;
    case LIM_VANLEER: all(std::integral_constant<int, LIM_VANLEER>{}); break;
    case LIM_VANALBADA: all(std::integral_constant<int, LIM_VANALBADA>{}); break;
    case LIM_SUPERBEE: all(std::integral_constant<int, LIM_SUPERBEE>{}); break;
    case LIM_MC: all(std::integral_constant<int, LIM_MC>{}); break;
    default: all(std::integral_constant<int, LIM_NONE>{}); break;
  }
}

// computeLocalSlopes + limitSlopes + extrapolate + verifyAndCorrectPhase on a
// uniform Cartesian cell: slope1 is the face's own slope, slope2 the opposite
// face's (zero on a boundary face that carries none, as the opposite alpha).  negate: right cell (changeSign,
// CellInterfaceO2Cartesian.cpp:151-156).  LK >= 0: every limiter of the case is
// of kind LK (no interface switch to evaluate); LK < 0: kinds from P.lim.  Slope
// element v at s1[v * S].
template <int MODEL, int N, int D, typename R, int LK, int S = 1>
__device__ __forceinline__ void extrapolate(const Params& P, Cell<N, R>& b, const R* s1, const R* s2,
                                            R aAfter, R aCell, R aOther, R dist, bool negate) {
  int lg = LK, lvf = LK;
  if (LK < 0) {
    if ((aCell >= R(1.e-4)) && (aCell <= R(1.) - R(1.e-4)) && ((aOther - aCell) * (aCell - aAfter) >= R(1.e-8))) {
      lg = P.lim[1]; lvf = P.lim[3];
    } else {
      lg = P.lim[0]; lvf = P.lim[2];
    }
  }
  // All the variables' limited slopes together, except in the three-phase kernels with the kind
  // fixed at compile time, where each waits until it is used: together they cost the 3D
  // second-order FP32 kernels 4-5 VGPRs more than the 128 of four waves (93 x 95 x 91, us a step
  // together / apart: FP64 671 / 639, FP32 244 / 239; two phases 119 x 113 x 117 FP32 330 / 334).
  constexpr bool LATE = LK >= 0 && N == 3;
  constexpr int NL = (MODEL == M_EULER ? 2 : 3 * N) + D;
  R lim[NL];
  if constexpr (LK < 0) {
    if (MODEL != M_EULER) limit_slopes<MODEL, N, D, R, S, true>(lvf, s1, s2, lim);
    limit_slopes<MODEL, N, D, R, S, false>(lg, s1, s2, lim);
  } else if constexpr (!LATE) {
#pragma unroll
    for (int v = 0; v < NL; v++) lim[v] = limit<R>(LK, s1[S * v], s2[S * v]);
  }
  auto late = [&](int v) {
    if constexpr (LATE) lim[v] = limit<R>(LK, s1[S * v], s2[S * v]);
  };
  int v = 0;
#pragma unroll
  for (int k = 0; k < N; k++) {
    R la = R(0.), lr, lp;
    if (MODEL != M_EULER) { late(v); la = lim[v]; v++; }
    late(v); lr = lim[v]; v++;
    late(v); lp = lim[v]; v++;
    if (negate) { la = -la; lr = -lr; lp = -lp; }
    if (MODEL != M_EULER) b.a[k] += la * dist;
    b.r[k] += lr * dist;
    b.p[k] += lp * dist;
    if (MODEL == M_EULER) {
#pragma unroll
      for (int d = 0; d < D; d++) {
        late(v + d);
        R lu = lim[v + d];
        if (negate) lu = lu * R(-1.);
        b.u[d] = b.u[d] + lu * dist;
      }
    }
    verify_correct<MODEL, N, R>(P, b, k);
  }
  if (MODEL != M_EULER) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      late(v + d);
      R lu = lim[v + d];
      if (negate) lu = lu * R(-1.);
      b.u[d] = b.u[d] + lu * dist;
    }
  }
}

// BoundCondWallO2Cartesian::computeSlopes (BoundCondWallO2Cartesian.cpp:88-112):
// every slope zero but the wall-normal velocity, u_n / (x_cell - x_face); dw is
// that signed distance (positive on the minus side); element v at o[v * S].
template <int MODEL, int N, int D, typename R, int S = 1>
__device__ __forceinline__ void wall_slope_vars(const Cell<N, R>& c, int ax, R dw, R* o) {
  constexpr int PV = (MODEL == M_EULER) ? 2 : 3 * N;
#pragma unroll
  for (int v = 0; v < PV + D; v++) o[S * v] = R(0.);
  if (fabs(dw) > R(1.e-8)) o[S * (PV + ax)] = fdiv(c.u[ax], dw);
}

// Second-order wall state (BoundCondWallO2Cartesian::solveRiemann,
// BoundCondWallO2Cartesian.cpp:116-151, with CellO2Cartesian::computeLocalSlopesLimite,
// CellO2Cartesian.cpp:173-277): slope 1 is the wall's, slope 2 the inner face's on
// the other side of the cell; the interface switch reads only the cell's own
// time-n volume fraction; the extrapolated phases are not checked.
template <int MODEL, int N, int D, typename R, int LK>
__device__ __forceinline__ void extrapolate_wall(const Params& P, Cell<N, R>& b, const R* s1, const R* s2, R aCell,
                                                 R dist) {
  int lg = LK, lvf = LK;
  if (LK < 0) {
    if ((aCell >= R(1.e-4)) && (aCell <= R(1.) - R(1.e-4))) {
      lg = P.lim[1]; lvf = P.lim[3];
    } else {
      lg = P.lim[0]; lvf = P.lim[2];
    }
  }
  R lim[(MODEL == M_EULER ? 2 : 3 * N) + D];
  if (MODEL != M_EULER) limit_slopes<MODEL, N, D, R, 1, true>(lvf, s1, s2, lim);
  limit_slopes<MODEL, N, D, R, 1, false>(lg, s1, s2, lim);
  int v = 0;
#pragma unroll
  for (int k = 0; k < N; k++) {
    if (MODEL != M_EULER) { b.a[k] += lim[v] * dist; v++; }
    b.r[k] += lim[v] * dist; v++;
    b.p[k] += lim[v] * dist; v++;
  }
#pragma unroll
  for (int d = 0; d < D; d++) b.u[d] = b.u[d] + lim[v + d] * dist;
}

// A staged face flux: element v at o[v * S].
template <int MODEL, int N, int D, int S, typename R>
__device__ __forceinline__ void flux_to_lds(const Flux<N, R>& F, R* o) {
  int v = 0;
  if (MODEL == M_EULER) {
    o[S * v++] = F.f.mass[0];
  } else {
#pragma unroll
    for (int k = 0; k < N; k++) { o[S * v++] = F.f.alpha[k]; o[S * v++] = F.f.mass[k]; o[S * v++] = F.f.energ[k]; }
  }
#pragma unroll
  for (int d = 0; d < D; d++) o[S * v++] = F.f.mom[d];
  o[S * v++] = F.f.energM;
  o[S * v++] = F.sM;
  o[S * v++] = F.uStar;
}

template <int MODEL, int N, int D, int S, typename R>
__device__ __forceinline__ void flux_from_lds(const R* o, Flux<N, R>& F) {
  int v = 0;
  if (MODEL == M_EULER) {
    F.f.mass[0] = o[S * v++];
  } else {
#pragma unroll
    for (int k = 0; k < N; k++) { F.f.alpha[k] = o[S * v++]; F.f.mass[k] = o[S * v++]; F.f.energ[k] = o[S * v++]; }
  }
#pragma unroll
  for (int d = 0; d < D; d++) F.f.mom[d] = o[S * v++];
  F.f.energM = o[S * v++];
  F.sM = o[S * v++];
  F.uStar = o[S * v++];
}

// Tile origin of the block among the launch's tile rows (row0, nrows of the
// outermost axis).
template <int MODEL, int N, int D, bool LEARN, int TK>
__device__ __forceinline__ void tile_origin(const Params& P, int row0, int nrows, int& i0, int& j0, int& k0) {
  const int tiles1 = tile_small(TK) ? (P.ny + Tile<D, TK>::Y - 1) / Tile<D, TK>::Y : P.tiles[1];
  const int t0 = (D == 1) ? nrows : tile_small(TK) ? (P.nx + Tile<D, TK>::X - 1) / Tile<D, TK>::X : P.tiles[0];
  const int t1 = (D == 2) ? nrows : (D == 3) ? tiles1 : 1;
  const int nb = t0 * t1 * ((D == 3) ? nrows : 1);
  // The rule's runs as constants, so that the order takes shifts.
  constexpr int RUN = tile_small(TK) ? 0 : tile_run(MODEL, N, D, tile_esize(TK), LEARN, 4096);
  constexpr int FEW = tile_small(TK) ? 0 : tile_run(MODEL, N, D, tile_esize(TK), LEARN, 1);
  const int run = tile_run(MODEL, N, D, tile_esize(TK), LEARN, nb);
  const int b = (RUN > 0 && run == RUN)   ? xcd_tile(nb, blockIdx.x, RUN)
                : (FEW > 0 && run == FEW) ? xcd_tile(nb, blockIdx.x, FEW)
                                          : xcd_tile(nb, blockIdx.x, 0);
  int tx = b % t0;
  const int rest = b / t0;
  int ty = rest % t1;
  int tz = rest / t1;
  if (D == 3 && TK == 4 && (t1 & 1) == 0 && (nrows & 1) == 0) {
    // 3D FP32 tiles (16 x 4 x 4): rows of x tiles in 2 x 2 groups over (y, z), so
    // that the y and the z neighbours of a row run close in time and meet their
    // shared halo planes in L2 (the 512^3 step fetches 13 % less).
    const int blk = rest >> 2, w = rest & 3, hy = P.tiles[1] >> 1;
    ty = 2 * (blk % hy) + (w & 1);
    tz = 2 * (blk / hy) + (w >> 1);
  }
  if (D == 1) tx += row0;
  else if (D == 2) ty += row0;
  else tz += row0;
  i0 = tx * Tile<D, TK>::X;
  j0 = ty * Tile<D, TK>::Y;
  k0 = tz * Tile<D, TK>::Z;
}

// Accumulators that wait in the thread's own LDS slots while the fluxes are evaluated.  The 3D
// three-phase FP64 kernels need 187 (first order) and 195 registers and have 168 (three
// waves per SIMD); what a third of a CU's LDS holds beside the staging, seven and six
// doubles a thread (nine in 2D), takes the accumulators out of the flux passes, where they had been
// spilled and reloaded in every pass (256^3 first order: 3186 -> 2657 us a step; two waves
// per SIMD without spills: 3242).  18 (VELOCITYEQ) or 32 VGPRs (Kapila) at first order and 38 to 90 at second
// order still spill.  The cold first-order FP32 kernel runs five waves that way (step_waves); the
// learned one gains no wave, runs 2 % faster without (256^3 13.73 -> 14.01 Gcell-updates/s), and its
// inference, whose rows start at offset 0 of the LDS, then meets no waiting accumulators.
template <int MODEL, int N, int D, bool O2, int TK, int LK, bool LEARN> constexpr int acc_stash() {
  if (LEARN || !(N == 3 && D >= 2 && (TK == 8 || (TK == 4 && !O2)) && LK != LK_FULL)) return 0;
  const int room = ((TK == 8 ? 53760 : 32256) - TK * Sizes<MODEL, N, D>::template lds_elems<TK>(O2)) / (256 * 8);
  return room < 3 * N ? room : 3 * N;
}
template <int NS, int N, typename R, class F> __device__ __forceinline__ void each_stashed(ConsAcc<N, R>& acc, F f) {
  int v = 0;
#pragma unroll
  for (int k = 0; k < N; k++) {
    if (v < NS) { f(acc.alpha[k].v, v); v++; }
    if (v < NS) { f(acc.mass[k].v, v); v++; }
    if (v < NS) { f(acc.energ[k].v, v); v++; }
  }
}

// One axis pass (steps A, B, C above) for axis AX with face frame FR, in
// batches of lines when the staging would exceed lds_batch_bytes.  The small tiles call
// one step at a time (STEPS) on the axis's own threads, with the barriers between them.
constexpr int STEP_A = 1, STEP_B = 2, STEP_C = 4, STEP_ABC = 7;
template <int MODEL, int N, int D, bool O2, typename R, int LK, int AX, int FR, bool LEARN, int TK = (int)sizeof(R), int STEPS = STEP_ABC>
__device__ __forceinline__ void axis_pass(const Params& P, const StepLaunchT<R>& L, R* lds, const int org[3],
                                          const int own[3], bool own_ok, const R* an, const R* pn, R& smax,
                                          ConsAcc<N, R>& acc) {
  using TA = TileAxis<D, AX, TK>;
  using SZ = Sizes<MODEL, N, D>;
  constexpr int T = TA::T;
  constexpr int NB = SZ::template batches<AX, TK>(O2);
  constexpr int LB = TA::LINES / NB;              // lines per batch
  constexpr int B = (AX == 0) ? 1 : 0;           // first line axis
  constexpr int C = (AX == 2) ? 1 : 2;           // second line axis
  constexpr int TB = (B == 0) ? Tile<D, TK>::X : Tile<D, TK>::Y;
  // Cell indices: 32-bit from the launch's first cell in FP32, 64-bit in FP64.
  using CI = typename std::conditional<off32<R>(), uint32_t, int64_t>::type;
  const int n3[3] = {P.nx, P.ny, P.nz};
  const CI st3[3] = {CI(1), (CI)P.nx, (CI)P.nx * (CI)P.ny};
  const CI cb0 = off32<R>() ? (CI)L.cbase : CI(0);
  const int na = n3[AX];
  const CI sa = st3[AX];
  R* s_slope = lds + SZ::template lds_base<AX, TK>(O2);
  R* s_flux = s_slope + (O2 ? (T + 3) * LB * SZ::NS : 0);
  // Face slopes: slot g of line lb is s = lb * (T + 3) + g + 2.  A slope of NS
  // elements whose bytes are a multiple of 32 (8 doubles in 2D with two phases,
  // 12 in 3D with three; 8 floats in 2D) is staged variable-major, element v at
  // v * NSLOT + s: as a record, neighbouring lanes' 16-byte accesses would fall
  // in the same banks.  Other sizes stay records of NS consecutive elements.
  constexpr int NSLOT = (T + 3) * LB;
  constexpr bool SVM = (SZ::NS * (int)sizeof(R)) % 32 == 0;
  constexpr int SRS = SVM ? 1 : SZ::NS;     // slot stride
  constexpr int SES = SVM ? NSLOT : 1;      // element stride
  // Face flux records r = line * (T + 1) + face.  FP32: NF consecutive floats per
  // record (48 bytes for two phases in 3D: neighbouring lanes' 16-byte accesses
  // fall in distinct banks).  FP64: variable-major, element v of record r at
  // v * NREC + r, so that the lanes' 8-byte accesses walk consecutive addresses
  // (records of 12 doubles put neighbouring lanes' 16-byte accesses 96 bytes
  // apart, in the same banks).
  constexpr int NREC = (T + 1) * LB;
  constexpr int FRS = (sizeof(R) == 8) ? 1 : SZ::NF;     // record stride
  constexpr int FES = (sizeof(R) == 8) ? NREC : 1;       // element stride
  const int tid = tile_small(TK) ? threadIdx.x % pass_threads<TK>() : threadIdx.x;
  const int lown = (own[B] - org[B]) + TB * (own[C] - org[C]);   // line of the own cell
  // Work slots of steps A and B run along the axis for x (contiguous cells), and
  // across the lines for y and z, whose consecutive lines are consecutive x: a
  // wave's loads then walk along x in every pass.
  constexpr bool ACROSS = (AX != 0);
  // Second-order walls: their slopes enter the neighbouring cells' limiters.
  const bool wall_m = O2 && LK == LK_FULL && P.bc[2 * AX] == BC_WALL;
  const bool wall_p = O2 && LK == LK_FULL && P.bc[2 * AX + 1] == BC_WALL;

#pragma unroll 1
  for (int bt = 0; bt < NB; bt++) {
    const int l0 = bt * LB;
    // A. face slopes s_g, g = -2 .. T (interior faces only)
    if constexpr (O2 && (STEPS & STEP_A)) {
      for (int q = tid; q < (T + 3) * LB; q += pass_threads<TK>()) {
        const int g = (ACROSS ? q / LB : q % (T + 3)) - 2;
        const int lb = ACROSS ? q % LB : q / (T + 3);
        const int l = l0 + lb;
        const int cb = org[B] + l % TB, cc = org[C] + l / TB;
        const int m = org[AX] + g;
        R* o = s_slope + (lb * (T + 3) + g + 2) * SRS;
        if (cb < n3[B] && cc < n3[C] && m >= 0 && m <= na - 2) {
          const CI cell = (CI)m * sa + (CI)cb * st3[B] + (CI)cc * st3[C] - cb0;
          Cell<N, R> cl, cr;
          load_prim<MODEL, N, D, off32<R>()>(P, L.wsrc, cell, cl);
          load_prim<MODEL, N, D, off32<R>()>(P, L.wsrc, cell + sa, cr);
          slope_vars<MODEL, N, D, R, AX, SES>(cl, cr, FaceDist<R, AX>(P, m), o);
        } else if (cb < n3[B] && cc < n3[C] && ((m == -1 && wall_m) || (m == na - 1 && wall_p))) {
          // Wall faces carry slopes (second order); the cell is the one inside.
          const CI cell = (CI)(m < 0 ? 0 : na - 1) * sa + (CI)cb * st3[B] + (CI)cc * st3[C] - cb0;
          Cell<N, R> cw;
          load_prim<MODEL, N, D, off32<R>()>(P, L.wsrc, cell, cw);
          wall_slope_vars<MODEL, N, D, R, SES>(cw, AX, m < 0 ? pv<R>(P.dwall[AX][0], P.f_dwall[AX][0]) : -pv<R>(P.dwall[AX][1], P.f_dwall[AX][1]), o);
        } else if (cb < n3[B] && cc < n3[C]) {
          // No slope beyond the mesh: the limiters read zeros, without a test per variable
          // (which kept the reads of a record apart, each behind its own mask).
#pragma unroll
          for (int v = 0; v < SZ::NS; v++) o[SES * v] = R(0.);
        }
      }
      if (STEPS == STEP_ABC) __syncthreads();
    }

    // B. interior face fluxes f = -1 .. T-1
    if constexpr (STEPS & STEP_B) {
      for (int q = tid; q < (T + 1) * LB; q += pass_threads<TK>()) {
        const int f = (ACROSS ? q / LB : q % (T + 1)) - 1;
        const int lb = ACROSS ? q % LB : q / (T + 1);
        const int l = l0 + lb;
        const int cb = org[B] + l % TB, cc = org[C] + l / TB;
        const int m = org[AX] + f;
        if (cb < n3[B] && cc < n3[C] && m >= 0 && m <= na - 2) {
          const CI cell = (CI)m * sa + (CI)cb * st3[B] + (CI)cc * st3[C] - cb0;
          Cell<N, R> bl, br;
          load_prim<MODEL, N, D, off32<R>()>(P, L.wsrc, cell, bl);
          load_prim<MODEL, N, D, off32<R>()>(P, L.wsrc, cell + sa, br);
          if (O2) {
            const R aL = (MODEL == M_EULER) ? R(0.) : bl.a[0];
            const R aR = (MODEL == M_EULER) ? R(0.) : br.a[0];
            const R* s1 = s_slope + (lb * (T + 3) + f + 2) * SRS;
            const bool hasm = (m >= 1) || wall_m, hasp = (m + 1 <= na - 2) || wall_p;
            // The far neighbours' time-n alpha only decides the interface limiter switch;
            // across a wall the "cell after" is the cell itself (CellO2Cartesian.cpp:75-79).
            const R aLL = (LK < 0 && MODEL != M_EULER && hasm) ? alpha0_at<R>(L.wn, (m >= 1) ? cell - sa : cell) : R(0.);
            const R aRR = (LK < 0 && MODEL != M_EULER && hasp)
                              ? alpha0_at<R>(L.wn, (m + 1 <= na - 2) ? cell + 2 * sa : cell + sa)
                              : R(0.);
            extrapolate<MODEL, N, D, R, LK, SES>(P, bl, s1, s1 - SRS, aLL, aL, aR, face_dfl<R, AX>(P, m), false);
            extrapolate<MODEL, N, D, R, LK, SES>(P, br, s1, s1 + SRS, aRR, aR, aL, face_dfr<R, AX>(P, m), true);
            if constexpr (LK == LK_FULL && MODEL != M_EULER && N == 2) {
              if (P.thinc) {
                // THINC replaces the extrapolated volume fractions at an interface.
                double na;
                if (thinc_alpha(P, 0, (double)aL, (double)aLL, (double)aR, na)) { bl.a[0] = R(na); bl.a[1] = R(1. - na); }
                if (thinc_alpha(P, 1, (double)aR, (double)aRR, (double)aL, na)) { br.a[0] = R(na); br.a[1] = R(1. - na); }
              }
            }
            derive<MODEL, N, R>(P, bl, MODEL == M_EULER);
            derive<MODEL, N, R>(P, br, MODEL == M_EULER);
          } else {
            derive<MODEL, N, R>(P, bl, false);
            derive<MODEL, N, R>(P, br, false);
          }
          Flux<N, R> F;
          face_flux<MODEL, N, FR, R, crpow<R, LK>()>(P, bl, bl.E, br, br.E, smax, F);
          flux_to_lds<MODEL, N, D, FES, R>(F, s_flux + (lb * (T + 1) + f + 1) * FRS);
        } else if (sizeof(R) == 4 && cb < n3[B] && cc < n3[C]) {
          // The FP32 gather reads both faces of every cell: a face outside the mesh is zero.
          R* o = s_flux + (lb * (T + 1) + f + 1) * SZ::NF;
  #pragma unroll
          for (int v = 0; v < SZ::NF; v++) o[v] = R(0.);
        }
      }
    }
    if (STEPS == STEP_ABC) __syncthreads();

    // C. gather: add the lower face, subtract the upper face
    constexpr int ST = acc_stash<MODEL, N, D, O2, TK, LK, LEARN>();
    double* st = reinterpret_cast<double*>(lds + SZ::template lds_elems<TK>(O2)) + threadIdx.x;
    if constexpr (ST > 0) each_stashed<ST, N, R>(acc, [&](double& x, int v) { x = st[256 * v]; });
    if ((STEPS & STEP_C) && own_ok && lown / LB == bt) {
      const int t = own[AX] - org[AX];
      const int lb = lown - l0;
      const R coef = pv<R>(P.coef[AX], P.f_coef[AX]);
      if constexpr (sizeof(R) == 4) {
        Flux<N, R> Fl, Fu;
        flux_from_lds<MODEL, N, D, FES, R>(s_flux + (lb * (T + 1) + t) * FRS, Fl);
        flux_from_lds<MODEL, N, D, FES, R>(s_flux + (lb * (T + 1) + t + 1) * FRS, Fu);
        add_flux_pair<MODEL, N, D>(acc, Fl, Fu, coef, an, pn);
      } else {
        Flux<N, R> F;
        if (own[AX] > 0) {
          flux_from_lds<MODEL, N, D, FES, R>(s_flux + (lb * (T + 1) + t) * FRS, F);
          add_flux<MODEL, N, D, R>(acc, F, coef, an, pn);
        }
        if (own[AX] < na - 1) {
          flux_from_lds<MODEL, N, D, FES, R>(s_flux + (lb * (T + 1) + t + 1) * FRS, F);
          sub_flux<MODEL, N, D, R>(acc, F, coef, an, pn);
        }
      }
    }
    if constexpr (ST > 0) each_stashed<ST, N, R>(acc, [&](double& x, int v) { st[256 * v] = x; });
    if (STEPS == STEP_ABC) __syncthreads();
  }
}

template <int MODEL, int N, int D, int FR, typename R, bool CRPOW>
__device__ __forceinline__ void boundary_face(const Params& P, const Cell<N, R>& b, int bc, R coef, const R* an,
                                              const R* pn, R& smax, ConsAcc<N, R>& acc) {
  Flux<N, R> F;
  const R EB = (MODEL == M_EULER) ? b.e[0] + R(0.5) * sqn3<R>(b.u) : b.E;
  boundary_flux<MODEL, N, FR, R, CRPOW>(P, b, EB, bc, smax, F);
  sub_flux<MODEL, N, D, R>(acc, F, coef, an, pn);
}

// The step kernel's side of an inlet-tank face: the record k_tank wrote for it.
template <int MODEL, int N, int D, int AX, int SIDE, typename R>
__device__ __forceinline__ void tank_face(const Params& P, const int* own, R coef, const R* an, const R* pn,
                                          ConsAcc<N, R>& acc) {
  // 32-bit (a side has fewer than 2^31 faces), recomputed here rather than kept
  // live from the cell index's products.
  const int f = (AX == 0) ? own[1] + P.ny * own[2] : (AX == 1) ? own[0] + P.nx * own[2] : own[0] + P.nx * own[1];
  const R* rec = reinterpret_cast<const R*>(P.tank_buf) + (P.tank_off[2 * AX + SIDE] + f) * TANK_REC;
  Flux<N, R> F;
#pragma unroll
  for (int k = 0; k < N; k++) { F.f.alpha[k] = R(rec[k]); F.f.mass[k] = R(rec[4 + k]); F.f.energ[k] = R(rec[8 + k]); }
  F.f.mom[0] = R(rec[12]); F.f.mom[1] = R(rec[13]); F.f.mom[2] = R(rec[14]);
  F.f.energM = R(rec[15]);
  F.sM = R(rec[16]);
  F.uStar = R(rec[17]);
  sub_flux<MODEL, N, D, R>(acc, F, coef, an, pn);
}

// Boundary face of axis AX, side SIDE (0: minus, 1: plus) of the own cell c
// (coordinates own).  A second-order wall first extrapolates the cell's stage
// state to the face (LK_FULL kernels); an inlet tank's flux comes from k_tank.
template <int MODEL, int N, int D, bool O2, int AX, int SIDE, int FR, typename R, int LK>
__device__ __forceinline__ void boundary_face_at(const Params& P, const StepLaunchT<R>& L, const Cell<N, R>& src,
                                                 int64_t c, const int* own, const R* an, const R* pn, R& smax,
                                                 ConsAcc<N, R>& acc) {
  const int bc = P.bc[2 * AX + SIDE];
  const R coef = pv<R>(P.coef[AX], P.f_coef[AX]);
  if (bc == BC_TANK) {
    tank_face<MODEL, N, D, AX, SIDE, R>(P, own, coef, an, pn, acc);
    return;
  }
  if (!O2 || LK != LK_FULL || bc != BC_WALL) {
    boundary_face<MODEL, N, D, FR, R, crpow<R, LK>()>(P, src, bc, coef, an, pn, smax, acc);
    return;
  }
  using SZ = Sizes<MODEL, N, D>;
  const int n3[3] = {P.nx, P.ny, P.nz};
  const int64_t sa = (AX == 0) ? 1 : (AX == 1) ? (int64_t)P.nx : (int64_t)P.nx * P.ny;
  const int na = n3[AX];
  R s1[SZ::NS], s2[SZ::NS];
  wall_slope_vars<MODEL, N, D, R>(src, AX, SIDE == 0 ? pv<R>(P.dwall[AX][0], P.f_dwall[AX][0]) : -pv<R>(P.dwall[AX][1], P.f_dwall[AX][1]), s1);
  // Slope of the inner face on the other side of the cell.
  Cell<N, R> nb;
  load_prim<MODEL, N, D, off32<R>()>(P, L.wsrc, SIDE == 0 ? c + sa : c - sa, nb);
  if (SIDE == 0) slope_vars<MODEL, N, D, R, AX>(src, nb, FaceDist<R, AX>(P, 0), s2);
  else slope_vars<MODEL, N, D, R, AX>(nb, src, FaceDist<R, AX>(P, na - 2), s2);
  const R aCell = (MODEL == M_EULER) ? R(0.) : alpha0_at<R>(L.wn, c);
  Cell<N, R> b = src;
  extrapolate_wall<MODEL, N, D, R, LK>(P, b, s1, s2, aCell, SIDE == 0 ? -pv<R>(P.dwall[AX][0], P.f_dwall[AX][0]) : pv<R>(P.dwall[AX][1], P.f_dwall[AX][1]));
  derive<MODEL, N, R>(P, b, MODEL == M_EULER);
  boundary_face<MODEL, N, D, FR, R, crpow<R, LK>()>(P, b, bc, coef, an, pn, smax, acc);
}

__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = dmin<double>(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ unsigned long long wave_sum(unsigned long long v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// The step kernels' wave reductions, by DPP moves (row shifts, then the row broadcasts of a
// 64-wide wave; lane 63 ends with the whole): no LDS pipe, and a few cycles a step where a
// cross-lane permute is a round trip of about a hundred.  Lanes without a source take 0, the
// identity of both reductions (speeds are not negative).
template <int CTRL, int ROWS> __device__ __forceinline__ uint32_t dpp0(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS> __device__ __forceinline__ float dpp0(float x) {
  return __builtin_bit_cast(float, dpp0<CTRL, ROWS>(__builtin_bit_cast(uint32_t, x)));
}
template <int CTRL, int ROWS> __device__ __forceinline__ double dpp0(double x) {
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  return __builtin_bit_cast(double, (uint64_t)dpp0<CTRL, ROWS>((uint32_t)b) |
                                        ((uint64_t)dpp0<CTRL, ROWS>((uint32_t)(b >> 32)) << 32));
}
template <typename T, class Op> __device__ __forceinline__ T wave_reduce63(T v, Op op) {
  v = op(v, dpp0<0x111, 0xf>(v));   // row_shr 1, 2, 4, 8
  v = op(v, dpp0<0x112, 0xf>(v));
  v = op(v, dpp0<0x114, 0xf>(v));
  v = op(v, dpp0<0x118, 0xf>(v));
  v = op(v, dpp0<0x142, 0xa>(v));   // row_bcast 15 into rows 1 and 3
  v = op(v, dpp0<0x143, 0xc>(v));   // row_bcast 31 into rows 2 and 3
  return v;
}

// Inlet-tank faces (BoundCondInletTank::solveRiemannBoundary,
// BoundCondInletTank.cpp:209-212), one thread each, ahead of the step kernel:
// the buffer cell is the stage state of the boundary cell, as for every
// first-order boundary class, and the tank solver runs in FP64.  Each face's
// flux goes to its record of P.tank_buf, where the step kernel picks it up in
// the reference's face order; the tank's wave speeds join the step's dtMax
// through the counter slots.  A Newton that spends its 50 iterations counts in
// tank_fail and leaves a zero flux.  Faces of a side are numbered in plane
// order: (j, k) for x sides, (i, k) for y sides, (i, j) for z sides.
template <int MODEL, int N, int FR, typename S>
__device__ __forceinline__ int tank_record(const Params& P, const TankDev& T, const Cell<N, double>& b, double& dtm,
                                           S* rec) {
  double lu[3];
  to_local<FR, double>(b.u, lu);
  Flux<N, double> F = {};
  const int it = tank_flux<MODEL, N>(P, T, b, lu, dtm, F);
  if (it < 0) F = Flux<N, double>{};
  const double loc[3] = {F.f.mom[0], F.f.mom[1], F.f.mom[2]};
  to_global<FR, double>(loc, F.f.mom);
#pragma unroll
  for (int k = 0; k < N; k++) { rec[k] = S(F.f.alpha[k]); rec[4 + k] = S(F.f.mass[k]); rec[8 + k] = S(F.f.energ[k]); }
  rec[12] = S(F.f.mom[0]); rec[13] = S(F.f.mom[1]); rec[14] = S(F.f.mom[2]);
  rec[15] = S(F.f.energM); rec[16] = S(F.sM); rec[17] = S(F.uStar);
  return it;
}

template <int MODEL, int N, int D, typename S>
__global__ __launch_bounds__(256, 4) void k_tank(ParamsPtr Pc, const S* __restrict__ wsrc, const Clock* __restrict__ clk,
                                              Counters* __restrict__ cnt, int64_t nfaces) {
  const Params& P = *(const Params*)Pc;
  __shared__ double s_dt[4];
  __shared__ int s_bad[4];
  if (clk->done) return;
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  double dtm = 1.e10;
  int bad = 0;
  if (g < nfaces) {
    // The sides' record ranges are disjoint and increasing: the last tank side starting at or before g owns it.
    int side = 0;
    for (int q = 0; q < 2 * D; q++)
      if (P.bc[q] == BC_TANK && P.tank_off[q] <= g) side = q;
    const int64_t f = g - P.tank_off[side];
    const int ax = side >> 1, hi = side & 1;
    const int64_t na = (ax == 0) ? P.ny : P.nx;                // first plane axis extent
    const int64_t u = f % na, v = f / na;
    int64_t i, j, k;
    if (ax == 0) { i = hi ? P.nx - 1 : 0; j = u; k = v; }
    else if (ax == 1) { i = u; j = hi ? P.ny - 1 : 0; k = v; }
    else { i = u; j = v; k = hi ? P.nz - 1 : 0; }
    const int64_t c = i + j * P.nx + k * (int64_t)P.nx * P.ny;
    Cell<N, double> b;
    load_prim<MODEL, N, D>(P, wsrc, c, b);
    derive<MODEL, N, double>(P, b, MODEL == M_EULER);
    // Records in the state's precision (the FP32 form's fluxes are float).
    S* rec = reinterpret_cast<S*>(P.tank_buf) + g * TANK_REC;
    const TankDev& T = P.tank[side];
    int it = 0;
    switch (side) {
      case 0: it = tank_record<MODEL, N, FR_XM, S>(P, T, b, dtm, rec); break;
      case 1: it = tank_record<MODEL, N, FR_XP, S>(P, T, b, dtm, rec); break;
      case 2: it = tank_record<MODEL, N, FR_YM, S>(P, T, b, dtm, rec); break;
      case 3: it = tank_record<MODEL, N, FR_YP, S>(P, T, b, dtm, rec); break;
      case 4: it = tank_record<MODEL, N, FR_ZM, S>(P, T, b, dtm, rec); break;
      default: it = tank_record<MODEL, N, FR_ZP, S>(P, T, b, dtm, rec); break;
    }
    bad = it < 0 ? 1 : 0;
  }
  const double m = wave_min(dtm);
  const int nb = (int)wave_sum((unsigned long long)bad);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0) { s_dt[wv] = m; s_bad[wv] = nb; }
  __syncthreads();
  if (threadIdx.x == 0) {
    double mm = s_dt[0];
    int bb = s_bad[0];
    for (int q = 1; q < 4; q++) { mm = dmin<double>(mm, s_dt[q]); bb += s_bad[q]; }
    Counters* slot = cnt + (blockIdx.x % ATOMIC_SLOTS);
    atomicMin(&slot->dtmax_bits, (unsigned long long)__double_as_longlong(mm));
    if (bb) atomicAdd(&slot->tank_fail, (unsigned long long)bb);
  }
}

// Wave-aggregated append of relaxation samples (one atomic per wave).
__device__ __forceinline__ void capture_samples(const SampleSink& K, bool cap, const float* feat, float target,
                                                int iters, float remainder, float sigma) {
  const unsigned long long mask = __ballot(cap);
  if (mask == 0ull) return;
  const int lane = threadIdx.x & 63;
  const int leader = __ffsll((long long)mask) - 1;
  unsigned long long base = 0ull;
  if (lane == leader) base = atomicAdd(K.seen, (unsigned long long)__popcll(mask));
  const unsigned int lo = __shfl((unsigned int)(base & 0xFFFFFFFFull), leader, 64);
  const unsigned int hi = __shfl((unsigned int)(base >> 32), leader, 64);
  base = ((unsigned long long)hi << 32) | lo;
  if (!cap) return;
  const unsigned long long idx = base + (unsigned long long)__popcll(mask & ((1ull << lane) - 1ull));
  if (idx % (unsigned long long)K.stride != 0ull) return;
  const unsigned long long slot = (unsigned long long)K.base + idx / (unsigned long long)K.stride;
  if (slot >= (unsigned long long)K.cap) return;
  float4* o = reinterpret_cast<float4*>(K.buf + slot * SAMPLE_FLOATS);
  o[0] = make_float4(feat[0], feat[1], feat[2], feat[3]);
  o[1] = make_float4(feat[4], feat[5], feat[6], feat[7]);
  o[2] = make_float4(feat[8], feat[9], feat[10], feat[11]);
  o[3] = make_float4(target, (float)iters, remainder, sigma);
}

// Waves per SIMD the step kernels are compiled for (at least): three in FP64 (168
// VGPRs) and in the FP32 LK_FULL kernels; five for the one- and two-phase FP32
// kernels (96 VGPRs; the 2D and 3D minmod kernels need 76-85 and spill nothing,
// the 2D first-order cold ones then run six waves; the 2D first-order learned ones
// need 82-86 and would spill 40 bytes per lane at six); four for the second-order,
// learned and capture three-phase FP32 kernels (128 VGPRs instead of 131: the 256^3 three-phase step runs 11 %
// faster than at three; at five they spill too much); five for the first-order
// three-phase ones, whose accumulators wait in LDS (acc_stash: 89 VGPRs; at 251 x 243 x 257
// 1205 -> 1166 us a step).
// LDS of one wave in the learned kernels after the flux passes: the inference's
// staging (MLP_WAVE_LDS) and two doubles per lane for the start's affine form.
constexpr int STEP_WAVE_LDS = MLP_WAVE_LDS + 64 * 2 * 8;
template <int TK> constexpr int step_block_lds() { return tile_cells<TK>() / 64 * STEP_WAVE_LDS; }   // waves with cells

template <typename R, int N, int D, bool O2, bool LEARN, int LK>
constexpr int step_waves() {
  return (sizeof(R) == 4 && LK != LK_FULL) ? (N <= 2 || (!O2 && !LEARN) ? 5 : 4) : 3;
}

// CAP: the instantiation that also captures warm-start training records (cold
// relaxing kernels with a sample buffer attached; the full-featured kernels
// always carry it).  Without it the capture path is not compiled: its features
// and slot arithmetic cost the FP64 benchmark kernel 1 % even when not taken.
template <int MODEL, int N, int D, bool O2, typename R, bool LEARN, int LK, bool CAP = false, int TK = (int)sizeof(R)>
__global__ __launch_bounds__((tile_threads<D, TK>()), (step_waves<R, N, D, O2, LEARN || CAP, LK>())) void k_step(ParamsPtr Pc, StepLaunchT<R> L, Clock* __restrict__ clk,
                                              Counters* __restrict__ cnt) {
  constexpr bool CAPTURE = !LEARN && MODEL != M_EULER && (CAP || LK == LK_FULL);
  const Params& P = *(const Params*)Pc;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  R* lds = reinterpret_cast<R*>(lds_raw);
  constexpr int NW = tile_threads<D, TK>() / 64;   // waves of the block
  __shared__ double s_dt[NW], s_res[NW];
  __shared__ unsigned long long s_c[6][NW];
  if (clk->done) return;
  const double dt = clk->dt;
  int org[3];
  tile_origin<MODEL, N, D, LEARN, TK>(P, L.row0, L.nrows, org[0], org[1], org[2]);
  const int tid = threadIdx.x;
  int own[3];
  own[0] = org[0] + tid % Tile<D, TK>::X;
  own[1] = org[1] + (tid / Tile<D, TK>::X) % Tile<D, TK>::Y;
  own[2] = org[2] + tid / (Tile<D, TK>::X * Tile<D, TK>::Y);
  const bool own_ok = (!tile_small(TK) || tid < tile_cells<TK>()) && own[0] < P.nx && own[1] < P.ny && own[2] < P.nz;
  const int64_t c = own[0] + (int64_t)own[1] * P.nx + (int64_t)own[2] * P.nx * P.ny;
  const int64_t lc = c - (off32<R>() ? (int64_t)L.cbase : 0);   // state index of the own cell

  R smax = R(0.);   // largest wave speed of the cell's faces (cfl_speed)
  unsigned long long n_it = 0, n_fail = 0, n_relax = 0, n_warm = 0, n_wfb = 0;
  double resid = 0.;
  // Time-n phases of the own cell for the non-conservative terms (Cell::getPhase default type).
  R an[N], pn[N];
#pragma unroll
  for (int q = 0; q < N; q++) { an[q] = R(0.); pn[q] = R(0.); }
  if (own_ok && MODEL != M_EULER) {
#pragma unroll
    for (int q = 0; q < N; q++) {
      an[q] = R(ld_var<off32<R>()>(L.wn, P.pitch, 3 * q, lc));
      pn[q] = R(ld_var<off32<R>()>(L.wn, P.pitch, 3 * q + 2, lc));
    }
  }
  ConsAcc<N, R> acc;

  // The accumulators' slots lie behind the staging.  They are read back without a barrier, so
  // nothing may write LDS after the passes (the learned kernels' inference does).
  constexpr int ST = acc_stash<MODEL, N, D, O2, TK, LK, LEARN>();
  constexpr int STAGED = (int)sizeof(R) * Sizes<MODEL, N, D>::template lds_elems<TK>(O2);
  static_assert(ST >= 0, "the staging leaves no room for the accumulators");
  static_assert(ST == 0 || STAGED % 8 == 0, "the accumulators' slots are doubles");
  static_assert(!LEARN || ST == 0, "the inference would write where accumulators may wait");
  double* st = reinterpret_cast<double*>(lds_raw + STAGED) + tid;
  if constexpr (ST > 0) each_stashed<ST, N, R>(acc, [&](double& x, int v) { st[256 * v] = x; });
  if constexpr (tile_small(TK)) {
    // Waves 0-1 take the x axis, 2-3 y, 4-5 z; the first wave gathers in the faces' order.
    const int grp = __builtin_amdgcn_readfirstlane(tid / pass_threads<TK>());
#define ECG_AXES(STEP)                                                                                               \
  do {                                                                                                               \
    if (grp == 0) axis_pass<MODEL, N, D, O2, R, LK, 0, FR_XI, LEARN, TK, STEP>(P, L, lds, org, own, own_ok, an, pn, smax, acc); \
    else if (grp == 1) axis_pass<MODEL, N, D, O2, R, LK, 1, FR_YI, LEARN, TK, STEP>(P, L, lds, org, own, own_ok, an, pn, smax, acc); \
    else if constexpr (D >= 3) axis_pass<MODEL, N, D, O2, R, LK, 2, FR_ZI, LEARN, TK, STEP>(P, L, lds, org, own, own_ok, an, pn, smax, acc); \
    __syncthreads();                                                                                                 \
  } while (0)
    if constexpr (O2) ECG_AXES(STEP_A);
    ECG_AXES(STEP_B);
#undef ECG_AXES
    axis_pass<MODEL, N, D, O2, R, LK, 0, FR_XI, LEARN, TK, STEP_C>(P, L, lds, org, own, own_ok, an, pn, smax, acc);
    axis_pass<MODEL, N, D, O2, R, LK, 1, FR_YI, LEARN, TK, STEP_C>(P, L, lds, org, own, own_ok, an, pn, smax, acc);
    if constexpr (D >= 3) axis_pass<MODEL, N, D, O2, R, LK, 2, FR_ZI, LEARN, TK, STEP_C>(P, L, lds, org, own, own_ok, an, pn, smax, acc);
    __syncthreads();
  } else {
    axis_pass<MODEL, N, D, O2, R, LK, 0, FR_XI, LEARN>(P, L, lds, org, own, own_ok, an, pn, smax, acc);
    if (D >= 2) axis_pass<MODEL, N, D, O2, R, LK, 1, FR_YI, LEARN>(P, L, lds, org, own, own_ok, an, pn, smax, acc);
    if (D >= 3) axis_pass<MODEL, N, D, O2, R, LK, 2, FR_ZI, LEARN>(P, L, lds, org, own, own_ok, an, pn, smax, acc);
  }
  if constexpr (ST > 0) each_stashed<ST, N, R>(acc, [&](double& x, int v) { x = st[256 * v]; });

  Cell<N> nw;
  bool relax_now = false, spread_ok = false;
  double relax_dt = 0.;   // dt of the stage's relaxation (dt/2 after the predictor)
  double p_cold = 0., spread = 0., sigma = 1e-9, t_lin_d = 0.;
  float feat[MLP_IN];
  float t_lin = 0.f;
  // Learned kernels: a relaxation that the first evaluation settles (relaxed1) is
  // finished before the inference and carries its final residual; an unsettled one
  // carries the reference procedure's next iterate.
  bool relaxed1 = false;
  double carry = 0.;
#pragma unroll
  for (int q = 0; q < MLP_IN; q++) feat[q] = 0.f;
  if (own_ok) {
    const int i = own[0], j = own[1], k = own[2];
    const bool on_bnd = (i == 0) || (i == P.nx - 1) || (D >= 2 && (j == 0 || j == P.ny - 1)) ||
                        (D >= 3 && (k == 0 || k == P.nz - 1));
    if (on_bnd) {
      // Boundary faces see the stage's own cell: W^n (first order / predictor) or W* (corrector).
      Cell<N, R> src;
      load_prim<MODEL, N, D, off32<R>()>(P, (O2 && L.stage == 2) ? L.wsrc : L.wn, lc, src);
      derive<MODEL, N, R>(P, src, false);
      if (i == 0) boundary_face_at<MODEL, N, D, O2, 0, 0, FR_XM, R, LK>(P, L, src, lc, own, an, pn, smax, acc);
      if (i == P.nx - 1) boundary_face_at<MODEL, N, D, O2, 0, 1, FR_XP, R, LK>(P, L, src, lc, own, an, pn, smax, acc);
      if (D >= 2) {
        if (j == 0) boundary_face_at<MODEL, N, D, O2, 1, 0, FR_YM, R, LK>(P, L, src, lc, own, an, pn, smax, acc);
        if (j == P.ny - 1) boundary_face_at<MODEL, N, D, O2, 1, 1, FR_YP, R, LK>(P, L, src, lc, own, an, pn, smax, acc);
      }
      if (D >= 3) {
        if (k == 0) boundary_face_at<MODEL, N, D, O2, 2, 0, FR_ZM, R, LK>(P, L, src, lc, own, an, pn, smax, acc);
        if (k == P.nz - 1) boundary_face_at<MODEL, N, D, O2, 2, 1, FR_ZP, R, LK>(P, L, src, lc, own, an, pn, smax, acc);
      }
    }

    // FP64 cell update from the time-n primitives.
    Cell<N> own64;
    load_prim<MODEL, N, D, off32<R>()>(P, L.wn, lc, own64);
    if (MODEL != M_EULER && sizeof(R) == 4) {
      // FP32 storage rounds a dominant volume fraction (1 - eps) by up to 3e-8
      // absolute, so the stored fractions no longer sum to one.  buildPrim's
      // renormalisation would turn that defect into a phase-density change,
      // which a stiff EOS amplifies to p_inf * 1e-8 of pressure and the
      // relaxation then pushes into the minority phase.  Restoring the sum in
      // FP64 here keeps the stored phase densities and pressures.
      double un = 0.;
#pragma unroll
      for (int k = 0; k < N; k++) un += own64.a[k];
      const double iun = rcp_ieee(un);
#pragma unroll
      for (int k = 0; k < N; k++) own64.a[k] = div_special(own64.a[k], un, iun);
    }
    // U^n needs the mixture density of the time-n cell (Cell::timeEvolution rebuilds
    // the conservative variables from the primitives, FluxUEq::buildCons).
    if (MODEL != M_EULER) mixture_density<N>(own64);
    const double scale = (O2 && L.stage == 1) ? 0.5 * dt : dt;
    relax_dt = scale;
    Cons<N> A;
    time_evolution<MODEL, N, D, R>(P, acc, A, own64, scale);
    build_prim<MODEL, N>(P, A, nw);
    if (MODEL != M_EULER && P.relax && !(MODEL == M_UEQ && LK == LK_FULL && P.relax_mu > 0.)) {
      relax_now = !relax_gated<N>(P, nw);
      if constexpr (LEARN) {
        // The reference procedure's first evaluation, at the cold guess: the network
        // is consulted only for a cell that it leaves short of the tolerance.
        if (relax_now) {
          double akS[N], rkS[N];
          NewtonState s1{relax_guess<N>(nw), 0., 1., 0};
          newton_resume<N, false>(P, nw, s1, akS, rkS, 1);
          if (fabs(s1.f) <= 1e-10) {
            relaxed1 = true;
            carry = s1.f;
            relax_end<N>(P, nw, s1, true, akS, rkS);
          } else {
            spread_ok = relax_features<N>(P, nw, WARM_MIN_RESIDUAL, true, p_cold, spread, feat, t_lin, t_lin_d, sigma);
            carry = s1.p - div1(s1.f, s1.df);
          }
        }
      } else if (relax_now && CAPTURE && L.sink.buf != nullptr) {
        spread_ok = relax_features<N>(P, nw, CAPTURE_MIN_RESIDUAL, false, p_cold, spread, feat, t_lin, t_lin_d, sigma);
      }
    }
  }

  // Learned warm start for the wave's cells that relax from distinct phase pressures.
  // The start's affine form, guess = ga + gb y, waits in the wave's LDS while the
  // inference needs the registers.
  float y = 0.f;
  double ga = 0., gb = 0.;
  if constexpr (LEARN && MODEL != M_EULER) {
    unsigned char* wl = lds_raw + (threadIdx.x >> 6) * STEP_WAVE_LDS;
    double* st = reinterpret_cast<double*>(wl + MLP_WAVE_LDS) + 2 * (threadIdx.x & 63);
    if (spread_ok) { st[0] = p_cold + spread * t_lin_d; st[1] = spread * sigma; }
    y = mlp_wave_infer(L.mlp, spread_ok, feat, wl);
    if (spread_ok) { ga = st[0]; gb = st[1]; }
  }

  int it = 0;
  unsigned long long n_warn = 0, n_bad = 0;
  if (own_ok && MODEL != M_EULER && P.relax) {
    // Relaxation: after the predictor (CellO2.cpp:128-134) and after the full step
    // (Run::advancingProcedure, Run.cpp:593).
    double fres = 0.;
    int flags = 0;
    if (MODEL == M_UEQ && LK == LK_FULL && P.relax_mu > 0.) {
      it = relax_finite<N>(P, nw, relax_dt, flags);
    } else if constexpr (LEARN) {
      if (relax_now && relaxed1) {
        it = 1;
        fres = carry;
      } else if (relax_now) {
        // After an unsettling first evaluation: a Newton from the network's guess
        // (WARM_MAX_IT evaluations; short of the tolerance, the reference procedure
        // continues from its first evaluation), or the reference procedure continued
        // (from its next iterate: f = 0 and f' = 1 make the resumed step take it).
        double akS[N], rkS[N];
        NewtonState nst{carry, 0., 1., 1};
        int total = nst.it;
        bool conv = false;
        if (spread_ok) {
          n_warm = 1;
          const double guess = ga + gb * (double)y;
          NewtonState w{guess, 0., 1., 0};
          if (guess == guess) {
            newton_resume<N, false>(P, nw, w, akS, rkS, WARM_MAX_IT);
            total += w.it;
          }
          if (guess == guess && fabs(w.f) <= 1e-10) {
            nst = w;
            conv = true;
          } else {
            n_wfb = 1;
          }
        }
        if (!conv) {
          const int before = nst.it;
          newton_resume<N, false>(P, nw, nst, akS, rkS, 100);
          total += nst.it - before;
          conv = nst.it < 100;
        }
        fres = nst.f;
        flags = relax_end<N>(P, nw, nst, conv, akS, rkS);
        it = total;
      }
    } else {
      bool fell = false;
      const double start = relax_guess<N>(nw);   // the reference's guess, sum alpha_k p_k
      it = relax_start<N>(P, nw, start, 100, start, fell, fres, flags);
    }
    if (it > 0) {
      n_relax = 1; n_it = (unsigned long long)it; resid = fabs(fres);
    }
    n_fail = (flags & RELAX_FAIL) ? 1 : 0;
    if (flags & RELAX_WARN) {
      n_warn = 1;
      const unsigned long long q = atomicAdd(P.warn_cnt, 1ull);
      if (q < (unsigned long long)P.warn_cap) {
        WarnRec r;
        r.iteration = clk->iteration; r.cell = c; r.stage = L.stage; r.kind = 0; r.value = fabs(fres);
        P.warn_rec[q] = r;
      }
    }
  }
  // Capture records cold solves only (the API keeps a warm start and a sink apart),
  // so the features need not stay live across the inference.
  if (CAPTURE && L.sink.buf != nullptr) {
    const bool cap = spread_ok && it > 0 && it < 100;
    const double t = cap ? (nw.p[0] - p_cold) / spread : 0.;
    const float rem = cap ? (float)((t - t_lin_d) / sigma) : 0.f;
    capture_samples(L.sink, cap, feat, (float)t, it, rem, (float)sigma);
  }
  if (own_ok) {
    if (MODEL != M_EULER && P.relax) correct_and_derive<MODEL, N>(P, nw);
    else if (O2 && L.stage == 1) correct_and_derive<MODEL, N>(P, nw);
    n_bad = nonfinite_prim<MODEL, N, D>(nw) ? 1 : 0;
    store_prim<MODEL, N, D, off32<R>()>(P, L.wout, lc, nw);
  }
  // Block reductions: largest wave speed (the CFL bound) and relaxation counters (per-cell
  // flags by ballot).
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const R wmax = wave_reduce63(smax, [](R a, R b) { return dmax<R>(a, b); });
  const unsigned nb_w = __popcll(__ballot(n_bad != 0));
  unsigned nr_w = 0, it_w = 0, nw_w = 0, nf_w = 0, fail_w = 0, warn_w = 0;
  if constexpr (MODEL != M_EULER) {
    nr_w = __popcll(__ballot(n_relax != 0));
    if (nr_w) {
      it_w = wave_reduce63((uint32_t)n_it, [](uint32_t a, uint32_t b) { return a + b; });
      resid = wave_reduce63(resid, [](double a, double b) { return a + b; });
      fail_w = __popcll(__ballot(n_fail != 0));
      warn_w = __popcll(__ballot(n_warn != 0));
      if constexpr (LEARN) {
        nw_w = __popcll(__ballot(n_warm != 0));
        nf_w = __popcll(__ballot(n_wfb != 0));
      }
    }
  }
  if (lane == 63) {
    s_dt[wv] = (double)wmax;
    s_c[5][wv] = nb_w;
    if constexpr (MODEL != M_EULER) {
      s_res[wv] = resid;
      s_c[0][wv] = it_w; s_c[1][wv] = fail_w | ((unsigned long long)warn_w << 32);   // warnings in the high half
      s_c[2][wv] = nr_w; s_c[3][wv] = nw_w; s_c[4][wv] = nf_w;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = s_dt[0], rs = 0.;
    unsigned long long a = 0, b = 0, r = 0, w = 0, wf = 0, nb = s_c[5][0];
    for (int q = 1; q < NW; q++) { m = dmax<double>(m, s_dt[q]); nb += s_c[5][q]; }
    if constexpr (MODEL != M_EULER)
      for (int q = 0; q < NW; q++) {
        rs += s_res[q];
        a += s_c[0][q]; b += s_c[1][q]; r += s_c[2][q]; w += s_c[3][q]; wf += s_c[4][q];
      }
    Counters* slot = cnt + (blockIdx.x % ATOMIC_SLOTS);
    const double dtb = cfl_dt(P.lcfl, m);
    atomicMin(&slot->dtmax_bits, (unsigned long long)__double_as_longlong(dtb));
    if (nb) atomicAdd(&slot->nonfinite, nb);
    if (r) {
      atomicAdd(&slot->newton_iters, a);
      if (b) {
        atomicAdd(&slot->newton_fail, b & 0xFFFFFFFFull);
        atomicAdd(&slot->newton_warn, b >> 32);
      }
      atomicAdd(&slot->relax_calls, r);
      atomicAdd(&slot->resid_sum, rs);
    }
    if (w) {
      atomicAdd(&slot->warm_calls, w);
      atomicAdd(&slot->warm_fallbacks, wf);
    }
  }
}

// Initial condition: Cell::fill over the domains (later ones override), then
// Cell::completeFulfillState (Cell.cpp:344-353) and E = e + |u|^2/2.
template <int MODEL, int N, int D, typename S>
__global__ __launch_bounds__(256) void k_fill(Params P, const DomainDev* __restrict__ doms, int ndom,
                                              S* __restrict__ W) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= P.ncell) return;
  const int i = (int)(c % P.nx);
  const int j = (int)((c / P.nx) % P.ny);
  const int k = (int)(c / ((int64_t)P.nx * P.ny));
  double x[3];
  x[0] = (i + 0.5) * P.d[0];
  x[1] = (j + 0.5) * P.d[1];
  x[2] = (k + 0.5) * P.d[2];
  Cell<N> s;
#pragma unroll
  for (int q = 0; q < N; q++) { s.a[q] = 0.; s.r[q] = 0.; s.p[q] = 0.; }
  s.u[0] = s.u[1] = s.u[2] = 0.;
  // The last domain containing the cell wins: scan backwards and stop at the first hit.
  for (int q = ndom - 1; q >= 0; q--) {
    const DomainDev& d = doms[q];
    bool in = false;
    if (d.kind == 0) {
      in = true;
    } else if (d.kind == 1) {
      in = (d.dir >= 0) ? (x[d.axis] >= d.origin) : (x[d.axis] <= d.origin);
    } else if (d.kind == 2) {
      const double a = x[d.axis] - d.center[d.axis], b = x[d.axis2] - d.center[d.axis2];
      double sum = 0.;
      sum += a * a;
      sum += b * b;
      in = (sum <= d.radius * d.radius);
    } else if (d.kind == 3) {
      const double a = x[0] - d.center[0], b = x[1] - d.center[1], e = x[2] - d.center[2];
      const double sum = a * a + b * b + e * e;
      in = (sum <= d.radius * d.radius);
    } else if (d.kind == 4) {
      in = !((x[d.axis] - d.lo[d.axis] < 0) || (x[d.axis] - d.lo[d.axis] > d.len[d.axis]) ||
             (x[d.axis2] - d.lo[d.axis2] < 0) || (x[d.axis2] - d.lo[d.axis2] > d.len[d.axis2]));
    } else if (d.kind == 5) {
      in = true;
      for (int a = 0; a < 3; a++)
        if ((x[a] - d.lo[a] < 0) || (x[a] - d.lo[a] > d.len[a])) in = false;
    }
    if (in) {
#pragma unroll
      for (int q2 = 0; q2 < N; q2++) {
        s.a[q2] = (MODEL == M_EULER) ? 1. : d.alpha[q2];
        s.r[q2] = d.rho[q2];
        s.p[q2] = d.p[q2];
      }
      s.u[0] = d.vel[0];
      s.u[1] = (D >= 2) ? d.vel[1] : 0.;
      s.u[2] = (D >= 3) ? d.vel[2] : 0.;
      break;
    }
  }
  derive<MODEL, N, double>(P, s, MODEL == M_EULER);
  if (MODEL != M_EULER) s.E = s.em + 0.5 * sqn3<double>(s.u);
  store_prim<MODEL, N, D>(P, W, c, s);
}

// The small tiles serve meshes of at most one ordinary tile per CU, where a stage lasts as
// long as one block: up to 256 ordinary tiles at second order in 2D and in cold FP32, up to 128 at
// first order, in 3D FP64 and in the learned 3D kernels, where a block's chain is shorter against
// the small tiles' extra faces and the inferences of four times the blocks.  Both sides measured, a
// step of a run, ordinary / small tiles (us).  Two phases: 2D O2 FP64 96^2 110/66, 256^2 89/86, FP32
// 256^2 124/95; 2D O1 FP64 160^2 48/35, 256^2 40/39; 3D O2 FP32 32^3 112/78, 40^3 (300 tiles) 117/105,
// FP64 24^3 138/73, 32^3 128/115, 40^3 131/158; 3D O1 FP64 32^3 31/26, 36^3 30/33, FP32 36^3 24/22;
// learned 3D O2 32^3 54/42, 36^3 (243 tiles) 54/59, 40^3 59/71, O1 36^3 26/34.  Three phases: 2D O2
// FP64 256^2 94/86; 3D O1 FP64 32^3 34/34, 40^3 56/67; 3D O2 FP64 36^3 206/155, FP32 40^3 176/117;
// learned 3D O2 36^3 62/68.  Euler: 3D O2 FP64 32^3 37/22, 48^3 78/91.  The full-featured and the
// capture kernels keep the ordinary tiles (their code is long; Euler's LK_FULL, the second-order
// walls, is the exception).
template <int MODEL, int D, int LK, bool CAP> constexpr bool has_small() {
  return D >= 2 && !CAP && (LK != LK_FULL || MODEL == M_EULER);
}
template <int D, bool O2, int ES, bool LEARN> inline bool step_small(const Params& P) {
  return (int64_t)P.tiles[0] * P.tiles[1] * P.tiles[2] <= ((O2 && (D == 2 || (ES == 4 && !LEARN))) ? 256 : 128);
}

// One stage of the step.  The FP32 kernels address the state by 32-bit byte
// offsets from the launch's first cell: when the tile rows of the outermost axis
// (with the two lines of halo on each side) span more than step_span_bytes of
// one variable, the stage runs as several launches over consecutive rows (an
// even count each, for the FP32 tile groups), each with its own first cell.
template <int MODEL, int N, int D, bool O2, typename R, bool LEARN, int LK, bool CAP = false, int TK = (int)sizeof(R)>
void launch_step_v(const Params& P, const StepLaunchT<R>& L, Clock* clk, Counters* cnt, hipStream_t s) {
  constexpr int ES = (int)sizeof(R);
  if constexpr (!tile_small(TK) && has_small<MODEL, D, LK, CAP>()) {
    if (step_small<D, O2, ES, LEARN>(P)) {
      launch_step_v<MODEL, N, D, O2, R, LEARN, LK, CAP, TK + SMALL_TILE>(P, L, clk, cnt, s);
      return;
    }
  }
  using SZ = Sizes<MODEL, N, D>;
  using TL = Tile<D, TK>;
  constexpr int T = (D == 3) ? TL::Z : (D == 2) ? TL::Y : TL::X;
  const int t3[3] = {(P.nx + TL::X - 1) / TL::X, (P.ny + TL::Y - 1) / TL::Y, (P.nz + TL::Z - 1) / TL::Z};
  const int rows = t3[D - 1];
  const int per_row = t3[0] * t3[1] * t3[2] / rows;   // blocks of one tile row
  const int64_t line = (D == 3) ? (int64_t)P.nx * P.ny : (D == 2) ? (int64_t)P.nx : 1;   // cells of one line
  int chunk = rows;
  if (off32<R>()) {
    const int64_t lines = step_span_bytes() / (line * ES);
    chunk = (int)std::min<int64_t>(rows, std::max<int64_t>((lines - 4) / T, 1));
    if (chunk < rows && chunk > 1) chunk &= ~1;
  }
  size_t lds = sizeof(R) * SZ::template lds_elems<TK>(O2) + 256 * sizeof(double) * acc_stash<MODEL, N, D, O2, TK, LK, LEARN>();
  if (LEARN && lds < (size_t)step_block_lds<TK>()) lds = step_block_lds<TK>();
  auto k = k_step<MODEL, N, D, O2, R, LEARN, LK, CAP, TK>;
  // A failure here surfaces as the launch error the caller checks next.
  (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  for (int r0 = 0; r0 < rows; r0 += chunk) {
    StepLaunchT<R> Ls = L;
    Ls.row0 = r0;
    Ls.nrows = std::min(chunk, rows - r0);
    Ls.cbase = 0;
    if (off32<R>()) {
      const int64_t first = std::max<int64_t>((int64_t)r0 * T - 2, 0) * line;
      Ls.cbase = (uint32_t)first;
      Ls.wn = L.wn + first;
      Ls.wsrc = L.wsrc + first;
      Ls.wout = L.wout + first;
    }
    hipLaunchKernelGGL(k, dim3(per_row * Ls.nrows), dim3(tile_threads<D, TK>()), lds, s, (ParamsPtr)L.pdev, Ls, clk, cnt);
  }
}


// Second order: a case with a wall, a THINC limiter or the finite-rate
// relaxation runs the LK_FULL instantiation; otherwise a case whose
// four limiters are all minmod (the common choice) runs the instantiation with
// the limiter fixed at compile time.  A capture (cap) runs the generic one with
// the capture path.
template <int MODEL, int N, int D, typename R, bool LEARN>
void launch_step_o2(const Params& P, const StepLaunchT<R>& L, bool cap, Clock* clk, Counters* cnt, hipStream_t s) {
  bool full = P.thinc != 0 || P.relax_mu > 0.;
  for (int a = 0; a < D; a++) full = full || P.bc[2 * a] == BC_WALL || P.bc[2 * a + 1] == BC_WALL;
  const bool all_minmod = P.lim[0] == LIM_MINMOD && P.lim[1] == LIM_MINMOD && P.lim[2] == LIM_MINMOD &&
                          P.lim[3] == LIM_MINMOD;
  if (full) {
    launch_step_v<MODEL, N, D, true, R, LEARN, LK_FULL>(P, L, clk, cnt, s);
    return;
  }
  if constexpr (!LEARN && MODEL != M_EULER) {
    if (cap) {
      launch_step_v<MODEL, N, D, true, R, false, LK_GENERIC, true>(P, L, clk, cnt, s);
      return;
    }
  }
  if (all_minmod) launch_step_v<MODEL, N, D, true, R, LEARN, LIM_MINMOD>(P, L, clk, cnt, s);
  else launch_step_v<MODEL, N, D, true, R, LEARN, LK_GENERIC>(P, L, clk, cnt, s);
}

template <int MODEL, int N, int D, typename R>
void launch_step_t(const Params& P, const StepLaunch& Lv, Clock* clk, Counters* cnt, hipStream_t s) {
  StepLaunchT<R> L;
  L.wn = (const R*)Lv.wn; L.wsrc = (const R*)Lv.wsrc; L.wout = (R*)Lv.wout; L.stage = Lv.stage;
  L.row0 = 0; L.nrows = P.tiles[D - 1]; L.cbase = 0;
  L.pdev = Lv.pdev;
  L.mlp = Lv.mlp;
  L.sink = Lv.sink;
  // Inlet-tank faces: launched on their own ahead of the step kernel, whose
  // gather reads their records.
  if (Lv.tank_only) {
    int64_t nf = 0;
    for (int q = 0; q < 2 * D; q++)
      if (P.bc[q] == BC_TANK) nf += tank_faces(P, q);
    if (nf > 0)
      hipLaunchKernelGGL((k_tank<MODEL, N, D, R>), dim3((unsigned)((nf + 255) / 256)), dim3(256), 0, s,
                         (ParamsPtr)Lv.pdev, L.wsrc, clk, cnt, nf);
    return;
  }
  // The learned warm start exists in the FP32 form of the relaxing models only.
  constexpr bool CAN_LEARN = (sizeof(R) == 4) && (MODEL != M_EULER);
  const bool learn = CAN_LEARN && Lv.mlp.frag != nullptr;
  const bool cap = (MODEL != M_EULER) && Lv.sink.buf != nullptr;
  if (Lv.stage == 0) {
    if constexpr (CAN_LEARN) {
      if (learn) { launch_step_v<MODEL, N, D, false, R, true, LK_GENERIC>(P, L, clk, cnt, s); return; }
    }
    // First order: the finite-rate relaxation lives in LK_FULL.
    if (MODEL == M_UEQ && P.relax_mu > 0.) {
      launch_step_v<MODEL, N, D, false, R, false, LK_FULL>(P, L, clk, cnt, s);
      return;
    }
    if constexpr (MODEL != M_EULER) {
      if (cap) {
        launch_step_v<MODEL, N, D, false, R, false, LK_GENERIC, true>(P, L, clk, cnt, s);
        return;
      }
    }
    launch_step_v<MODEL, N, D, false, R, false, LK_GENERIC>(P, L, clk, cnt, s);
  } else {
    if constexpr (CAN_LEARN) {
      if (learn) { launch_step_o2<MODEL, N, D, R, true>(P, L, false, clk, cnt, s); return; }
    }
    launch_step_o2<MODEL, N, D, R, false>(P, L, cap, clk, cnt, s);
  }
}

template <int MODEL, int N, int D, typename S>
void launch_fill_t(const Params& P, const DomainDev* doms, int ndom, void* w, hipStream_t s) {
  const int blocks = (int)((P.ncell + 255) / 256);
  hipLaunchKernelGGL((k_fill<MODEL, N, D, S>), dim3(blocks), dim3(256), 0, s, P, doms, ndom, (S*)w);
}

}  // namespace ecg
