// Kernel entry points of the finite-volume step (gfx950), shared by the
// per-model translation units and the C ABI layer.
#pragma once

#include "ecg_mlp.hpp"

namespace ecg {

// Domain description on the device (Cell::fill, GeometricalDomain.cpp:64-83).
struct DomainDev {
  int kind, axis, axis2, dir;
  double origin;
  double center[3];
  double radius;
  double lo[3], len[3];
  double alpha[4], rho[4], p[4];
  double vel[3];
};

// Relaxation samples written while a sink is attached: every stride-th cell
// that relaxes from distinct phase pressures, up to cap records.
struct SampleSink {
  float* buf;                  // cap * SAMPLE_FLOATS
  unsigned long long* seen;    // candidates met since the attachment
  long long cap;
  long long base;              // records held before the attachment
  int stride;
};

// The step kernels read their parameters from a device copy through a pointer into
// the constant address space: the compiler then reloads a field where it is used
// (scalar loads) instead of keeping every parameter in scalar registers through the
// whole kernel, which spilled them into vector-register lanes.
typedef const __attribute__((address_space(4))) Params* ParamsPtr;

// Buffers of one launch; the element type is the state type of the precision form.
struct StepLaunch {
  const Params* pdev;   // device copy of the context's parameters
  const void* wn;       // state at time n
  const void* wsrc;     // state the fluxes are evaluated on (== wn for first order / predictor)
  void* wout;           // written state
  int stage;            // 0: first order; 1: predictor; 2: corrector
  MlpDev mlp;           // learned warm start (frag == nullptr: cold start)
  SampleSink sink;      // relaxation sample capture (buf == nullptr: off)
  int tank_only;        // 1: launch only k_tank for this stage's inlet-tank faces
};

template <typename R>
struct StepLaunchT {
  const Params* pdev;
  const R* wn;
  const R* wsrc;
  R* wout;
  int stage;
  MlpDev mlp;
  SampleSink sink;
  // The launch's tile rows along the outermost axis (z in 3D, y in 2D, x in 1D):
  // row0 .. row0 + nrows - 1.  cbase: the cell the launch's state indices count
  // from; wn, wsrc and wout point at it (FP32 kernels; 0 in FP64).
  int row0, nrows;
  uint32_t cbase;
};

// Per (model, phases, dimension, precision) launchers; defined in ecg_step_<model>_<precision>.hip.
typedef void (*step_fn)(const Params& P, const StepLaunch& L, Clock* clk, Counters* cnt, hipStream_t s);
typedef void (*fill_fn)(const Params& P, const DomainDev* doms, int ndom, void* w, hipStream_t s);

// Tile that block `block` of a launch over nb tiles works on.  The chip hands block i to XCD
// i % 8, and neighbouring tiles share halo lines in an XCD's L2.  run = 0: one range of nb / 8
// consecutive tiles per XCD (the first nb % 8 one tile longer).  run > 0: runs of that many
// tiles dealt to the XCDs in turn, what is left over in eight ranges, so that a region whose
// cells cost more (a shock's relaxation) is shared by all XCDs.
__host__ __device__ inline int xcd_tile(int nb, int block, int run) {
  const int xcd = block & 7, full = run > 0 ? nb / (8 * run) * (8 * run) : 0;
  if (run > 0 && block < full) {
    const int i = block >> 3;
    return (i / run * 8 + xcd) * run + i % run;
  }
  const int rest = nb - full, rem = rest & 7;
  return full + xcd * (rest >> 3) + (xcd < rem ? xcd : rem) + ((block - full) >> 3);
}

// Tiles per run of xcd_tile for a step launch over nb tiles of 256 cells, of a case with n phases
// in d dimensions and a state of esize bytes an element; 0: one range per XCD.  Ranges share the
// most halos, and where every tile costs the same they are the fastest: Euler 3D O1 FP64 at
// 121 x 119 x 117 97 us a step, dealt singly 157.
// A two-phase step's relaxation makes the tiles around a shock and the interfaces cost a multiple
// of the others, and ranges leave them to one or two XCDs: 2D O1 FP64 at 701 x 683 (1892 tiles) 73
// us in ranges, 64 dealt singly, 62 in runs of 32 (2048^2 379 / 363 / 367); O2 FP32 113 / 110 / 99
// (1361 x 1283 233 / 281 / 213; beyond 8192 tiles FP32 ranges win: 2048^2 O1 196 us, in runs 201).
// Below 512 tiles runs of 16 (208^2, 169 tiles, O1 FP64 48.5 us in ranges, 46.3).  In 3D runs of
// 64 keep the x and y neighbours together: O2 FP64 at 93 x 95 x 91 449 / 472 / 423, FP32 222 / 239 /
// 204; beyond 6144 tiles (eight rounds of three blocks a CU) the costs even out within a range, and
// its shared z halos win (O1 FP32 at 119 x 113 x 117 144 us, in runs of 64 150).  Three-phase steps
// gain nothing (2D O1 FP64 at 907 x 883 109 us in ranges and in runs), nor do learned ones in 3D,
// whose relaxations are short (O1 at 101 x 99 x 97 112 us in ranges, 122 in runs of 32), nor the
// small tiles, all resident at once.
__host__ __device__ constexpr int tile_run(int model, int n, int d, int esize, bool learned, int nb) {
  if (model == M_EULER || n != 2 || d == 1) return 0;
  if (d == 2) return nb < 512 ? 16 : esize == 8 || nb <= 8192 ? 32 : 0;
  return !learned && nb <= 6144 ? 64 : 0;
}

// Tile extents (cells per block along x, y, z) for a problem dimension and state element size.
void tile_extent(int dim, int esize, int t[3]);

void launch_clock(Clock* clk, Counters* cnt, double cfl, hipStream_t s);

// Bytes of one state variable a launch of the FP32 step kernels addresses from its
// first cell: 4 GiB (32-bit offsets); a test may lower it to split small grids.
int64_t step_span_bytes();

}  // namespace ecg
