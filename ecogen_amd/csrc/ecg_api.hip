// C ABI of the finite-volume step (include/ecogen_amd.h): context, device
// memory, the device-side time loop and the state transfers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "../../include/ecogen_amd.h"
#include "ecg_kernels.hpp"
#include "ecg_learn.hpp"

namespace ecg {
step_fn get_step_fn_euler_f64(int nph, int dim);
step_fn get_step_fn_pueq_f64(int nph, int dim);
step_fn get_step_fn_ueq_f64(int nph, int dim);
step_fn get_step_fn_euler_f32(int nph, int dim);
step_fn get_step_fn_pueq_f32(int nph, int dim);
step_fn get_step_fn_ueq_f32(int nph, int dim);
fill_fn get_fill_fn_euler_f64(int nph, int dim);
fill_fn get_fill_fn_pueq_f64(int nph, int dim);
fill_fn get_fill_fn_ueq_f64(int nph, int dim);
fill_fn get_fill_fn_euler_f32(int nph, int dim);
fill_fn get_fill_fn_pueq_f32(int nph, int dim);
fill_fn get_fill_fn_ueq_f32(int nph, int dim);

static step_fn get_step_fn(int model, int nph, int dim, bool f32) {
  if (model == M_EULER) return f32 ? get_step_fn_euler_f32(nph, dim) : get_step_fn_euler_f64(nph, dim);
  if (model == M_PUEQ) return f32 ? get_step_fn_pueq_f32(nph, dim) : get_step_fn_pueq_f64(nph, dim);
  if (model == M_UEQ) return f32 ? get_step_fn_ueq_f32(nph, dim) : get_step_fn_ueq_f64(nph, dim);
  return nullptr;
}

static fill_fn get_fill_fn(int model, int nph, int dim, bool f32) {
  if (model == M_EULER) return f32 ? get_fill_fn_euler_f32(nph, dim) : get_fill_fn_euler_f64(nph, dim);
  if (model == M_PUEQ) return f32 ? get_fill_fn_pueq_f32(nph, dim) : get_fill_fn_pueq_f64(nph, dim);
  if (model == M_UEQ) return f32 ? get_fill_fn_ueq_f32(nph, dim) : get_fill_fn_ueq_f64(nph, dim);
  return nullptr;
}

// Cells per 256-thread tile (must match Tile<D, ES> in ecg_step_impl.hpp).
void tile_extent(int dim, int esize, int t[3]) {
  if (dim == 1) { t[0] = 256; t[1] = 1; t[2] = 1; }
  else if (dim == 2) { t[0] = 16; t[1] = 16; t[2] = 1; }
  else if (esize == 8) { t[0] = 8; t[1] = 8; t[2] = 4; }
  else { t[0] = 16; t[1] = 4; t[2] = 4; }
}

// Run::solver bookkeeping after a step (Run.cpp:417-486): t += dt, dt = cfl*dtMax.
// One wave: lane l reduces and resets counter slot l.
// Errors over the counter slots (one lane per slot): inlet-tank solves that did not
// converge and cells left with a non-finite state.
__device__ __forceinline__ unsigned long long fatal_total(const Counters* cnt) {
  const int l = threadIdx.x;
  unsigned long long f = (l < ATOMIC_SLOTS) ? cnt[l].tank_fail + cnt[l].nonfinite : 0ull;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) f += __shfl_xor(f, o, 64);
  return f;
}

// Bound by latency: the slots and the clock are loaded together and reduced side by side
// (one after the other they took 2.6 to 4.5 us a step, a sixth of a small mesh's).
__global__ __launch_bounds__(64) void k_clock(Clock* clk, Counters* cnt, double cfl) {
  static_assert(ATOMIC_SLOTS == 64, "one lane per slot");
  const int l = threadIdx.x;
  unsigned long long b = cnt[l].dtmax_bits, fatal = cnt[l].tank_fail + cnt[l].nonfinite;
  Clock k = *clk;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long q = __shfl_xor(b, o, 64);
    fatal += __shfl_xor(fatal, o, 64);
    b = (q < b) ? q : b;
  }
  if (k.done) return;
  cnt[l].dtmax_bits = (uint64_t)__double_as_longlong(1.e10);
  if (l != 0) return;
  const double dtmax = __longlong_as_double((long long)b);
  k.dt_max = dtmax;
  k.t += k.dt;
  k.iteration += 1;
  k.dt_next = cfl * dtmax;
  if (k.max_iter > 0) {
    if (k.iteration >= k.max_iter) k.done = 1;
  } else if (k.t >= k.t_end) {
    k.done = 1;
  }
  // A step that left an error ends the run there (Run::verifyErrors stops the reference
  // before its next step); the steps enqueued behind it return at once.
  if (fatal != k.fatal_seen) {
    k.done = 1;
    k.fatal = 1;
    k.fatal_seen = fatal;
  }
  k.dt = k.dt_next;
  *clk = k;
}

// Host-set clock: reset or explicit-dt steps; the dtMax slots restart at 1e10 and
// the error baseline is the counters' current total.
__global__ void k_clock_set(Clock* clk, Counters* cnt, Clock v) {
  const unsigned long long fatal = fatal_total(cnt);
  if (threadIdx.x == 0) {
    v.fatal = 0;
    v.fatal_seen = fatal;
    *clk = v;
  }
  if (threadIdx.x < ATOMIC_SLOTS) cnt[threadIdx.x].dtmax_bits = (uint64_t)__double_as_longlong(1.e10);
}

// Enqueued steps run even after a run's clock stopped: a stopped clock reopens
// without a limit, keeping its time, dt and error baseline.
__global__ void k_clock_open(Clock* clk) {
  if (threadIdx.x == 0 && clk->done && !clk->fatal) {
    clk->done = 0;
    clk->max_iter = 0;
    clk->t_end = INFINITY;
  }
}

// Plain streaming copy (16 bytes per lane per iteration), used to calibrate byte counters.
__global__ __launch_bounds__(256) void k_copy(const double2* __restrict__ src, double2* __restrict__ dst, int64_t n2) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n2; i += stride) dst[i] = src[i];
}

// Field-wise differences of two states of one mesh: for every persistent
// variable and, last, the mixture density sum_k alpha_k rho_k (Euler: rho),
// out[4f..4f+3] accumulates sum|a-b|, sum|b|, max|a-b|, max|b| (maxima as
// the bits of non-negative doubles).
template <typename SA, typename SB>
__global__ __launch_bounds__(256) void k_state_diff(const SA* __restrict__ a, const SB* __restrict__ b, int64_t ncell,
                                                    int64_t pa, int64_t pb, int nvar, int nph, int multiphase,
                                                    double* __restrict__ out) {
  __shared__ double red[4][4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int f = 0; f <= nvar; f++) {
    double sd = 0., sb = 0., md = 0., mb = 0.;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < ncell; i += stride) {
      double va, vb;
      if (f < nvar) {
        va = (double)a[f * pa + i];
        vb = (double)b[f * pb + i];
      } else if (multiphase) {
        va = 0.; vb = 0.;
        for (int k = 0; k < nph; k++) {
          va += (double)a[(3 * k) * pa + i] * (double)a[(3 * k + 1) * pa + i];
          vb += (double)b[(3 * k) * pb + i] * (double)b[(3 * k + 1) * pb + i];
        }
      } else {
        va = (double)a[i];
        vb = (double)b[i];
      }
      const double d = fabs(va - vb), ab = fabs(vb);
      sd += d; sb += ab; md = fmax(md, d); mb = fmax(mb, ab);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      sd += __shfl_xor(sd, o, 64); sb += __shfl_xor(sb, o, 64);
      md = fmax(md, __shfl_xor(md, o, 64)); mb = fmax(mb, __shfl_xor(mb, o, 64));
    }
    if (lane == 0) { red[wv][0] = sd; red[wv][1] = sb; red[wv][2] = md; red[wv][3] = mb; }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < 4; w++) {
        sd += red[w][0]; sb += red[w][1]; md = fmax(md, red[w][2]); mb = fmax(mb, red[w][3]);
      }
      atomicAdd(&out[4 * f + 0], sd);
      atomicAdd(&out[4 * f + 1], sb);
      atomicMax(reinterpret_cast<unsigned long long*>(&out[4 * f + 2]), (unsigned long long)__double_as_longlong(md));
      atomicMax(reinterpret_cast<unsigned long long*>(&out[4 * f + 3]), (unsigned long long)__double_as_longlong(mb));
    }
    __syncthreads();
  }
}

void launch_clock(Clock* clk, Counters* cnt, double cfl, hipStream_t s) {
  hipLaunchKernelGGL(k_clock, dim3(1), dim3(64), 0, s, clk, cnt, cfl);
}

}  // namespace ecg

using namespace ecg;

static thread_local std::string g_err;

static int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

namespace ecg {
int api_fail(int code, const std::string& msg) { return fail(code, msg); }
static std::atomic<int64_t> g_step_span{(int64_t)1 << 32};
int64_t step_span_bytes() { return g_step_span.load(std::memory_order_relaxed); }
}  // namespace ecg

#define HIPCHK(expr)                                                                                   \
  do {                                                                                                 \
    hipError_t e_ = (expr);                                                                            \
    if (e_ != hipSuccess) return fail(ECG_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

struct ecg_ctx {
  ecg_config cfg;
  Params P;
  int D = 1, nvar = 0;
  int64_t ncell = 0, pitch = 0;
  hipStream_t stream = nullptr;
  void* W[3] = {nullptr, nullptr, nullptr};    // two time levels + second-order predicted state
  int esize = 8;                               // bytes per state element (8: FP64 form, 4: FP32 forms)
  int cur = 0;                                 // W[cur] holds the current state
  double* tank_buf = nullptr;                  // flux records of the inlet-tank faces (k_tank)
  int64_t ntank = 0;                           // inlet-tank faces
  Params* pdev = nullptr;                      // device copy of P (the step kernels' parameters)
  Clock* clk = nullptr;                        // device clock
  Counters* cnt = nullptr;
  Clock* hclk = nullptr;                       // pinned host mirror
  Counters* hcnt = nullptr;
  step_fn step = nullptr;
  fill_fn fill = nullptr;
  int64_t pending = 0;                         // steps enqueued since the clock was last read
  int cur_at_sync = 0;                         // cur and the clock's iteration when last read
  int64_t iter_at_sync = 0;
  WarnRec* warn_rec = nullptr;                 // warning log of the step kernels (WARN_CAP records)
  unsigned long long* warn_cnt = nullptr;      // its append counter (device)
  std::vector<ecg_warning> warn_host;          // records read back, not yet taken
  int64_t warn_dropped = 0;                    // warnings beyond the log's capacity
  int64_t warn_seen = 0;                       // newton_warn total when the log was last drained
  // Kernel timing (ecg_set_profiling): event pairs per launch, resolved at synchronisation.
  bool profiling = false;
  std::vector<hipEvent_t> ev_pool;
  std::vector<std::pair<int, std::pair<hipEvent_t, hipEvent_t>>> ev_pending;
  double kt_ms[ECG_K_KINDS] = {};
  int64_t kt_n[ECG_K_KINDS] = {};
  MlpDev mlp = {nullptr, nullptr};                // learned warm start (ecg_set_warm_start)
  SampleSink sink = {nullptr, nullptr, 0, 0, 1};  // relaxation sample capture (ecg_attach_samples)
  // Staging buffers of the state download, allocated by the first one (at most 8 MB).
  unsigned char* bounce[8] = {};
  hipEvent_t bounce_ev[8] = {};
  const ecg_mlp* mlp_obj = nullptr;               // the attached objects (their attachment counts)
  ecg_samples* sink_obj = nullptr;
};

// Records the step kernels' warning log holds per context; further warnings are
// counted (Counters::newton_warn) but not recorded.
constexpr int64_t WARN_CAP = 4096;

static hipEvent_t take_event(ecg_ctx* c) {
  if (!c->ev_pool.empty()) {
    hipEvent_t e = c->ev_pool.back();
    c->ev_pool.pop_back();
    return e;
  }
  hipEvent_t e = nullptr;
  hipEventCreate(&e);
  return e;
}

// Launch f() between two recorded events when profiling.
template <class F>
static void timed(ecg_ctx* c, int kind, F f) {
  if (!c->profiling) {
    f();
    return;
  }
  hipEvent_t a = take_event(c), b = take_event(c);
  hipEventRecord(a, c->stream);
  f();
  hipEventRecord(b, c->stream);
  c->ev_pending.push_back({kind, {a, b}});
}

static void resolve_events(ecg_ctx* c) {
  for (auto& r : c->ev_pending) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, r.second.first, r.second.second) == hipSuccess) {
      c->kt_ms[r.first] += ms;
      c->kt_n[r.first] += 1;
    }
    c->ev_pool.push_back(r.second.first);
    c->ev_pool.push_back(r.second.second);
  }
  c->ev_pending.clear();
}

extern "C" {

const char* ecg_last_error(void) { return g_err.c_str(); }

const char* ecg_version(void) { return "ecogen_amd 0.1 (gfx950)"; }

int ecg_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

static bool valid_eos(const ecg_eos& e) {
  return (e.type == ECG_EOS_IG || e.type == ECG_EOS_SG) && std::isfinite(e.gamma) && e.gamma > 1.0 &&
         std::isfinite(e.pinf) && std::isfinite(e.eref);
}

static EosDev make_eos(const ecg_eos& e) {
  EosDev q;
  q.sg = (e.type == ECG_EOS_SG);
  q.g = e.gamma;
  q.pinf = q.sg ? e.pinf : 0.;
  q.gm1 = e.gamma - 1.;
  q.gpinf = e.gamma * q.pinf;
  q.eref = e.eref;
  q.mixg = q.sg ? e.gamma * q.pinf / (e.gamma - 1.) : 0.;
  q.mixinv = 1. / (e.gamma - 1.);
  q.pclamp = q.sg ? -(1. - 1.e-15) * q.pinf + 1.e-15 : 1.e-8;
  q.fg = (float)q.g; q.fpinf = (float)q.pinf; q.fgm1 = (float)q.gm1; q.fgpinf = (float)q.gpinf;
  q.feref = (float)q.eref; q.fmixinv = (float)q.mixinv; q.fpclamp = (float)q.pclamp;
  return q;
}

// Tank constants (BoundCondInletTank.cpp:56, 121 for the densities; ModUEq.cpp:562-569
// and ModEuler.cpp:474-476 for the mixture density, mass fractions and total
// enthalpy, whose zero tank velocity adds exactly nothing).
static TankDev make_tank(const ecg_config& g, double eps, const ecg_tank& t) {
  TankDev T;
  std::memset(&T, 0, sizeof(T));
  T.p0 = t.p0;
  auto energy = [&](const ecg_eos& q, double rho, double p) {
    if (q.type == ECG_EOS_SG) return (p + q.gamma * q.pinf) / (q.gamma - 1.) / std::max(rho, eps) + q.eref;
    return p / (q.gamma - 1.) / std::max(rho, eps) + q.eref;
  };
  for (int k = 0; k < g.nph; k++) {
    const ecg_eos& q = g.eos[k];
    const double num = (q.type == ECG_EOS_SG) ? t.p0 + q.pinf : t.p0;
    T.rhok0[k] = num / std::max(((q.gamma - 1.) * q.cv * t.T0), eps);
  }
  if (g.model == ECG_EULER) {
    T.Yk0[0] = 1.;
    T.H0 = energy(g.eos[0], T.rhok0[0], T.p0) + T.p0 / std::max(T.rhok0[0], eps);
    return T;
  }
  double rho0 = 0.;
  for (int k = 0; k < g.nph; k++) rho0 += t.alpha[k] * T.rhok0[k];
  T.H0 = 0.;
  for (int k = 0; k < g.nph; k++) {
    T.Yk0[k] = t.alpha[k] * T.rhok0[k] / rho0;
    T.H0 += T.Yk0[k] * (energy(g.eos[k], T.rhok0[k], T.p0) + T.p0 / std::max(T.rhok0[k], eps));
  }
  return T;
}

static int check_config(const ecg_config* c) {
  if (!c) return fail(ECG_E_ARG, "null config");
  if (c->nx < 2) return fail(ECG_E_ARG, "Number of cells in the x-direction has to be superior to 1");
  if (c->ny < 1 || c->nz < 1) return fail(ECG_E_ARG, "cell counts must be positive");
  if (c->nz > 1 && c->ny <= 1)
    return fail(ECG_E_ARG, "Number of cells in the z-direction can't be superior to 1 if number of cells in the "
                           "y-direction is equal to 1");
  if (!(c->lx > 0 && c->ly > 0 && c->lz > 0)) return fail(ECG_E_ARG, "domain lengths must be positive");
  if (c->model < ECG_EULER || c->model > ECG_UEQ) return fail(ECG_E_ARG, "unknown model");
  if (c->model == ECG_EULER && c->nph != 1) return fail(ECG_E_ARG, "Euler model has exactly one phase");
  if (c->model != ECG_EULER && (c->nph < 2 || c->nph > 3))
    return fail(ECG_E_UNSUPPORTED, "multiphase models are built for 2 or 3 phases");
  for (int k = 0; k < c->nph; k++)
    if (!valid_eos(c->eos[k])) return fail(ECG_E_ARG, "invalid EOS parameters for phase " + std::to_string(k));
  if (c->order != 1 && c->order != 2) return fail(ECG_E_ARG, "order must be 1 or 2");
  if (c->order == 2) {
    for (int i = 0; i < 4; i++) {
      if (c->lim[i] == ECG_LIM_THINC) {
        if (i < 2) return fail(ECG_E_ARG, "THINC can only be a volume-fraction limiter");
        if (c->model == ECG_EULER || c->nph != 2) return fail(ECG_E_ARG, "Limiter THINC only works for 2 phases");
        continue;
      }
      if (c->lim[i] < ECG_LIM_MINMOD || c->lim[i] > ECG_LIM_MC)
        return fail(ECG_E_UNSUPPORTED, "second order needs minmod/vanleer/vanalbada/superbee/mc/THINC limiters");
    }
  }
  for (int i = 0; i < 6; i++) {
    if (c->bc[i] != ECG_BC_NONREFLECTING && c->bc[i] != ECG_BC_WALL && c->bc[i] != ECG_BC_INLET_TANK)
      return fail(ECG_E_ARG, "unknown boundary");
    if (c->bc[i] != ECG_BC_INLET_TANK) continue;
    const ecg_tank& t = c->tank[i];
    if (!(t.p0 > 0.) || !std::isfinite(t.p0) || !(t.T0 > 0.) || !std::isfinite(t.T0))
      return fail(ECG_E_ARG, "inlet tank " + std::to_string(i) + ": p0 and T0 must be positive");
    for (int k = 0; k < c->nph; k++)
      if (!(c->eos[k].cv > 0.)) return fail(ECG_E_ARG, "inlet tank: the EOS of phase " + std::to_string(k) +
                                                           " needs cv > 0 for its density at (p0, T0)");
    if (c->model != ECG_EULER) {
      double sum = 0.;
      for (int k = 0; k < c->nph; k++) {
        if (!(t.alpha[k] >= 0. && t.alpha[k] <= 1.)) return fail(ECG_E_ARG, "alpha should be in [0,1]");
        sum += t.alpha[k];
      }
      if (std::fabs(sum - 1.) > 1.e-6) return fail(ECG_E_ARG, "sum of alpha should be 1");
    }
  }
  if (!(c->cfl > 0)) return fail(ECG_E_ARG, "CFL must be positive");
  if (c->precision != ECG_FP64 && c->precision != ECG_FP32_RELAX64 && c->precision != ECG_FP32_LEARNED)
    return fail(ECG_E_ARG, "unknown precision form");
  if (c->precision == ECG_FP32_LEARNED && (c->model == ECG_EULER || (c->model == ECG_UEQ && !c->relax_p)))
    return fail(ECG_E_ARG, "the learned warm start needs a relaxing multiphase model");
  if (!(c->relax_rate >= 0.) || !std::isfinite(c->relax_rate)) return fail(ECG_E_ARG, "relax_rate must be >= 0");
  if (c->relax_rate > 0. && (c->model != ECG_UEQ || !c->relax_p))
    return fail(ECG_E_ARG, "finite-rate pressure relaxation belongs to VELOCITYEQ with relax_p");
  if (c->relax_rate > 0. && c->precision == ECG_FP32_LEARNED)
    return fail(ECG_E_ARG, "the learned warm start accelerates the infinite relaxation only");
  if (c->precision != ECG_FP64) {
    // The FP32 step kernels index cells in 32 bits and address one tile row of the
    // outermost axis with its halo (two lines of cells on each side) by 32-bit byte
    // offsets: 3D rows are 4 planes deep, 2D rows 16 lines, 1D rows 256 cells.
    const int dims = (c->nx > 1) + (c->ny > 1) + (c->nz > 1);
    const int64_t row = (dims == 3) ? 8 * (int64_t)c->nx * c->ny : (dims == 2) ? 20 * (int64_t)c->nx : 260;
    if ((int64_t)c->nx * c->ny * c->nz >= ((int64_t)1 << 32))
      return fail(ECG_E_UNSUPPORTED, "the FP32 forms index at most 2^32 cells per GPU");
    if (row * 4 > ((int64_t)1 << 32))
      return fail(ECG_E_UNSUPPORTED, "a plane of " + std::to_string(c->nx) + " x " + std::to_string(c->ny) +
                                         " cells is too large for the FP32 forms' 32-bit state offsets");
  }
  return ECG_OK;
}

// Sizes of a case's state.
struct Layout {
  int D, nvar, esize;
  int64_t ncell, pitch, ntank;
};

// Everything the step kernels' parameters hold that needs no device memory: geometry,
// EOS, limiters, boundaries, tanks, tiles and the uniform-axis constants.  The device
// pointers (tank records, warning log) are the caller's to set.  Allocates
// nothing.  g is a checked configuration with relax_p normalised.
static void build_params(const ecg_config& g, Params& P, Layout& Ly) {
  Ly.D = (g.nx > 1) + (g.ny > 1) + (g.nz > 1);
  Ly.ncell = (int64_t)g.nx * g.ny * g.nz;
  Ly.pitch = (Ly.ncell + 63) / 64 * 64;
  Ly.nvar = (g.model == ECG_EULER) ? (2 + Ly.D + 1) : (3 * g.nph + Ly.D + 1);
  Ly.esize = (g.precision != ECG_FP64) ? 4 : 8;
  std::memset(&P, 0, sizeof(P));
  P.nx = g.nx; P.ny = g.ny; P.nz = g.nz;
  P.ncell = Ly.ncell;
  P.pitch = Ly.pitch;
  // MeshCartesian::meshStretching / initializeGeometrieMonoCpu (MeshCartesian.cpp:168-246)
  const int n3[3] = {g.nx, g.ny, g.nz};
  const double L3[3] = {g.lx, g.ly, g.lz};
  for (int a = 0; a < 3; a++) P.d[a] = L3[a] / (double)n3[a];
  const double volume = P.d[0] * P.d[1] * P.d[2];
  P.coef[0] = P.d[1] * P.d[2] / volume;
  P.coef[1] = P.d[0] * P.d[2] / volume;
  P.coef[2] = P.d[0] * P.d[1] / volume;
  double lcfl = 1.e10;
  if (g.nx != 1) lcfl = std::min(lcfl, P.d[0]);
  if (g.ny != 1) lcfl = std::min(lcfl, P.d[1]);
  if (g.nz != 1) lcfl = std::min(lcfl, P.d[2]);
  if (Ly.D > 1) lcfl *= 0.6;
  P.lcfl = lcfl;
  P.eps = (g.model != ECG_EULER && g.alpha_null) ? 1.e-15 : 0.;  // Eos.cpp:88-97
  // verifyAndCorrectPhase (PhaseUEq.cpp:355-370), in each arithmetic.
  CellFloors& q = P.floors;
  const bool an = P.eps > 1.e-20;
  q.alo = an ? 0. : 1e-15;       q.f_alo = an ? 0.f : (float)1e-15;
  q.alo_v = an ? 0. : 1e-14;     q.f_alo_v = an ? 0.f : (float)1e-14;
  q.ahi = an ? 1. : 1. - 1e-15;  q.f_ahi = an ? 1.f : 1.f - (float)1e-15;
  q.ahi_v = an ? 1. : 1. - 1e-14; q.f_ahi_v = an ? 1.f : 1.f - (float)1e-14;
  q.rho_v = an ? 1.e-15 : 1.e-14; q.f_rho_v = an ? (float)1.e-15 : (float)1.e-14;
  P.cfl = g.cfl;
  P.alpha_null = g.alpha_null;
  P.relax = g.relax_p;
  P.relax_mu = (g.model == ECG_UEQ && g.relax_p) ? g.relax_rate : 0.;
  for (int i = 0; i < 6; i++) P.bc[i] = g.bc[i];
  for (int i = 0; i < 4; i++) P.lim[i] = g.lim[i];
  P.thinc = (g.order == 2 && (g.lim[2] == ECG_LIM_THINC || g.lim[3] == ECG_LIM_THINC)) ? 1 : 0;
  P.thinc_cosh = std::cosh(1.6);
  P.thinc_tanh = std::tanh(1.6);
  for (int k = 0; k < g.nph; k++) P.eos[k] = make_eos(g.eos[k]);
  for (int i = 0; i < 6; i++)
    if (g.bc[i] == ECG_BC_INLET_TANK) P.tank[i] = make_tank(g, P.eps, g.tank[i]);
  int tex[3];
  tile_extent(Ly.D, Ly.esize, tex);
  for (int a = 0; a < 3; a++) P.tiles[a] = (n3[a] + tex[a] - 1) / tex[a];

  // Boundary faces at 0 and at the last centre + d/2 (MeshCartesian.cpp:395-552):
  // Face::distance to the adjacent centre, used by second-order walls.
  for (int a = 0; a < 3; a++) {
    const double first = (0 + 0.5) * P.d[a], last = (n3[a] - 1 + 0.5) * P.d[a];
    const double x0 = 0. - first;
    const double fp = last + 0.5 * P.d[a];
    const double x1 = fp - last;
    P.dwall[a][0] = std::sqrt(x0 * x0 + 0. * 0. + 0. * 0.);
    P.dwall[a][1] = std::sqrt(x1 * x1 + 0. * 0. + 0. * 0.);
  }
  // The axes where each of the three face distances is one value.
  P.dist_uniform = 0;
  P.dcc_pow2 = 0;
  for (int a = 0; a < 3; a++) {
    if (n3[a] < 2) continue;
    const double c0 = face_distance(P.d[a], 0, 0), l0 = face_distance(P.d[a], 0, 1), r0 = face_distance(P.d[a], 0, 2);
    bool uni = true;
    for (int m = 1; m + 1 < n3[a] && uni; m++)
      uni = face_distance(P.d[a], m, 0) == c0 && face_distance(P.d[a], m, 1) == l0 && face_distance(P.d[a], m, 2) == r0;
    if (!uni) continue;
    P.dist_uniform |= 1 << a;
    P.dcc_c[a] = c0; P.dfl_c[a] = l0; P.dfr_c[a] = r0;
    int ex = 0;
    const double fr = std::frexp(c0, &ex);
    if (fr == 0.5 && std::isnormal(c0) && ex > -1000) {
      P.dcc_pow2 |= 1 << a;
      P.inv_dcc[a] = std::ldexp(1.0, 1 - ex);     // 1 / 2^(ex-1), exact
    } else {
      P.inv_dcc[a] = 1.0 / c0;
    }
  }
  // Float copies for the FP32 kernels.
  P.f_eps = (float)P.eps;
  for (int a = 0; a < 3; a++) {
    P.f_coef[a] = (float)P.coef[a];
    P.f_dcc_c[a] = (float)P.dcc_c[a]; P.f_dfl_c[a] = (float)P.dfl_c[a]; P.f_dfr_c[a] = (float)P.dfr_c[a];
    P.f_inv_dcc[a] = (float)P.inv_dcc[a];
    P.f_dwall[a][0] = (float)P.dwall[a][0]; P.f_dwall[a][1] = (float)P.dwall[a][1];
  }
  // Inlet-tank face records, sides in order (the step kernels read them back by side and plane index).
  Ly.ntank = 0;
  for (int q = 0; q < 2 * Ly.D; q++)
    if (P.bc[q] == BC_TANK) { P.tank_off[q] = Ly.ntank; Ly.ntank += tank_faces(P, q); }
}

ecg_ctx* ecg_create(const ecg_config* cfg) {
  if (check_config(cfg) != ECG_OK) return nullptr;
  ecg_ctx* c = new ecg_ctx();
  c->cfg = *cfg;
  if (cfg->model == ECG_PUEQ) c->cfg.relax_p = 1;
  if (cfg->model == ECG_EULER) c->cfg.relax_p = 0;
  const ecg_config& g = c->cfg;
  Params& P = c->P;
  Layout Ly;
  build_params(g, P, Ly);
  c->D = Ly.D;
  c->ncell = Ly.ncell;
  c->pitch = Ly.pitch;
  c->nvar = Ly.nvar;
  c->esize = Ly.esize;
  const bool f32 = (g.precision != ECG_FP64);
  c->step = get_step_fn(g.model, g.nph, c->D, f32);
  c->fill = get_fill_fn(g.model, g.nph, c->D, f32);
  if (!c->step || !c->fill) {
    fail(ECG_E_UNSUPPORTED, "no kernel built for this model/phase/dimension combination");
    delete c;
    return nullptr;
  }
  bool ok = true;
  auto chk = [&](hipError_t e, const char* what) {
    if (e != hipSuccess && ok) {
      ok = false;
      fail(ECG_E_HIP, std::string(what) + ": " + hipGetErrorString(e));
    }
  };
  chk(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking), "hipStreamCreate");
  const size_t bytes = (size_t)c->esize * (size_t)c->pitch * c->nvar;
  const int nbuf = (g.order == 2) ? 3 : 2;
  for (int b = 0; b < nbuf && ok; b++) chk(hipMalloc(&c->W[b], bytes), "hipMalloc(state)");
  const int64_t ntank = Ly.ntank;
  if (ok && ntank > 0) chk(hipMalloc(&c->tank_buf, sizeof(double) * TANK_REC * ntank), "hipMalloc(tank records)");
  c->ntank = ntank;
  P.tank_buf = c->tank_buf;
  if (ok) chk(hipMalloc(&c->clk, sizeof(Clock)), "hipMalloc(clock)");
  if (ok) chk(hipMalloc(&c->cnt, sizeof(Counters) * ATOMIC_SLOTS), "hipMalloc(counters)");
  if (ok) chk(hipHostMalloc(&c->hclk, sizeof(Clock), hipHostMallocDefault), "hipHostMalloc(clock)");
  if (ok) chk(hipHostMalloc(&c->hcnt, sizeof(Counters) * ATOMIC_SLOTS, hipHostMallocDefault), "hipHostMalloc(counters)");
  if (ok) chk(hipMalloc(&c->warn_rec, sizeof(WarnRec) * WARN_CAP), "hipMalloc(warning log)");
  if (ok) chk(hipMalloc(&c->warn_cnt, sizeof(unsigned long long)), "hipMalloc(warning counter)");
  P.warn_rec = c->warn_rec;
  P.warn_cnt = c->warn_cnt;
  P.warn_cap = WARN_CAP;
  if (!ok) {
    ecg_destroy(c);
    return nullptr;
  }
  // The host copies mirror the zeroed device counters until the first read (pinned
  // memory can come back from an earlier context with its old contents).
  std::memset(c->hclk, 0, sizeof(Clock));
  std::memset(c->hcnt, 0, sizeof(Counters) * ATOMIC_SLOTS);
  // The step kernels' parameters, complete from here on.
  if (hipMalloc(&c->pdev, sizeof(Params)) != hipSuccess ||
      hipMemcpy(c->pdev, &c->P, sizeof(Params), hipMemcpyHostToDevice) != hipSuccess) {
    fail(ECG_E_HIP, "device copy of the parameters");
    ecg_destroy(c);
    return nullptr;
  }
  // Zero the state and counters, reset the clock.
  for (int b = 0; b < nbuf; b++) hipMemset(c->W[b], 0, bytes);
  hipMemset(c->cnt, 0, sizeof(Counters) * ATOMIC_SLOTS);
  hipMemset(c->warn_cnt, 0, sizeof(unsigned long long));
  if (ecg_reset_clock(c) != ECG_OK) {
    ecg_destroy(c);
    return nullptr;
  }
  hipStreamSynchronize(c->stream);
  return c;
}

void ecg_destroy(ecg_ctx* c) {
  if (!c) return;
  if (c->stream) hipStreamSynchronize(c->stream);
  if (c->mlp_obj) mlp_detach(c->mlp_obj);
  if (c->sink_obj) samples_detach(c->sink_obj);
  if (c->warn_rec) hipFree(c->warn_rec);
  if (c->pdev) hipFree(c->pdev);
  if (c->warn_cnt) hipFree(c->warn_cnt);
  for (int b = 0; b < 3; b++)
    if (c->W[b]) hipFree(c->W[b]);
  if (c->tank_buf) hipFree(c->tank_buf);
  if (c->clk) hipFree(c->clk);
  if (c->cnt) hipFree(c->cnt);
  if (c->hclk) hipHostFree(c->hclk);
  if (c->hcnt) hipHostFree(c->hcnt);
  for (int b = 0; b < 8; b++) {
    if (c->bounce[b]) hipHostFree(c->bounce[b]);
    if (c->bounce_ev[b]) hipEventDestroy(c->bounce_ev[b]);
  }
  for (auto& r : c->ev_pending) { c->ev_pool.push_back(r.second.first); c->ev_pool.push_back(r.second.second); }
  for (hipEvent_t e : c->ev_pool) hipEventDestroy(e);
  if (c->stream) hipStreamDestroy(c->stream);
  delete c;
}

int ecg_nvar(const ecg_ctx* c) { return c ? c->nvar : ECG_E_ARG; }
int64_t ecg_ncell(const ecg_ctx* c) { return c ? c->ncell : ECG_E_ARG; }
void* ecg_stream(ecg_ctx* c) { return c ? (void*)c->stream : nullptr; }

static Clock fresh_clock(double dt, int64_t max_iter, double t_end) {
  Clock k;
  std::memset(&k, 0, sizeof(k));
  k.t = 0.;
  k.dt = dt;
  k.dt_next = dt;
  k.dt_max = 1.e10;
  k.t_end = t_end;
  k.iteration = 0;
  k.max_iter = max_iter;
  k.done = 0;
  return k;
}

static int set_clock(ecg_ctx* c, const Clock& k) {
  hipLaunchKernelGGL(k_clock_set, dim3(1), dim3(64), 0, c->stream, c->clk, c->cnt, k);
  HIPCHK(hipGetLastError());
  return ECG_OK;
}

int ecg_reset_clock(ecg_ctx* c) {
  if (!c) return fail(ECG_E_ARG, "null context");
  c->pending = 0;
  c->cur_at_sync = c->cur;
  c->iter_at_sync = 0;
  return set_clock(c, fresh_clock(1.e-15, 0, INFINITY));
}

int ecg_fill(ecg_ctx* c, const ecg_domain* doms, int ndom) {
  if (!c || !doms || ndom < 1) return fail(ECG_E_ARG, "ecg_fill needs at least one domain");
  std::vector<DomainDev> dd(ndom);
  for (int q = 0; q < ndom; q++) {
    const ecg_domain& s = doms[q];
    DomainDev& d = dd[q];
    std::memset(&d, 0, sizeof(d));
    if (s.kind < ECG_DOM_ENTIRE || s.kind > ECG_DOM_CUBOID) return fail(ECG_E_ARG, "unknown domain kind");
    if (s.axis < 0 || s.axis > 2 || s.axis2 < 0 || s.axis2 > 2) return fail(ECG_E_ARG, "domain axis out of range");
    d.kind = s.kind; d.axis = s.axis; d.axis2 = s.axis2; d.dir = s.dir; d.origin = s.origin; d.radius = s.radius;
    for (int a = 0; a < 3; a++) {
      d.center[a] = s.center[a]; d.lo[a] = s.lo[a]; d.len[a] = s.len[a]; d.vel[a] = s.vel[a];
      if (a >= c->D && s.vel[a] != 0.)
        return fail(ECG_E_ARG, "velocity along an inactive axis must be zero (state keeps active axes only)");
    }
    for (int k = 0; k < ECG_MAX_PHASES; k++) { d.alpha[k] = s.alpha[k]; d.rho[k] = s.rho[k]; d.p[k] = s.p[k]; }
  }
  DomainDev* ddev = nullptr;
  HIPCHK(hipMalloc(&ddev, sizeof(DomainDev) * ndom));
  HIPCHK(hipMemcpyAsync(ddev, dd.data(), sizeof(DomainDev) * ndom, hipMemcpyHostToDevice, c->stream));
  c->fill(c->P, ddev, ndom, c->W[c->cur], c->stream);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(c->stream));
  HIPCHK(hipFree(ddev));
  return ECG_OK;
}

int ecg_upload_state(ecg_ctx* c, const double* const* soa, int nvars) {
  if (!c || !soa) return fail(ECG_E_ARG, "null argument");
  if (nvars != c->nvar) return fail(ECG_E_ARG, "expected " + std::to_string(c->nvar) + " state arrays");
  std::vector<float> tmp;
  for (int v = 0; v < nvars; v++) {
    if (!soa[v]) return fail(ECG_E_ARG, "null state array");
    char* dst = (char*)c->W[c->cur] + (size_t)v * c->pitch * c->esize;
    if (c->esize == 8) {
      HIPCHK(hipMemcpyAsync(dst, soa[v], sizeof(double) * c->ncell, hipMemcpyHostToDevice, c->stream));
    } else {
      tmp.resize(c->ncell);
      for (int64_t i = 0; i < c->ncell; i++) tmp[i] = (float)soa[v][i];
      HIPCHK(hipMemcpyAsync(dst, tmp.data(), sizeof(float) * c->ncell, hipMemcpyHostToDevice, c->stream));
    }
    HIPCHK(hipStreamSynchronize(c->stream));
  }
  HIPCHK(hipStreamSynchronize(c->stream));
  return ECG_OK;
}

static int settle(ecg_ctx* c);

// Elements [e, e + n) of the state array (variables pitch apart), staged at src, to the
// caller's arrays of doubles.
static void unpack_state(const ecg_ctx* c, double* const* soa, const unsigned char* src, int64_t e, int64_t n) {
  for (int64_t at = e; at < e + n;) {
    const int64_t v = at / c->pitch, i = at % c->pitch, k = std::min(c->pitch - i, e + n - at);
    const int64_t cells = std::min(k, c->ncell - i);   // the rest pads the variable
    if (cells > 0) {
      const unsigned char* s = src + (at - e) * c->esize;
      if (c->esize == 8) std::memcpy(soa[v] + i, s, sizeof(double) * cells);
      else for (int64_t q = 0; q < cells; q++) soa[v][i + q] = (double)reinterpret_cast<const float*>(s)[q];
    }
    at += k;
  }
}

// Whether p is memory that the device copies to directly: page-locked, or the device's own or
// managed memory (*device), which the host threads need not reach.
static bool device_reachable(const void* p, bool* device) {
  hipPointerAttribute_t at;
  if (hipPointerGetAttributes(&at, p) != hipSuccess) {
    (void)hipGetLastError();   // an address the runtime does not know: ordinary host memory
    return false;
  }
  *device = at.type == hipMemoryTypeManaged || at.type == hipMemoryTypeDevice;
  return *device || at.type == hipMemoryTypeHost;
}

// Whether two of the caller's arrays share memory: the later variable's values then stand.
static bool arrays_overlap(const ecg_ctx* c, double* const* soa) {
  uintptr_t at[3 * ECG_MAX_PHASES + 3];
  for (int v = 0; v < c->nvar; v++) at[v] = reinterpret_cast<uintptr_t>(soa[v]);
  std::sort(at, at + c->nvar);
  for (int v = 1; v < c->nvar; v++)
    if (at[v] - at[v - 1] < sizeof(double) * (uintptr_t)c->ncell) return true;
  return false;
}

// One variable after the other, by the runtime's own copies.
static int download_plain(ecg_ctx* c, double* const* soa) {
  std::unique_ptr<float[]> tmp;
  if (c->esize == 4) {
    tmp.reset(new (std::nothrow) float[c->ncell]);
    if (!tmp) return fail(ECG_E_ARG, "no host memory for the state's conversion");
  }
  for (int v = 0; v < c->nvar; v++) {
    const char* src = static_cast<const char*>(c->W[c->cur]) + (size_t)v * c->pitch * c->esize;
    void* dst = c->esize == 8 ? static_cast<void*>(soa[v]) : tmp.get();
    HIPCHK(hipMemcpyAsync(dst, src, (size_t)c->esize * c->ncell, hipMemcpyDeviceToHost, c->stream));
    if (c->esize == 8 && v + 1 < c->nvar) continue;
    HIPCHK(hipStreamSynchronize(c->stream));
    if (c->esize == 4)
      for (int64_t i = 0; i < c->ncell; i++) soa[v][i] = (double)tmp[i];
  }
  return ECG_OK;
}

// The state through pinned buffers of 1 MB: large states by up to eight threads, each with a
// buffer of its own, that copy and unpack every eighth piece.  The host side is the bound:
// the caller's arrays are usually fresh pages, and one thread converting floats into them
// took 8 ms for the ten variables of a 104^3 mesh, half of a 32-step run.  FP64 states of
// 2 MB and more go straight into page-locked arrays (eight variables, through the buffers /
// straight, ms: 128^2 (1 MB) 0.070 / 0.104, 181^2 0.115 / 0.115, 512^2 0.67 / 0.41, 160^3 10.4 /
// 5.8), and any into device memory.  Where page-locked memory is refused, as many threads
// as got a buffer share the pieces, and without any the runtime copies.
static int download_state(ecg_ctx* c, double* const* soa) {
  const bool large = (int64_t)c->esize * c->pitch * c->nvar >= (int64_t(2) << 20);
  for (int v = 0; v < c->nvar && c->esize == 8; v++) {
    bool device = false;
    if (device_reachable(soa[v], &device) && (large || device)) return download_plain(c, soa);
  }
  const int64_t total = c->pitch * c->nvar, piece = std::min<int64_t>(total, (int64_t(1) << 20) / c->esize);
  const int64_t npiece = (total + piece - 1) / piece;
  const int want = arrays_overlap(c, soa)   // in order
                       ? 1
                       : (int)std::min<int64_t>(std::min(8u, std::max(1u, std::thread::hardware_concurrency())), npiece);
  int team = 0;
  while (team < want) {
    if (!c->bounce_ev[team] && hipEventCreateWithFlags(&c->bounce_ev[team], hipEventDisableTiming) != hipSuccess) break;
    if (!c->bounce[team] &&
        hipHostMalloc((void**)&c->bounce[team], (size_t)piece * c->esize, hipHostMallocDefault) != hipSuccess) {
      c->bounce[team] = nullptr;
      break;
    }
    team++;
  }
  if (team < want) (void)hipGetLastError();
  if (team == 0) return download_plain(c, soa);
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  const unsigned char* src = static_cast<const unsigned char*>(c->W[c->cur]);
  hipError_t err[8] = {};
  std::atomic<int64_t> next{0};
  auto work = [&](int b) {
    if (b > 0) err[b] = hipSetDevice(dev);
    for (int64_t p; err[b] == hipSuccess && (p = next.fetch_add(1)) < npiece;) {
      const int64_t e = p * piece, n = std::min(piece, total - e);
      err[b] = hipMemcpyAsync(c->bounce[b], src + e * c->esize, (size_t)n * c->esize, hipMemcpyDeviceToHost, c->stream);
      if (err[b] == hipSuccess) err[b] = hipEventRecord(c->bounce_ev[b], c->stream);
      if (err[b] == hipSuccess) err[b] = hipEventSynchronize(c->bounce_ev[b]);
      if (err[b] == hipSuccess) unpack_state(c, soa, c->bounce[b], e, n);
    }
  };
  std::vector<std::thread> threads;
  try {
    threads.reserve((size_t)team);
    for (int b = 1; b < team; b++) threads.emplace_back(work, b);
  } catch (const std::exception&) {   // the threads that could be started share the pieces
  }
  work(0);
  for (std::thread& t : threads) t.join();
  for (int b = 0; b < team; b++) HIPCHK(err[b]);
  return ECG_OK;
}

int ecg_download_state(ecg_ctx* c, double* const* soa, int nvars) {
  if (!c || !soa) return fail(ECG_E_ARG, "null argument");
  if (nvars != c->nvar) return fail(ECG_E_ARG, "expected " + std::to_string(c->nvar) + " state arrays");
  int rc = settle(c);
  if (rc != ECG_OK) return rc;
  for (int v = 0; v < nvars; v++)
    if (!soa[v]) return fail(ECG_E_ARG, "null state array");
  return download_state(c, soa);
}

// Enqueue one step on the device clock.  Buffers ping-pong; a step the clock
// marks done is skipped by every kernel, so the current buffer is settled from
// the executed iteration count after synchronising.
static int enqueue_one(ecg_ctx* c) {
  const int nxt = 1 - c->cur;
  StepLaunch L;
  L.pdev = c->pdev;
  L.mlp = c->mlp;
  L.sink = c->sink;
  L.tank_only = 0;
  // Inlet-tank face records of the stage, then the step kernel that reads them.
  auto tank = [&] {
    if (c->ntank == 0) return;
    L.tank_only = 1;
    timed(c, ECG_K_TANK, [&] { c->step(c->P, L, c->clk, c->cnt, c->stream); });
    L.tank_only = 0;
  };
  if (c->cfg.order == 1) {
    L.wn = c->W[c->cur]; L.wsrc = c->W[c->cur]; L.wout = c->W[nxt]; L.stage = 0;
    tank();
    timed(c, ECG_K_STEP, [&] { c->step(c->P, L, c->clk, c->cnt, c->stream); });
  } else {
    L.wn = c->W[c->cur]; L.wsrc = c->W[c->cur]; L.wout = c->W[2]; L.stage = 1;
    tank();
    timed(c, ECG_K_PREDICT, [&] { c->step(c->P, L, c->clk, c->cnt, c->stream); });
    L.wn = c->W[c->cur]; L.wsrc = c->W[2]; L.wout = c->W[nxt]; L.stage = 2;
    tank();
    timed(c, ECG_K_CORRECT, [&] { c->step(c->P, L, c->clk, c->cnt, c->stream); });
  }
  timed(c, ECG_K_CLOCK, [&] { launch_clock(c->clk, c->cnt, c->cfg.cfl, c->stream); });
  HIPCHK(hipGetLastError());
  c->cur = nxt;
  c->pending += 1;
  return ECG_OK;
}

// Moves the records of the device warning log to the host list and empties the log.
static int drain_warnings(ecg_ctx* c) {
  unsigned long long n = 0;
  HIPCHK(hipMemcpyAsync(&n, c->warn_cnt, sizeof(n), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  if (n == 0) return ECG_OK;
  const int64_t k = std::min<int64_t>((int64_t)n, WARN_CAP);
  std::vector<WarnRec> r((size_t)k);
  HIPCHK(hipMemcpyAsync(r.data(), c->warn_rec, sizeof(WarnRec) * k, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipMemsetAsync(c->warn_cnt, 0, sizeof(unsigned long long), c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  for (const WarnRec& w : r) {
    ecg_warning o;
    o.iteration = w.iteration; o.cell = w.cell; o.stage = w.stage; o.kind = w.kind; o.value = w.value;
    c->warn_host.push_back(o);
  }
  c->warn_dropped += (int64_t)n - k;
  return ECG_OK;
}

static int read_clock(ecg_ctx* c) {
  HIPCHK(hipMemcpyAsync(c->hclk, c->clk, sizeof(Clock), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipMemcpyAsync(c->hcnt, c->cnt, sizeof(Counters) * ATOMIC_SLOTS, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  resolve_events(c);
  int64_t warn = 0;
  for (int q = 0; q < ATOMIC_SLOTS; q++) warn += (int64_t)c->hcnt[q].newton_warn;
  if (warn != c->warn_seen) {
    c->warn_seen = warn;
    return drain_warnings(c);
  }
  return ECG_OK;
}

// The clock has just been read and nothing is enqueued behind it.
static void mark_synced(ecg_ctx* c) {
  c->pending = 0;
  c->cur_at_sync = c->cur;
  c->iter_at_sync = c->hclk->iteration;
}

// Resolve which buffer holds the state after the enqueued steps: steps the clock
// skipped (after a run's end or an error) did not swap the buffers.
static int settle(ecg_ctx* c) {
  if (c->pending == 0) return ECG_OK;
  int rc = read_clock(c);
  if (rc != ECG_OK) return rc;
  const int64_t executed = c->hclk->iteration - c->iter_at_sync;
  c->cur = (int)((c->cur_at_sync + executed) % 2);
  mark_synced(c);
  return ECG_OK;
}

// Errors::errorMessage of ModEuler.cpp:487 / ModUEq.cpp:586 (the reference stops there).
static const char* const TANK_FAIL = "solveRiemannInletTank not converged (50 Newton iterations)";

// Host sum of the counter slots (fixed order).
static Counters sum_counters(const ecg_ctx* c) {
  Counters s;
  std::memset(&s, 0, sizeof(s));
  for (int q = 0; q < ATOMIC_SLOTS; q++) {
    const Counters& h = c->hcnt[q];
    s.newton_warn += h.newton_warn;
    s.nonfinite += h.nonfinite;
    s.newton_fail += h.newton_fail;
    s.newton_iters += h.newton_iters;
    s.relax_calls += h.relax_calls;
    s.warm_calls += h.warm_calls;
    s.warm_fallbacks += h.warm_fallbacks;
    s.resid_sum += h.resid_sum;
    s.tank_fail += h.tank_fail;
  }
  return s;
}

static void fill_stats(ecg_ctx* c, ecg_step_stats* st) {
  if (!st) return;
  st->t = c->hclk->t;
  st->dt_next = c->hclk->dt_next;
  st->dt_max = c->hclk->dt_max;
  st->iteration = c->hclk->iteration;
  const Counters s = sum_counters(c);
  st->newton_fail = (int64_t)s.newton_fail;
  st->newton_iters = (int64_t)s.newton_iters;
  st->relax_calls = (int64_t)s.relax_calls;
  st->warm_calls = (int64_t)s.warm_calls;
  st->warm_fallbacks = (int64_t)s.warm_fallbacks;
  st->resid_sum = s.resid_sum;
  st->newton_warn = (int64_t)s.newton_warn;
  st->nonfinite = (int64_t)s.nonfinite;
}

// Outcome of the steps between two counter snapshots: an error (ECG_E_STATE) when an
// inlet-tank solve failed or a cell's state became non-finite, else the number of the
// reference's warnings (non-converged relaxation Newton solves).
static int step_outcome(const Counters& before, const Counters& after) {
  if (after.tank_fail != before.tank_fail) return fail(ECG_E_STATE, TANK_FAIL);
  if (after.nonfinite != before.nonfinite)
    return fail(ECG_E_STATE, "non-finite state in " + std::to_string(after.nonfinite - before.nonfinite) +
                                 " cell updates");
  const unsigned long long w = after.newton_warn - before.newton_warn;
  return w > 0 ? (int)std::min<unsigned long long>(w, (unsigned long long)INT32_MAX) : ECG_OK;
}

int ecg_step(ecg_ctx* c, double dt, double* dtmax_out, ecg_step_stats* st) {
  if (!c) return fail(ECG_E_ARG, "null context");
  if (!(dt > 0) || !std::isfinite(dt)) return fail(ECG_E_ARG, "dt must be positive and finite");
  int rc = settle(c);
  if (rc == ECG_OK) rc = read_clock(c);
  if (rc != ECG_OK) return rc;
  Clock k = *c->hclk;
  const Counters before = sum_counters(c);
  k.dt = dt;
  k.done = 0;
  k.max_iter = 0;
  k.t_end = INFINITY;
  rc = set_clock(c, k);
  if (rc != ECG_OK) return rc;
  rc = enqueue_one(c);
  if (rc != ECG_OK) return rc;
  rc = read_clock(c);
  if (rc != ECG_OK) return rc;
  mark_synced(c);
  if (dtmax_out) *dtmax_out = c->hclk->dt_max;
  fill_stats(c, st);
  return step_outcome(before, sum_counters(c));
}

// Runs clock k until the device marks it done (or max_steps steps, when > 0,
// have been enqueued).  The executed steps decide which buffer holds the state.
static int run_clock(ecg_ctx* c, const Clock& k, int64_t max_steps, ecg_step_stats* st) {
  const int start = c->cur;
  const int64_t it0 = k.iteration;
  const Counters before = sum_counters(c);
  int rc = set_clock(c, k);
  if (rc != ECG_OK) return rc;
  int64_t enq = 0;
  int batch = 8;
  for (;;) {
    for (int b = 0; b < batch; b++) {
      rc = enqueue_one(c);
      if (rc != ECG_OK) return rc;
      enq++;
      if (max_steps > 0 && enq >= max_steps) break;
    }
    rc = read_clock(c);
    if (rc != ECG_OK) return rc;
    if (c->hclk->done) break;
    if (batch < 256) batch *= 2;
  }
  const int64_t done_steps = c->hclk->iteration - it0;
  c->cur = (int)((start + done_steps) % 2);
  mark_synced(c);
  fill_stats(c, st);
  return step_outcome(before, sum_counters(c));
}

int ecg_run(ecg_ctx* c, int64_t max_iter, double t_end, ecg_step_stats* st) {
  if (!c) return fail(ECG_E_ARG, "null context");
  if (max_iter <= 0 && !(t_end > 0)) return fail(ECG_E_ARG, "need max_iter > 0 or t_end > 0");
  // A fresh read: run_clock compares the counters against their values before the run.
  int rc = settle(c);
  if (rc == ECG_OK) rc = read_clock(c);
  if (rc != ECG_OK) return rc;
  mark_synced(c);
  return run_clock(c, fresh_clock(1.e-15, max_iter, max_iter > 0 ? INFINITY : t_end), max_iter, st);
}

int ecg_tile_of_block(const ecg_config* cfg, int ntiles, int block) {
  if (!cfg || ntiles < 1 || block < 0 || block >= ntiles) return fail(ECG_E_ARG, "block outside the launch");
  const int d = (cfg->nx > 1) + (cfg->ny > 1) + (cfg->nz > 1);
  const int esize = cfg->precision == ECG_FP64 ? 8 : 4;
  return xcd_tile(ntiles, block, tile_run(cfg->model, cfg->nph, d, esize, cfg->precision == ECG_FP32_LEARNED, ntiles));
}

double ecg_exp(double x) { return exp_cr(x); }
double ecg_log(double x) { return log_pos(x); }
double ecg_pow(double x, double y) { return pow_cr(x, y); }

int64_t ecg_set_step_span(int64_t bytes) {
  const int64_t lim = (int64_t)1 << 32;
  if (bytes <= 0) return ecg::g_step_span.load();
  return ecg::g_step_span.exchange(std::min(bytes, lim));
}

int ecg_run_to(ecg_ctx* c, int64_t until_iter, double until_t, ecg_step_stats* st) {
  if (!c) return fail(ECG_E_ARG, "null context");
  if (until_iter <= 0 && !(until_t > 0)) return fail(ECG_E_ARG, "need until_iter > 0 or until_t > 0");
  int rc = settle(c);
  if (rc == ECG_OK) rc = read_clock(c);
  if (rc != ECG_OK) return rc;
  mark_synced(c);
  Clock k = *c->hclk;
  if (until_iter > 0 && k.iteration >= until_iter) return fail(ECG_E_ARG, "the clock is already at until_iter");
  if (until_iter <= 0 && k.t >= until_t) return fail(ECG_E_ARG, "the clock is already at until_t");
  k.max_iter = until_iter > 0 ? until_iter : 0;
  k.t_end = until_iter > 0 ? INFINITY : until_t;
  k.done = 0;
  return run_clock(c, k, until_iter > 0 ? until_iter - k.iteration : 0, st);
}

int ecg_set_time(ecg_ctx* c, double t, double dt, int64_t iteration) {
  if (!c) return fail(ECG_E_ARG, "null context");
  if (!(dt > 0) || !std::isfinite(dt) || !std::isfinite(t) || iteration < 0)
    return fail(ECG_E_ARG, "need a finite time, a positive dt and a non-negative iteration");
  int rc = settle(c);
  if (rc != ECG_OK) return rc;
  Clock k = fresh_clock(dt, 0, INFINITY);
  k.t = t;
  k.iteration = iteration;
  rc = set_clock(c, k);
  if (rc != ECG_OK) return rc;
  rc = read_clock(c);
  if (rc != ECG_OK) return rc;
  mark_synced(c);
  return ECG_OK;
}

int ecg_enqueue_steps(ecg_ctx* c, int n) {
  if (!c || n < 0) return fail(ECG_E_ARG, "bad arguments");
  if (n > 0) {
    hipLaunchKernelGGL(k_clock_open, dim3(1), dim3(64), 0, c->stream, c->clk);
    HIPCHK(hipGetLastError());
  }
  for (int i = 0; i < n; i++) {
    int rc = enqueue_one(c);
    if (rc != ECG_OK) return rc;
  }
  return ECG_OK;
}

int ecg_synchronize(ecg_ctx* c, ecg_step_stats* st) {
  if (!c) return fail(ECG_E_ARG, "null context");
  int rc = settle(c);
  if (rc == ECG_OK) rc = read_clock(c);
  if (rc != ECG_OK) return rc;
  mark_synced(c);
  fill_stats(c, st);
  return ECG_OK;
}

int64_t ecg_take_warnings(ecg_ctx* c, ecg_warning* out, int64_t max, int64_t* dropped) {
  if (!c || max < 0 || (max > 0 && !out)) return fail(ECG_E_ARG, "bad arguments");
  int rc = settle(c);
  if (rc == ECG_OK) rc = read_clock(c);
  if (rc != ECG_OK) return rc;
  // The reference's order: steps in turn, the predictor's relaxations before the
  // corrector's, cells in index order within a stage.
  std::stable_sort(c->warn_host.begin(), c->warn_host.end(), [](const ecg_warning& a, const ecg_warning& b) {
    if (a.iteration != b.iteration) return a.iteration < b.iteration;
    if (a.stage != b.stage) return a.stage < b.stage;
    return a.cell < b.cell;
  });
  const int64_t n = std::min<int64_t>(max, (int64_t)c->warn_host.size());
  std::copy(c->warn_host.begin(), c->warn_host.begin() + n, out);
  c->warn_host.erase(c->warn_host.begin(), c->warn_host.begin() + n);
  if (dropped) *dropped = c->warn_dropped;
  c->warn_dropped = 0;
  return n;
}

int ecg_calibration_copy(ecg_ctx* c, int64_t nbytes) {
  if (!c) return fail(ECG_E_ARG, "null context");
  const int64_t cap = (int64_t)c->esize * c->pitch * c->nvar;
  if (nbytes <= 0 || nbytes > cap || nbytes % 16) return fail(ECG_E_ARG, "nbytes must be a positive multiple of 16 "
                                                                       "not larger than one state buffer");
  const int64_t n2 = nbytes / 16;
  const int threads = 256;
  const int blocks = (int)std::min<int64_t>((n2 + threads - 1) / threads, 256 * 1024);
  hipLaunchKernelGGL(k_copy, dim3(blocks), dim3(threads), 0, c->stream, (const double2*)c->W[c->cur],
                     (double2*)c->W[1 - c->cur], n2);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(c->stream));
  return ECG_OK;
}

int ecg_state_diff(ecg_ctx* a, ecg_ctx* b, double* out, int nfields) {
  if (!a || !b || !out) return fail(ECG_E_ARG, "null argument");
  if (a->ncell != b->ncell || a->nvar != b->nvar || a->cfg.model != b->cfg.model || a->cfg.nph != b->cfg.nph ||
      a->cfg.nx != b->cfg.nx || a->cfg.ny != b->cfg.ny || a->cfg.nz != b->cfg.nz)
    return fail(ECG_E_ARG, "the two contexts hold different meshes or models");
  if (nfields != a->nvar + 1) return fail(ECG_E_ARG, "nfields must be nvar + 1");
  int rc = settle(a);
  if (rc != ECG_OK) return rc;
  rc = settle(b);
  if (rc != ECG_OK) return rc;
  HIPCHK(hipStreamSynchronize(b->stream));
  double* d = nullptr;
  const size_t bytes = sizeof(double) * 4 * (size_t)nfields;
  HIPCHK(hipMalloc(&d, bytes));
  hipError_t e = hipMemsetAsync(d, 0, bytes, a->stream);
  const int blocks = (int)std::min<int64_t>((a->ncell + 255) / 256, 4096);
  const int mp = a->cfg.model != ECG_EULER;
  if (e == hipSuccess) {
    if (a->esize == 8 && b->esize == 8)
      hipLaunchKernelGGL((k_state_diff<double, double>), dim3(blocks), dim3(256), 0, a->stream, (const double*)a->W[a->cur],
                         (const double*)b->W[b->cur], a->ncell, a->pitch, b->pitch, a->nvar, a->cfg.nph, mp, d);
    else if (a->esize == 4 && b->esize == 8)
      hipLaunchKernelGGL((k_state_diff<float, double>), dim3(blocks), dim3(256), 0, a->stream, (const float*)a->W[a->cur],
                         (const double*)b->W[b->cur], a->ncell, a->pitch, b->pitch, a->nvar, a->cfg.nph, mp, d);
    else if (a->esize == 8 && b->esize == 4)
      hipLaunchKernelGGL((k_state_diff<double, float>), dim3(blocks), dim3(256), 0, a->stream, (const double*)a->W[a->cur],
                         (const float*)b->W[b->cur], a->ncell, a->pitch, b->pitch, a->nvar, a->cfg.nph, mp, d);
    else
      hipLaunchKernelGGL((k_state_diff<float, float>), dim3(blocks), dim3(256), 0, a->stream, (const float*)a->W[a->cur],
                         (const float*)b->W[b->cur], a->ncell, a->pitch, b->pitch, a->nvar, a->cfg.nph, mp, d);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(out, d, bytes, hipMemcpyDeviceToHost, a->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(a->stream);
  hipFree(d);
  if (e != hipSuccess) return fail(ECG_E_HIP, std::string("state comparison: ") + hipGetErrorString(e));
  return ECG_OK;
}

int ecg_attach_samples(ecg_ctx* c, ecg_samples* smp, int stride) {
  if (!c) return fail(ECG_E_ARG, "null context");
  if (!smp) {
    int rc = settle(c);
    if (rc != ECG_OK) return rc;
    c->sink = SampleSink{nullptr, nullptr, 0, 0, 1};
    if (c->sink_obj) samples_detach(c->sink_obj);
    c->sink_obj = nullptr;
    return ECG_OK;
  }
  if (stride < 1) return fail(ECG_E_ARG, "sample stride must be at least 1");
  if (c->cfg.model == ECG_EULER || !c->cfg.relax_p) return fail(ECG_E_ARG, "the case has no pressure relaxation");
  if (c->mlp.frag) return fail(ECG_E_ARG, "samples record cold solves: detach the warm start first");
  if (c->cfg.relax_rate > 0.) return fail(ECG_E_ARG, "samples record infinite relaxations; the case relaxes at a finite rate");
  // Records written so far stay; the candidate counter restarts for this attachment.
  const long long held = samples_count(smp);
  if (held < 0) return fail(ECG_E_HIP, "reading the sample counter failed");
  HIPCHK(hipMemset(smp->seen, 0, sizeof(unsigned long long)));
  smp->base = held;
  smp->stride = stride;
  smp->uploaded = -1;
  c->sink = SampleSink{smp->buf, smp->seen, smp->cap, held, stride};
  if (c->sink_obj != smp) {
    if (c->sink_obj) samples_detach(c->sink_obj);
    samples_attach(smp);
    c->sink_obj = smp;
  }
  return ECG_OK;
}

int ecg_set_warm_start(ecg_ctx* c, const ecg_mlp* m) {
  if (!c) return fail(ECG_E_ARG, "null context");
  if (!m) {
    int rc = settle(c);
    if (rc != ECG_OK) return rc;
    c->mlp = MlpDev{nullptr, nullptr};
    if (c->mlp_obj) mlp_detach(c->mlp_obj);
    c->mlp_obj = nullptr;
    return ECG_OK;
  }
  if (c->cfg.precision != ECG_FP32_LEARNED) return fail(ECG_E_ARG, "the warm start belongs to the ECG_FP32_LEARNED form");
  if (c->sink.buf) return fail(ECG_E_ARG, "samples record cold solves: detach the sample buffer first");
  HIPCHK(hipStreamSynchronize(m->stream));
  c->mlp = MlpDev{m->frag, m->bias};
  if (c->mlp_obj != m) {
    if (c->mlp_obj) mlp_detach(c->mlp_obj);
    mlp_attach(m);
    c->mlp_obj = m;
  }
  return ECG_OK;
}

int ecg_set_profiling(ecg_ctx* c, int on) {
  if (!c) return fail(ECG_E_ARG, "null context");
  int rc = read_clock(c);
  if (rc != ECG_OK) return rc;
  c->profiling = (on != 0);
  for (int k = 0; k < ECG_K_KINDS; k++) { c->kt_ms[k] = 0.; c->kt_n[k] = 0; }
  return ECG_OK;
}

int ecg_kernel_times(ecg_ctx* c, double* ms_total, int64_t* launches, int nkinds) {
  if (!c || nkinds < 0) return fail(ECG_E_ARG, "bad arguments");
  int rc = read_clock(c);
  if (rc != ECG_OK) return rc;
  for (int k = 0; k < nkinds && k < ECG_K_KINDS; k++) {
    if (ms_total) ms_total[k] = c->kt_ms[k];
    if (launches) launches[k] = c->kt_n[k];
  }
  return ECG_OK;
}


// ---------------------------------------------------------------------------
// Allocation-free step (ecg_step_noalloc)
// ---------------------------------------------------------------------------
// Everything the step needs beyond the caller's two state buffers lives in this
// file-scope device array: the parameter copy, the clock, the counter slots, the
// warning counter, the inlet-tank records and, at second order,
// the predicted state W*.  Each GPU the library runs on holds its own copy until the
// process ends.  In host code `scratch` names a host-side stand-in, not device memory:
// the device address of each GPU's copy comes from hipGetSymbolAddress, once per device
// (noalloc_scratch), and only that address is handed to kernels and copies.  Calls that
// overlap on one GPU share the array and race.
constexpr size_t NOALLOC_SCRATCH_BYTES = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];
constexpr int NOALLOC_MAX_DEVICES = 64;
static unsigned char* g_scratch_dev[NOALLOC_MAX_DEVICES];
static std::mutex g_scratch_mtx;

// Device address of the current device's scratch array.
static int noalloc_scratch(unsigned char** out) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) return fail(ECG_E_ARG, "device index beyond the scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mtx);
  if (!g_scratch_dev[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(ECG_E_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch_dev[dev] = static_cast<unsigned char*>(p);
  }
  *out = g_scratch_dev[dev];
  return ECG_OK;
}

// Everything a step on caller buffers finds in the scratch array, in one launch: the
// parameter copy, zeroed counter slots (dtMax slots at 1e10), the zeroed warning counter and
// the given clock.  Bound by latency alone: as a host copy and two kernels it took three
// dependent submissions ahead of every step.
__global__ __launch_bounds__(256) void k_noalloc_open(Params P, Params* pdev, Clock* clk, Counters* cnt,
                                                      unsigned long long* warn_cnt, Clock v) {
  const int l = threadIdx.x;
  constexpr int PW = sizeof(Params) / sizeof(uint64_t);
  static_assert(sizeof(Params) % sizeof(uint64_t) == 0, "the parameters are copied in 8-byte words");
  const uint64_t* src = reinterpret_cast<const uint64_t*>(&P);
  for (int i = l; i < PW; i += 256) reinterpret_cast<uint64_t*>(pdev)[i] = src[i];
  if (l < ATOMIC_SLOTS) {
    Counters z = {};
    z.dtmax_bits = (uint64_t)__double_as_longlong(1.e10);
    cnt[l] = z;
  }
  if (l == 0) {
    v.fatal = 0;
    v.fatal_seen = 0;
    *clk = v;
    *warn_cnt = 0ull;
  }
}

int ecg_step_noalloc(const ecg_config* cfg, const void* state_in, void* state_out, double dt, void* stream,
                     double* dtmax_out) {
  const int checked = check_config(cfg);
  if (checked != ECG_OK) return checked;
  if (!state_in || !state_out || state_in == state_out)
    return fail(ECG_E_ARG, "ecg_step_noalloc needs two distinct device state buffers");
  if (!(dt > 0) || !std::isfinite(dt)) return fail(ECG_E_ARG, "dt must be positive and finite");
  if (cfg->precision == ECG_FP32_LEARNED)
    return fail(ECG_E_ARG, "ecg_step_noalloc has no warm-start network: use ECG_FP32_RELAX64");
  ecg_config g = *cfg;
  if (g.model == ECG_PUEQ) g.relax_p = 1;
  if (g.model == ECG_EULER) g.relax_p = 0;
  Params P;
  Layout Ly;
  build_params(g, P, Ly);
  const step_fn step = get_step_fn(g.model, g.nph, Ly.D, Ly.esize == 4);
  if (!step) return fail(ECG_E_UNSUPPORTED, "no kernel built for this model/phase/dimension combination");
  // Scratch layout, 256-byte aligned pieces.
  size_t used = 0;
  auto take = [&](size_t bytes) {
    const size_t at = used;
    used = (used + bytes + 255) / 256 * 256;
    return at;
  };
  const size_t o_par = take(sizeof(Params)), o_clk = take(sizeof(Clock));
  const size_t o_cnt = take(sizeof(Counters) * ATOMIC_SLOTS), o_wc = take(sizeof(unsigned long long));
  // Three doubles per face of an axis' line that nothing reads: they are part of the size
  // above which a case is refused.
  size_t nface = 0;
  for (int n : {g.nx, g.ny, g.nz}) nface += (size_t)std::max(n - 1, 1);
  take(3 * sizeof(double) * nface);
  const size_t o_tank = take(sizeof(double) * TANK_REC * (size_t)Ly.ntank);
  const size_t o_ws = (g.order == 2) ? take((size_t)Ly.esize * (size_t)Ly.pitch * (size_t)Ly.nvar) : 0;
  if (used > NOALLOC_SCRATCH_BYTES)
    return fail(ECG_E_ARG, "the case needs " + std::to_string(used) + " bytes of scratch; ecg_step_noalloc holds " +
                               std::to_string(NOALLOC_SCRATCH_BYTES) + " (a context from ecg_create has no such limit)");
  unsigned char* S = nullptr;
  int rc = noalloc_scratch(&S);
  if (rc != ECG_OK) return rc;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  P.tank_buf = reinterpret_cast<double*>(S + o_tank);
  P.warn_rec = nullptr;   // warnings are counted, not recorded
  P.warn_cnt = reinterpret_cast<unsigned long long*>(S + o_wc);
  P.warn_cap = 0;
  Clock* clk = reinterpret_cast<Clock*>(S + o_clk);
  Counters* cnt = reinterpret_cast<Counters*>(S + o_cnt);
  hipLaunchKernelGGL(k_noalloc_open, dim3(1), dim3(256), 0, st, P, reinterpret_cast<Params*>(S + o_par), clk, cnt,
                     P.warn_cnt, fresh_clock(dt, 0, INFINITY));
  StepLaunch L;
  std::memset(&L, 0, sizeof(L));
  L.pdev = reinterpret_cast<const Params*>(S + o_par);
  L.mlp = MlpDev{nullptr, nullptr};
  L.sink = SampleSink{nullptr, nullptr, 0, 0, 1};
  auto tank = [&] {
    if (Ly.ntank == 0) return;
    L.tank_only = 1;
    step(P, L, clk, cnt, st);
    L.tank_only = 0;
  };
  if (g.order == 1) {
    L.wn = state_in; L.wsrc = state_in; L.wout = state_out; L.stage = 0;
    tank();
    step(P, L, clk, cnt, st);
  } else {
    void* ws = S + o_ws;
    L.wn = state_in; L.wsrc = state_in; L.wout = ws; L.stage = 1;
    tank();
    step(P, L, clk, cnt, st);
    L.wn = state_in; L.wsrc = ws; L.wout = state_out; L.stage = 2;
    tank();
    step(P, L, clk, cnt, st);
  }
  HIPCHK(hipGetLastError());
  // The caller keeps the time: of the clock's bookkeeping only dtMax is left, the least of
  // the slots (non-negative doubles order as integers), taken here from the one copy.
  Counters hc[ATOMIC_SLOTS];
  HIPCHK(hipMemcpyAsync(hc, cnt, sizeof(hc), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  Counters zero, sum;
  std::memset(&zero, 0, sizeof(zero));
  std::memset(&sum, 0, sizeof(sum));
  uint64_t dtb = UINT64_MAX;
  for (int q = 0; q < ATOMIC_SLOTS; q++) {
    sum.tank_fail += hc[q].tank_fail;
    sum.nonfinite += hc[q].nonfinite;
    sum.newton_warn += hc[q].newton_warn;
    dtb = std::min(dtb, hc[q].dtmax_bits);
  }
  if (dtmax_out) std::memcpy(dtmax_out, &dtb, sizeof(dtb));
  return step_outcome(zero, sum);
}

}  // extern "C"
