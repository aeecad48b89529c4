/*
 * ecogen_amd -- C ABI of the MI355X (gfx950) finite-volume step.
 *
 * Drop-in boundary for ECOGEN's explicit Cartesian step.  The reference calls
 * its physics through virtual C++ interfaces at face/cell granularity:
 *   Model::solveRiemannIntern / solveRiemannWall       src/Models/Model.h:109,127
 *   Flux::{addFlux,subtractFlux,buildCons,buildPrim,
 *          addNonCons,schemeCorrection,correctionEnergy} src/Models/Flux.h:48-100
 *   Relaxation::relaxation                              src/Relaxations/Relaxation.h:58
 *   Eos::compute*                                       src/Eos/Eos.h:104-164
 *   Limiter::limiteSlope                                src/Order2/Limiter.h:43
 * driven by Run::integrationProcedure / solveHyperbolic[O2] / solveRelaxations
 * (src/Run.cpp:502-804).  Per-face virtual calls cannot cross a device
 * boundary, so this ABI works at sweep/step granularity: one call advances the
 * whole mesh by one reference time step (faces, cells, relaxation, energy
 * correction, CFL reduction), on the context's HIP stream.
 *
 * Plain pointers and sizes only.  Host buffers are SoA double arrays of the
 * persistent primitive set, variable-major:
 *   multiphase (PUEQ/UEQ): [alpha_k, rho_k, p_k] for k = 0..N-1, then the
 *                          velocity components of the active axes, then the
 *                          mixture total energy E          (3N + D + 1 arrays)
 *   Euler:                 rho, p, velocity (active axes), E (D + 3 arrays)
 * Cells are indexed i + j*nx + k*nx*ny (MeshCartesian.cpp:141-147).
 *
 * Error policy: functions returning int give 0 on success, a negative ECG_E_*
 * code on failure (message in ecg_last_error()).  ecg_step, ecg_run and
 * ecg_run_to return, when positive, the number of the reference's warnings
 * during their steps (a relaxation Newton that spent its 100 iterations with
 * |p*| > 1e-7, RelaxationP.cpp:62-68; ecg_take_warnings gives them one by one),
 * and ECG_E_STATE when a step left a cell with a non-finite state or an inlet
 * tank's Newton failed (the reference's errors stop its run, Run.cpp:808-842).
 */
#ifndef ECOGEN_AMD_H
#define ECOGEN_AMD_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define ECG_MAX_PHASES 4

enum ecg_model { ECG_EULER = 0, ECG_PUEQ = 1, ECG_UEQ = 2 };
enum ecg_eos_type { ECG_EOS_IG = 0, ECG_EOS_SG = 1 };
/* ECG_LIM_THINC: volume-fraction limiters only (lim[2], lim[3]), two-phase models; its slope
 * limiter is minmod and at interfaces the extrapolated volume fractions are replaced by the THINC
 * profile's face value (LimiterTHINC.cpp, CellInterfaceO2Cartesian.cpp:133-180). */
enum ecg_limiter { ECG_LIM_NONE = 0, ECG_LIM_MINMOD = 1, ECG_LIM_VANLEER = 2, ECG_LIM_VANALBADA = 3,
                   ECG_LIM_SUPERBEE = 4, ECG_LIM_MC = 5, ECG_LIM_THINC = 6 };
/* ECG_BC_INLET_TANK: subsonic inflow from a stagnation tank (BoundCondInletTank.cpp,
 * ModEuler.cpp:413-545, ModUEq.cpp:496-673) with the state of ecg_config.tank[side]. */
enum ecg_bc { ECG_BC_NONREFLECTING = 0, ECG_BC_WALL = 1, ECG_BC_INLET_TANK = 2 };
/* Arithmetic of the hot path:
 *   ECG_FP64          plain double precision, the parity path
 *   ECG_FP32_RELAX64  state, reconstruction and fluxes in float, the face contributions
 *                     accumulated in double; update, relaxation and EOS inversions in double
 *   ECG_FP32_LEARNED  as ECG_FP32_RELAX64 with the Newton warm start predicted by the MLP */
enum ecg_precision { ECG_FP64 = 0, ECG_FP32_RELAX64 = 1, ECG_FP32_LEARNED = 2 };
enum ecg_domain_kind { ECG_DOM_ENTIRE = 0, ECG_DOM_HALFSPACE = 1, ECG_DOM_DISC = 2, ECG_DOM_SPHERE = 3,
                       ECG_DOM_RECTANGLE = 4, ECG_DOM_CUBOID = 5 };

enum {
  ECG_OK = 0,
  ECG_E_ARG = -1,       /* invalid argument or configuration */
  ECG_E_HIP = -2,       /* HIP runtime error */
  ECG_E_STATE = -3,     /* invalid / non-finite state */
  ECG_E_UNSUPPORTED = -4
};

/* Eos::assignParametersEos (EosSG.cpp:48-57, EosIG.cpp:47-55) */
typedef struct {
  int type;               /* ecg_eos_type */
  double gamma, pinf, cv, eref;
} ecg_eos;

/* Tank of an inletTank boundary (BoundCondInletTank.cpp:37-165): stagnation pressure
 * and temperature, and the tank's volume fractions (summing to one; Euler: alpha[0] = 1).
 * The phase densities are each EOS's computeDensity(p0, T0). */
typedef struct {
  double p0, T0;
  double alpha[ECG_MAX_PHASES];
} ecg_tank;

/* What Input::readInputXML assembles for the hot path (Input.cpp:77-1193). */
typedef struct {
  int nx, ny, nz;         /* cells per axis; nx > 1, nz > 1 requires ny > 1 (Input.cpp:459-467) */
  double lx, ly, lz;      /* domain lengths */
  int model;              /* ecg_model */
  int nph;                /* phases (1 for Euler) */
  ecg_eos eos[ECG_MAX_PHASES];
  int order;              /* 1: Godunov, 2: MUSCL + explicit midpoint */
  int lim[4];             /* global, interface, global volume-fraction, interface volume-fraction */
  int alpha_null;         /* flowModel alphaNull attribute */
  int relax_p;            /* <relaxation type="P" speed="infinite"/> (forced for PUEQ) */
  int bc[6];              /* X-, X+, Y-, Y+, Z-, Z+ (ecg_bc) */
  double cfl;
  int precision;          /* ecg_precision */
  double relax_rate;      /* > 0 (VELOCITYEQ with relax_p): <relaxation type="P" speed="finite" rate=...
                             solver="Euler"> (RelaxationPFinite) instead of the infinite relaxation */
  ecg_tank tank[6];       /* stagnation state of each ECG_BC_INLET_TANK side (ignored elsewhere) */
} ecg_config;

/* One initial-condition domain with its state (GeometricalDomain + Phase/Mixture states). */
typedef struct {
  int kind;               /* ecg_domain_kind */
  int axis, axis2, dir;   /* half-space axis/direction, disc axes */
  double origin;          /* half-space origin */
  double center[3];
  double radius;
  double lo[3], len[3];   /* rectangle / cuboid lower corner and lengths */
  double alpha[ECG_MAX_PHASES], rho[ECG_MAX_PHASES], p[ECG_MAX_PHASES];
  double vel[3];
} ecg_domain;

typedef struct {
  double t;               /* physical time after the last step */
  double dt_next;         /* cfl * dtMax of the last step (Run.cpp:439) */
  double dt_max;          /* min over the last step's Riemann calls of lCFL/|s| */
  int64_t iteration;
  int64_t newton_fail;    /* relaxations that fell back to the interface pressure (cumulative) */
  int64_t newton_iters;   /* total Newton iterations (cumulative) */
  int64_t relax_calls;    /* relaxed cells (cumulative) */
  int64_t warm_calls;     /* relaxations started from the learned guess (cumulative) */
  int64_t warm_fallbacks; /* of those, continued by the reference procedure (cumulative) */
  double resid_sum;       /* sum over relaxed cells of |f| when Newton stopped (cumulative) */
  int64_t newton_warn;    /* of newton_fail, those with |p*| > 1e-7: the reference's warnings (cumulative) */
  int64_t nonfinite;      /* cell updates that produced a non-finite state (cumulative) */
} ecg_step_stats;

/* One warning of the reference's Run::verifyErrors log (Run.cpp:808-842,
 * Errors.cpp:142-160): RelaxationP::NewtonRaphson did not converge
 * (RelaxationP.cpp:62-68) and the cell took the interface pressure. */
enum { ECG_WARN_NEWTON = 0 };
typedef struct {
  int64_t iteration;      /* steps completed before the step that warned */
  int64_t cell;           /* i + j*nx + k*nx*ny */
  int32_t stage;          /* 0 first-order step, 1 second-order predictor, 2 corrector */
  int32_t kind;           /* ECG_WARN_NEWTON */
  double value;           /* convergence error |f| after the last iteration */
} ecg_warning;

typedef struct ecg_ctx ecg_ctx;

/* Time control of a case's main.xml (Input.cpp:179-203). */
typedef struct {
  char run_name[128];
  int iterations_mode;    /* 1: stop after `iterations` steps; 0: at physical time total_time */
  int64_t iterations;
  int iter_freq;
  double total_time, time_freq;
} ecg_run_control;

/* Library / device ------------------------------------------------------- */
const char* ecg_last_error(void);
const char* ecg_version(void);
int ecg_device_count(void);

/* Input::readInputXML (src/InputOutput/Input.cpp:54-73) for the hot path: reads
 * case_dir/{main,mesh,model,initialConditions}.xml and the EOS files of eos_dir
 * (NULL: the first libEOS directory in case_dir or its parents) into *cfg (with
 * the given precision form), doms[0..*ndoms) and *rc (may be NULL).  Features the
 * library does not build (AMR, stretching, other models/EOS/limiters/boundaries,
 * transports, additional physics) return ECG_E_UNSUPPORTED with the reason; when
 * max_doms is too small, *ndoms holds the count needed and ECG_E_ARG is returned. */
int ecg_read_case(const char* case_dir, const char* eos_dir, int precision, ecg_config* cfg, ecg_domain* doms,
                  int max_doms, int* ndoms, ecg_run_control* rc);

/* The exponential the kernels use where the reference calls exp (the THINC
 * reconstruction, CellInterfaceO2Cartesian.cpp:139,171): correctly rounded for
 * -708 < x < 709.78, the same code on the host and the device. */
double ecg_exp(double x);
/* The logarithm of the star-state isentropes x^g = exp(g log x) in the FP64 kernels
 * outside the full-featured ones (EosSG.cpp:129-132 calls std::pow): within 2 ulp of
 * the exact logarithm for positive finite arguments; zero, negative, infinite and NaN
 * arguments give what the C library's log gives; the same code on the host and the
 * device. */
double ecg_log(double x);
/* Tile that block `block` of a step launch over `ntiles` tiles of 256 cells of the case works on
 * (the kernels' own order, for tests): a permutation of 0 .. ntiles - 1. */
int ecg_tile_of_block(const ecg_config* cfg, int ntiles, int block);
/* The pow the full-featured FP64 kernels use in the star-state isentropes
 * (EosSG.cpp:129-132 calls std::pow): correctly rounded for a positive finite base and
 * a result between 2^-1010 and 2^1010, the library's pow otherwise; the same code on
 * the host and the device. */
double ecg_pow(double x, double y);
/* The bytes of one state variable a launch of the FP32 step kernels may address
 * (32-bit offsets from the launch's first cell; default and maximum 4 GiB): a stage
 * whose tile rows span more runs as several launches over consecutive rows.  No
 * counterpart in the reference; for tests of the split launches on small grids.
 * Takes effect on the next step; returns the previous value (bytes <= 0: no change). */
int64_t ecg_set_step_span(int64_t bytes);

/* Result files in the reference's formats (src/InputOutput/Output*.cpp) for the
 * case in case_dir, under work_dir/results/<run>/: opening does what
 * Run::initialize does before the first print (folders, savesInput copies,
 * ParaView/VisIt collections, global-quantity files, and unless the case
 * restarts, empty infoCalcul.out and infoMesh files).  Host-side only; needs no GPU. */
typedef struct ecg_output ecg_output;
ecg_output* ecg_output_open(const char* case_dir, const char* eos_dir, const char* work_dir);
/* One print of Run::solver (Run.cpp:441-467) from a host state in the layout above:
 * infoCalcul.out line, infoMesh line, global quantities, then the dataset (GNU
 * columns + gnuplot script, or VTK XML .vtr + collections) numbered 0, 1, ... */
int ecg_output_write(ecg_output* o, const double* const* soa, int nvars, int64_t iteration, double t,
                     double dt_next, double seconds);
/* Restart point of the case's <restartSimulation restartFileNumber="n"> (Run::restartSimulation,
 * Run.cpp:345-381): the infoCalcul.out line of file n (iteration, time, dt; the file is cut
 * after it) and the XML dataset n rebuilt into a state (Cell::fulfillStateRestart +
 * completeFulfillState).  Later writes continue with file n + 1. */
int ecg_output_restart(ecg_output* o, double* const* soa, int nvars, int64_t* iteration, double* t, double* dt);
void ecg_output_close(ecg_output* o);

/* Context lifetime (Run::Run / Run::initialize / Run::finalize). */
ecg_ctx* ecg_create(const ecg_config* cfg);
void ecg_destroy(ecg_ctx* ctx);
int ecg_nvar(const ecg_ctx* ctx);
int64_t ecg_ncell(const ecg_ctx* ctx);

/* Initial condition: Cell::fill over the domains in order, then completeFulfillState
 * (Run.cpp:128-140).  Runs on the device. */
int ecg_fill(ecg_ctx* ctx, const ecg_domain* doms, int ndom);

/* State transfer, host SoA double arrays (layout above). soa[v] points at ncell doubles.
 * Downloaded arrays may share memory: the later variable's values then stand.  The first download
 * allocates up to 8 MB of page-locked memory, freed by ecg_destroy; it works without, more slowly. */
int ecg_upload_state(ecg_ctx* ctx, const double* const* soa, int nvars);
int ecg_download_state(ecg_ctx* ctx, double* const* soa, int nvars);

/* One reference step with an explicit dt: the work of Run::integrationProcedure +
 * advancingProcedure (Run.cpp:502-623).  Synchronous; *dtmax_out receives dtMax.
 * Returns the step's warning count when positive, ECG_E_STATE after an error. */
int ecg_step(ecg_ctx* ctx, double dt, double* dtmax_out, ecg_step_stats* st);

/* Reference time loop (Run::solver, Run.cpp:385-498) with dt0 = 1e-15 and the lagged
 * dt_{n+1} = cfl*dtMax_n kept on the device.  Stops after max_iter steps when
 * max_iter > 0, else at the first step with t >= t_end.  Restarts the clock.
 * A step that leaves an error stops the run after it (ECG_E_STATE); a positive
 * return is the number of warnings during the run. */
int ecg_run(ecg_ctx* ctx, int64_t max_iter, double t_end, ecg_step_stats* st);
/* Continues the device clock (time, dt, iteration) of the last run instead of
 * starting afresh: runs until the first step with iteration >= until_iter
 * (until_iter > 0) or t >= until_t.  The runner's output schedule
 * (Run::solver, src/Run.cpp:385-498) is built from these calls. */
int ecg_run_to(ecg_ctx* ctx, int64_t until_iter, double until_t, ecg_step_stats* st);
/* Sets the clock a restart resumes from (Output::readInfos, src/InputOutput/Output.cpp:525-573):
 * physical time, the dt of the next step and the iteration count. */
int ecg_set_time(ecg_ctx* ctx, double t, double dt, int64_t iteration);

/* ecg_step for callers that cannot allocate (code under HIP graph capture, serving
 * loops, harnesses that forbid it).  No counterpart in the reference.  No context:
 * the caller passes the case and two distinct device buffers holding the state in the
 * library's layout (the variables above, each over pitch = ncell rounded up to 64
 * elements; double for ECG_FP64, float for ECG_FP32_RELAX64) and gets the state after
 * one step of size dt in state_out.  Everything else (parameters, clock, counters,
 * inlet-tank records, the second-order predicted state) lives in a
 * fixed 64 MiB device array of the library, one per GPU, held until the process ends;
 * a case that needs more is refused with ECG_E_ARG.  The call allocates nothing, runs
 * on `stream` (NULL: the null stream) and waits for it; *dtmax_out receives dtMax.
 * Returns like ecg_step (warning count, ECG_E_STATE); warnings are counted, not
 * recorded.  Calls that overlap on one GPU share the array and race.
 * ECG_FP32_LEARNED is refused (no network). */
int ecg_step_noalloc(const ecg_config* cfg, const void* state_in, void* state_out, double dt, void* stream,
                     double* dtmax_out);

/* Enqueue n steps of the device-clocked loop without synchronising (benchmarking).
 * A clock a run left stopped continues without a limit; after an error it stays stopped. */
int ecg_enqueue_steps(ecg_ctx* ctx, int n);
int ecg_synchronize(ecg_ctx* ctx, ecg_step_stats* st);
int ecg_reset_clock(ecg_ctx* ctx);

/* Run::verifyErrors (Run.cpp:808-842): the warnings of the steps run so far that
 * were not taken yet, in the reference's order (steps in turn; within a step the
 * predictor's cells before the corrector's, cells in index order).  Copies at
 * most max into out and returns the count copied; the context records at most
 * 4096 warnings between two calls and *dropped (may be NULL) receives how many
 * were not recorded since the last call. */
int64_t ecg_take_warnings(ecg_ctx* ctx, ecg_warning* out, int64_t max, int64_t* dropped);

/* Stream the context runs on (a hipStream_t), for event timing by the caller. */
void* ecg_stream(ecg_ctx* ctx);

/* Per-kernel timing with HIP events recorded around every launch on the
 * context's stream.  Kinds: 0 first-order step, 1 second-order predictor,
 * 2 second-order corrector, 3 clock update, 4 inlet-tank faces (ahead of each
 * step kernel).  ecg_kernel_times accumulates the elapsed milliseconds and
 * launch counts since profiling was switched on. */
enum { ECG_K_STEP = 0, ECG_K_PREDICT = 1, ECG_K_CORRECT = 2, ECG_K_CLOCK = 3, ECG_K_TANK = 4, ECG_K_KINDS = 5 };
int ecg_set_profiling(ecg_ctx* ctx, int on);
int ecg_kernel_times(ecg_ctx* ctx, double* ms_total, int64_t* launches, int nkinds);

/* Byte-counter calibration: one launch of a plain streaming copy kernel that reads
 * and writes nbytes (at most one state buffer) between the context's two state
 * buffers.  Profilers divide a kernel's FETCH_SIZE / WRITE_SIZE by what they
 * report for this launch to turn counter units into bytes. */
int ecg_calibration_copy(ecg_ctx* ctx, int64_t nbytes);

/* Field-wise comparison of two contexts on the same mesh and model (any
 * precision forms): for f = 0..nvar-1 the persistent variables, f = nvar the
 * mixture density sum_k alpha_k rho_k (Euler: rho); out[4f .. 4f+3] =
 * sum|a-b|, sum|b|, max|a-b|, max|b| over the cells.  nfields = nvar + 1.
 * A diagnostic of this library (error of the FP32 forms against the FP64 path);
 * the reference has no counterpart. */
int ecg_state_diff(ecg_ctx* a, ecg_ctx* b, double* out, int nfields);

/* Learned Newton warm start ---------------------------------------------
 * Extends RelaxationPInfinite::relaxation (src/Relaxations/RelaxationPInfinite.cpp:43-98),
 * whose Newton (src/Relaxations/RelaxationP.cpp:43-70) starts from sum_k alpha_k p_k.
 * The reference has no learned guess: these entry points have no counterpart there.
 *
 * A sample record is ECG_SAMPLE_FLOATS floats: 12 scale-free features of the
 * pre-relaxation phase states (3 phase slots x [alpha_k, (p_k - p_cold)/s,
 * linearised weight w_k, s/(s + rho_k c_k^2)], s = max_k |p_k - p_cold|), the
 * normalised relaxed pressure t = (p* - p_cold)/s, the cold-start Newton
 * evaluations, the remainder u = (t - t_lin)/sigma computed in FP64, and the
 * second-order scale sigma = max(|sum_k w_k (t_lin - x_k1)^2 s/(rho_k c_k^2)|,
 * 1e-9), t_lin = sum_k w_k x_k1. */
#define ECG_MLP_INPUTS 12
#define ECG_MLP_HIDDEN 64
#define ECG_MLP_NPARAM 5057    /* W1[12][64], b1[64], W2[64][64], b2[64], w3[64], b3 */
#define ECG_SAMPLE_FLOATS 16

typedef struct ecg_samples ecg_samples;
typedef struct ecg_mlp ecg_mlp;

/* Device buffer of relaxation samples. */
ecg_samples* ecg_samples_create(int64_t capacity);
/* ECG_E_ARG (and nothing freed) while a context has the buffer attached. */
int ecg_samples_destroy(ecg_samples* s);
int ecg_samples_reset(ecg_samples* s);
int64_t ecg_samples_count(ecg_samples* s);   /* records held */
int64_t ecg_samples_seen(ecg_samples* s);    /* candidate cells met while attached (every stride) */
int ecg_samples_download(ecg_samples* s, float* host, int64_t n);
int ecg_samples_upload(ecg_samples* s, const float* host, int64_t n);

/* While attached, the context's steps append one record for every stride-th
 * cell that relaxes (cold start, any precision form) from distinct phase
 * pressures, after the records the buffer already holds (attaching restarts
 * the candidate count; records beyond the capacity are dropped).  One buffer
 * serves one attached context at a time.  NULL detaches.  Records come from cold
 * solves: a context with a warm start set (ecg_set_warm_start) refuses a buffer. */
int ecg_attach_samples(ecg_ctx* ctx, ecg_samples* s, int stride);

/* 12 -> 64 -> 64 -> 1 GELU network predicting u = (t - t_lin) / sigma (clipped to +-4 in training).
 * Parameters are FP32 on the device; inference packs them as BF16 for MFMA. */
ecg_mlp* ecg_mlp_create(uint64_t seed);
/* ECG_E_ARG (and nothing freed) while a context uses the network as its warm start.
 * ecg_mlp_set_params and ecg_mlp_train wait for the device first in that case. */
int ecg_mlp_destroy(ecg_mlp* m);
int ecg_mlp_get_params(ecg_mlp* m, float* host);          /* ECG_MLP_NPARAM floats */
int ecg_mlp_set_params(ecg_mlp* m, const float* host);    /* resets the optimiser */
/* Mean squared error over the first n records (phase slots as stored) and its gradient. */
int ecg_mlp_gradient(ecg_mlp* m, ecg_samples* s, int64_t n, float* grad, double* loss);
/* Adam on every record of s, phase slots permuted at random per record; epoch_loss[e]
 * receives the mean loss of epoch e. */
int ecg_mlp_train(ecg_mlp* m, ecg_samples* s, int epochs, int batch, float lr, uint64_t seed,
                  double* epoch_loss);
/* BF16-MFMA inference (the device function fused into the relaxation): the network
 * output y for the first n records (the warm start uses t = t_lin + sigma * y). */
int ecg_mlp_predict(ecg_mlp* m, ecg_samples* s, int64_t n, float* out);
/* Use m's guess, p = p_cold + s (t_lin + sigma y), in the relaxations of an
 * ECG_FP32_LEARNED context; Newton still runs to |f| <= 1e-10 and restarts from
 * the cold guess after 30 evaluations.  NULL returns to the cold start.  Refused
 * while a sample buffer is attached. */
int ecg_set_warm_start(ecg_ctx* ctx, const ecg_mlp* m);

#ifdef __cplusplus
}
#endif
#endif
