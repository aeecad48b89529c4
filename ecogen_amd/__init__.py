"""ecogen_amd: MI355X-native explicit finite-volume step of ECOGEN (Cartesian).

Python host binding of ``libecogen_amd.so`` (C ABI in ``include/ecogen_amd.h``).
The library is required: every entry point raises if it is missing, there is
no CPU fallback.

A *case* is a plain dict (see :mod:`ecogen_amd.case`) holding what ECOGEN's
XML inputs describe for the hot path: mesh, flow model, EOS per phase,
order/limiters, boundary conditions, CFL and the initial-condition domains.
"""
import ctypes as C
import os

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
# ECOGEN_AMD_LIB selects another build of the library (a path to its .so).
LIB_PATH = os.environ.get("ECOGEN_AMD_LIB") or os.path.join(_HERE, "libecogen_amd.so")
_LIB = None

MAX_PHASES = 4
MODELS = {"euler": 0, "pueq": 1, "ueq": 2}
EOS_TYPES = {"IG": 0, "SG": 1}
LIMITERS = {"none": 0, "minmod": 1, "vanleer": 2, "vanalbada": 3, "superbee": 4, "mc": 5, "thinc": 6}
BCS = {"nonreflecting": 0, "wall": 1, "symmetry": 1, "inlettank": 2}
DOMAINS = {"entire": 0, "halfspace": 1, "disc": 2, "sphere": 3, "rectangle": 4, "cuboid": 5}
PRECISIONS = {"fp64": 0, "fp32": 1, "fp32_learned": 2}


class EcgEos(C.Structure):
    _fields_ = [("type", C.c_int), ("gamma", C.c_double), ("pinf", C.c_double), ("cv", C.c_double),
                ("eref", C.c_double)]


class EcgTank(C.Structure):
    _fields_ = [("p0", C.c_double), ("T0", C.c_double), ("alpha", C.c_double * MAX_PHASES)]


class EcgConfig(C.Structure):
    _fields_ = [("nx", C.c_int), ("ny", C.c_int), ("nz", C.c_int),
                ("lx", C.c_double), ("ly", C.c_double), ("lz", C.c_double),
                ("model", C.c_int), ("nph", C.c_int), ("eos", EcgEos * MAX_PHASES), ("order", C.c_int),
                ("lim", C.c_int * 4), ("alpha_null", C.c_int), ("relax_p", C.c_int), ("bc", C.c_int * 6),
                ("cfl", C.c_double), ("precision", C.c_int), ("relax_rate", C.c_double), ("tank", EcgTank * 6)]


class EcgDomain(C.Structure):
    _fields_ = [("kind", C.c_int), ("axis", C.c_int), ("axis2", C.c_int), ("dir", C.c_int),
                ("origin", C.c_double), ("center", C.c_double * 3), ("radius", C.c_double),
                ("lo", C.c_double * 3), ("len", C.c_double * 3),
                ("alpha", C.c_double * MAX_PHASES), ("rho", C.c_double * MAX_PHASES),
                ("p", C.c_double * MAX_PHASES), ("vel", C.c_double * 3)]


class EcgRunControl(C.Structure):
    _fields_ = [("run_name", C.c_char * 128), ("iterations_mode", C.c_int), ("iterations", C.c_int64),
                ("iter_freq", C.c_int), ("total_time", C.c_double), ("time_freq", C.c_double)]


class EcgStepStats(C.Structure):
    _fields_ = [("t", C.c_double), ("dt_next", C.c_double), ("dt_max", C.c_double), ("iteration", C.c_int64),
                ("newton_fail", C.c_int64), ("newton_iters", C.c_int64), ("relax_calls", C.c_int64),
                ("warm_calls", C.c_int64), ("warm_fallbacks", C.c_int64), ("resid_sum", C.c_double),
                ("newton_warn", C.c_int64), ("nonfinite", C.c_int64)]

    def as_dict(self):
        return {k: getattr(self, k) for k, _ in self._fields_}


class EcgWarning(C.Structure):
    _fields_ = [("iteration", C.c_int64), ("cell", C.c_int64), ("stage", C.c_int32), ("kind", C.c_int32),
                ("value", C.c_double)]


# Exported symbols and their ctypes signatures (checked by the CPU test-suite).
_DP = C.POINTER(C.c_double)
_FP = C.POINTER(C.c_float)
SIGNATURES = {
    "ecg_last_error": (C.c_char_p, []),
    "ecg_version": (C.c_char_p, []),
    "ecg_device_count": (C.c_int, []),
    "ecg_create": (C.c_void_p, [C.POINTER(EcgConfig)]),
    "ecg_destroy": (None, [C.c_void_p]),
    "ecg_nvar": (C.c_int, [C.c_void_p]),
    "ecg_ncell": (C.c_int64, [C.c_void_p]),
    "ecg_fill": (C.c_int, [C.c_void_p, C.POINTER(EcgDomain), C.c_int]),
    "ecg_upload_state": (C.c_int, [C.c_void_p, C.POINTER(_DP), C.c_int]),
    "ecg_download_state": (C.c_int, [C.c_void_p, C.POINTER(_DP), C.c_int]),
    "ecg_step": (C.c_int, [C.c_void_p, C.c_double, _DP, C.POINTER(EcgStepStats)]),
    "ecg_run": (C.c_int, [C.c_void_p, C.c_int64, C.c_double, C.POINTER(EcgStepStats)]),
    "ecg_run_to": (C.c_int, [C.c_void_p, C.c_int64, C.c_double, C.POINTER(EcgStepStats)]),
    "ecg_exp": (C.c_double, [C.c_double]),
    "ecg_pow": (C.c_double, [C.c_double, C.c_double]),
    "ecg_log": (C.c_double, [C.c_double]),
    "ecg_tile_of_block": (C.c_int, [C.POINTER(EcgConfig), C.c_int, C.c_int]),
    "ecg_set_step_span": (C.c_int64, [C.c_int64]),
    "ecg_set_time": (C.c_int, [C.c_void_p, C.c_double, C.c_double, C.c_int64]),
    "ecg_output_open": (C.c_void_p, [C.c_char_p, C.c_char_p, C.c_char_p]),
    "ecg_output_write": (C.c_int, [C.c_void_p, C.c_void_p, C.c_int, C.c_int64, C.c_double, C.c_double,
                                   C.c_double]),
    "ecg_output_restart": (C.c_int, [C.c_void_p, C.c_void_p, C.c_int, C.POINTER(C.c_int64),
                                     C.POINTER(C.c_double), C.POINTER(C.c_double)]),
    "ecg_output_close": (None, [C.c_void_p]),
    "ecg_enqueue_steps": (C.c_int, [C.c_void_p, C.c_int]),
    "ecg_synchronize": (C.c_int, [C.c_void_p, C.POINTER(EcgStepStats)]),
    "ecg_reset_clock": (C.c_int, [C.c_void_p]),
    "ecg_step_noalloc": (C.c_int, [C.POINTER(EcgConfig), C.c_void_p, C.c_void_p, C.c_double, C.c_void_p, _DP]),
    "ecg_take_warnings": (C.c_int64, [C.c_void_p, C.POINTER(EcgWarning), C.c_int64, C.POINTER(C.c_int64)]),
    "ecg_stream": (C.c_void_p, [C.c_void_p]),
    "ecg_set_profiling": (C.c_int, [C.c_void_p, C.c_int]),
    "ecg_kernel_times": (C.c_int, [C.c_void_p, _DP, C.POINTER(C.c_int64), C.c_int]),
    "ecg_calibration_copy": (C.c_int, [C.c_void_p, C.c_int64]),
    "ecg_state_diff": (C.c_int, [C.c_void_p, C.c_void_p, _DP, C.c_int]),
    "ecg_read_case": (C.c_int, [C.c_char_p, C.c_char_p, C.c_int, C.POINTER(EcgConfig), C.POINTER(EcgDomain), C.c_int,
                                C.POINTER(C.c_int), C.POINTER(EcgRunControl)]),
    "ecg_samples_create": (C.c_void_p, [C.c_int64]),
    "ecg_samples_destroy": (C.c_int, [C.c_void_p]),
    "ecg_samples_reset": (C.c_int, [C.c_void_p]),
    "ecg_samples_count": (C.c_int64, [C.c_void_p]),
    "ecg_samples_seen": (C.c_int64, [C.c_void_p]),
    "ecg_samples_download": (C.c_int, [C.c_void_p, _FP, C.c_int64]),
    "ecg_samples_upload": (C.c_int, [C.c_void_p, _FP, C.c_int64]),
    "ecg_attach_samples": (C.c_int, [C.c_void_p, C.c_void_p, C.c_int]),
    "ecg_mlp_create": (C.c_void_p, [C.c_uint64]),
    "ecg_mlp_destroy": (C.c_int, [C.c_void_p]),
    "ecg_mlp_get_params": (C.c_int, [C.c_void_p, _FP]),
    "ecg_mlp_set_params": (C.c_int, [C.c_void_p, _FP]),
    "ecg_mlp_gradient": (C.c_int, [C.c_void_p, C.c_void_p, C.c_int64, _FP, _DP]),
    "ecg_mlp_train": (C.c_int, [C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_float, C.c_uint64, _DP]),
    "ecg_mlp_predict": (C.c_int, [C.c_void_p, C.c_void_p, C.c_int64, _FP]),
    "ecg_set_warm_start": (C.c_int, [C.c_void_p, C.c_void_p]),
}
MLP_NPARAM = 5057
SAMPLE_FLOATS = 16
KERNEL_KINDS = ("step", "predict", "correct", "clock", "tank")


def library(path=None):
    """Load the HIP library (raises when it has not been built)."""
    global _LIB
    if _LIB is None:
        p = path or LIB_PATH
        if not os.path.exists(p):
            raise RuntimeError(f"{p} is missing: build it with `python -m ecogen_amd.build`")
        L = C.CDLL(p)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(L, name)
            fn.restype = res
            fn.argtypes = args
        _LIB = L
    return _LIB


class EcgError(RuntimeError):
    pass


def _check(rc):
    if rc < 0:
        raise EcgError(library().ecg_last_error().decode())
    return rc


def make_config(case):
    c = EcgConfig()
    c.nx, c.ny, c.nz = case["nx"], case["ny"], case["nz"]
    c.lx, c.ly, c.lz = case["lx"], case["ly"], case["lz"]
    c.model = MODELS[case["model"]]
    c.nph = len(case["eos"])
    for k, e in enumerate(case["eos"]):
        c.eos[k] = EcgEos(EOS_TYPES[e["type"].upper()], float(e["gamma"]), float(e.get("pinf", 0.0)),
                          float(e.get("cv", 0.0)), float(e.get("eref", 0.0)))
    c.order = case.get("order", 1)
    lims = case.get("limiters", ("none",) * 4)
    for i in range(4):
        c.lim[i] = LIMITERS[lims[i].lower()]
    c.alpha_null = int(bool(case.get("alpha_null", False)))
    c.relax_p = int(bool(case.get("relax_p", case["model"] == "pueq")))
    for i, b in enumerate(case.get("bc", ("nonreflecting",) * 6)):
        c.bc[i] = BCS[b.lower()]
    c.cfl = case.get("cfl", 0.8)
    c.precision = PRECISIONS[case.get("precision", "fp64")]
    c.relax_rate = float(case.get("relax_rate", 0.0))
    # "tanks": {side: dict(p0=, T0=, alpha=[...])} for the "inletTank" sides (0..5 = X-, X+, Y-, Y+, Z-, Z+)
    for side, t in case.get("tanks", {}).items():
        o = c.tank[int(side)]
        o.p0, o.T0 = float(t["p0"]), float(t["T0"])
        for k, a in enumerate(t.get("alpha", [1.0])):
            o.alpha[k] = float(a)
    return c


def make_domains(case):
    doms = case["domains"]
    arr = (EcgDomain * len(doms))()
    for i, d in enumerate(doms):
        o = arr[i]
        o.kind = DOMAINS[d["kind"]]
        o.axis = d.get("axis", 0)
        o.axis2 = d.get("axis2", 1)
        o.dir = d.get("dir", 1)
        o.origin = d.get("origin", 0.0)
        o.radius = d.get("radius", 0.0)
        for a in range(3):
            o.center[a] = d.get("center", (0.0, 0.0, 0.0))[a]
            o.lo[a] = d.get("lo", (0.0, 0.0, 0.0))[a]
            o.len[a] = d.get("len", (0.0, 0.0, 0.0))[a]
            o.vel[a] = d.get("vel", (0.0, 0.0, 0.0))[a]
        n = len(d["rho"])
        for k in range(n):
            o.alpha[k] = d.get("alpha", [1.0] * n)[k]
            o.rho[k] = d["rho"][k]
            o.p[k] = d["p"][k]
    return arr


def read_case(case_dir, eos_dir=None, precision="fp64"):
    """A case directory in the reference's XML input format (main.xml, mesh.xml,
    model.xml, initialConditions.xml + libEOS files), read by the library's
    ecg_read_case, as a case dict; run control under "control"."""
    L = library()
    cfg = EcgConfig()
    rc = EcgRunControl()
    nd = C.c_int(0)
    args = (str(case_dir).encode(), eos_dir.encode() if eos_dir else None, PRECISIONS[precision])
    r = L.ecg_read_case(*args, C.byref(cfg), None, 0, C.byref(nd), C.byref(rc))
    if r < 0 and nd.value == 0:
        _check(r)
    doms = (EcgDomain * max(nd.value, 1))()
    _check(L.ecg_read_case(*args, C.byref(cfg), doms, nd.value, C.byref(nd), C.byref(rc)))
    inv = lambda m, v: next(k for k, x in m.items() if x == v)
    eos = []
    for k in range(cfg.nph):
        e = cfg.eos[k]
        eos.append(dict(type=inv(EOS_TYPES, e.type), gamma=e.gamma, pinf=e.pinf, cv=e.cv, eref=e.eref))
    kinds = {v: k for k, v in DOMAINS.items()}
    domains = []
    for i in range(nd.value):
        d = doms[i]
        domains.append(dict(kind=kinds[d.kind], axis=d.axis, axis2=d.axis2, dir=d.dir, origin=d.origin,
                            radius=d.radius, center=tuple(d.center), lo=tuple(d.lo), len=tuple(d.len),
                            vel=tuple(d.vel), alpha=list(d.alpha[:cfg.nph]), rho=list(d.rho[:cfg.nph]),
                            p=list(d.p[:cfg.nph])))
    bcs = ("nonreflecting", "wall", "inletTank")
    tanks = {i: dict(p0=cfg.tank[i].p0, T0=cfg.tank[i].T0, alpha=list(cfg.tank[i].alpha[:cfg.nph]))
             for i in range(6) if cfg.bc[i] == BCS["inlettank"]}
    return dict(name=rc.run_name.decode(), nx=cfg.nx, ny=cfg.ny, nz=cfg.nz, lx=cfg.lx, ly=cfg.ly, lz=cfg.lz,
                model=inv(MODELS, cfg.model), eos=eos, order=cfg.order,
                limiters=tuple(inv(LIMITERS, cfg.lim[i]) for i in range(4)), alpha_null=bool(cfg.alpha_null),
                relax_p=bool(cfg.relax_p), relax_rate=cfg.relax_rate, bc=tuple(bcs[cfg.bc[i]] for i in range(6)),
                tanks=tanks, cfl=cfg.cfl,
                precision=precision, domains=domains,
                control=dict(iterations_mode=bool(rc.iterations_mode), iterations=rc.iterations,
                             iter_freq=rc.iter_freq, total_time=rc.total_time, time_freq=rc.time_freq))


class Solver:
    """One case on the GPU: the Run object of the reference, reduced to its hot path."""

    def __init__(self, case, fill=True):
        self.L = library()
        self.case = case
        self.cfg = make_config(case)
        self.h = self.L.ecg_create(C.byref(self.cfg))
        if not self.h:
            raise EcgError(self.L.ecg_last_error().decode())
        self.nvar = self.L.ecg_nvar(self.h)
        self.ncell = self.L.ecg_ncell(self.h)
        self.stats = EcgStepStats()
        self.warnings = 0          # warning count returned by the last step / run call
        self._mlp = None           # the attached warm-start network and sample buffer: kept
        self._samples = None       # alive while the device reads or writes them
        if fill and "domains" in case:
            doms = make_domains(case)
            _check(self.L.ecg_fill(self.h, doms, len(doms)))

    def close(self):
        if getattr(self, "h", None):
            self.L.ecg_destroy(self.h)
            self.h = None
            for o in (self._mlp, self._samples):
                if o is not None:
                    o._users.discard(id(self))
            self._mlp = self._samples = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def _ptrs(self, arr):
        return (_DP * self.nvar)(*[arr[v].ctypes.data_as(_DP) for v in range(self.nvar)])

    def get_state(self):
        out = np.empty((self.nvar, self.ncell), dtype=np.float64)
        _check(self.L.ecg_download_state(self.h, self._ptrs(out), self.nvar))
        return out

    def set_state(self, st):
        st = np.ascontiguousarray(st, dtype=np.float64)
        if st.shape != (self.nvar, self.ncell):
            raise ValueError(f"state must have shape {(self.nvar, self.ncell)}")
        _check(self.L.ecg_upload_state(self.h, self._ptrs(st), self.nvar))

    def step(self, dt):
        """One step of size dt: (dtMax, number of the reference's warnings during it)."""
        dtm = np.zeros(1)
        rc = _check(self.L.ecg_step(self.h, float(dt), dtm.ctypes.data_as(_DP), C.byref(self.stats)))
        self.warnings = rc
        return float(dtm[0]), rc

    def run(self, max_iter=0, t_end=0.0):
        self.warnings = _check(self.L.ecg_run(self.h, int(max_iter), float(t_end), C.byref(self.stats)))
        return self.stats.as_dict()

    def run_to(self, until_iter=0, until_t=0.0):
        """Continue the device clock until iteration until_iter (> 0) or time until_t."""
        self.warnings = _check(self.L.ecg_run_to(self.h, int(until_iter), float(until_t), C.byref(self.stats)))
        return self.stats.as_dict()

    def take_warnings(self):
        """Warnings of the steps so far not taken yet, in the reference's order, as
        (iteration, cell, stage, |f|) tuples, and how many the context did not record."""
        out, buf = [], (EcgWarning * 1024)()
        dropped = C.c_int64(0)
        while True:
            n = _check(self.L.ecg_take_warnings(self.h, buf, 1024, C.byref(dropped)))
            out += [(buf[i].iteration, buf[i].cell, buf[i].stage, buf[i].value) for i in range(n)]
            if n < 1024:
                return out, dropped.value

    def set_time(self, t, dt, iteration):
        """Clock of a restart: time, dt of the next step, iteration count."""
        _check(self.L.ecg_set_time(self.h, float(t), float(dt), int(iteration)))

    def reset_clock(self):
        _check(self.L.ecg_reset_clock(self.h))

    def enqueue(self, n):
        _check(self.L.ecg_enqueue_steps(self.h, int(n)))

    def refill(self):
        """Re-apply the case's initial condition (ecg_fill)."""
        doms = make_domains(self.case)
        _check(self.L.ecg_fill(self.h, doms, len(doms)))

    def synchronize(self):
        _check(self.L.ecg_synchronize(self.h, C.byref(self.stats)))
        return self.stats.as_dict()

    def calibration_copy(self, nbytes):
        _check(self.L.ecg_calibration_copy(self.h, int(nbytes)))

    def set_profiling(self, on=True):
        _check(self.L.ecg_set_profiling(self.h, int(bool(on))))

    def kernel_times(self):
        """{kind: (total ms, launches)} since profiling was switched on."""
        nk = len(KERNEL_KINDS)
        ms = np.zeros(nk)
        n = (C.c_int64 * nk)()
        _check(self.L.ecg_kernel_times(self.h, ms.ctypes.data_as(_DP), n, nk))
        return {k: (float(ms[i]), int(n[i])) for i, k in enumerate(KERNEL_KINDS)}

    @property
    def stream(self):
        return self.L.ecg_stream(self.h)

    def diff(self, ref):
        """{field: (rel L1, rel Linf)} of this state against `ref` (same mesh, any form); the
        relative L-infinity error is max|a-b| / max|b|; field 'mixture_rho' last."""
        from .case import variable_names
        nf = self.nvar + 1
        out = np.zeros(4 * nf)
        _check(self.L.ecg_state_diff(self.h, ref.h, out.ctypes.data_as(_DP), nf))
        names = variable_names(self.case) + ["mixture_rho"]
        res = {}
        for f, nm in enumerate(names):
            sd, sb = out[4 * f], out[4 * f + 1]
            md, mb = out[4 * f + 2:4 * f + 4].copy().view(np.float64)
            res[nm] = (sd / sb if sb > 0 else float(sd > 0) * np.inf, md / mb if mb > 0 else float(md > 0) * np.inf)
        return res

    def attach_samples(self, samples, stride=1):
        """Append relaxation samples of the following steps to `samples` (None detaches)."""
        _check(self.L.ecg_attach_samples(self.h, samples.h if samples is not None else None, int(stride)))
        self._swap_attached("_samples", samples)

    def set_warm_start(self, mlp):
        """Relax from the network's guess (fp32_learned cases; None: cold start)."""
        _check(self.L.ecg_set_warm_start(self.h, mlp.h if mlp is not None else None))
        self._swap_attached("_mlp", mlp)

    def _swap_attached(self, slot, obj):
        old = getattr(self, slot)
        if old is not None and old is not obj:
            old._users.discard(id(self))
        if obj is not None:
            obj._users.add(id(self))
        setattr(self, slot, obj)


def _fp(a):
    return a.ctypes.data_as(_FP)


class Output:
    """The reference's result files for a case (ecg_output_*): host-side, no GPU needed."""

    def __init__(self, case_dir, work_dir, eos_dir=None):
        self.L = library()
        self.h = self.L.ecg_output_open(str(case_dir).encode(), eos_dir.encode() if eos_dir else None,
                                        str(work_dir).encode())
        if not self.h:
            raise EcgError(self.L.ecg_last_error().decode())

    def write(self, state, iteration, t, dt_next, seconds=0.0):
        st = np.ascontiguousarray(state, dtype=np.float64)
        ptrs = (_DP * st.shape[0])(*[st[v].ctypes.data_as(_DP) for v in range(st.shape[0])])
        _check(self.L.ecg_output_write(self.h, ptrs, st.shape[0], int(iteration), float(t), float(dt_next),
                                       float(seconds)))

    def restart(self, nvar, ncell):
        """(state, iteration, t, dt) of the case's restart file."""
        out = np.empty((nvar, ncell), dtype=np.float64)
        ptrs = (_DP * nvar)(*[out[v].ctypes.data_as(_DP) for v in range(nvar)])
        it, t, dt = C.c_int64(), C.c_double(), C.c_double()
        _check(self.L.ecg_output_restart(self.h, ptrs, nvar, C.byref(it), C.byref(t), C.byref(dt)))
        return out, it.value, t.value, dt.value

    def close(self):
        if getattr(self, "h", None):
            self.L.ecg_output_close(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class Samples:
    """Device buffer of relaxation samples (records of SAMPLE_FLOATS floats)."""

    def __init__(self, capacity):
        self.L = library()
        self._users = set()
        self.h = self.L.ecg_samples_create(int(capacity))
        if not self.h:
            raise EcgError(self.L.ecg_last_error().decode())
        self.capacity = int(capacity)

    def close(self):
        """Free the device buffer; raises while a Solver has it attached."""
        if getattr(self, "h", None):
            if self._users:
                raise EcgError("the sample buffer is attached to a solver (detach it first)")
            _check(self.L.ecg_samples_destroy(self.h))
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def __len__(self):
        return int(_check(self.L.ecg_samples_count(self.h)))

    def reset(self):
        _check(self.L.ecg_samples_reset(self.h))

    @property
    def seen(self):
        """Candidate cells met while attached."""
        return int(_check(self.L.ecg_samples_seen(self.h)))

    def download(self, n=None):
        n = len(self) if n is None else int(n)
        out = np.empty((n, SAMPLE_FLOATS), dtype=np.float32)
        _check(self.L.ecg_samples_download(self.h, _fp(out), n))
        return out

    def upload(self, rec):
        rec = np.ascontiguousarray(rec, dtype=np.float32)
        if rec.ndim != 2 or rec.shape[1] != SAMPLE_FLOATS:
            raise ValueError(f"records must have shape (n, {SAMPLE_FLOATS})")
        _check(self.L.ecg_samples_upload(self.h, _fp(rec), rec.shape[0]))


class Mlp:
    """The warm-start network on the device (FP32 parameters, BF16 MFMA inference)."""

    def __init__(self, seed=1):
        self.L = library()
        self._users = set()
        self.h = self.L.ecg_mlp_create(int(seed))
        if not self.h:
            raise EcgError(self.L.ecg_last_error().decode())

    def close(self):
        """Free the network; raises while a Solver uses it as its warm start."""
        if getattr(self, "h", None):
            if self._users:
                raise EcgError("the network is the warm start of a solver (detach it first)")
            _check(self.L.ecg_mlp_destroy(self.h))
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def get_params(self):
        out = np.empty(MLP_NPARAM, dtype=np.float32)
        _check(self.L.ecg_mlp_get_params(self.h, _fp(out)))
        return out

    def set_params(self, prm):
        prm = np.ascontiguousarray(prm, dtype=np.float32)
        if prm.shape != (MLP_NPARAM,):
            raise ValueError(f"parameters must have shape ({MLP_NPARAM},)")
        _check(self.L.ecg_mlp_set_params(self.h, _fp(prm)))

    def gradient(self, samples, n):
        g = np.empty(MLP_NPARAM, dtype=np.float32)
        loss = np.zeros(1)
        _check(self.L.ecg_mlp_gradient(self.h, samples.h, int(n), _fp(g), loss.ctypes.data_as(_DP)))
        return g, float(loss[0])

    def train(self, samples, epochs=4, batch=4096, lr=1e-3, seed=1):
        losses = np.zeros(int(epochs))
        _check(self.L.ecg_mlp_train(self.h, samples.h, int(epochs), int(batch), float(lr), int(seed),
                                    losses.ctypes.data_as(_DP)))
        return losses

    def predict(self, samples, n=None):
        n = len(samples) if n is None else int(n)
        out = np.empty(n, dtype=np.float32)
        _check(self.L.ecg_mlp_predict(self.h, samples.h, n, _fp(out)))
        return out
