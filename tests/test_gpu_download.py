"""ecg_download_state into every kind of array a caller may hold, and where page-locked memory is
refused (needs a GPU).  The state itself is what ecg_upload_state stored."""
import ctypes as C
import os
import subprocess
import sys
import textwrap

import numpy as np
import pytest

from ecogen_amd.case import IG_AIR, SG_WATER

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DP = C.POINTER(C.c_double)


def _solver(nx, ny, precision):
    """A two-phase 2D solver (eight variables) holding known values, exact in float."""
    from ecogen_amd import Solver
    case = dict(nx=nx, ny=ny, nz=1, lx=1., ly=1., lz=1., model="ueq", eos=[dict(SG_WATER), dict(IG_AIR)], order=1,
                relax_p=True, precision=precision)
    s = Solver(case, fill=False)
    st = (np.arange(s.nvar)[:, None] * 1000 + np.arange(s.ncell)[None, :] % 997 + 0.5).astype(np.float64)
    s.set_state(st)
    return s, st


def _download(s, arrays):
    from ecogen_amd import library
    return library().ecg_download_state(s.h, (DP * s.nvar)(*[C.cast(a.ctypes.data, DP) for a in arrays]), s.nvar)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("mesh", [(8, 4), (512, 256), (701, 683)])
def test_arrays_that_share_memory_hold_the_last_variable(mesh, precision):
    """One dummy array for every variable, and for all but the first.  (512 x 256 cells make one
    variable a whole number of staging pieces: every piece goes to the same addresses.)"""
    s, st = _solver(*mesh, precision)
    print(f"[download] shared arrays {mesh} {precision}", flush=True)
    for _ in range(3):
        one, first = np.zeros(s.ncell), np.zeros(s.ncell)
        assert _download(s, [one] * s.nvar) == 0
        np.testing.assert_array_equal(one, st[-1])
        assert _download(s, [first] + [one] * (s.nvar - 1)) == 0
        np.testing.assert_array_equal(first, st[0])
        np.testing.assert_array_equal(one, st[-1])


# A library that stands before the HIP runtime in the child's symbol order: it counts the copies
# and, when told to, refuses page-locked allocations of 4 KB or more, the runtime's own answer
# when there is no such memory left.
SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static void* sym(const char* n) { return dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY), n); }
int refuse, refused;
size_t copied_to_caller, copied_elsewhere;
char *caller_lo, *caller_hi;
int hipHostMalloc(void** p, size_t n, unsigned f) {
  if (refuse && n >= 4096) { refused++; if (refused > refuse - 1) return 2; }
  return ((int (*)(void**, size_t, unsigned))sym("hipHostMalloc"))(p, n, f);
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) {
  if (k == 2) { if ((char*)d >= caller_lo && (char*)d < caller_hi) copied_to_caller += n; else copied_elsewhere += n; }
  return ((int (*)(void*, const void*, size_t, int, void*))sym("hipMemcpyAsync"))(d, s, n, k, st);
}
"""
CHILD = textwrap.dedent("""
    import ctypes as C, sys
    import numpy as np
    sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
    shim = C.CDLL(sys.argv[2], mode=C.RTLD_GLOBAL)
    var = lambda n, t=C.c_int: t.in_dll(shim, n)
    from test_gpu_download import _download, _solver
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    for precision in ("fp64", "fp32"):
        for refuse in (1, 4):   # from the first buffer on, from the fourth on
            s, st = _solver(701, 683, precision)
            var("refused").value, var("refuse").value = 0, refuse
            print("[download] refused", precision, refuse, flush=True)
            assert np.array_equal(s.get_state(), st) and var("refused").value >= 1
            var("refuse").value = 0
            s.close()
        s, st = _solver(701, 683, precision)
        p = C.c_void_p()
        assert hip.hipHostMalloc(C.byref(p), st.nbytes, 0) == 0
        locked = np.frombuffer((C.c_char * st.nbytes).from_address(p.value)).reshape(st.shape)
        locked[:] = 0
        var("caller_lo", C.c_void_p).value, var("caller_hi", C.c_void_p).value = p.value, p.value + st.nbytes
        to, other = var("copied_to_caller", C.c_size_t), var("copied_elsewhere", C.c_size_t)
        to.value = other.value = 0
        print("[download] page-locked", precision, flush=True)
        assert _download(s, list(locked)) == 0 and np.array_equal(locked, st)
        if precision == "fp64":   # no detour through the staging buffers
            assert to.value == s.nvar * s.ncell * 8, (to.value, other.value)
        mixed = [locked[v] if v % 2 else np.zeros(s.ncell) for v in range(s.nvar)]
        locked[:] = 0
        assert _download(s, mixed) == 0 and all(np.array_equal(a, b) for a, b in zip(mixed, st))
        s.close()
    print("ok")
""")


@pytest.mark.gpu
def test_refused_staging_and_page_locked_arrays(tmp_path):
    src, lib = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(src), "-o", str(lib), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-u", "-c", CHILD, ROOT, str(lib)], capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and r.stdout.rstrip().endswith("ok"), r.stdout + r.stderr
