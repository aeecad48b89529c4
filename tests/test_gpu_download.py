"""ecg_download_state into every kind of array a caller may hold (needs a GPU).  The state itself is
what ecg_upload_state stored."""
import ctypes as C

import numpy as np
import pytest

from ecogen_amd.case import IG_AIR, SG_WATER

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
