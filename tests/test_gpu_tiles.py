"""Meshes on both sides of the line between the step kernels' small tiles (64 cells, the
axes side by side) and their ordinary ones, with ragged edges, against the oracle (needs a
GPU).  FP64 within the parity bar of 1e-12 relative L1 per variable; FP32 within 1e-5 of the
mixture density, the bar of the FP32 form."""
import numpy as np
import pytest

from small_cases import all_cases

CASES = all_cases()
# Ordinary tiles (16 x 16; FP64 8 x 8 x 4; FP32 16 x 4 x 4) are split into small ones up to
# 256 of them at second order in 2D and in FP32, up to 128 otherwise: meshes on the line and past it.
MESH = {(2, 256): ((256, 255, 1), (257, 243, 1)), (2, 128): ((125, 256, 1), (129, 243, 1)),
        (3, "fp32", 256): ((62, 31, 31), (65, 31, 30)), (3, "fp32", 128): ((63, 31, 14), (65, 30, 14)),
        (3, "fp64", 128): ((31, 32, 29), (33, 31, 27))}
TILE = {2: (16, 16, 1), (3, "fp64"): (8, 8, 4), (3, "fp32"): (16, 4, 4)}
NAMES = ["euler_2d_o1", "euler_2d_o2_wall", "pueq_2d_o1", "pueq_2d_o2", "ueq_2d_o2", "pueq_2d_o2_tank",
         "euler_3d_o2", "euler_3d_o2_wall", "ueq3_3d_o1", "ueq2_3d_o2", "pueq3_3d_o2"]


def rel_l1(a, b):
    return float(np.sum(np.abs(a - b)) / max(np.sum(np.abs(b)), 1e-300))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("side", ["small", "large"])
@pytest.mark.parametrize("name", NAMES)
def test_both_tile_kinds_match_the_oracle(name, side, precision):
    from ecogen_amd import Solver
    from ecogen_amd.case import variable_names
    from oracle.pyoracle import Oracle, lib

    case = dict(CASES[name])
    three = case["nz"] > 1
    line = 256 if case["order"] == 2 and (not three or precision == "fp32") else 128
    n = MESH[(3, precision, line) if three else (2, line)][side == "large"]
    case["nx"], case["ny"], case["nz"] = n
    tile = TILE[(3, precision) if three else 2]
    assert (np.prod([-(-a // b) for a, b in zip(n, tile)]) <= line) == (side == "small")
    names = variable_names(case)
    print(f"[tiles] {name} {n} {precision}", flush=True)
    lib().orc_set_exact_exp(0)
    lib().orc_set_pow_mode(1 if name.endswith("wall") else 0)
    o = Oracle(case)
    g = Solver(dict(case, precision=precision))
    dt = 1.e-15
    for _ in range(3):
        dtm_g, _ = g.step(dt)
        dtm_o = o.step(dt)
        assert abs(dtm_g - dtm_o) <= (1e-12 if precision == "fp64" else 1e-5) * dtm_o
        dt = case["cfl"] * dtm_o
    lib().orc_set_pow_mode(0)
    sg, so = g.get_state(), o.get_state()
    if precision == "fp64":
        for v, nm in enumerate(names):
            assert rel_l1(sg[v], so[v]) <= 1e-12, nm
        return
    mix = [sum(s[names.index(f"alpha{k}")] * s[names.index(f"rho{k}")] for k in range(len(case["eos"])))
           if case["model"] != "euler" else s[names.index("rho")] for s in (sg, so)]
    assert np.all(np.isfinite(sg))
    assert rel_l1(*mix) <= 1e-5


# Split launches of the ordinary tiles (a launch of n tile rows of T lines reads n T + 4 lines), and of
# small ones in 2D (T = 8): one row, two, uneven rests.
@pytest.mark.gpu
@pytest.mark.parametrize("name,mesh,lines", [("ueq2_3d_o2", (65, 31, 30), 8), ("ueq2_3d_o2", (65, 31, 30), 13),
                                             ("ueq2_3d_o2", (65, 31, 30), 24), ("pueq_2d_o2", (257, 243, 1), 20),
                                             ("pueq_2d_o2", (257, 243, 1), 53), ("pueq_2d_o2", (100, 90, 1), 12),
                                             ("pueq_2d_o2", (100, 90, 1), 29)])
def test_split_launches_of_both_tile_kinds(name, mesh, lines):
    from ecogen_amd import Solver, library
    case = dict(CASES[name], precision="fp32")
    case["nx"], case["ny"], case["nz"] = mesh
    line_cells = mesh[0] * mesh[1] if mesh[2] > 1 else mesh[0]
    out = []
    for span in (1 << 32, lines * line_cells * 4):
        prev = library().ecg_set_step_span(span)
        try:
            g = Solver(case)
            dt = 1.e-15
            for _ in range(3):
                dt = case["cfl"] * g.step(dt)[0]
            out.append((dt, g.get_state()))
        finally:
            library().ecg_set_step_span(prev)
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[1][1], out[0][1])
