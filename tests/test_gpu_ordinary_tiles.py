"""The ordinary tiles (256 cells) of step kernels that small meshes run with small ones, against
the oracle (needs a GPU): limiters chosen per variable, alphaNull, first-order walls and three
phases in 2D, on ragged meshes just past the line between the two kinds of tiles; the three-phase 2D
kernels on both sides of it.  FP64 within the parity bar of 1e-12 relative L1 per variable; FP32
within 1e-5 of the mixture density, the bar of the FP32 form."""
import numpy as np
import pytest

from small_cases import all_cases, euler_2d, mixed_limiters, pueq3_3d, pueq_2d, ueq2_3d, ueq_2d, wall_variant

# Past 256 ordinary tiles at second order in 2D and in FP32, past 128 otherwise.
LARGE = {(2, 1): (129, 243, 1), (2, 2): (257, 243, 1), (3, "fp32", 1): (65, 30, 14), (3, "fp32", 2): (65, 31, 30),
         (3, "fp64", 1): (33, 31, 27), (3, "fp64", 2): (33, 31, 27)}
SMALL = {1: (125, 130, 1), 2: (125, 123, 1)}


def _three_phase_2d(model, order, lims=("minmod",) * 4):
    """A 2D plane of the three-phase case: discs of epoxy and air in water behind a shock."""
    c = pueq3_3d(order)
    c["model"], c["nz"], c["lz"] = model, 1, 0.1
    doms = []
    for d in c["domains"]:
        d = dict(d)
        if d["kind"] == "sphere":
            d.update(kind="disc", axis=0, axis2=1)
        doms.append(d)
    c["domains"], c["relax_p"] = doms, True
    if order == 2:
        c["limiters"] = lims
    c["name"] = f"{model}3_2d_o{order}" + ("" if lims[0] == lims[1] else "_mixlim")
    return c


def _all_vanleer(case):
    return dict(case, limiters=("vanleer",) * 4, name=case["name"] + "_vanleer")


MIX = ("vanalbada", "minmod", "mc", "superbee")
THREE = [_three_phase_2d(m, o) for m in ("pueq", "ueq") for o in (1, 2)] + [_three_phase_2d("ueq", 2, MIX)]
CASES = {c["name"]: c for c in [
    mixed_limiters(pueq_2d(2)), mixed_limiters(ueq2_3d(2), MIX), mixed_limiters(pueq3_3d(2), MIX), euler_2d(2, lim="superbee"),
    _all_vanleer(euler_2d(2)), _all_vanleer(ueq_2d(2)), pueq_2d(1, alpha_null=True), pueq_2d(2, alpha_null=True),
    ueq_2d(2, alpha_null=True), wall_variant(pueq_2d(1)), wall_variant(all_cases()["ueq3_3d_o1"]),
    wall_variant(euler_2d(1))] + THREE}
RUNS = [(n, "large", p) for n in CASES for p in ("fp64", "fp32")] + \
       [(c["name"], "small", p) for c in THREE for p in ("fp64", "fp32")]


def rel_l1(a, b):
    return float(np.sum(np.abs(a - b)) / max(np.sum(np.abs(b)), 1e-300))


@pytest.mark.gpu
@pytest.mark.parametrize("name,side,precision", RUNS)
def test_matches_the_oracle(name, side, precision):
    from ecogen_amd import Solver
    from ecogen_amd.case import variable_names
    from oracle.pyoracle import Oracle, lib

    case = dict(CASES[name])
    order = case["order"]
    case["nx"], case["ny"], case["nz"] = (SMALL[order] if side == "small" else
                                          LARGE[(2, order) if case["nz"] == 1 else (3, precision, order)])
    names = variable_names(case)
    print(f"[ordinary tiles] {name} {case['nx']}x{case['ny']}x{case['nz']} {precision}", flush=True)
    lib().orc_set_exact_exp(0)
    lib().orc_set_pow_mode(0)
    o, g = Oracle(case), Solver(dict(case, precision=precision))
    dt = 1.e-15
    for _ in range(3):
        dtm_g, _ = g.step(dt)
        dtm_o = o.step(dt)
        assert abs(dtm_g - dtm_o) <= (1e-12 if precision == "fp64" else 1e-5) * dtm_o
        dt = case["cfl"] * dtm_o
    sg, so = g.get_state(), o.get_state()
    if precision == "fp64":
        for v, nm in enumerate(names):
            assert rel_l1(sg[v], so[v]) <= 1e-12, nm
        return
    mix = [sum(s[names.index(f"alpha{k}")] * s[names.index(f"rho{k}")] for k in range(len(case["eos"])))
           if case["model"] != "euler" else s[names.index("rho")] for s in (sg, so)]
    assert np.all(np.isfinite(sg))
    assert rel_l1(*mix) <= 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("name,mesh", [("pueq_2d_o1", (129, 243, 1)), ("pueq_2d_o2", (257, 243, 1)),
                                       ("pueq_2d_o2", (125, 123, 1)), ("pueq3_2d_o1", (129, 243, 1)),
                                       ("pueq3_2d_o1", (125, 130, 1)), ("ueq3_3d_o1", (33, 31, 27)),
                                       ("ueq2_3d_o2", (65, 29, 29)), ("ueq2_3d_o2", (31, 31, 29)),
                                       ("ueq2_3d_o2", (36, 36, 36))])
def test_learned_kernels_track_the_cold_ones(name, mesh):
    """Learned kernels of both tile kinds, states included (3D second order: ordinary tiles past 128, where
    the cold kernels still take small ones up to 256): with the network output at zero (the
    linearised guess) the relaxed state is that of the cold FP32 form to the Newton tolerance
    (1e-10 of the saturation per relaxation; 6e-8 the rounding of the stored floats), so 1e-5 of the
    mixture density, the FP32 form's bar, over ten steps."""
    from ecogen_amd import Mlp, Solver
    from oracle import mlp_oracle as mo
    case = dict({**all_cases(), **CASES}[name])
    case["nx"], case["ny"], case["nz"] = mesh
    print(f"[ordinary tiles] learned {name} {mesh}", flush=True)
    states, stats = [], []
    for precision in ("fp32", "fp32_learned"):
        g = Solver(dict(case, precision=precision))
        if precision == "fp32_learned":
            net = Mlp(seed=1)
            net.set_params(np.zeros(mo.N_PARAM, dtype=np.float32))
            g.set_warm_start(net)
        stats.append(g.run(max_iter=10))
        states.append(g.get_state())
        g.close()
    n = len(case["eos"])
    assert stats[1]["newton_fail"] == 0 and np.all(np.isfinite(states[1]))
    if name.startswith("pueq_2d"):   # (the other cases' gates may leave the network no cell in ten steps)
        assert stats[1]["warm_calls"] > 0
    mix = [sum(s[3 * k] * s[3 * k + 1] for k in range(n)) for s in states]
    assert rel_l1(mix[1], mix[0]) <= 1e-5
