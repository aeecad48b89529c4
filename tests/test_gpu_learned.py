"""Learned Newton warm start on the GPU: sample capture, training gradients and
BF16-MFMA inference against the CPU checker, and what the trained network
saves over the cold start (needs a GPU)."""
import ctypes as C

import numpy as np
import pytest

import oracle.pyoracle as po
from oracle import mlp_oracle as mo
from ecogen_amd.case import IG_AIR, SG_EPOXY, SG_WATER, kapila_bubbles_2d

DP = C.POINTER(C.c_double)
EOS3 = [SG_WATER, SG_EPOXY, IG_AIR]


def _uniform_case(model, eos, alpha, rho, p, nx=64):
    return dict(name=f"uniform_{model}_{len(eos)}", nx=nx, ny=1, nz=1, lx=1.0, ly=1.0, lz=1.0, model=model,
                eos=[dict(e) for e in eos], order=1, limiters=("none",) * 4, cfl=0.8, alpha_null=False,
                relax_p=True, bc=("nonreflecting",) * 6,
                domains=[dict(kind="entire", alpha=list(alpha), rho=list(rho), p=list(p), vel=[0., 0., 0.])])


def _random_records(rng, n):
    rec = np.zeros((n, mo.SAMPLE_FLOATS), dtype=np.float32)
    for i in range(n):
        k = int(rng.integers(2, 4))
        a = rng.dirichlet(np.ones(k))
        p = 10 ** rng.uniform(4.5, 9, size=k)
        f = mo.features(a, p, EOS3[:k])
        rec[i, :12] = f[0]
        u = rng.normal(0, 1.5)
        rec[i, 15] = f[5]
        rec[i, 14] = u
        rec[i, 12] = f[3] + f[5] * u
    return rec


@pytest.mark.gpu
@pytest.mark.parametrize("model,eos,alpha,rho,p", [
    ("pueq", [SG_WATER, IG_AIR], (0.3, 0.7), (1000.0, 1.2), (3.e5, 1.e5)),
    ("ueq", EOS3, (0.5, 0.3, 0.2), (1000.0, 1185.0, 1.2), (2.e5, 5.e6, 1.e5)),
])
def test_capture_matches_oracle_relaxation(model, eos, alpha, rho, p):
    """A uniform state out of pressure equilibrium has no fluxes: every cell's
    pre-relaxation state is the initial one, so each record must carry the
    features of that state and the oracle relaxation's root and iteration count."""
    from ecogen_amd import Samples, Solver
    print(f"[learned] capture {model} {len(eos)} phases", flush=True)
    case = _uniform_case(model, eos, alpha, rho, p)
    s = Solver(case)
    smp = Samples(1000)
    s.attach_samples(smp, 1)
    s.step(1.e-15)
    rec = smp.download()
    assert rec.shape[0] == case["nx"]
    x, pc, sp, tl, fl, sg = mo.features(alpha, p, eos)
    assert abs(fl) > 1e-6          # above the library's warm-start gate
    L = po.lib()
    n = len(eos)
    oe = (po.OrcEos * n)(*[po.make_eos(e) for e in eos])
    a, r, pp, ps = np.array(alpha, float), np.array(rho, float), np.array(p, float), np.zeros(1)
    it = L.orc_relax_cell(n, oe, 0.0, 0, a.ctypes.data_as(DP), r.ctypes.data_as(DP), pp.ctypes.data_as(DP),
                          ps.ctypes.data_as(DP))
    t = (ps[0] - pc) / sp
    np.testing.assert_allclose(rec[:, :12], np.broadcast_to(x.astype(np.float32), (rec.shape[0], 12)),
                               rtol=0, atol=2e-7)
    np.testing.assert_allclose(rec[:, 12], t, rtol=2e-6, atol=2e-7)
    assert np.all(rec[:, 13] == it)
    np.testing.assert_allclose(rec[:, 15], sg, rtol=1e-6)
    # remainder over the linearised root in units of sigma; the root is known to the Newton tolerance
    Zmax = max(e["gamma"] * (p[k] + e.get("pinf", 0.)) for k, e in enumerate(eos))
    np.testing.assert_allclose(rec[:, 14], (t - tl) / sg, rtol=1e-5, atol=2e-10 * Zmax / sp / sg)


@pytest.mark.gpu
def test_training_gradient_matches_oracle():
    from ecogen_amd import Mlp, Samples
    print("[learned] gradient", flush=True)
    rng = np.random.default_rng(21)
    rec = _random_records(rng, 1000)
    prm = rng.normal(0, 0.2, mo.N_PARAM).astype(np.float32)
    smp = Samples(rec.shape[0])
    smp.upload(rec)
    m = Mlp(seed=5)
    m.set_params(prm)
    g, loss = m.gradient(smp, rec.shape[0])
    loss_o, g_o = mo.loss_and_grad(prm.astype(np.float64), rec.astype(np.float64))
    assert abs(loss - loss_o) <= 1e-5 * loss_o
    err = np.linalg.norm(g - g_o) / np.linalg.norm(g_o)
    print(f"[learned] gradient relative L2 error {err:.2e}", flush=True)
    assert err <= 1e-4
    assert np.all(np.abs(g - g_o) <= 1e-4 * np.abs(g_o).max() + 1e-4 * np.abs(g_o))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 63, 65, 1023, 1025, 4160, 32768, 32769, 70001])
def test_gradient_at_chunk_and_segment_edges(n):
    """Partial chunks (64 records), partial groups of 16 chunks, lane groups of 64 chunks and
    segments of 512 chunks.  The bound: a chain of 64 products per unit, twice, and one sum of
    at most 64 + 1094 float additions (each 6e-8), so 1e-4 of the gradient's norm."""
    from ecogen_amd import Mlp, Samples
    rng = np.random.default_rng(n)
    rec = _random_records(rng, min(n, 2000))
    rec = rec[rng.integers(0, len(rec), size=n)]
    prm = rng.normal(0, 0.2, mo.N_PARAM).astype(np.float32)
    smp = Samples(n)
    smp.upload(rec)
    m = Mlp(seed=5)
    m.set_params(prm)
    g, loss = m.gradient(smp, n)
    loss_o, g_o = mo.loss_and_grad(prm.astype(np.float64), rec.astype(np.float64))
    assert abs(loss - loss_o) <= 1e-4 * loss_o
    assert np.linalg.norm(g - g_o) <= 1e-4 * np.linalg.norm(g_o)


@pytest.mark.gpu
def test_mfma_inference_matches_bf16_oracle():
    from ecogen_amd import Mlp, Samples
    print("[learned] inference", flush=True)
    rng = np.random.default_rng(22)
    rec = _random_records(rng, 3001)          # partial last wave
    prm = rng.normal(0, 0.3, mo.N_PARAM).astype(np.float32)
    smp = Samples(rec.shape[0])
    smp.upload(rec)
    m = Mlp(seed=6)
    m.set_params(prm)
    out = m.predict(smp)
    ref = mo.forward_bf16(prm, rec[:, :12])
    ref64 = mo.forward(prm.astype(np.float64), rec[:, :12].astype(np.float64))
    d = np.abs(out - ref)
    scale = 1.0 + np.abs(ref)
    print(f"[learned] inference |gpu - bf16 oracle| max {np.max(d / scale):.2e} mean {np.mean(d / scale):.2e}; "
          f"|bf16 oracle - fp64 network| mean {np.mean(np.abs(ref - ref64) / scale):.2e}", flush=True)
    assert np.max(d / scale) <= 1e-2
    assert np.mean(d / scale) <= 2e-4


@pytest.mark.gpu
def test_samples_and_warm_start_are_exclusive():
    """Sample records describe cold solves: a context takes a sample buffer or a
    warm start, not both at once."""
    from ecogen_amd import EcgError, Mlp, Samples, Solver
    print("[learned] sample buffer / warm start exclusivity", flush=True)
    c = dict(kapila_bubbles_2d(n=32, nbub=2, order=1))
    c["precision"] = "fp32_learned"
    s = Solver(c)
    smp = Samples(1000)
    m = Mlp(seed=2)
    s.set_warm_start(m)
    with pytest.raises(EcgError, match="detach the warm start"):
        s.attach_samples(smp, 1)
    s.set_warm_start(None)
    s.attach_samples(smp, 1)
    with pytest.raises(EcgError, match="detach the sample buffer"):
        s.set_warm_start(m)
    s.attach_samples(None)
    s.set_warm_start(m)
    s.run(max_iter=2)


@pytest.mark.gpu
def test_trained_warm_start_saves_newton_iterations():
    """Train on samples of the plain FP64 solver, then compare the FP32 form's
    Newton work with the cold guess, the linearised guess (network output zero)
    and the learned guess on the same case."""
    from ecogen_amd import Mlp, Samples, Solver
    print("[learned] capture + train", flush=True)
    case = kapila_bubbles_2d(n=128, nbub=8, order=1)
    steps = 40
    s = Solver(case)
    smp = Samples(2_000_000)
    s.attach_samples(smp, 1)
    s.run(max_iter=steps)
    n = len(smp)
    print(f"[learned] {n} samples from {steps} FP64 steps", flush=True)
    assert n > 2000
    rec = smp.download()
    assert np.all(np.isfinite(rec))
    m = Mlp(seed=3)
    nchk = min(n, 50000)
    loss0 = m.gradient(smp, nchk)[1]
    losses = m.train(smp, epochs=12, batch=1024, lr=2e-3, seed=4)
    loss1 = m.gradient(smp, nchk)[1]
    print(f"[learned] loss {loss0:.3e} -> {loss1:.3e} (epochs {', '.join(f'{v:.2e}' for v in losses)})", flush=True)
    assert loss1 < 0.5 * loss0

    def run(precision, mlp):
        c = dict(case)
        c["precision"] = precision
        g = Solver(c)
        if mlp is not None:
            g.set_warm_start(mlp)
        st = g.run(max_iter=steps)
        return st, g.get_state()

    zero = Mlp(seed=1)
    zero.set_params(np.zeros(mo.N_PARAM, dtype=np.float32))
    cold, s_cold = run("fp32", None)
    lin, s_lin = run("fp32_learned", zero)
    warm, s_warm = run("fp32_learned", m)
    for nm, st in (("cold", cold), ("linearised", lin), ("learned", warm)):
        print(f"[learned] {nm}: newton evaluations {st['newton_iters']} over {st['relax_calls']} relaxations "
              f"({st['newton_iters'] / st['relax_calls']:.4f} each), warm-started {st['warm_calls']}, "
              f"fallbacks {st['warm_fallbacks']}, mean |f| at exit {st['resid_sum'] / st['relax_calls']:.2e}",
              flush=True)
    saved = cold["newton_iters"] - warm["newton_iters"]
    print(f"[learned] evaluations saved over the cold start: {saved} "
          f"({saved / max(warm['warm_calls'], 1):.3f} per warm-started relaxation)", flush=True)
    assert warm["warm_calls"] > 0
    assert warm["newton_iters"] < cold["newton_iters"]
    assert warm["warm_fallbacks"] <= 0.01 * warm["warm_calls"]
    assert warm["newton_fail"] == 0

    def mix(st):
        return st[0] * st[1] + st[3] * st[4]
    err = np.sum(np.abs(mix(s_warm) - mix(s_cold))) / np.sum(np.abs(mix(s_cold)))
    print(f"[learned] mixture density rel L1 learned vs cold FP32 form: {err:.2e}", flush=True)
    assert err <= 1e-5


@pytest.mark.gpu
def test_learned_second_order_kernels_with_an_inlet_tank():
    """The learned form of a second-order case with an inlet tank runs the
    full-featured kernel instantiation; with the network output at zero (the
    linearised guess) it must track the cold FP32 form."""
    from ecogen_amd import Mlp, Solver
    from small_cases import pueq_2d_tank
    print("[learned] second order with an inlet tank", flush=True)
    case = pueq_2d_tank(2)
    states, stats = [], []
    for precision in ("fp32", "fp32_learned"):
        c = dict(case)
        c["precision"] = precision
        g = Solver(c)
        if precision == "fp32_learned":
            m = Mlp(seed=1)
            m.set_params(np.zeros(mo.N_PARAM, dtype=np.float32))
            g.set_warm_start(m)
        stats.append(g.run(max_iter=10))
        states.append(g.get_state())
    assert stats[1]["warm_calls"] > 0 and np.all(np.isfinite(states[1]))
    mix = lambda s: s[0] * s[1] + s[3] * s[4]
    err = np.sum(np.abs(mix(states[1]) - mix(states[0]))) / np.sum(np.abs(mix(states[0])))
    print(f"[learned] tank case: mixture density rel L1 learned vs cold {err:.2e}", flush=True)
    assert err <= 1e-5


@pytest.mark.gpu
def test_three_phase_warm_start_saves_newton_iterations():
    """The three-phase pressure-non-equilibrium case (water, epoxy, air inclusions hit by a
    1e9 Pa shock; a 48^3 replica of the 256^3 configuration): trained on relaxation records
    of its own plain FP64 run and of the 2D Kapila case, the learned warm start must need
    fewer Newton evaluations than the cold start of the same FP32 form, stop every
    relaxation at the reference tolerance (mean |f| at exit below 1e-10) and never fall
    back to the interface pressure."""
    from ecogen_amd import learned
    from ecogen_amd.case import ueq3_spheres_3d
    print("[learned] three-phase capture + train", flush=True)
    case = ueq3_spheres_3d(n=48, nsph=12)
    steps = 12
    sources = [(case, steps), (kapila_bubbles_2d(n=128, nbub=8, order=1), 20)]
    smp, info = learned.collect_samples(sources, target=400_000)
    print(f"[learned] {info}", flush=True)
    assert info["records"] > 20000
    fsmp, kept = learned.focus(smp)
    smp.close()
    print(f"[learned] {kept} records above the inference gate", flush=True)
    assert kept > 2000
    m, tinfo = learned.train(fsmp, batch=1024, lr=2e-3, seed=5, updates=3000)
    fsmp.close()
    print(f"[learned] training {tinfo['loss_initial']:.3e} -> {tinfo['loss_final']:.3e}", flush=True)
    from ecogen_amd import Solver
    res = {}
    for form in ("fp32", "fp32_learned"):
        g = Solver(dict(case, precision=form))
        if form == "fp32_learned":
            g.set_warm_start(m)
        res[form] = g.run(max_iter=steps)
        g.close()
    cold, warm = res["fp32"], res["fp32_learned"]
    for nm, st in (("cold", cold), ("learned", warm)):
        print(f"[learned] three-phase {nm}: {st['newton_iters']} evaluations over {st['relax_calls']} relaxations "
              f"({st['newton_iters'] / st['relax_calls']:.5f} each), warm-started {st['warm_calls']}, "
              f"fallbacks {st['warm_fallbacks']}, mean |f| at exit {st['resid_sum'] / st['relax_calls']:.2e}",
              flush=True)
    assert warm["warm_calls"] > 0
    assert warm["newton_iters"] < cold["newton_iters"]
    assert warm["resid_sum"] / warm["relax_calls"] <= 1e-10
    assert warm["newton_fail"] == 0 and cold["newton_fail"] == 0
