"""Production-mode parity on the GPU.

* FP64 kernel vs the oracle's CPU twin on the same Philox-4x32-10 stream:
  identical discrete history, k and E within 1e-12 relative.
* GPU-side ensemble reductions vs the same sums taken on the CPU.
* FP32 and FP64 kernels vs the reference-RNG (mt19937_64) CPU ensemble:
  drift velocity, mean energy and subvalley occupancy within 3 sigma of the
  combined statistical error.
(FP32 against FP64 on the same stream: test_gpu_precision.py.)
"""
import numpy as np
import pytest

from emc_models import MODELS, field_force
from oracle import oracle_py as O

pytestmark = pytest.mark.gpu

REL_TOL = 1e-12


def _emc():
    from viennaemc_amd import emcgpu
    return emcgpu


def _ctx(name, n, precision, n_instances=1):
    emcgpu = _emc()
    ctx = emcgpu.Context(precision=precision, n_instances=n_instances)
    for i in range(n_instances):
        ctx.setup(i, MODELS[name])
    ctx.resize([n] * n_instances)
    return ctx


def _rel_k(a, b):
    return np.linalg.norm(a - b, axis=-1) / np.maximum(np.linalg.norm(b, axis=-1), 1e-300)


@pytest.mark.parametrize("ppl", [1, 2, 4, 8])
@pytest.mark.parametrize("name", ["si_jacoboni", "polar_gamma", "two_valley", "para_iso",
                                  "screened_polar"])
def test_fp64_production_matches_oracle_twin(name, ppl):
    emcgpu = _emc()
    spec = MODELS[name]
    n, ns, seed = 4096, 100, 0x5EED1234ABCD
    print("fp64 production vs oracle twin:", name, flush=True)
    M = O.OracleModel(spec)
    Vt = O.thermal_voltage(spec["T"])
    ref = M.init_philox(n, Vt, seed)
    ctx = _ctx(name, n, emcgpu.FP64)
    ctx.init_particles(0, seed, spec["T"])
    g0 = ctx.get_particles(0)
    assert (g0["valley"] == ref["valley"]).all() and (g0["sub"] == ref["sub"]).all()
    assert _rel_k(g0["k"].reshape(-1, 3), ref["k"].reshape(-1, 3)).max() < REL_TOL
    assert (np.abs(g0["E"] - ref["E"]) / ref["E"]).max() < REL_TOL
    assert (np.abs(g0["tau"] - ref["tau"]) / ref["tau"]).max() < REL_TOL
    # run both from the oracle's state so the comparison isolates the step
    ctx.set_particles(0, ref["k"], ref["E"], ref["tau"], ref["valley"], ref["sub"])
    force, d = field_force(spec)
    ctx.step(1e-15, ns, seed=seed, step0=7, steps_per_launch=32, ppl=ppl)
    obs_ref = M.run_philox(ref, ns, 1e-15, force, d, seed, instance=0, step0=7)
    g = ctx.get_particles(0)
    assert (g["valley"] == ref["valley"]).all()
    assert (g["sub"] == ref["sub"]).all()
    assert _rel_k(g["k"].reshape(-1, 3), ref["k"].reshape(-1, 3)).max() < REL_TOL
    assert (np.abs(g["E"] - ref["E"]) / ref["E"]).max() < REL_TOL
    av = ctx.averages(0)
    nv = len(spec["valleys"])
    # getAvgEnergy / getAvgDriftVelocity / occupancy per step, GPU Kahan sums
    # vs the oracle's serial FP64 sums over identical particles
    assert np.allclose(av["avgE"], obs_ref[:, 0, :nv], rtol=1e-11, atol=0)
    assert np.allclose(av["avgV"], obs_ref[:, 1, :nv], rtol=1e-9, atol=1e-6)
    assert (av["occ"] == obs_ref[:, 2, :nv]).all()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name", ["si_jacoboni", "two_valley"])
def test_positions_match_oracle_twin(name, precision):
    """Positions in the periodic box on the Philox stream: initial positions
    uniform in the box (draws 8-10 of the particle's initial stream) and
    their drift with the free flights, against the oracle's twin; FP64
    within 1e-12 of the box, FP32 draws bit-identical initially and within
    1e-5 of the box after 50 steps on the FP32 trajectory (the FP32 kernel
    follows the same history as long as no draw lands within rounding of a
    decision boundary, so the FP32 comparison takes the particles whose
    final valley, subvalley and k (1e-4) agree with the twin, at least 90 %
    of them)."""
    emcgpu = _emc()
    spec = MODELS[name]
    n, ns, seed = 4096, 50, 0xB0C5
    box = (3e-7, 2e-7, 4e-7)
    print("positions vs oracle twin:", name, precision, flush=True)
    M = O.OracleModel(spec)
    M.set_box(box)
    ref = M.init_philox(n, O.thermal_voltage(spec["T"]), seed, positions=True)
    ctx = _ctx(name, n, precision)
    ctx.set_box(0, box)
    ctx.init_particles(0, seed, spec["T"])
    p0 = ctx.get_positions(0)
    rp = ref["pos"].reshape(-1, 3)
    if precision == emcgpu.FP64:
        assert (np.abs(p0 - rp) <= 1e-12 * np.array(box)).all()
    else:
        # 24-bit uniforms times the box, rounded to FP32
        assert (np.abs(p0 - rp) <= 2.0 ** -23 * np.array(box)).all()
    assert (p0 >= 0).all() and (p0 <= np.array(box)).all()
    # the step from the oracle's state
    ctx.set_particles(0, ref["k"], ref["E"], ref["tau"], ref["valley"], ref["sub"])
    ctx.set_positions(0, rp)
    force, d = field_force(spec)
    ctx.step(1e-15, ns, seed=seed, step0=3)
    M.run_philox(ref, ns, 1e-15, force, d, seed, instance=0, step0=3, obs=False)
    g = ctx.get_particles(0)
    p1 = ctx.get_positions(0)
    rp1 = ref["pos"].reshape(-1, 3)
    same = (g["valley"] == ref["valley"]) & (g["sub"] == ref["sub"])
    same &= _rel_k(g["k"].reshape(-1, 3), ref["k"].reshape(-1, 3)) < 1e-4
    dp = np.abs(p1 - rp1)
    dp = np.minimum(dp, np.array(box) - dp)
    tol = 1e-12 if precision == emcgpu.FP64 else 1e-5
    print("same history %.4f, max position diff / box %.2e"
          % (same.mean(), (dp[same] / np.array(box)).max()), flush=True)
    assert same.mean() > (0.999999 if precision == emcgpu.FP64 else 0.9)
    assert (dp[same] <= tol * np.array(box)).all(), dp[same].max(axis=0)
    assert (p1 >= 0).all() and (p1 <= np.array(box)).all()
    # the particles moved: mean displacement against the field
    assert np.abs(p1 - rp).mean() > 0


def test_observe_matches_cpu_sums():
    """emcgpu_observe: the ensemble sums of the current state without a step
    (the step-0 row of the bulk example) equal the sums of the returned state."""
    emcgpu = _emc()
    spec = MODELS["two_valley"]
    counts = [50_001, 777]
    ctx = emcgpu.Context(precision=emcgpu.FP64, n_instances=2)
    for i in range(2):
        ctx.setup(i, spec)
    ctx.resize(counts)
    for i in range(2):
        ctx.init_particles(i, 5 + i, spec["T"])
    o = ctx.observe()
    _, mv, md = ctx.obs_layout()
    M = O.OracleModel(spec)
    _, d = field_force(spec)
    for i in range(2):
        g = ctx.get_particles(i)
        vdir = np.array([M.velocity(int(v), int(s), k, e) @ np.array(d) for v, s, k, e in
                         zip(g["valley"], g["sub"], g["k"].reshape(-1, 3), g["E"])])
        assert o[i, 0] == 0 and o[i, 1] == 0
        for v in range(len(spec["valleys"])):
            m = g["valley"] == v
            assert o[i, 2 + 3 * v] == m.sum()
            assert np.isclose(o[i, 3 + 3 * v], g["E"][m].sum(), rtol=1e-13)
            assert np.isclose(o[i, 4 + 3 * v], vdir[m].sum(), rtol=1e-9, atol=1e-3)
            for s in range(spec["valleys"][v]["deg"]):
                assert o[i, 2 + 3 * mv + v * md + s] == ((g["valley"] == v) & (g["sub"] == s)).sum()


def test_reductions_match_cpu_sums():
    """Per-step sums of the last step equal the sums of the returned state."""
    emcgpu = _emc()
    name = "two_valley"
    spec = MODELS[name]
    n = 100_003  # ragged: not a multiple of the tile
    ctx = _ctx(name, n, emcgpu.FP64)
    ctx.init_particles(0, 99, spec["T"])
    ctx.step(1e-15, 40, seed=99)
    g = ctx.get_particles(0)
    av = ctx.averages(0)
    M = O.OracleModel(spec)
    _, d = field_force(spec)
    vdir = np.array([M.velocity(int(v), int(s), k, e) @ np.array(d) for v, s, k, e in
                     zip(g["valley"], g["sub"], g["k"].reshape(-1, 3), g["E"])])
    for v in range(len(spec["valleys"])):
        m = g["valley"] == v
        assert av["count"][-1, v] == m.sum()
        assert np.isclose(av["sumE"][-1, v], g["E"][m].sum(), rtol=1e-13)
        assert np.isclose(av["sumV"][-1, v], vdir[m].sum(), rtol=1e-9, atol=1e-3)
        for s in range(spec["valleys"][v]["deg"]):
            assert av["sub_occ"][-1, v, s] * n == pytest.approx(((g["valley"] == v) & (g["sub"] == s)).sum())


def _stat_compare(a_mean, a_sig, b_mean, b_sig, nsig=3.0):
    return np.abs(a_mean - b_mean) <= nsig * np.sqrt(a_sig ** 2 + b_sig ** 2)


@pytest.mark.parametrize("precision", [0, 1])
def test_ensemble_matches_reference_rng(precision):
    """Si, 50 kV/cm: GPU (Philox) vs CPU ensemble on the reference engine."""
    emcgpu = _emc()
    name = "si_jacoboni"
    spec = MODELS[name]
    nsteps, dt = 800, 1e-15
    n_gpu, n_cpu = 400_000, 20_000
    print("ensemble vs reference rng, precision", precision, flush=True)
    M = O.OracleModel(spec)
    force, d = field_force(spec)
    obs_cpu, fin = M.run_mt(n_cpu, 20261202, O.thermal_voltage(spec["T"]), nsteps, dt, force, d,
                            threads=8, final=True)
    vel = np.array([M.velocity(int(v), int(s), k, e) @ np.array(d) for v, s, k, e in
                    zip(fin["valley"], fin["sub"], fin["k"].reshape(-1, 3), fin["E"])])
    sig_v, sig_e = vel.std(), fin["E"].std()
    ctx = _ctx(name, n_gpu, precision)
    ctx.init_particles(0, 4242, spec["T"])
    ctx.step(dt, nsteps, seed=4242)
    av = ctx.averages(0)
    for s in (99, 199, 399, 599, 799):
        assert _stat_compare(av["avgV"][s, 0], sig_v / np.sqrt(n_gpu),
                             obs_cpu[s, 1, 0], sig_v / np.sqrt(n_cpu)), (s, av["avgV"][s, 0], obs_cpu[s, 1, 0])
        assert _stat_compare(av["avgE"][s, 0], sig_e / np.sqrt(n_gpu),
                             obs_cpu[s, 0, 0], sig_e / np.sqrt(n_cpu)), (s, av["avgE"][s, 0], obs_cpu[s, 0, 0])
    # subvalley occupancy (valley repopulation: the pair with m_l along the
    # field is favoured at 50 kV/cm) agrees with the reference ensemble, and
    # the two pairs transverse to [100] are equally occupied
    occ = av["sub_occ"][-1, 0, :3]
    occ_cpu = np.array([(fin["sub"] == s).mean() for s in range(3)])
    sig = np.sqrt(occ * (1 - occ) / n_gpu + occ_cpu * (1 - occ_cpu) / n_cpu)
    assert np.all(np.abs(occ - occ_cpu) < 3 * sig), (occ, occ_cpu)
    assert abs(occ[1] - occ[2]) < 3 * np.sqrt(2 * occ[1] * (1 - occ[1]) / n_gpu)
    assert occ[0] > occ[1] + 10 * sig[0]


@pytest.mark.parametrize("precision", [0, 1])
def test_screened_ensemble_matches_reference_rng(precision):
    """Screened polar optical scattering (q_s^2 = 1e17 / m^2, 20 kV/cm): GPU
    (Philox) vs the oracle's ensemble on the reference engine."""
    emcgpu = _emc()
    name = "screened_polar"
    spec = MODELS[name]
    nsteps, dt = 400, 1e-15
    n_gpu, n_cpu = 200_000, 20_000
    print("screened ensemble vs reference rng, precision", precision, flush=True)
    M = O.OracleModel(spec)
    force, d = field_force(spec)
    obs_cpu, fin = M.run_mt(n_cpu, 20261203, O.thermal_voltage(spec["T"]), nsteps, dt, force, d,
                            threads=8, final=True)
    vel = np.array([M.velocity(int(v), int(s), k, e) @ np.array(d) for v, s, k, e in
                    zip(fin["valley"], fin["sub"], fin["k"].reshape(-1, 3), fin["E"])])
    sig_v, sig_e = vel.std(), fin["E"].std()
    ctx = _ctx(name, n_gpu, precision)
    ctx.init_particles(0, 99, spec["T"])
    ctx.step(dt, nsteps, seed=99)
    av = ctx.averages(0)
    for s in (49, 149, 299, 399):
        assert _stat_compare(av["avgV"][s, 0], sig_v / np.sqrt(n_gpu),
                             obs_cpu[s, 1, 0], sig_v / np.sqrt(n_cpu)), (s, av["avgV"][s, 0], obs_cpu[s, 1, 0])
        assert _stat_compare(av["avgE"][s, 0], sig_e / np.sqrt(n_gpu),
                             obs_cpu[s, 0, 0], sig_e / np.sqrt(n_cpu)), (s, av["avgE"][s, 0], obs_cpu[s, 0, 0])


def test_batched_instances_are_independent():
    """Three instances with ragged counts in one arena: each evolves exactly
    as it does alone (same instance index, seed and counts)."""
    emcgpu = _emc()
    name = "si_jacoboni"
    spec = MODELS[name]
    counts = [1000, 257, 3001]
    ctx = emcgpu.Context(precision=emcgpu.FP64, n_instances=3)
    for i in range(3):
        ctx.setup(i, spec)
    ctx.set_field(1, (0, 1, 0), 20e5)
    ctx.resize(counts)
    for i in range(3):
        ctx.init_particles(i, 11, spec["T"])
    ctx.step(1e-15, 50, seed=11)
    M = O.OracleModel(spec)
    for i, n in enumerate(counts):
        ref = M.init_philox(n, O.thermal_voltage(spec["T"]), 11, instance=i)
        if i == 1:
            force = [0.0, 20e5 * -O.Q, 0.0]
            d = (0, 1, 0)
        else:
            force, d = field_force(spec)
        M.run_philox(ref, 50, 1e-15, force, d, 11, instance=i, obs=False)
        g = ctx.get_particles(i)
        assert (g["valley"] == ref["valley"]).all() and (g["sub"] == ref["sub"]).all()
        assert _rel_k(g["k"].reshape(-1, 3), ref["k"].reshape(-1, 3)).max() < REL_TOL


@pytest.mark.parametrize("precision", [0, 1])
def test_field_step_and_tables_changed_between_calls(precision):
    """a context whose field, time step and tables change from call to call
    against contexts that are set up with them: bit-identical"""
    import copy
    emcgpu = _emc()
    base = MODELS["si_jacoboni"]
    other = copy.deepcopy(base)
    other["mechs"] = other["mechs"][:5]
    n, state = 777, None
    ctx = _ctx("si_jacoboni", n, precision)
    ctx.init_particles(0, 9, 300.0)
    # (model, field, dt): the tables change with the model only
    for i, (spec, kv, dt) in enumerate([(base, 10, 1e-15), (base, 50, 1e-15), (base, 50, 2e-15),
                                        (other, 50, 2e-15), (other, 20, 2e-15), (base, 20, 1e-15)]):
        spec = dict(spec, field_kvcm=kv)
        fresh = emcgpu.Context(precision=precision)
        fresh.setup(0, spec)
        fresh.resize([n])
        if i == 0 or spec["mechs"] is not last["mechs"]:
            ctx.setup(0, spec)
        else:
            ctx.set_field(0, spec["field_dir"], kv * 1e5)
        last = spec
        state = ctx.get_particles(0)
        for c in (ctx, fresh):
            c.set_particles(0, state["k"], state["E"], state["tau"], state["valley"], state["sub"])
            c.step(dt, 9, seed=4, step0=9 * i)
        g, f = ctx.get_particles(0), fresh.get_particles(0)
        assert all(np.array_equal(g[key], f[key]) for key in g)
        assert np.array_equal(ctx.observables(0), fresh.observables(0))
        fresh.close()
    ctx.close()
