"""Bath tallies, bath updates and plasma screening with every number of
particles per lane: the kernels that keep a lane's particles (1; 2 in FP32 with
several valleys), stream them (FP64, one valley) or exchange them through LDS
(the others).  The oracle's twin on the same random numbers at ragged counts,
so that events that change lanes are tallied exactly once."""
import copy

import numpy as np
import pytest

from emc_models import MODELS, ZERO_IV_AB, ZERO_IV_EM, field_force
from oracle import oracle_py as O

pytestmark = pytest.mark.gpu

PPL = [1, 2, 4, 8]


def _two_valleys():
    """hot_polar with a second valley, its own Froehlich pair on the same bath
    and exchange between the valleys"""
    spec = copy.deepcopy(MODELS["hot_polar"])
    spec["valleys"].append(dict(spec["valleys"][0], bottom=0.25, mass=(0.4, 0.4, 0.4)))
    spec["mechs"] += [dict(m, valley=1, mrel=0.4) for m in spec["mechs"]]
    for a, b in ((0, 1), (1, 0)):
        for kind in (ZERO_IV_AB, ZERO_IV_EM):
            spec["mechs"].append(dict(kind=kind, valley=a, final=b, defpot=5e10, hw=0.05, fmap=[[0]]))
    return spec


def _twin(spec, n, ns, dt, seed, ppl, update, every=1, screened=False):
    from viennaemc_amd import emcgpu
    M = O.OracleModel(spec)
    M.set_bath_mode(update=update, rebuild_every=every, step_count=0)
    ref = M.init_philox_energy(n, spec["init_energy"], 0.05, seed)
    ctx = emcgpu.Context(precision=emcgpu.FP64)
    ctx.setup(0, spec)
    ctx.resize([n])
    ctx.set_particles(0, ref["k"], ref["E"], ref["tau"], ref["valley"], ref["sub"])
    if screened:
        M.seed_screening(ref["E"], ref["valley"])
        ctx.update_screening(0)
    force, d = field_force(spec)
    ctx.step(dt, ns, seed=seed, ppl=ppl, bath_record_only=not update, rebuild_every=every)
    hist, obs = [], []
    for s in range(ns):
        obs.append(M.run_philox(ref, 1, dt, force, d, seed, step0=s)[0])
        hist.append(M.bath(0)["mean"])
    g = ctx.get_particles(0)
    assert (g["valley"] == ref["valley"]).all() and (g["sub"] == ref["sub"]).all()
    # the sums of every step are those of the particles of that step
    assert (ctx.averages(0)["occ"] == np.array(obs)[:, 2, :len(spec["valleys"])]).all()
    return ctx, M, ref, g, np.array(hist)


def _same_state(g, ref):
    k, kr = g["k"].reshape(-1, 3), ref["k"].reshape(-1, 3)
    assert (np.linalg.norm(k - kr, axis=1) <= 1e-12 * np.linalg.norm(kr, axis=1)).all()


@pytest.mark.parametrize("ppl", PPL)
@pytest.mark.parametrize("dt", [0.5e-15, 8e-15])
@pytest.mark.parametrize("n", [65, 3001])
@pytest.mark.parametrize("valleys", [1, 2])
def test_tallies_are_exact(valleys, n, dt, ppl):
    """few and, at 8 fs, several events per particle and step"""
    spec = MODELS["hot_polar"] if valleys == 1 else _two_valleys()
    ctx, M, ref, g, _ = _twin(spec, n, 12, dt, 0x7A11, ppl, update=False)
    _same_state(g, ref)
    em, ab = ctx.bath_tallies(0, 0)
    o = M.bath(0)
    assert em.sum() > 0
    assert (em == o["n_em"].astype(np.uint64)).all()
    assert (ab == o["n_abs"].astype(np.uint64)).all()
    ctx.close()


@pytest.mark.parametrize("ppl", PPL)
@pytest.mark.parametrize("valleys,every", [(1, 1), (1, 4), (2, 1)])
def test_bath_follows_the_twin(valleys, every, ppl):
    spec = MODELS["hot_polar"] if valleys == 1 else _two_valleys()
    ctx, M, ref, g, hist = _twin(spec, 2777, 22, 0.5e-15, 0x5712, ppl, update=True, every=every)
    _same_state(g, ref)
    assert np.allclose(ctx.bath_history(0, 0), hist, rtol=1e-12, atol=0)
    assert np.allclose(ctx.get_bath(0, 0)["nq"], M.bath(0)["nq"], rtol=1e-12, atol=0)
    ctx.close()


@pytest.mark.parametrize("ppl", PPL)
def test_screening_follows_the_twin(ppl):
    """history, bath and q_s^2; the q-resolved angle turns rounding at the
    window's edge into direction noise of about its square root, so that k is
    held to 1e-6 and what follows from the energies to 1e-10"""
    ctx, M, ref, g, hist = _twin(MODELS["screened_hot_polar"], 3001, 30, 0.5e-15, 0x5C4EE, ppl,
                                 update=True, screened=True)
    k, kr = g["k"].reshape(-1, 3), ref["k"].reshape(-1, 3)
    assert (np.linalg.norm(k - kr, axis=1) <= 1e-6 * np.linalg.norm(kr, axis=1)).all()
    assert np.allclose(ctx.bath_history(0, 0), hist, rtol=1e-10, atol=0)
    assert np.allclose(ctx.get_bath(0, 0)["nq"], M.bath(0)["nq"], rtol=1e-10, atol=0)
    assert abs(ctx.get_screening(0) - M.qs2()) <= 1e-10 * M.qs2()
    ctx.close()


@pytest.mark.parametrize("ppl", PPL)
def test_screened_instances_are_independent(ppl):
    """two instances with ragged counts evolve as each does alone, the
    screening of each from its own tiles of the step partials"""
    from viennaemc_amd import emcgpu
    specs = [MODELS["screened_hot_polar"], copy.deepcopy(MODELS["screened_hot_polar"])]
    specs[1]["field_kvcm"] = 30.0
    specs[1]["screening"]["volume"] = 1.0e-23
    counts, out = [4097, 1500], []
    for which in ((0, 1), (0,), (1,)):
        ctx = emcgpu.Context(precision=emcgpu.FP64, n_instances=2)
        for i in range(2):
            ctx.setup(i, specs[i])
        ctx.resize([counts[i] if i in which else 0 for i in range(2)])
        for i in which:
            ctx.init_particles_energy(i, 17, 0.5, 0.05)
            ctx.update_screening(i)
        ctx.step(0.5e-15, 20, seed=17, ppl=ppl)
        out.append({i: (ctx.get_particles(i), ctx.bath_history(i, 0), ctx.get_screening(i)) for i in which})
        ctx.close()
    for i in range(2):
        (p, h, q), (ps, hs, qs) = out[0][i], out[1 + i][i]
        assert all(np.array_equal(p[key], ps[key]) for key in p)
        assert np.array_equal(h, hs) and q == qs


@pytest.mark.parametrize("ppl", PPL)
@pytest.mark.parametrize("valleys", [1, 2])
def test_fp32_tallies_hold_every_event(valleys, ppl):
    """FP32 has no twin: the tallies of a record-only run are the tallies of
    the run with one particle per lane, whose histories part only where a draw
    falls within the rounding of a decision (about once in 2^20 events)"""
    from viennaemc_amd import emcgpu
    spec = MODELS["hot_polar"] if valleys == 1 else _two_valleys()
    n, out = 6001, []
    for p in (1, ppl):
        ctx = emcgpu.Context(precision=emcgpu.FP32)
        ctx.setup(0, spec)
        ctx.resize([n])
        ctx.init_particles_energy(0, 5, 0.5, 0.05)
        ctx.step(4e-15, 15, seed=5, ppl=p, bath_record_only=True)
        out.append((np.concatenate(ctx.bath_tallies(0, 0)).astype(np.int64), ctx.observables(0)))
        ctx.close()
    (t1, o1), (t, o) = out
    total = t1.sum()
    assert total > 1000
    # 90 k particle steps of about one event: an odd history moves a few of them
    assert np.abs(t - t1).sum() <= 1e-3 * total
    assert np.abs(o[:, :2] - o1[:, :2]).sum() <= 1e-3 * o1[:, :2].sum()
    assert (o[:, 2:3] == n).all() if valleys == 1 else (o[:, 2] + o[:, 5] == n).all()
