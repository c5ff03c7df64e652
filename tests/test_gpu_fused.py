"""The production step kernel where its bookkeeping can go wrong: waves that
are partly or barely filled, steps around the depth of its step-sum ring,
event rates at which particles lag behind or share passes, and table rows of
every grouping.  FP64 against the oracle's twin on the same random numbers:
histories identical, k and E within rounding, the per-step sums of exactly
the particles of each step."""
import copy

import numpy as np
import pytest

from emc_models import MODELS, field_force
from oracle import oracle_py as O

pytestmark = pytest.mark.gpu


def _run(spec, n, steps, dt, ppl, spl, seed=77):
    from viennaemc_amd import emcgpu
    M = O.OracleModel(spec)
    ref = M.init_philox(n, O.thermal_voltage(spec["T"]), seed)
    ctx = emcgpu.Context(precision=emcgpu.FP64)
    ctx.setup(0, spec)
    ctx.resize([n])
    ctx.set_particles(0, ref["k"], ref["E"], ref["tau"], ref["valley"], ref["sub"])
    ctx.step(dt, steps, seed=seed, step0=3, steps_per_launch=spl, ppl=ppl)
    force, d = field_force(spec)
    obs = M.run_philox(ref, steps, dt, force, d, seed, step0=3)
    got = ctx.get_particles(0)
    assert (got["valley"] == ref["valley"]).all() and (got["sub"] == ref["sub"]).all()
    # one rounding per drift and event accumulates like the 1e-12 of the long
    # twin runs over 100 steps
    k, kr = got["k"].reshape(-1, 3), ref["k"].reshape(-1, 3)
    assert (np.linalg.norm(k - kr, axis=1) <= 1e-12 * np.linalg.norm(kr, axis=1)).all()
    assert (np.abs(got["tau"] - ref["tau"]) <= 1e-12 * dt + 1e-12 * np.abs(ref["tau"])).all()
    av = ctx.averages(0)
    nv = len(spec["valleys"])
    assert (av["occ"] == obs[:, 2, :nv]).all()
    assert np.allclose(av["avgE"], obs[:, 0, :nv], rtol=1e-11, atol=0)
    # velocities cancel: within rounding of the thermal ones (1e5 m/s)
    assert np.allclose(av["avgV"], obs[:, 1, :nv], rtol=1e-9, atol=1e-6)
    # the last step's subvalley counts are those of the final state
    cnt = np.array([[np.sum((ref["valley"] == v) & (ref["sub"] == s)) for s in range(av["sub_occ"].shape[2])]
                    for v in range(nv)])
    assert (np.rint(av["sub_occ"][-1] * n) == cnt).all()
    ctx.close()


@pytest.mark.parametrize("ppl", [1, 2, 4, 8])
@pytest.mark.parametrize("n", [1, 63, 65, 257, 2049])
def test_partly_filled_waves(n, ppl):
    _run(MODELS["two_valley"], n, 21, 2e-15, ppl, 0)


@pytest.mark.parametrize("spl", [1, 2, 15, 16, 17, 40])
@pytest.mark.parametrize("dt", [0.05e-15, 12e-15])
def test_rare_and_frequent_events(dt, spl):
    """dt = 0.05 fs: about three pending events per wave and step, so that
    they wait for each other; 12 fs: most particles scatter, several times"""
    _run(MODELS["si_jacoboni"], 1500, 40, dt, 4, spl)


@pytest.mark.parametrize("nt", [1, 3, 4, 5, 8, 9, 16, 17, 32])
def test_table_rows(nt):
    """rows of one to eight groups, the last one full or not"""
    spec = copy.deepcopy(MODELS["si_jacoboni"])
    base = spec["mechs"]
    spec["mechs"] = []
    for j in range(nt):
        m = dict(base[j % len(base)])
        scale = 0.3 + 0.07 * j
        if "sigma" in m:
            m["sigma"] *= scale
        else:
            m["defpot"] *= scale
        spec["mechs"].append(m)
    _run(spec, 700, 30, 2e-15, 2, 16)


@pytest.mark.parametrize("ppl", [1, 2, 4, 8])
@pytest.mark.parametrize("model,dt", [("screened_polar", 0.5e-15), ("two_valley", 15e-15)])
def test_one_step_launches(model, dt, ppl):
    """one-step launches with few events (one valley: streamed in one to eight
    chunks of 64, the last one ragged; in registers with one per lane) and with
    mostly scattering particles (two valleys: held in LDS)"""
    _run(MODELS[model], 1801, 12, dt, ppl, 1)


@pytest.mark.parametrize("ppl", [2, 4, 8])
@pytest.mark.parametrize("n", [127, 1801, 4097])
def test_streaming_with_many_events(n, ppl):
    """most particles of a chunk wait when the next 64 arrive: the queue holds
    up to 59 + 64 of its 128 entries and wraps"""
    _run(MODELS["si_jacoboni"], n, 8, 15e-15, ppl, 1)


# dt such that about 4 % and most of the particles scatter in a step
RARE, MANY = {"si_jacoboni": 0.2e-15, "two_valley": 1e-15}, 12e-15


@pytest.mark.parametrize("spl", [1, 3, 4, 5])
@pytest.mark.parametrize("n", [1, 65, 1801])
@pytest.mark.parametrize("model", ["si_jacoboni", "two_valley"])
def test_short_launches_one_per_lane(model, n, spl):
    """one particle per lane: in registers up to four steps per launch, in LDS
    from five on"""
    _run(MODELS[model], n, 10, MANY, 1, spl)


@pytest.mark.parametrize("ppl", [1, 2, 4, 8])
@pytest.mark.parametrize("dt", [RARE["two_valley"], MANY])
@pytest.mark.parametrize("n", [63, 1801])
def test_one_step_launches_of_several_valleys(n, dt, ppl):
    """two and four per lane: in registers while events are rare, else in LDS"""
    _run(MODELS["two_valley"], n, 20, dt, ppl, 1)


@pytest.mark.parametrize("model,ppl,spl", [("two_valley", 1, 1), ("two_valley", 2, 1), ("two_valley", 4, 1),
                                           ("si_jacoboni", 1, 1), ("si_jacoboni", 1, 4),
                                           ("si_jacoboni", 2, 1)])
def test_fp32_launch_shapes_agree(model, ppl, spl):
    """the kernels of short launches in FP32 against eight per lane held in LDS
    for all steps.  The same arithmetic, but the compiler may contract it
    differently in each kernel: a last bit decides a draw about once in 2^20
    events, and k differs by a rounding (6e-8) per flight"""
    from viennaemc_amd import emcgpu
    spec, n, steps, out = MODELS[model], 5001, 12, []
    for p, k in ((ppl, spl), (8, steps)):
        for dt in (RARE[model], MANY):
            ctx = emcgpu.Context(precision=emcgpu.FP32)
            ctx.setup(0, spec)
            ctx.resize([n])
            ctx.init_particles(0, 11, spec["T"])
            ctx.step(dt, steps, seed=5, steps_per_launch=k, ppl=p)
            out.append((ctx.get_particles(0), ctx.averages(0)))
            ctx.close()
    for (g, av), (h, bv) in zip(out[:2], out[2:]):
        same = (g["valley"] == h["valley"]) & (g["sub"] == h["sub"])
        x, y = g["k"].reshape(-1, 3), h["k"].reshape(-1, 3)
        # 12 steps of up to about four flights, each rounding twice
        same &= np.linalg.norm(x - y, axis=1) <= 1e-5 * np.linalg.norm(y, axis=1)
        # the share of a particle whose 50 events each meet such a draw
        assert same.mean() > 1 - 1e-3
        assert np.abs(av["occ"] - bv["occ"]).max() <= 1e-3
        nv = len(spec["valleys"])
        cnt = np.array([[np.sum((g["valley"] == v) & (g["sub"] == s)) for s in range(av["sub_occ"].shape[2])]
                        for v in range(nv)])
        assert (np.rint(av["sub_occ"][-1] * n) == cnt).all()


@pytest.mark.parametrize("n,spl", [(70001, 1), (70001, 3), (70001, 10), (163841, 1), (163841, 10),
                                   (327681, 1), (327681, 10)])
@pytest.mark.parametrize("model,dt", [("si_jacoboni", 1e-15), ("two_valley", 1e-15), ("si_jacoboni", 9e-15)])
def test_tracked_positions_at_every_default(model, dt, n, spl):
    """positions with one, two and four particles per lane, which follow from
    the size of the ensemble"""
    from viennaemc_amd import emcgpu
    spec, steps, seed = MODELS[model], 10, 21
    box = np.array([3e-7, 2e-7, 4e-7])
    M = O.OracleModel(spec)
    M.set_box(tuple(box))
    ref = M.init_philox(n, O.thermal_voltage(spec["T"]), seed, positions=True)
    ctx = emcgpu.Context(precision=emcgpu.FP64)
    ctx.setup(0, spec)
    ctx.resize([n])
    ctx.set_box(0, tuple(box))
    ctx.set_particles(0, ref["k"], ref["E"], ref["tau"], ref["valley"], ref["sub"])
    ctx.set_positions(0, ref["pos"])
    ctx.step(dt, steps, seed=seed, step0=3, steps_per_launch=spl)
    force, d = field_force(spec)
    obs = M.run_philox(ref, steps, dt, force, d, seed, step0=3)
    got, pos = ctx.get_particles(0), ctx.get_positions(0)
    assert (got["valley"] == ref["valley"]).all() and (got["sub"] == ref["sub"]).all()
    k, kr = got["k"].reshape(-1, 3), ref["k"].reshape(-1, 3)
    assert (np.linalg.norm(k - kr, axis=1) <= 1e-12 * np.linalg.norm(kr, axis=1)).all()
    dp = np.abs(pos - ref["pos"].reshape(-1, 3))
    assert (np.minimum(dp, box - dp) <= 1e-12 * box).all()
    av = ctx.averages(0)
    assert (av["occ"] == obs[:, 2, :len(spec["valleys"])]).all()
    ctx.close()


def test_two_threads_with_workgroups_of_different_lds():
    """contexts of different models step side by side in the same kernel, each
    with its own amount of LDS above 64 KB"""
    import threading
    from viennaemc_amd import emcgpu
    names, n, calls = ("si_jacoboni", "para_iso"), 4096, 40

    def run(name, out):
        ctx = emcgpu.Context(precision=emcgpu.FP64)
        ctx.setup(0, MODELS[name])
        ctx.resize([n])
        ctx.init_particles(0, 2, 300.0)
        for c in range(calls):
            ctx.step(1e-15, 8, seed=6, step0=8 * c, steps_per_launch=8, ppl=8)
        out[name] = (ctx.get_particles(0), ctx.observables(0))
        ctx.close()

    alone, together = {}, {}
    for name in names:
        run(name, alone)
    threads = [threading.Thread(target=run, args=(name, together)) for name in names]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for name in names:
        (p, obs), (q, want) = together[name], alone[name]
        assert all(np.array_equal(p[key], q[key]) for key in p)
        assert np.array_equal(obs, want)


def test_reserve_covers_a_shorter_call():
    """positions in FP64: two steps take four particles per lane, one step
    takes one and four times the partials.  A context that reserved two steps
    runs one without taking device memory"""
    import ctypes as C
    from test_zz_no_alloc import _hip
    from viennaemc_amd import emcgpu
    hip = _hip()  # the runtime that the library is linked against

    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    spec, n, used = MODELS["si_jacoboni"], 4_000_000, []
    for _ in range(2):  # the first context also loads the kernels
        ctx = emcgpu.Context(precision=emcgpu.FP64)
        ctx.setup(0, spec)
        ctx.resize([n])
        ctx.set_box(0, (3e-7, 2e-7, 4e-7))
        ctx.init_particles(0, 2, spec["T"])
        ctx.reserve(1e-15, 2)
        ctx.synchronize()
        free = free_bytes()
        ctx.step(1e-15, 1, seed=3)
        ctx.synchronize()
        used.append(free - free_bytes())
        ctx.close()
    assert used[1] <= 0
