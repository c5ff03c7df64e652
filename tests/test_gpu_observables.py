"""The per-step sums that a call leaves in its context: readable until the next
call, whatever comes between."""
import numpy as np
import pytest

from emc_models import MODELS

pytestmark = pytest.mark.gpu

DT = 1e-15


def _ctx(n=1000, n_instances=1, precision=1):
    from viennaemc_amd import emcgpu
    spec = MODELS["si_jacoboni"]
    ctx = emcgpu.Context(precision=precision, n_instances=n_instances)
    for i in range(n_instances):
        ctx.setup(i, spec)
    ctx.resize([n] * n_instances)
    for i in range(n_instances):
        ctx.init_particles(i, 3 + i, spec["T"])
    return ctx


def test_a_model_of_another_layout_drops_the_sums():
    """four subvalleys of two valleys take more values per step than were
    written: no read past them"""
    ctx = _ctx()
    ctx.step(DT, 7, seed=1)
    assert ctx.observables(0).shape[0] == 7
    ctx.setup(0, MODELS["si_vasileska"])  # the same layout: kept
    assert ctx.observables(0).shape[0] == 7
    ctx.setup(0, MODELS["two_valley"])
    assert ctx.observables(0).shape[0] == 0
    ctx.close()


def test_reserve_keeps_the_sums():
    """more steps reserved between a call and its read; into device memory
    (64 instances x 20000 steps x 8 values: 82 MB and more)"""
    ctx = _ctx(n=300, n_instances=64)
    ctx.step(DT, 7, seed=1)
    ctx.synchronize()
    want = [ctx.observables(i).copy() for i in (0, 63)]
    assert want[0].shape[0] == 7 and (want[0][:, 2] == 300).all()
    for steps in (100, 20000):
        ctx.reserve(DT, steps)
        for i, w in zip((0, 63), want):
            assert np.array_equal(ctx.observables(i), w)
    ctx.close()


def test_a_failed_reserve_keeps_the_sums():
    """2^31 - 1 steps of 64 instances are terabytes of sums: an error, the last
    call's sums stay, and the next call runs"""
    from viennaemc_amd import emcgpu
    ctx = _ctx(n=300, n_instances=64)
    ctx.step(DT, 7, seed=1)
    want = ctx.observables(63).copy()
    with pytest.raises(emcgpu.EmcGpuError):
        ctx.reserve(DT, 2**31 - 1)
    assert np.array_equal(ctx.observables(63), want)
    ctx.step(DT, 9, seed=1, step0=7)
    assert ctx.observables(63).shape[0] == 9
    ctx.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_sums_beyond_the_pinned_limit(precision):
    """the sums of a long call, held in device memory, are those of the same
    steps in two calls whose sums are pinned"""
    steps, inst = 18000, 64
    ctx = _ctx(n=65, n_instances=inst, precision=precision)
    assert 8 * steps * inst * ctx.obs_layout()[0] > 64 << 20 > 4 * steps * inst * ctx.obs_layout()[0]
    ctx.step(DT, steps, seed=4, steps_per_launch=60)
    got = [ctx.observables(i) for i in (0, 31, 63)]
    ctx.close()
    ctx = _ctx(n=65, n_instances=inst, precision=precision)
    for half in (0, 1):
        ctx.step(DT, steps // 2, seed=4, step0=half * steps // 2, steps_per_launch=60)
        for i, g in zip((0, 31, 63), got):
            assert np.array_equal(ctx.observables(i), g[half * steps // 2:(half + 1) * steps // 2])
    ctx.close()
