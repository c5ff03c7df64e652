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
