"""The Poisson workgroup's multigrid data in each of its places: all in LDS,
the fine residual in global memory, everything there.  The solution meets the
stopping rule max |F| <= tol max h^2 (|C| + n + p) of the discrete equations
(PoissonSolver/emcSORSolver.hpp:49-197), F formed here in FP64."""
import numpy as np
import pytest

from emc_models import MODELS_DEVICE, resistor_device

pytestmark = pytest.mark.gpu

Q, EPS0 = 1.60219e-19, 8.85419e-12


@pytest.mark.parametrize("equilibrium", [True, False])
@pytest.mark.parametrize("nx,ny", [(110, 97), (127, 99), (131, 113), (150, 121)])
def test_solution_meets_the_stopping_rule(nx, ny, equilibrium):
    from viennaemc_amd import emcgpu
    dev = resistor_device(nx=nx, ny=ny, n_particles=1000)
    # spacings that differ, so that the two directions cannot be mixed up
    dev["spacing"] = (1e-9, 1.25e-9)
    dev["max_pos"] = ((nx - 1) * 1e-9, (ny - 1) * 1.25e-9)
    top = dev["max_pos"][1]
    dev["doping"] = [((lo[0], 0.0), (hi[0], top), n) for lo, hi, n in dev["doping"]]
    dev["contacts"] = [(b, v, 0.0, top) for b, v, _, _ in dev["contacts"]]
    tol = 1e-11
    ctx = emcgpu.Context(precision=emcgpu.FP64)
    ctx.setup(0, MODELS_DEVICE["device_para"])
    ctx.device_setup(dev, poisson_tol=tol)
    g = ctx.device_grids()
    dop = g["doping"] / dev["ni"]
    conc = dop * (1.0 + 0.1 * np.sin(np.arange(dop.size)))
    pot, iters, resid = ctx.poisson(np.arcsinh(0.5 * dop), None if equilibrium else conc, equilibrium)
    assert resid <= tol and iters > 0
    hx, hy = (s / ctx.debye for s in dev["spacing"])
    f = np.pad(pot.reshape(ny, nx), 1, mode="reflect")
    lap = (hy / hx * (f[1:-1, :-2] + f[1:-1, 2:] - 2 * f[1:-1, 1:-1]) +
           hx / hy * (f[:-2, 1:-1] + f[2:, 1:-1] - 2 * f[1:-1, 1:-1])).reshape(-1)
    p = np.exp(-pot)
    n = np.exp(pot) if equilibrium else conc
    F = lap + hx * hy * (p - n + dop)
    free = g["contact"] < 0
    scale = (hx * hy * (np.abs(dop) + n + p))[free].max()
    # the terms of F cancel: forming it here rounds at 1e-16 of their sum
    slack = 1e-15 * np.abs(pot).max() * 2 * (hx / hy + hy / hx)
    assert np.abs(F[free]).max() <= 1.01 * tol * scale + slack
    ctx.close()
