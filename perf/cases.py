"""The work that users of this library have it do, as cases to be timed and compared.

Each case goes through the public entry points of ``viennaemc_amd.emcgpu``: bulk ensembles from ten
thousand to ten million carriers, a batched parameter sweep, hot-phonon cooling, the self-consistent 2-D
device, and the particle-mesh and Poisson operators on host data.  Sizes, models and options are those of
the workload descriptions, the tests and the benchmark of this repository.

``exact`` follows the same carriers in 64 bits with torch and numpy alone: the random numbers are
Philox-4x32-10 keyed by the seed, so the carriers' histories are determined, not just their statistics.
"""
import copy
import math

import numpy as np
import torch

from viennaemc_amd import emcgpu, workloads

Q, KB, HBAR, EPS0, ME = 1.60219e-19, 1.38066e-23, 1.05459e-34, 8.85419e-12, 9.11e-31
PM_NAMES = {"ngp": 0, "cic": 1, "nec": 2}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the plain bulk silicon run of the reference's bulk example: ten thousand electrons at low field in
        # FP64, a stretch of it with the averages of every step, then the particle dump
        dict(name="bulk_10k_fp64", kind="bulk", model="si_jacoboni", particles=10_000, precision="f64",
             steps=100, field=10.0, t_init=340.0, read="state", graph=False),
        # a program that keeps the reference's loop: one moveParticles(dt) and the averages after it, per call
        dict(name="bulk_call_fp32", kind="bulk", model="si_vasileska", particles=50_001, precision="f32",
             steps=1, field=10.0, t_init=340.0, read="averages", graph=False),
        # the bulk example with positions in the periodic box and its files at the end
        dict(name="bulk_box_200k_fp32", kind="bulk", model="si_jacoboni", particles=200_003, precision="f32",
             steps=50, field=30.0, t_init=1200.0, read="positions", graph=False),
        # the benchmark's ensemble: ten million electrons at 50 kV/cm, 64 steps fused
        dict(name="bulk_10m_fp32", kind="bulk", model="si_jacoboni", particles=10_000_000, precision="f32",
             steps=64, field=50.0, t_init=2000.0, read="averages", graph=False),
        # two valleys (an anisotropic one and a raised Kane valley) in double precision, an odd size
        dict(name="two_valley_4m_fp64", kind="bulk", model="two_valley", particles=3_999_971, precision="f64",
             steps=16, field=30.0, t_init=1000.0, read="averages", graph=False),
        # the 64-instance bias / temperature / size sweep, one arena, one HIP graph per call
        dict(name="sweep_64_fp32", kind="sweep", instances=64, precision="f32", steps=32, n_min=10_000,
             n_max=2_000_000, graph=True),
        # photoexcited cooling on a 256-bin hot-phonon bath, updated with the tables after every step
        dict(name="cooling_4m_fp32", kind="cooling", screened=False, particles=4_000_000, precision="f32",
             steps=24, graph=True),
        # the hot-carrier default: screened, q-resolved, with plasma screening, in double precision
        dict(name="screened_1m_fp64", kind="cooling", screened=True, particles=1_000_003, precision="f64",
             steps=16, graph=True),
        # the 2-D resistor of the benchmark: Poisson, deposit and contacts every 0.1 fs step
        dict(name="resistor_2m_fp32", kind="device", nx=200, ny=50, particles=2_000_000, precision="f32",
             steps=40, gated=False, pm="cic", bias=0.5, graph=True),
        # a smaller resistor with a gate over part of one boundary (no separable inverse), double precision
        dict(name="gated_60k_fp64", kind="device", nx=81, ny=31, particles=60_000, precision="f64", steps=20,
             gated=True, pm="cic", bias=0.3, graph=False),
        # the start of a MOSFET run: the equilibrium potential on the 126 x 101 grid by Newton and multigrid
        dict(name="mosfet_equilibrium", kind="poisson", nx=126, ny=101, width=1e-6),
        # 3-D charge assignment and force interpolation on the caller's arrays
        dict(name="mesh3_200k", kind="mesh3", nx=48, ny=40, nz=33, particles=200_001, pm="cic"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["bulk"] * 6 + ["sweep"] + ["cooling"] * 2 + ["device"] * 3 + ["poisson", "mesh3"])
    prec = rng.choice(["f32", "f32", "f64"])
    if kind == "bulk":
        n = _log(rng, 8_000, 8_000_000 if prec == "f32" else 3_000_000)
        most = (300 if prec == "f32" else 60) * 1_000_000 // n
        read = rng.choice(["averages", "averages", "state", "positions"]) if n <= 250_000 else "averages"
        steps = max(1, min(_log(rng, 1, 128), most))
        model = rng.choice(["si_jacoboni", "si_jacoboni", "si_vasileska", "two_valley", "polar_gamma",
                            "para_iso", "screened_polar"])
        # a carrier temperature near what the field holds, and fields the models' energy grids cover
        field = round(math.exp(rng.uniform(math.log(1.0), math.log(40.0))), 3)
        field = min(field, 8.0) if model == "para_iso" else field
        return dict(kind="bulk", model=model, particles=n, precision=prec, steps=steps, field=field,
                    t_init=round(300.0 + 25.0 * field, 1), read=read, graph=rng.random() < 0.3)
    if kind == "sweep":
        return dict(kind="sweep", instances=rng.randint(3, 64), precision=prec, steps=rng.randint(2, 12),
                    n_min=_log(rng, 2_000, 20_000), n_max=_log(rng, 50_000, 400_000), graph=rng.random() < 0.5)
    if kind == "cooling":
        return dict(kind="cooling", screened=rng.random() < 0.5, particles=_log(rng, 50_000, 2_000_000),
                    precision=prec, steps=rng.randint(4, 16), graph=rng.random() < 0.5)
    if kind == "device":
        gated = rng.random() < 0.4
        return dict(kind="device", nx=rng.randint(41, 160), ny=rng.randint(11, 48),
                    particles=_log(rng, 30_000, 300_000 if gated else 1_500_000), precision=prec,
                    steps=rng.randint(4, 24), gated=gated, pm=rng.choice(["cic", "cic", "ngp", "nec"]),
                    bias=round(rng.uniform(0.05, 0.6), 3), graph=rng.random() < 0.5)
    if kind == "poisson":
        # the junction depths keep their proportions on a grid of another resolution
        return dict(kind="poisson", nx=rng.randint(90, 126), ny=rng.randint(60, 101), width=1e-6)
    return dict(kind="mesh3", nx=rng.randint(17, 64), ny=rng.randint(9, 48), nz=rng.randint(5, 40),
                particles=_log(rng, 20_000, 400_000), pm=rng.choice(["cic", "ngp"]))


# ---------------------------------------------------------------------------
# what a program has in hand before the call
# ---------------------------------------------------------------------------
def _precision(case):
    return emcgpu.FP32 if case["precision"] == "f32" else emcgpu.FP64


def _bulk_spec(case):
    spec = copy.deepcopy(workloads.MODELS[case["model"]])
    spec["field_kvcm"] = case["field"]
    return spec


def _sweep(case, seed):
    # the seed of the sweep fixes sizes and conditions; a run's seed draws its carriers and random numbers
    return workloads.batched_instances(case["instances"], 20261202, case["n_min"], case["n_max"])


def _cooling_spec(case):
    n = case["particles"]
    return workloads.screened_cooling(n) if case["screened"] else workloads.photoexcited_cooling(n)


def _device_dict(case):
    dev = workloads.resistor_device(nx=case["nx"], ny=case["ny"], n_particles=case["particles"],
                                    contact_nodes=max(3, case["nx"] // 20), bias=case["bias"])
    if case["gated"]:
        # an oxide gate over the middle of the upper boundary, as in the gated resistor of the tests
        x0, x1 = (case["nx"] // 4) * 1e-9, (case["nx"] - 1 - case["nx"] // 4) * 1e-9
        dev["contacts"] = dev["contacts"] + [(3, 0.4, x0, x1, 3.9, 1e-9, 0.3)]
    return dev


def _mosfet_dict(case, seed):
    # the mosfet2D device; the grid's spacing scales so that the extents stay those of the example, and the
    # bulk doping varies by a few percent from wafer to wafer
    dev = workloads.mosfet_device(width=case["width"])
    nx, ny = case["nx"], case["ny"]
    dev["spacing"] = (dev["max_pos"][0] / (nx - 1), dev["max_pos"][1] / (ny - 1))
    f = 1.0 + 0.05 * (2.0 * np.random.RandomState(seed % (1 << 32)).rand() - 1.0)
    dev["doping"] = [(lo, hi, n * f) for lo, hi, n in dev["doping"]]
    return dev


DEVICE_DT = 0.1e-15
COOLING_DT = 0.5e-15
BULK_DT = 1e-15


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case, seed=seed, at=0)
    if kind == "mesh3":
        rs = np.random.RandomState(seed % (1 << 32))
        ext = (case["nx"], case["ny"], case["nz"])
        nn = ext[0] * ext[1] * ext[2]
        h = (1.0e-9, 1.5e-9, 2.0e-9)
        top = np.array([(e - 1) * d for e, d in zip(ext, h)])
        st.update(ctx=emcgpu.Context(precision=emcgpu.FP64), ext=ext, h=h,
                  pos=rs.rand(case["particles"], 3) * top * (1.0 - 1e-9),
                  E=[1e6 * rs.standard_normal(nn) for _ in range(3)])
        return st
    ctx = emcgpu.Context(precision=emcgpu.FP64 if kind == "poisson" else _precision(case),
                         n_instances=case["instances"] if kind == "sweep" else 1)
    st["ctx"] = ctx
    if kind == "bulk":
        ctx.setup(0, _bulk_spec(case))
        ctx.resize([case["particles"]])
        if case["read"] == "positions":
            ctx.set_box(0, BOX)
        # carriers at the temperature that the field holds them at
        ctx.init_particles(0, seed, case["t_init"])
        ctx.reserve(BULK_DT, case["steps"])
    elif kind == "sweep":
        inst = _sweep(case, seed)
        for i, (m, _) in enumerate(inst):
            ctx.setup(i, m)
        ctx.resize([n for _, n in inst])
        for i, (m, _) in enumerate(inst):
            ctx.init_particles(i, seed, _sweep_t_init(m))
        ctx.reserve(BULK_DT, case["steps"])
    elif kind == "cooling":
        ctx.setup(0, _cooling_spec(case))
        ctx.resize([case["particles"]])
        ctx.init_particles_energy(0, seed, 0.5, 0.05)
        if case["screened"]:
            ctx.update_screening(0)
        ctx.reserve(COOLING_DT, case["steps"])
    elif kind == "device":
        ctx.setup(0, workloads.MODELS_DEVICE["device_para"])
        ctx.device_setup(_device_dict(case), pm=PM_NAMES[case["pm"]], poisson_tol=1e-10, poisson_max_iter=50)
        ctx.device_init(seed)
    elif kind == "poisson":
        ctx.setup(0, workloads.MODELS_DEVICE["device_para"])
        ctx.device_setup(_mosfet_dict(case, seed), pm=emcgpu.PM_CIC, poisson_tol=1e-10, poisson_max_iter=50)
        # the charge-neutral guess, as the simulation starts from it
        st["guess"] = np.arcsinh(0.5 * ctx.device_grids()["doping"] / workloads.SI_NI)
    ctx.synchronize()
    return st


BOX = (200e-9, 100e-9, 150e-9)


def _sweep_t_init(m):
    return m["T"] + 25.0 * m["field_kvcm"]


def _padded(a, case):
    """rows of the ensemble, whose size varies from seed to seed, filled up with zeros"""
    out = np.zeros((case["particles"] * 5 // 4,) + a.shape[1:], dtype=a.dtype)
    out[:a.shape[0]] = a
    return out


# ---------------------------------------------------------------------------
# one pass
#
# The averages of every step are what emcgpu_step hands out; the carriers themselves stay on the GPU from
# call to call, and a program copies them to the host once per run, if at all.  The cases of the sizes for
# which the examples write particle files do that at the end of the pass; the ones of millions of carriers
# return what the program reads after each call, which every carrier enters at every step.
# ---------------------------------------------------------------------------
def run(st):
    case, ctx, seed = st["case"], st["ctx"], st["seed"]
    kind = case["kind"]
    if kind in ("bulk", "sweep"):
        ctx.step(BULK_DT, case["steps"], seed=seed, step0=st["at"], graph=case["graph"])
        st["at"] += case["steps"]
        if kind == "sweep":
            av = [ctx.averages(i) for i in range(case["instances"])]
            return {k: np.stack([a[k] for a in av]) for k in av[0]}
        out = dict(ctx.averages(0))
        if case["read"] in ("state", "positions"):
            out["particles"] = ctx.get_particles(0)
        if case["read"] == "positions":
            out["pos"] = ctx.get_positions(0)
        return out
    if kind == "cooling":
        ctx.step(COOLING_DT, case["steps"], seed=seed, step0=st["at"], graph=case["graph"])
        st["at"] += case["steps"]
        out = dict(ctx.averages(0))
        out["history"] = ctx.bath_history(0, 0)
        out["bath"] = {k: float(v) if k != "nq" else v for k, v in ctx.get_bath(0, 0).items()}
        out["energy"] = ctx.bath_energy(0, 0)
        if case["screened"]:
            out["qs2"] = float(ctx.get_screening(0))
        return out
    if kind == "device":
        rec = ctx.device_step(DEVICE_DT, case["steps"], seed=seed, graph=case["graph"])
        out = ctx.device_fields()
        out["E"] = np.stack([out.pop("ex"), out.pop("ey")])
        # the contact currents that the simulation reports: charge through each contact up to every step
        net = rec["exits"].astype(np.float64) + rec["deleted"] - rec["injected"]
        t = DEVICE_DT * np.arange(1, case["steps"] + 1)[:, None]
        out["current"] = Q * np.cumsum(net, axis=0) / t
        out["carriers"] = rec["n_particles"].astype(np.float64)
        if case["particles"] <= 100_000 and case["precision"] == "f64":
            out["particles"] = {k: _padded(v, case) for k, v in ctx.device_get_particles().items()}
        return out
    if kind == "poisson":
        pot, _, _ = ctx.poisson(st["guess"], equilibrium=True)
        ex, ey = ctx.efield(pot)
        return dict(pot=pot, ex=ex, ey=ey)
    pm = PM_NAMES[case["pm"]]
    grid = ctx.deposit3(st["ext"], st["h"], st["pos"], pm=pm)
    force = ctx.interpolate3(st["ext"], st["h"], st["E"][0], st["E"][1], st["E"][2], st["pos"], pm=pm)
    return dict(grid=grid, force=force)


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far a correct result may be off
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "mesh3":
        nn = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": case["particles"] * (24.0 * 2 + 24.0) + nn * 8.0 * 5, "flops": case["particles"] * 150.0}
    if kind == "poisson":
        nn = case["nx"] * case["ny"]
        # eight Newton systems of a five-point operator, each the work of a few tens of sweeps
        return {"bytes": nn * 8.0 * 5, "flops": nn * 8 * 30 * 12.0}
    word = 4 if case["precision"] == "f32" else 8
    if kind == "sweep":
        n = sum(c for _, c in _sweep(case, 0))
    else:
        n = case["particles"]
    state = 5 * word + 4
    if kind == "device":
        # the deposit needs the whole ensemble at every step: the state moves through memory each time
        return {"bytes": case["steps"] * n * (2.0 * (state + 2 * word) + 4), "flops": case["steps"] * n * 80.0}
    if case.get("read") == "positions":
        state += 3 * word
    once = 2.0 * n * state
    if case.get("read") in ("state", "positions"):
        once += n * 48.0 + (n * 24.0 if case["read"] == "positions" else 0.0)
    if kind == "cooling":
        # the bath couples the carriers after every step
        return {"bytes": case["steps"] * 2.0 * n * state, "flops": case["steps"] * n * 120.0}
    return {"bytes": once, "flops": case["steps"] * n * 100.0}


def tolerance(case):
    """Four times what the library's results are off ``exact`` by, rounded up.

    In FP64 every carrier follows the exact history, so only sums and roundings differ.  In FP32 a draw that
    falls within rounding of a decision sends a carrier down another path, about one in 2e7 carrier steps:
    averages over few carriers then move by that carrier's share, states by its whole state."""
    kind = case["kind"]
    if kind == "mesh3":
        return {"rel": 1e-13}
    if kind == "poisson":
        return {"rel": 1e-9}  # the solver's stopping rule, not rounding, sets it
    single = case["precision"] == "f32"
    if kind == "device":
        if not single:
            return {"rel": 1e-9}  # atomic deposits: another order of the sums from run to run
        # one carrier more or less at a contact renumbers those injected after it
        return {"rel": 0.01 if case["particles"] >= 1_000_000 else 0.03, "max": 0.999}
    if kind == "cooling":
        # no field: the mean velocity is what is left of the carriers' cancelling ones
        return {"rel": 6e-3 if single else 1e-8}
    if not single:
        return {"rel": 1e-11}
    if kind == "sweep":
        return {"rel": 2e-4, "differ": 1e-3}
    if case["read"] != "averages":
        return {"rel": 0.015, "max": 0.999, "differ": 1e-3}
    return {"rel": min(0.02, max(5e-5, 100.0 / case["particles"]))}


# ---------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------
DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64, I64 = torch.float64, torch.int64
M32 = 0xFFFFFFFF


def _t(x, dtype=F64):
    return torch.as_tensor(x, dtype=dtype, device=DEV)


def _philox(c, seed):
    """Philox-4x32-10 on int64 tensors holding 32-bit words."""
    k0, k1 = seed & M32, (seed >> 32) & M32
    c0, c1, c2, c3 = c
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = (((p1 >> 32) & M32) ^ c1 ^ k0, p1 & M32, ((p0 >> 32) & M32) ^ c3 ^ k1, p0 & M32)
        k0, k1 = (k0 + 0x9E3779B9) & M32, (k1 + 0xBB67AE85) & M32
    return c0, c1, c2, c3


def _unit(w):
    return ((w >> 8) | 1).to(F64) * 2.0 ** -24


def _stream(j, step, pid, inst, seed):
    """uniform j of a (step, particle) stream"""
    return _unit(_philox((torch.full_like(pid, j >> 2), torch.full_like(pid, step), pid, inst), seed)[j & 3])


def _gamma(v, E):
    return E * (1 + v["alpha"] * E)


def _valley(v):
    aniso = v["kind"] in (2, 3)
    m = [x * ME for x in v["mass"]]
    alpha = v.get("alpha", 0.0) if v["kind"] in (1, 3) else 0.0
    if aniso:
        dos = np.cbrt(v["mass"][0] * v["mass"][1] * v["mass"][2]) * ME
        cond = 3.0 / sum(1.0 / x for x in m)
        vogt = [math.sqrt(cond / x) for x in m]
    else:
        dos = cond = m[0]
        vogt = [1.0] * 3
    metric = []
    for s in range(v["deg"]):
        if aniso:
            R = np.array(v["axes"][s], dtype=np.float64)
            R = R / np.linalg.norm(R, axis=1, keepdims=True)
            metric.append(R.T @ np.diag(vogt) @ R)
        else:
            metric.append(np.eye(3))
    return dict(alpha=alpha, dos=dos, cond=cond, bottom=v.get("bottom", 0.0), deg=v["deg"], metric=metric,
                c2=HBAR * HBAR * 1e18 / (2.0 * cond * Q), cv=HBAR * 1e9 / cond)


class Model:
    """Valleys, scatter tables and final states of one or more instances; the valleys of all instances share
    one index, so a sweep is one ensemble."""

    def __init__(self, specs, temps):
        self.specs, self.temps = specs, temps
        self.nl = specs[0]["n_levels"]
        self.dE = specs[0]["max_energy"] / self.nl
        self.valleys, self.first, mechs = [], [], []
        for spec in specs:
            base = len(self.valleys)
            self.first.append(base)
            self.valleys += [_valley(v) for v in spec["valleys"]]
            mechs += [[] for _ in spec["valleys"]]
            for m in spec["mechs"]:
                mechs[base + m["valley"]].append(dict(m, fv=base + m.get("final", m["valley"])))
        nv, nt = len(self.valleys), max(len(m) for m in mechs)
        self.mechs, self.nt = mechs, nt
        self.n_tab = _t([len(m) for m in mechs], I64)
        deg = max(v["deg"] for v in self.valleys)
        self.deg = deg
        par = lambda k: _t([v[k] for v in self.valleys])
        self.alpha, self.c2, self.cv, self.vdeg = par("alpha"), par("c2"), par("cv"), par("deg").to(I64)
        self.metric = torch.zeros(nv, deg, 3, 3, dtype=F64)
        self.accel, self.wdir = torch.zeros(nv, deg, 3, dtype=F64), torch.zeros(nv, deg, 3, dtype=F64)
        inst_of = [i for i, s in enumerate(specs) for _ in s["valleys"]]
        self.inst_of = inst_of
        for k, v in enumerate(self.valleys):
            d = np.array(specs[inst_of[k]]["field_dir"], dtype=np.float64)
            d = d / np.linalg.norm(d)
            F = d * specs[inst_of[k]]["field_kvcm"] * 1e5 * -Q
            for s, met in enumerate(v["metric"]):
                self.metric[k, s] = torch.as_tensor(met)
                self.accel[k, s] = torch.as_tensor(met @ F / HBAR * 1e-24)
                self.wdir[k, s] = torch.as_tensor(met @ d)
        self.metric, self.accel, self.wdir = self.metric.to(DEV), self.accel.to(DEV), self.wdir.to(DEV)
        # final states: 0 elastic, 1 intervalley, 2 polar, 3 screened polar
        self.kind, self.shift, self.z, self.fv, self.hot, self.qres = (np.zeros((nv, nt)) for _ in range(6))
        fsub = np.zeros((nv, nt, 8, 8))
        for k in range(nv):
            for j, m in enumerate(mechs[k]):
                a = m["kind"]
                self.fv[k, j], self.z[k, j] = k, 1
                if 1 <= a <= 4:
                    delta = self.valleys[m["fv"]]["bottom"] - self.valleys[k]["bottom"]
                    self.kind[k, j], self.fv[k, j], self.z[k, j] = 1, m["fv"], len(m["fmap"][0])
                    self.shift[k, j] = m["hw"] - delta if a in (1, 3) else -(m["hw"] + delta)
                    for s, row in enumerate(m["fmap"]):
                        fsub[k, j, s, :len(row)] = row
                elif a >= 5:
                    self.kind[k, j] = 3 if a >= 9 else 2
                    self.shift[k, j] = m["hw"] if a in (5, 7, 9, 11) else -m["hw"]
                    self.hot[k, j] = a in (7, 8, 11, 12)
                    self.qres[k, j] = a in (11, 12)
        self.emits = _t(self.shift < 0, I64)
        self.kind, self.z, self.fv, self.hot, self.qres = (_t(x, I64) for x in (self.kind, self.z, self.fv,
                                                                               self.hot, self.qres))
        self.shift, self.fsub = _t(self.shift), _t(fsub, I64)
        self.E = (torch.arange(1, self.nl + 1, dtype=F64)) * self.dE
        self.bath = None

    def build(self, qs2=0.0, bath=None):
        """the normalised cumulative tables and tau0 [fs] of every valley"""
        nv = len(self.valleys)
        cum = torch.full((nv, self.nl, self.nt), math.inf, dtype=F64)
        tau0 = torch.full((nv,), 2.0, dtype=F64)
        for k, v in enumerate(self.valleys):
            if not self.mechs[k]:
                continue
            r = torch.stack([self._rate(v, m, self.temps[self.inst_of[k]], self.specs[self.inst_of[k]], qs2, bath)
                             for m in self.mechs[k]], dim=1)
            c = torch.cumsum(r, dim=1)
            mx = c[:, -1].max()
            cum[k, :, :r.shape[1]] = c / mx
            tau0[k] = 1e15 / mx
        self.cum, self.tau0, self.qs2, self.bath = cum.to(DEV), tau0.to(DEV), qs2, bath

    def _rate(self, v, m, T, spec, qs2, bath):
        E, a = self.E, m["kind"]
        bose = lambda hw: 1.0 / (math.exp(Q * hw / (KB * T)) - 1.0)
        rho = spec.get("rho", 2329.0)
        if a == 0:
            C = (math.sqrt(2 * Q) * (m["sigma"] * Q) ** 2 * KB * T /
                 (math.pi * rho * spec.get("v_sound", 9040.0) ** 2 * HBAR ** 4))
            return C * v["dos"] ** 1.5 * torch.sqrt(_gamma(v, E)) * (2 * v["alpha"] * E + 1)
        ab = a in (1, 3, 5, 7, 9, 11)
        hw = m["hw"]
        if a <= 4:
            f = self.valleys[m["fv"]]
            Ef = E + (hw if ab else -hw) - (f["bottom"] - v["bottom"])
            ok = Ef > 0
            Ep = torch.where(ok, Ef, torch.zeros_like(Ef))
            N = bose(hw) + (0 if ab else 1)
            z, g = len(m["fmap"][0]), torch.sqrt(_gamma(f, Ep)) * (2 * f["alpha"] * Ep + 1)
            if a <= 2:
                C = z * math.sqrt(Q) * (m["defpot"] / HBAR) ** 2 * Q / (math.pi * rho * hw * math.sqrt(2)) * N
                r = C * f["dos"] ** 1.5 * g
            else:
                C = z * math.sqrt(2) * Q ** 2.5 * m["defpot"] ** 2 / (math.pi * rho * HBAR ** 4 * hw) * N
                r = C * f["dos"] ** 2.5 * g * (_gamma(v, E) + _gamma(f, Ep))
            return torch.where(ok, r, torch.zeros_like(r))
        meff = m["mrel"] * ME
        C = (Q * Q * (hw * Q / HBAR) * meff / (4 * math.pi * HBAR ** 2) *
             (1 / m["eps_hi"] - 1 / m["eps_lo"]) / EPS0)
        ok = (E > 0) if ab else (E > hw)
        Ef = torch.where(ok, E + (hw if ab else -hw), E)
        kI, kF = torch.sqrt(2 * meff * _gamma(v, E) * Q) / HBAR, torch.sqrt(2 * meff * _gamma(v, Ef) * Q) / HBAR
        N = bose(hw)
        if a in (7, 8):
            N = bath.mean()
        elif a >= 11:
            N = bath.window((kI - kF).abs(), kI + kF)
        if a >= 9 and qs2 > 0:
            ln = 0.5 * torch.log(((kI + kF) ** 2 + qs2) / ((kI - kF) ** 2 + qs2))
        else:
            ln = torch.log((kI + kF) / (kI - kF).abs())
        r = C * (N if ab else N + 1) / kI * ln
        return torch.where(ok & (Ef > 0), r, torch.zeros_like(r))

    # -- kinematics (k in 1/nm, E in eV, t in fs) --
    def energy(self, k, v):
        g = self.c2[v] * (k * k).sum(1)
        return 2 * g / (1 + torch.sqrt(1 + 4 * self.alpha[v] * g))

    def normk(self, E, v):
        return torch.sqrt(E * (1 + self.alpha[v] * E) / self.c2[v])

    def scatter(self, k, E, v, s, u):
        """one event of each carrier given; (k, E, v, s, real) after it, and q of bath events"""
        x = torch.floor(E / self.dE) - 1
        lev = torch.where(x == -1, torch.zeros_like(x), torch.where((x >= 0) & (x <= self.nl - 1), x,
                                                                   torch.full_like(x, self.nl - 1))).to(I64)
        row = self.cum[v, lev]
        t = (row <= u[0][:, None]).sum(1)
        real = torch.nonzero(t < self.n_tab[v])[:, 0]
        k, E, v, s = k.clone(), E.clone(), v.clone(), s.clone()
        if real.numel() == 0:
            return k, E, v, s, real
        t = t[real]
        low = torch.where(t > 0, row[real].gather(1, (t - 1).clamp(min=0)[:, None])[:, 0], torch.zeros_like(E[real]))
        up = row[real].gather(1, t[:, None])[:, 0]
        kind = self.kind[v[real], t]
        for which in (0, 1, 2, 3):
            at = torch.nonzero(kind == which)[:, 0]
            if at.numel() == 0:
                continue
            i, j = real[at], t[at]
            vi, ua, ub = v[i], u[1][i], u[2][i]
            if which <= 1:
                if which == 0:
                    n = torch.sqrt((k[i] * k[i]).sum(1))
                else:
                    z = self.z[vi, j]
                    zi = ((u[0][i] - low[at]) / (up[at] - low[at]) * z).to(I64)
                    s[i] = self.fsub[vi, j, s[i], torch.minimum(zi, z - 1)]
                    v[i] = self.fv[vi, j]
                    E[i] = E[i] + self.shift[vi, j]
                    n = self.normk(E[i], v[i])
                k[i] = self._random(n, ua, ub)
                continue
            k0, ei = k[i], E[i]
            ef = ei + self.shift[vi, j]
            E[i] = ef
            kn = self.normk(ef, vi)
            if which == 2:
                d = torch.sqrt(ei) - torch.sqrt(ef)
                f = 2 * torch.sqrt(ei * ef) / d / d
                ct = (1 + f - (1 + 2 * f) ** ua) / f
            else:
                ki = self.normk(ei, vi)
                B = 2 * ki * kn
                if bool(self.qres[vi[0], j[0]]):
                    q = self.bath.sample((ki - kn).abs(), ki + kn, self.emits[vi, j] > 0, ua)
                    ct = (ki * ki + kn * kn - q * q) / B
                else:
                    qn = self.qs2 * 1e-18
                    num, den = (ki - kn) ** 2 + qn, ki * ki + kn * kn + qn + B
                    ct = (ki * ki + kn * kn + qn - den * (num / den) ** ua) / B
            ct = ct.clamp(-1.0, 1.0)
            kk = self._about(k0, ct, ub)
            nk = torch.sqrt((kk * kk).sum(1))
            k[i] = kk * (kn / nk)[:, None]
            if bool(self.hot.any()):
                dk = k[i] - k0
                self.bath.record(torch.sqrt((dk * dk).sum(1)), self.emits[vi, j] > 0)
        return k, E, v, s, real

    @staticmethod
    def _random(n, uphi, ucos):
        ct = 1 - 2 * ucos
        st, phi = torch.sqrt(1 - ct * ct), 2 * math.pi * uphi
        return torch.stack([n * st * torch.cos(phi), n * st * torch.sin(phi), n * ct], 1)

    @staticmethod
    def _about(k, ct, uphi):
        kxy = torch.sqrt(k[:, 0] ** 2 + k[:, 1] ** 2)
        nk = torch.sqrt(kxy ** 2 + k[:, 2] ** 2)
        c0, s0 = k[:, 2] / nk, kxy / nk
        cf, sf = k[:, 0] / kxy, k[:, 1] / kxy
        st, phi = torch.sqrt(1 - ct * ct), 2 * math.pi * uphi
        x, y, z = nk * st * torch.cos(phi), nk * st * torch.sin(phi), nk * ct
        return torch.stack([x * cf * c0 - y * sf + z * cf * s0, x * sf * c0 + y * cf + z * sf * s0,
                            -x * s0 + z * c0], 1)

    def event(self, e, step, pid, inst, seed, k, E, v, s):
        w = _philox((torch.full_like(pid, e), torch.full_like(pid, step), pid, inst), seed)
        u = [_unit(x) for x in w]
        k, E, v, s, real = self.scatter(k, E, v, s, u)
        ut = u[3] * (1 - 1e-6) + 1e-6
        return k, E, v, s, -torch.log(ut) * self.tau0[v], real


class Bath:
    """LO phonons on wavevector bins, decaying into an acoustic reservoir"""

    def __init__(self, b, T):
        self.b, self.T, self.nb = b, T, b["n_bins"]
        bose = lambda hw: 1.0 / (math.exp(Q * hw / (KB * T)) - 1.0)
        self.n0, self.ac0 = bose(b["hw"]), bose(b["ac_hw"])
        self.ac = self.ac0
        self.q = (torch.arange(self.nb, dtype=F64) + 0.5) * b["dq"]
        self.n = torch.full((self.nb,), self.n0, dtype=F64)
        self.clear()

    def clear(self):
        self.em, self.ab = torch.zeros(self.nb, dtype=F64), torch.zeros(self.nb, dtype=F64)

    def record(self, q, emits):
        i = (q / (self.b["dq"] * 1e-9)).to(I64).clamp(max=self.nb - 1)
        self.em += torch.bincount(i[emits], minlength=self.nb).to(F64).cpu()
        self.ab += torch.bincount(i[~emits], minlength=self.nb).to(F64).cpu()

    def mean(self):
        w = self.q ** 2
        return float((w * self.n).sum() / w.sum())

    def windows(self, qs2):
        w = self.q / (self.q ** 2 + qs2)
        zero = torch.zeros(1, dtype=F64)
        self.cw, self.cwn = torch.cat([zero, torch.cumsum(w, 0)]), torch.cat([zero, torch.cumsum(w * self.n, 0)])

    def window(self, lo, hi):
        dq = self.b["dq"]
        a, b = torch.floor(lo / dq).to(I64).clamp(0, self.nb), torch.ceil(hi / dq).to(I64).clamp(0, self.nb)
        w = self.cw[b] - self.cw[a]
        ok = (b > a) & (w > 0)
        return torch.where(ok, (self.cwn[b] - self.cwn[a]) / torch.where(ok, w, torch.ones_like(w)),
                           torch.full_like(w, self.mean()))

    def sample(self, lo, hi, emits, u):
        dq = self.b["dq"] * 1e-9
        a, b = torch.floor(lo / dq).to(I64).clamp(0, self.nb), torch.ceil(hi / dq).to(I64).clamp(0, self.nb)
        out = lo.clone()
        for em in (False, True):
            at = torch.nonzero((emits == em) & (b > a))[:, 0]
            if at.numel() == 0:
                continue
            S = (self.cwn + self.cw if em else self.cwn).to(lo.device)
            s0, s1 = S[a[at]], S[b[at]]
            target = s0 + u[at] * (s1 - s0)
            i = (torch.searchsorted(S, target, right=True) - 1)
            i = torch.minimum(torch.maximum(i, a[at]), b[at] - 1)
            q = (i.to(F64) + (target - S[i]) / (S[i + 1] - S[i])) * dq
            out[at] = torch.maximum(torch.minimum(q, hi[at]), lo[at])
        return out

    def update(self, dt):
        b = self.b
        target = self.n0
        if self.ac > self.ac0:
            t = Q * b["ac_hw"] / (KB * math.log(1 + 1 / self.ac))
            target = 1.0 / (math.exp(Q * b["hw"] / (KB * t)) - 1.0)
        dph = self.q ** 2 * b["dq"] * b["volume"] / (2 * math.pi ** 2)
        old = self.n
        new = (old + (self.em - self.ab) / dph - dt / b["tau_lo"] * (old - target)).clamp(min=0.0)
        src = float((self.q ** 2 * (old - target)).sum() / (self.q ** 2).sum())
        self.ac = max(self.ac + dt * src / b["tau_lo"] - dt * (self.ac - self.ac0) / b["tau_ac"], self.ac0)
        energy = [float((self.em - self.ab).sum()), float((dph * (new - old)).sum()),
                  float((dph * (dt / b["tau_lo"]) * (old - target)).sum())]
        self.n = new
        self.clear()
        return [b["hw"] * x for x in energy]


class Ensemble:
    """carriers of all instances of a model: k [1/nm], E [eV], tau [fs], valley, subvalley"""

    def __init__(self, model, counts, seed, vts=None, mean=0.0, sigma=0.0, box=None):
        self.m, self.seed, self.box = model, seed, box
        self.at = torch.cumsum(torch.tensor([0] + list(counts)), 0)
        self.pid = torch.cat([torch.arange(n, device=DEV) for n in counts])
        self.inst = torch.cat([torch.full((n,), i, dtype=I64, device=DEV) for i, n in enumerate(counts)])
        u = lambda j: _stream(j, M32, self.pid, self.inst, seed)
        lo, sc = 1e-6, 1 - 1e-6
        nv = _t([len(s["valleys"]) for s in model.specs], I64)[self.inst]
        first = _t(model.first, I64)[self.inst]
        self.v = first + torch.minimum(torch.floor(nv * (u(0) * sc + lo)).to(I64), nv - 1)
        deg = model.vdeg[self.v]
        self.s = torch.minimum(torch.floor(deg * (u(1) * sc + lo)).to(I64), deg - 1)
        ue = u(2) * sc + lo
        if mean > 0:
            E = mean + sigma * torch.sqrt(-2 * torch.log(ue)) * torch.cos(2 * math.pi * u(6))
            self.E = E.abs()
        else:
            self.E = -1.5 * _t(vts)[self.inst] * torch.log(ue)
        self.k = model._random(model.normk(self.E, self.v), u(3), u(4))
        self.tau = -torch.log(u(5) * sc + lo) * model.tau0[self.v]
        self.pos = torch.stack([u(8 + d) * box[d] * 1e9 for d in range(3)], 1) if box else None

    def drift(self, t, k, E, v, s, pos):
        m = self.m
        k1 = k + m.accel[v, s] * t[:, None]
        E1 = m.energy(k1, v)
        if pos is not None:
            mid = torch.einsum("nij,nj->ni", m.metric[v, s], 0.5 * (k + k1))
            x = pos + mid * (m.cv[v] * t * 1e-6 / (1 + 2 * m.alpha[v] * E1))[:, None]
            box = _t([b * 1e9 for b in self.box])
            pos = torch.where(x < 0, x + box, torch.where(x > box, x - box, x))
        return k1, E1, pos

    def step(self, dt, step):
        """one step; events and real events per instance"""
        m, n_inst = self.m, len(self.m.specs)
        ev, re = torch.zeros(n_inst, dtype=F64, device=DEV), torch.zeros(n_inst, dtype=F64, device=DEV)
        t = torch.minimum(self.tau, torch.full_like(self.tau, dt))
        self.k, self.E, self.pos = self.drift(t, self.k, self.E, self.v, self.s, self.pos)
        rem = dt - self.tau
        i = torch.nonzero(rem > 0)[:, 0]
        rem, e = rem[i], 0
        while i.numel():
            k, E, v, s, nt, real = m.event(e, step, self.pid[i], self.inst[i], self.seed, self.k[i], self.E[i],
                                           self.v[i], self.s[i])
            ev += torch.diff(torch.searchsorted(i, self.at.to(DEV)))
            re += torch.diff(torch.searchsorted(i[real], self.at.to(DEV)))
            pos = self.pos[i] if self.pos is not None else None
            k, E, pos = self.drift(torch.minimum(rem, nt), k, E, v, s, pos)
            self.k[i], self.E[i], self.v[i], self.s[i] = k, E, v, s
            self.tau[i] += nt
            if pos is not None:
                self.pos[i] = pos
            rem = rem - nt
            go = rem > 0
            i, rem, e = i[go], rem[go], e + 1
        self.tau -= dt
        return ev, re

    def sums(self, ev, re):
        """the step's averages in the layout of Context.averages, an instance per row; the carriers of an
        instance are contiguous"""
        m = self.m
        vel = m.cv[self.v] * (self.k * m.wdir[self.v, self.s]).sum(1) / (1 + 2 * m.alpha[self.v] * self.E)
        per = len(m.valleys) // len(m.specs)
        rows = []
        for i in range(len(m.specs)):
            a, b = self.at[i], self.at[i + 1]
            E, V, v, sub = self.E[a:b], vel[a:b], self.v[a:b] - m.first[i], self.s[a:b]
            for k in range(per):
                in_k = v == k
                rows += [(E * in_k).sum(), (V * in_k).sum()] + [(in_k & (sub == j)).sum().to(F64)
                                                                for j in range(m.deg)]
        r = torch.stack(rows).view(len(m.specs), per, 2 + m.deg)
        sE, sV, sub = r[:, :, 0], r[:, :, 1], r[:, :, 2:]
        cnt = sub.sum(2)
        n = (self.at[1:] - self.at[:-1]).to(F64)[:, None].to(DEV)
        one, zero = cnt.clamp(min=1), torch.zeros_like(cnt)
        return dict(avgE=torch.where(cnt > 0, sE / one, zero), avgV=torch.where(cnt > 0, sV / one, zero),
                    occ=cnt / n, sub_occ=sub / n[:, :, None], events=ev, real_events=re, sumE=sE, sumV=sV,
                    count=cnt)

    def particles(self):
        return dict(k=(self.k / 1e-9).reshape(-1), E=self.E, tau=self.tau / 1e15, valley=None, sub=None)


def _exact_bulk(case, seed):
    sweep = case["kind"] == "sweep"
    if sweep:
        inst = _sweep(case, seed)
        specs, counts = [s for s, _ in inst], [n for _, n in inst]
        vts = [KB / Q * _sweep_t_init(s) for s in specs]
    else:
        specs, counts, vts = [_bulk_spec(case)], [case["particles"]], [KB / Q * case["t_init"]]
    m = Model(specs, [s["T"] for s in specs])
    m.build(specs[0].get("screening", {}).get("qs2", 0.0))
    ens = Ensemble(m, counts, seed, vts, box=BOX if case.get("read") == "positions" else None)
    got = [ens.sums(*ens.step(BULK_DT * 1e15, s)) for s in range(case["steps"])]
    if sweep:
        return {k: torch.stack([g[k] for g in got], 1) for k in got[0]}
    out = {k: torch.stack([g[k][0] for g in got]) for k in got[0]}
    if case["read"] in ("state", "positions"):
        out["particles"] = ens.particles()
    if case["read"] == "positions":
        out["pos"] = ens.pos * 1e-9
    return out


def _exact_cooling(case, seed):
    spec = _cooling_spec(case)
    m = Model([spec], [spec["T"]])
    bath = Bath(spec["baths"][0], spec["T"])
    n = case["particles"]

    def qs2_of(E, v):
        if not case["screened"]:
            return 0.0
        scr = spec["screening"]
        ts = 2.0 * float(E[v == 0].mean()) * Q / (3.0 * KB)
        return n / scr["volume"] * Q * Q / (scr["eps"] * EPS0 * KB * ts)

    # the carriers start with free-flight times of the tables at the starting screening
    qs2 = spec["screening"]["qs2"] if case["screened"] else 0.0
    bath.windows(qs2)
    m.build(qs2, bath)
    ens = Ensemble(m, [n], seed, mean=0.5, sigma=0.05)
    qs2 = qs2_of(ens.E, ens.v)
    bath.windows(qs2)
    m.build(qs2, bath)
    got, hist, energy = [], [], []
    for s in range(case["steps"]):
        got.append(ens.sums(*ens.step(COOLING_DT * 1e15, s)))
        qs2 = qs2_of(ens.E, ens.v)
        energy.append(bath.update(COOLING_DT))
        hist.append(bath.mean())
        bath.windows(qs2)
        m.build(qs2, bath)
    out = {k: torch.stack([g[k][0] for g in got]) for k in got[0]}
    out["history"], out["energy"] = _t(hist), _t(energy)
    b = spec["baths"][0]
    t_ac = Q * b["ac_hw"] / (KB * math.log(1 + 1 / bath.ac))
    out["bath"] = dict(nq=bath.n, mean=bath.mean(), n_ac=bath.ac, n_to=None, n0=bath.n0, t_ac=t_ac, t_to=None)
    if case["screened"]:
        out["qs2"] = float(qs2)
    return out


class Grid2:
    """geometry, boundary conditions and the discrete Poisson equation of a 2-D device"""

    def __init__(self, dev):
        self.dev, self.h = dev, dev["spacing"]
        self.nx, self.ny = (int(round(dev["max_pos"][d] / self.h[d])) + 1 for d in range(2))
        nx, ny = self.nx, self.ny
        self.vt = KB / Q * dev["T"]
        self.debye = math.sqrt(EPS0 * dev["eps_r"] * self.vt / Q / dev["ni"])
        self.volume = self.h[0] * self.h[1] * dev["width"]
        at = lambda x, d: int(math.floor(x / self.h[d] + 0.5))
        dop = np.full((ny, nx), dev["ni"])
        for lo, hi, n in dev["doping"]:
            dop[at(lo[1], 1):at(hi[1], 1) + 1, at(lo[0], 0):at(hi[0], 0) + 1] = n
        self.doping = dop
        lines = [np.full(ny, -1), np.full(ny, -1), np.full(nx, -1), np.full(nx, -1)]
        node = lambda b, s: ((0, s), (nx - 1, s), (s, 0), (s, ny - 1))[b]
        for c, ct in enumerate(dev["contacts"]):
            b = ct[0]
            for s in range(at(ct[2], 1 if b < 2 else 0), at(ct[3], 1 if b < 2 else 0) + 1):
                lines[b][s] = c
                x, y = node(b, s)
                if len(ct) == 4:
                    for bb, on, o in ((0, x == 0, y), (1, x == nx - 1, y), (2, y == 0, x), (3, y == ny - 1, x)):
                        if on:
                            lines[bb][o] = c
        self.lines = lines
        # the contact of a node is that of the first boundary it lies on
        self.contact = np.full((ny, nx), -1)
        for b in (3, 2, 1, 0):
            for s in range(len(lines[b])):
                x, y = node(b, s)
                self.contact[y, x] = lines[b][s]
        gate = np.array([len(ct) == 7 for ct in dev["contacts"]] + [False])
        self.ohmic = (self.contact >= 0) & ~gate[self.contact]
        # the edge factor of a node's cell
        self.half = np.ones((ny, nx))
        self.half[:, 0] *= 0.5
        self.half[:, -1] *= 0.5
        self.half[0] *= 0.5
        self.half[-1] *= 0.5

    def solve(self, pot, conc, applied, tol=1e-13):
        """Newton on the five-point equations, each system by block elimination over the rows"""
        nx, ny, dev = self.nx, self.ny, self.dev
        hn = [self.h[0] / self.debye, self.h[1] / self.debye]
        hf, hp = [hn[1] / hn[0], hn[0] / hn[1]], hn[0] * hn[1]
        dop = self.doping / dev["ni"]
        pot = pot.copy()
        shift, rhs = np.zeros((ny, nx)), np.zeros((ny, nx))
        node = lambda b, s: ((0, s), (nx - 1, s), (s, 0), (s, ny - 1))[b]
        for b in range(4):
            for s, c in enumerate(self.lines[b]):
                if c >= 0 and len(dev["contacts"][c]) == 7:
                    ct, (x, y) = dev["contacts"][c], node(b, s)
                    g = 2 * (ct[4] / dev["eps_r"]) / (ct[5] / self.debye) * hf[b // 2] * hn[b // 2]
                    shift[y, x] += g
                    rhs[y, x] += g * (ct[6] / self.vt + (ct[1] / self.vt if applied else 0.0))
        volts = np.array([ct[1] for ct in dev["contacts"]] + [0.0]) / self.vt
        fixed = self.ohmic
        bi = np.arcsinh(0.5 * dop)
        pot[fixed] = (bi + (volts[self.contact] if applied else 0.0))[fixed]
        for it in range(200):
            p = np.exp(-pot)
            n = conc if conc is not None else 1.0 / p
            F = hp * (p - n + dop) + rhs - shift * pot - 2 * (hf[0] + hf[1]) * pot
            L = np.pad(pot, 1, mode="reflect")
            F += hf[0] * (L[1:-1, :-2] + L[1:-1, 2:]) + hf[1] * (L[:-2, 1:-1] + L[2:, 1:-1])
            F[fixed] = 0.0
            diag = 2 * (hf[0] + hf[1]) + shift + hp * (p + (n if conc is None else 0.0))
            # blocks over the longer extent
            d = self._rows(diag, hf, F, ~fixed) if nx <= ny else self._rows(diag.T, hf[::-1], F.T, ~fixed.T).T
            step = min(1.0, 3.0 / max(np.abs(d).max(), 1e-300)) if it < 60 else 1.0
            pot = pot + step * d
            if np.abs(d).max() < tol * max(1.0, np.abs(pot).max()):
                break
        return pot

    @staticmethod
    def _rows(diag, hf, F, free):
        ny, nx = diag.shape
        lo, up = np.full(nx, -hf[0]), np.full(nx, -hf[0])
        lo[-1], up[0] = -2 * hf[0], -2 * hf[0]
        inv, y = [None] * ny, [None] * ny
        for j in range(ny):
            A = np.diag(diag[j]) + np.diag(lo[1:], -1) + np.diag(up[:-1], 1)
            A = np.where(free[j][:, None], A, np.eye(nx))
            b = F[j].copy()
            if j:
                w = -hf[1] * (2 if j == ny - 1 else 1) * free[j]
                u = -hf[1] * (2 if j - 1 == 0 else 1) * free[j - 1]
                A -= w[:, None] * inv[j - 1] * u[None, :]
                b -= w * y[j - 1]
            inv[j] = np.linalg.inv(A)
            y[j] = inv[j] @ b
        x = [None] * ny
        x[-1] = y[-1]
        for j in range(ny - 2, -1, -1):
            u = -hf[1] * (2 if j == 0 else 1) * free[j]
            x[j] = y[j] - inv[j] @ (u * x[j + 1])
        return np.array(x)

    def efield(self, pot, pm):
        ny, nx = pot.shape
        ex, ey = np.zeros((ny, nx)), np.zeros((ny, nx))
        if pm == "nec":
            ex[:, 1:-1] = (pot[:, 1:-1] - pot[:, 2:]) * self.vt / self.h[0]
            ey[1:-1] = (pot[1:-1] - pot[2:]) * self.vt / self.h[1]
        else:
            ex[:, 1:-1] = (pot[:, :-2] - pot[:, 2:]) * self.vt / (2 * self.h[0])
            ey[1:-1] = (pot[:-2] - pot[2:]) * self.vt / (2 * self.h[1])
        ln = self.lines
        ex[:, 0], ex[:, -1] = np.where(ln[0] < 0, 0, ex[:, 1]), np.where(ln[1] < 0, 0, ex[:, -2])
        ey[0], ey[-1] = np.where(ln[2] < 0, 0, ey[1]), np.where(ln[3] < 0, 0, ey[-2])
        return ex, ey


class Device:
    """the self-consistent device loop on the carriers of a resistor"""

    def __init__(self, case, seed):
        self.case, self.seed = case, seed
        self.dev = _device_dict(case)
        self.g = Grid2(self.dev)
        spec = workloads.MODELS_DEVICE["device_para"]
        self.m = Model([spec], [spec["T"]])
        self.m.build()
        g = self.g
        self.pot = g.solve(np.arcsinh(0.5 * g.doping / self.dev["ni"]), None, False)
        nr = (g.doping * g.half * g.volume).reshape(-1)
        node = torch.arange(nr.size, device=DEV)
        w = _philox((torch.zeros_like(node), torch.full_like(node, 0xFFFFFFFE), node,
                     torch.full_like(node, 0x40000002)), seed)
        whole = np.where(nr >= 1, np.floor(nr), 0)
        cnt = (whole + (_unit(w[0]).cpu().numpy() < nr - whole)).astype(np.int64)
        nodes = torch.repeat_interleave(node, _t(cnt, I64))
        self.pid = torch.arange(nodes.numel(), device=DEV)
        self.next = int(nodes.numel())
        self.x, self.k, self.E, self.tau, self.v, self.s = self.create(nodes, self.pid, M32)
        self.assign()

    def create(self, nodes, pid, step):
        g, m, h = self.g, self.m, self.g.h
        dom = torch.full_like(pid, 0x40000001)
        u = [_stream(j, step, pid, dom, self.seed) for j in range(8)]
        c, ext = [nodes % g.nx, nodes // g.nx], (g.nx, g.ny)
        x = []
        for d in range(2):
            f = c[d].to(F64)
            x.append(torch.where(c[d] == ext[d] - 1, f - u[d] * 0.5,
                                 torch.where(c[d] == 0, u[d] * 0.5, f + u[d] - 0.5)) * (h[d] * 1e9))
        v = torch.zeros_like(pid)
        s = torch.zeros_like(pid)
        E = -1.5 * g.vt * torch.log(u[4] * (1 - 1e-6) + 1e-6)
        k = m._random(m.normk(E, v), u[5], u[6])
        for d in range(2):
            flip = ((c[d] == 0) & (k[:, d] < 0)) | ((c[d] == ext[d] - 1) & (k[:, d] > 0))
            k[:, d] = torch.where(flip, -k[:, d], k[:, d])
        tau = -torch.log(u[7] * (1 - 1e-6) + 1e-6) * m.tau0[v]
        return torch.stack(x, 1), k, E, tau, v, s

    def _cell(self, x):
        r = [x[:, d] / (self.g.h[d] * 1e9) for d in range(2)]
        i = [torch.floor(a) for a in r]
        return [a.to(I64) for a in i], [a - b for a, b in zip(r, i)]

    def _nearest(self, x):
        return [torch.floor(x[:, d] / (self.g.h[d] * 1e9) + 0.5).to(I64) for d in range(2)]

    def assign(self):
        g, pm = self.g, self.case["pm"]
        grid = torch.zeros(g.nx * g.ny, dtype=F64, device=DEV)

        def add(ix, iy, w):
            ok = (ix < g.nx) & (iy < g.ny)
            grid.index_add_(0, (iy * g.nx + ix)[ok], w[ok])

        if pm == "ngp":
            ix, iy = self._nearest(self.x)
            add(ix, iy, torch.ones_like(self.E))
        else:
            (ix, iy), (wx, wy) = self._cell(self.x)
            if pm == "nec":
                wx = wy = torch.full_like(wx, 0.5)
            add(ix, iy, wx * wy)
            add(ix + 1, iy, (1 - wx) * wy)
            add(ix, iy + 1, wx * (1 - wy))
            add(ix + 1, iy + 1, (1 - wx) * (1 - wy))
        self.nr = grid.cpu().numpy().reshape(g.ny, g.nx)
        self.conc = self.nr / (g.half * g.volume) / self.dev["ni"]

    def force(self, x):
        """acceleration dk/dt [1/nm per fs] from the field at the position"""
        g, pm = self.g, self.case["pm"]
        E = [self.Ex, self.Ey]

        def get(f, ix, iy):
            ok = (ix < g.nx) & (iy < g.ny)
            return torch.where(ok, f[(iy * g.nx + ix).clamp(max=g.nx * g.ny - 1)], torch.zeros_like(x[:, 0]))

        if pm == "ngp":
            ix, iy = self._nearest(x)
            F = [get(f, ix, iy) for f in E]
        else:
            (ix, iy), (wx, wy) = self._cell(x)
            if pm == "nec":
                F = [(get(E[0], ix, iy) + get(E[0], ix, iy + 1)) / 2, (get(E[1], ix, iy) + get(E[1], ix + 1, iy)) / 2]
            else:
                F = [get(f, ix, iy) * wx * wy + get(f, ix + 1, iy) * (1 - wx) * wy + get(f, ix, iy + 1) * wx * (1 - wy) +
                     get(f, ix + 1, iy + 1) * (1 - wy) * (1 - wy) for f in E]
        return torch.stack([F[0], F[1], torch.zeros_like(F[0])], 1) * (-Q / HBAR * 1e-24)

    def drift(self, t, x, k, E, v):
        g, m = self.g, self.m
        k1 = k + self.force(x) * t[:, None]
        E1 = m.energy(k1, v)
        f = m.cv[v] * t * 1e-6 / (1 + 2 * m.alpha[v] * E1)
        x1 = x + 0.5 * (k + k1)[:, :2] * f[:, None]
        top = _t([d * 1e9 for d in self.dev["max_pos"]])
        inside = torch.minimum(x1.clamp(min=0.0), top)
        out = (inside != x1).any(1)
        cx, cy = self._nearest(inside)
        node = cy * g.nx + cx
        gone = out & _t(g.ohmic.reshape(-1), torch.bool)[node]
        for d in range(2):
            low, high = out & ~gone & (x1[:, d] < 0), out & ~gone & (x1[:, d] > top[d])
            k1[:, d] = torch.where(low | high, -k1[:, d], k1[:, d])
            x1[:, d] = torch.where(low, -x1[:, d], torch.where(high, 2 * top[d] - x1[:, d], x1[:, d]))
        x1 = torch.where(gone[:, None], inside, x1)
        return x1, k1, E1, gone, node

    def step(self, s):
        g, m, dt = self.g, self.m, DEVICE_DT * 1e15
        nc = len(self.dev["contacts"])
        self.pot = g.solve(self.pot, self.conc, True)
        ex, ey = g.efield(self.pot, self.case["pm"])
        self.field = (ex, ey)
        self.Ex, self.Ey = _t(ex.reshape(-1)), _t(ey.reshape(-1))
        t = torch.minimum(self.tau, torch.full_like(self.tau, dt))
        self.x, self.k, self.E, gone, node = self.drift(t, self.x, self.k, self.E, self.v)
        rem = dt - self.tau
        i, e = torch.nonzero((rem > 0) & ~gone)[:, 0], 0
        rem = rem[i]
        dom = torch.full_like(self.pid, 0x40000000)
        while i.numel():
            k, E, v, sv, nt, _ = m.event(e, s, self.pid[i], dom[i], self.seed, self.k[i], self.E[i], self.v[i],
                                         self.s[i])
            x, k, E, out, nd = self.drift(torch.minimum(rem, nt), self.x[i], k, E, v)
            self.x[i], self.k[i], self.E[i], self.v[i], self.s[i] = x, k, E, v, sv
            self.tau[i] += nt
            gone[i], node[i] = out, nd
            rem = rem - nt
            go = (rem > 0) & ~out
            i, rem, e = i[go], rem[go], e + 1
        self.tau -= dt
        contact = _t(g.contact.reshape(-1), I64)
        net = torch.bincount(contact[node[gone]], minlength=nc).to(F64)
        self._keep(~gone)
        # contact equilibrium: the first carriers in array order stay, the rest go; the missing ones come in
        expect = _t(np.where(g.ohmic, g.doping * g.half * g.volume, 0.0).reshape(-1))
        cx, cy = self._nearest(self.x)
        here = cy * g.nx + cx
        at = torch.nonzero(_t(g.ohmic.reshape(-1), torch.bool)[here])[:, 0]
        order = torch.argsort(here[at], stable=True)
        hs = here[at][order]
        total = torch.bincount(hs, minlength=g.nx * g.ny)
        start = torch.cumsum(total, 0) - total
        rank = torch.arange(hs.numel(), device=DEV) - start[hs]
        want = torch.ceil(expect).to(I64)
        extra = at[order][rank >= want[hs]]
        net += torch.bincount(contact[here[extra]], minlength=nc)
        keep = torch.ones_like(self.pid, dtype=torch.bool)
        keep[extra] = False
        self._keep(keep)
        miss = torch.where(expect > 0, (want - total).clamp(min=0), torch.zeros_like(want))
        nodes = torch.repeat_interleave(torch.arange(g.nx * g.ny, device=DEV), miss)
        net -= torch.bincount(contact[nodes], minlength=nc)
        pid = self.next + torch.arange(nodes.numel(), device=DEV)
        self.next += int(nodes.numel())
        new = self.create(nodes, pid, s)
        cat = lambda a, b: torch.cat([a, b])
        self.x, self.k, self.E, self.tau, self.v, self.s = (cat(a, b) for a, b in zip(
            (self.x, self.k, self.E, self.tau, self.v, self.s), new))
        self.pid = cat(self.pid, pid)
        self.assign()
        return net.cpu().numpy(), float(self.pid.numel())

    def _keep(self, mask):
        for name in ("x", "k", "E", "tau", "v", "s", "pid"):
            setattr(self, name, getattr(self, name)[mask])


def _exact_device(case, seed):
    d = Device(case, seed)
    got = [d.step(s) for s in range(case["steps"])]
    net = np.cumsum([n for n, _ in got], axis=0)
    out = dict(pot=d.pot.reshape(-1), E=np.stack([f.reshape(-1) for f in d.field]), conc=d.conc.reshape(-1),
               nr_part=d.nr.reshape(-1),
               current=Q * net / (DEVICE_DT * np.arange(1, case["steps"] + 1)[:, None]),
               carriers=np.array([n for _, n in got]))
    if case["particles"] <= 100_000 and case["precision"] == "f64":
        own = dict(pos=d.x * 1e-9, k=d.k / 1e-9, E=d.E, tau=d.tau / 1e15)
        out["particles"] = {k: _padded(v.cpu().numpy(), case) for k, v in own.items()}
    return out


def _exact_poisson(case, seed):
    g = Grid2(_mosfet_dict(case, seed))
    pot = g.solve(np.arcsinh(0.5 * g.doping / workloads.SI_NI), None, False)
    ex, ey = g.efield(pot, "cic")
    return dict(pot=pot.reshape(-1), ex=ex.reshape(-1), ey=ey.reshape(-1))


def _exact_mesh3(case, seed):
    rs = np.random.RandomState(seed % (1 << 32))
    ext, h = (case["nx"], case["ny"], case["nz"]), (1.0e-9, 1.5e-9, 2.0e-9)
    nn = ext[0] * ext[1] * ext[2]
    top = np.array([(e - 1) * d for e, d in zip(ext, h)])
    pos = rs.rand(case["particles"], 3) * top * (1.0 - 1e-9)
    E = [1e6 * rs.standard_normal(nn) for _ in range(3)]
    r = pos / np.array(h)
    grid, force = np.zeros(nn), np.zeros((case["particles"], 3))
    if case["pm"] == "ngp":
        i = np.floor(r + 0.5).astype(np.int64)
        m = i[:, 0] + ext[0] * (i[:, 1] + ext[1] * i[:, 2])
        grid += np.bincount(m, minlength=nn)
        for d in range(3):
            force[:, d] = -Q * E[d][m]
        return dict(grid=grid, force=force)
    i = np.floor(r).astype(np.int64)
    w = r - i
    for c in range(8):
        b = [c & 1, (c >> 1) & 1, c >> 2]
        f = [w[:, d] if b[d] == 0 else 1 - w[:, d] for d in range(3)]
        j = [i[:, d] + b[d] for d in range(3)]
        ok = (j[0] < ext[0]) & (j[1] < ext[1]) & (j[2] < ext[2])
        m = np.where(ok, j[0] + ext[0] * (j[1] + ext[1] * j[2]), 0)
        grid += np.bincount(m[ok], weights=(f[0] * f[1] * f[2])[ok], minlength=nn)
        # the scheme weights the (x+1, y+1) nodes by the y weight twice
        wf = (f[1] * f[1] if b[0] and b[1] else f[0] * f[1]) * f[2]
        for d in range(3):
            force[:, d] += np.where(ok, E[d][m], 0.0) * wf
    return dict(grid=grid, force=force * -Q)


def exact(case, seed):
    return {"bulk": _exact_bulk, "sweep": _exact_bulk, "cooling": _exact_cooling, "device": _exact_device,
            "poisson": _exact_poisson, "mesh3": _exact_mesh3}[case["kind"]](case, seed)
