"""The work that users of this framework have it do, through its public entry
points (aurora_pic.hip, aurora_pic.serving), as cases that can be timed.

A case is a dict of plain values; "kind" names the workload:

  beam_1d      1D1V periodic plasma (two-stream), spectral solve
  discharge    1D3V bounded RF discharge: null-collision MCC with ionization
               products, electrode drive, wall and power ledgers; with
               "ion_model" a second model (elastic and charge exchange off a
               300 K gas) acts on the ions
  ensemble     many discharges advanced together in captured graphs
  plasma_2d    2D3V periodic plasma, FFT solve, leapfrog or Boris push
  plasma_3d    3D3V periodic electron-ion plasma, tabulated or uniform B
  collide      the null-collision operator alone on device-resident
               velocities
  swarm        homogeneous electron-swarm requests advanced together
  branching    one swarm request with the branching population model

A pass of a particle-in-cell kind is one output interval of a run: the steps,
then what such a program writes there -- the node fields and the energies
(and, for the 1D beam, the particles).  The state goes on from pass to pass,
as a run does.  Sizes come from this repository's workloads, its tests and
bench.py, or are generic; mesh extents and particle counts that are not powers
of two, and meshes that the tiles do not divide, are as common in use as the
others.

exact() is a plain FP64 particle-in-cell restatement in torch.  It is None
where Monte-Carlo collisions act: there a random number within rounding of a
decision (does the particle collide, through which channel) sends a particle
to a different outcome, so the FP64 result is another sample rather than a
more exact one.  The integer tallies of those kinds are left out of the
outputs for the same reason (the energies, rates and fields that follow from
them are in).
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "aurora-pic_amd"))

from aurora_pic import hip, serving, workloads  # noqa: E402


def listed():
    return [
        # the smallest call: the 1D two-stream configuration in FP64, where
        # launches and their latency are the cost (100 of its 2,000 steps)
        dict(name="beam_1d_256", kind="beam_1d", nodes=256, particles=25600, precision=64,
             steps=100),
        # the RF discharge configuration at its full size, 50 steps (an
        # eighth of an RF period)
        dict(name="discharge_513", kind="discharge", nodes=513, particles=500000, steps=50,
             ion_model=False),
        # the discharge of the collision tests, with its ion collisions off a
        # 300 K gas: a small run on which a parameter study spends its time
        dict(name="discharge_129_ions", kind="discharge", nodes=129, particles=20000, steps=200,
             ion_model=True),
        # the batched form of the discharge: 64 instances, graphs of 50 steps
        dict(name="ensemble_64", kind="ensemble", instances=64, particles=100000, steps=100),
        # the 2D Langmuir configuration as bench.py runs it
        dict(name="plasma_2d_256", kind="plasma_2d", nx=256, ny=256, ppc=64, ions=False, b=1,
             precision=32, tuned=True, steps=50),
        # a 2D electron-ion run on a mesh of no special size, with the
        # defaults of the Simulation2D class (sort every 20 steps)
        dict(name="plasma_2d_odd", kind="plasma_2d", nx=210, ny=125, ppc=16, ions=True, b=1,
             precision=32, tuned=False, steps=20),
        # the headline 3D configuration: 67 million particles, tabulated B,
        # the tile shape and push variant the autotuner settles on
        dict(name="plasma_3d_128", kind="plasma_3d", nx=128, ny=128, nz=128, ppc=16, b=2,
             precision=32, tuned=True, steps=100),
        # a 3D run whose mesh is not made of powers of two and that the tiles
        # do not divide, with the defaults of the Simulation3D class
        dict(name="plasma_3d_odd", kind="plasma_3d", nx=90, ny=75, nz=60, ppc=8, b=2,
             precision=32, tuned=False, steps=20),
        # FP64 particles (a species option): a small 3D run kept for accuracy
        dict(name="plasma_3d_f64", kind="plasma_3d", nx=48, ny=48, nz=48, ppc=8, b=1,
             precision=64, tuned=False, steps=20),
        # NullCollisionModel::collide on a million device-resident velocities
        dict(name="collide_1m", kind="collide", count=1000000, thermal=False),
        # the served stream: 64 requests of its distribution, 1,000 steps
        dict(name="swarm_64", kind="swarm", requests=64, particles=0, steps=1000, thermal=False),
        # the branching swarm off a 300 K gas, of the size of the reference's
        # example: thousands of tiny dependent steps
        dict(name="branching_512", kind="branching", particles=512, steps=2000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["beam_1d", "discharge", "ensemble", "plasma_2d", "plasma_2d", "plasma_3d",
                       "plasma_3d", "collide", "swarm", "swarm", "branching"])
    if kind == "beam_1d":
        return dict(kind=kind, nodes=_log(rng, 32, 1024), particles=_log(rng, 2000, 2000000),
                    precision=rng.choice([32, 64]), steps=rng.randint(20, 100))
    if kind == "discharge":
        return dict(kind=kind, nodes=_log(rng, 65, 1025), particles=_log(rng, 10000, 1000000),
                    steps=rng.randint(20, 60), ion_model=rng.random() < 0.5)
    if kind == "ensemble":
        m = _log(rng, 1, 64)
        return dict(kind=kind, instances=m,
                    particles=2 * _log(rng, 5000, min(500000, 4000000 // m)), steps=100)
    if kind == "plasma_2d":
        return dict(kind=kind, nx=_log(rng, 24, 400), ny=_log(rng, 24, 400),
                    ppc=_log(rng, 4, 64) // 2 + 2, ions=rng.random() < 0.5,
                    b=rng.choice([0, 1, 2]), precision=rng.choice([32, 32, 32, 64]), tuned=False,
                    steps=rng.randint(10, 40))
    if kind == "plasma_3d":
        return dict(kind=kind, nx=_log(rng, 20, 100), ny=_log(rng, 20, 100),
                    nz=_log(rng, 20, 100), ppc=rng.randint(2, 8), b=rng.choice([0, 1, 2, 2]),
                    precision=rng.choice([32, 32, 32, 64]), tuned=False,
                    steps=rng.randint(10, 30))
    if kind == "collide":
        return dict(kind=kind, count=_log(rng, 5000, 5000000), thermal=rng.random() < 0.5)
    if kind == "swarm":
        m = _log(rng, 1, 64)
        return dict(kind=kind, requests=m, particles=_log(rng, 5000, 2000000 // m),
                    steps=_log(rng, 200, 1000), thermal=rng.random() < 0.5)
    return dict(kind=kind, particles=_log(rng, 256, 50000), steps=10 * rng.randint(20, 200))


# ----------------------------------------------------------------- inputs
def _rng(seed):
    return torch.Generator(device="cpu").manual_seed(int(seed))


def _dims(case):
    if case["kind"] == "beam_1d":
        return [case["nodes"]]
    if case["kind"] == "plasma_2d":
        return [case["nx"], case["ny"]]
    return [case["nx"], case["ny"], case["nz"]]


def _big(case):
    """Too many particles to place from the host: loaded on the device."""
    return case["kind"] == "plasma_3d" and math.prod(_dims(case)) * case["ppc"] > 8000000


def _plasma(case):
    """Mesh and species of a particle-in-cell case: (L, eps, dt, species),
    each species (charge, mass, weight, particles, thermal velocity)."""
    n = _dims(case)
    if case["kind"] == "beam_1d":
        L = 2.0 * math.pi / 0.5
        N = case["particles"]
        return [L], 1.0, 0.1, [(-1.0, 1.0, L / N, N, 0.1)]
    te = 1.0 if case["kind"] == "plasma_2d" else 5.0
    density = 1.0e16
    lam = workloads.debye_length(density, te)
    L = [c * lam for c in n]
    N = math.prod(n) * case["ppc"]
    w = density * math.prod(L) / N
    mi = 131.0 * workloads.AMU
    species = [(-workloads.EV, workloads.ME, w, N, workloads.maxwellian_sigma(te, workloads.ME))]
    if case.get("ions", True):
        species.append((workloads.EV, mi, w, N, workloads.maxwellian_sigma(0.1, mi)))
    return L, workloads.EPS0, 0.05 / workloads.plasma_frequency(density), species


def _particles(case, seed):
    """Positions and velocities of every species (FP64, host)."""
    L, _, _, species = _plasma(case)
    g, out = _rng(seed), []
    for k, (_, _, _, N, vth) in enumerate(species):
        x = torch.rand(N, len(L), generator=g, dtype=torch.float64) * torch.tensor(
            L, dtype=torch.float64)
        v = torch.randn(N, 3, generator=g, dtype=torch.float64) * vth
        if case["kind"] == "beam_1d":
            v[:, 1:] = 0.0
            v[::2, 0] += 3.0
            v[1::2, 0] -= 3.0
        if k == 0:        # the seeded wave of the two-stream and Langmuir set-ups
            amp = 1.0e-3 if case["kind"] == "beam_1d" else 1.0e-2
            kx = 2.0 * math.pi / L[0]
            x[:, 0] = torch.remainder(x[:, 0] + amp / kx * torch.sin(kx * x[:, 0]), L[0])
            x[:, 0].clamp_(max=math.nextafter(L[0], 0.0))
        out.append((x.numpy(), v.numpy()))
    return out


def _field_b(case, L):
    """Prescribed magnetic field: None, a uniform vector, or (x, values)."""
    b = case.get("b", 0)
    if b == 1:
        return [0.0, 0.0, 0.01]
    if b == 2:
        return workloads.gaussian_by_profile(L[0])
    return None


def _attaching_gas(density):
    """The synthetic gas with an attachment channel, heavy neutrals at 300 K."""
    channels = workloads.synthetic_gas_tables(200)
    e = channels[0][2]
    channels.append((workloads.ATTACHMENT, 0.0, e.copy(),
                     2.0e-21 / (1.0 + (e / workloads.EV / 4.0) ** 2)))
    return dict(channels=channels, neutral_density=density, neutral_mass=workloads.HELIUM_MASS,
                max_frequency=workloads.max_collision_frequency(channels, density),
                max_candidates=64, neutral_temperature=300.0)


def _swarm_gas(thermal):
    gas = workloads.synthetic_gas(1000, 1.0e21)
    gas["neutral_temperature"] = 300.0 if thermal else 0.0
    return gas


def _ion_gas():
    """Ions on the discharge's gas at 300 K: elastic and charge exchange."""
    mi = 6.67e-27
    e = np.geomspace(1.0e-3, 1.0e3, 200) * workloads.EV
    channels = [(hip.ELASTIC, 0.0, e, np.full(e.size, 2.0e-19)),
                (hip.CHARGE_EXCHANGE, 0.0, e.copy(),
                 3.0e-19 / (1.0 + np.sqrt(e / (100.0 * workloads.EV))))]
    return dict(channels=channels, neutral_density=1.0e21, neutral_mass=mi,
                max_frequency=workloads.max_collision_frequency(channels, 1.0e21, mi),
                max_candidates=64)


def _swarm_requests(case, seed):
    """Requests of the served stream's distribution (E/N from 100 Td up where
    few run, so that every channel is met), or of one particle count."""
    cfg = workloads.config_swarm_requests(case["requests"], seed=seed)
    reqs = serving.make_requests(cfg, steps=case["steps"], burn_in=case["steps"] // 2)
    for i, r in enumerate(reqs):
        r.seed = seed * 4099 + i
        if case["particles"]:
            r.particles = case["particles"]
        if case["requests"] < 16:
            r.reduced_field_td = 100.0 * 10.0 ** ((i + 0.5) / case["requests"])
    return reqs


# ---------------------------------------------------------------- prepare
def _prepare_pic(case, seed):
    n = _dims(case)
    L, eps, dt, species = _plasma(case)
    ctx = hip.Context(0)
    ctx.mesh(n, L, hip.PERIODIC, eps)
    b = _field_b(case, L)
    if isinstance(b, list):
        ctx.uniform_b(b)
    elif b is not None:
        ctx.b_profile(0, *b)
    if case.get("tuned") and case["kind"] == "plasma_3d":
        ctx.tiling(8, 8, 4, 2)
        ctx.push_variant(512, 5)
        ctx.sort_policy(hip.SORT_ADAPTIVE)
    elif case.get("tuned"):
        ctx.tiling(16, 8, 1, 2)
        ctx.push_variant(512, 1)
        ctx.sort_policy(hip.SORT_ADAPTIVE)
    elif case["kind"] != "beam_1d":
        ctx.sort_interval(20)
    loaded = None if _big(case) else _particles(case, seed)
    sids = []
    for k, (q, m, w, N, vth) in enumerate(species):
        sid = ctx.add_species(q, m, w, N, case["precision"])
        if loaded is None:
            ctx.init_maxwellian(sid, N, vth, seed * 8 + k)
        else:
            ctx.upload(sid, *loaded[k], kind=hip.VELOCITY_CENTRED)
        sids.append(sid)
    if case["kind"] != "beam_1d":
        ctx.sort()
    ctx.initialize(dt)
    ctx.sync()
    return dict(case=case, ctx=ctx, dt=dt, sids=sids)


def _prepare_discharge(case, seed):
    cfg = workloads.config_discharge()
    N = case["particles"]
    ctx = hip.Context(0)
    ctx.mesh([case["nodes"]], cfg["L"], hip.DIRICHLET, cfg["eps"])
    ctx.electrodes([0.0, 0.0, 0.0, 0.0], [0.0, cfg["phi_right_amplitude"], cfg["frequency"], 0.0])
    sids = []
    for k, s in enumerate(cfg["species"]):
        sid = ctx.add_species(s["charge"], s["mass"], 2.56e14 * cfg["L"][0] / N, 3 * N)
        ctx.init_maxwellian(sid, N, workloads.maxwellian_sigma(s["temperature_ev"], s["mass"]),
                            seed * 8 + k)
        sids.append(sid)
    ctx.mcc_load(sids[0], cfg["gas"], product_species=(sids[0], sids[1]), seed=seed)
    if case["ion_model"]:
        ctx.mcc_add(sids[1], _ion_gas(), seed=seed, neutral_temperature=300.0)
    ctx.initialize(cfg["dt"])
    ctx.sync()
    return dict(case=case, ctx=ctx, dt=cfg["dt"], sids=sids)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("beam_1d", "plasma_2d", "plasma_3d"):
        return _prepare_pic(case, seed)
    if kind == "discharge":
        return _prepare_discharge(case, seed)
    if kind == "ensemble":
        ctx, ens, dt = serving.discharge_ensemble(case["instances"], case["particles"],
                                                  capacity_factor=3, seed=seed % 1000003)
        return dict(case=case, ctx=ctx, ens=ens, dt=dt)
    ctx = hip.Context(0)
    if kind == "collide":
        # electrons of 1 to 40 eV, some above the ionization threshold, and a
        # step at which a tenth of them meet a candidate
        gas = workloads.synthetic_gas(1000, 1.0e21)
        ctx.mesh([65], [0.067], hip.DIRICHLET, workloads.EPS0)
        ctx.add_species(-workloads.EV, workloads.ME, 1.0, 16)
        # (a collide alone places no products; the model names its species)
        ctx.mcc_load(0, gas, product_species=(0, 0), seed=seed,
                     neutral_temperature=300.0 if case["thermal"] else 0.0)
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        n = case["count"]
        sigma = workloads.maxwellian_sigma(8.0, workloads.ME)
        s = dict(case=case, ctx=ctx, dt=0.1 / gas["max_frequency"], step=0,
                 v=torch.randn(n, 3, generator=g, device="cuda") * sigma,
                 counts=torch.zeros(16, dtype=torch.int64, device="cuda"),
                 energy=torch.zeros(8, dtype=torch.float64, device="cuda"),
                 status=torch.zeros(1, dtype=torch.int32, device="cuda"))
        torch.cuda.synchronize()      # the context works on a stream of its own
        return s
    if kind == "swarm":
        ctx.swarm_gas(_swarm_gas(case["thermal"]))
        return dict(case=case, ctx=ctx, reqs=_swarm_requests(case, seed))
    gas = _attaching_gas(1.0e22)
    ctx.swarm_gas(gas)
    req = hip.SwarmRequest(reduced_field_td=300.0, timestep=0.099 / gas["max_frequency"],
                           particles=case["particles"], steps=case["steps"],
                           burn_in=case["steps"] // 2, blocks=5, initial_mean_energy_ev=1.0,
                           max_energy_ev=500.0, seed=seed)
    return dict(case=case, ctx=ctx, req=req)


# -------------------------------------------------------------------- run
def _run_pic(s):
    case, ctx = s["case"], s["ctx"]
    ctx.step(s["dt"], case["steps"])
    ke, fe, l1, _ = ctx.energy(s["dt"])
    rho, phi, E = ctx.fields()
    out = dict(rho=rho, phi=phi, E=E, kinetic=ke, field_energy=fe, charge_l1=l1)
    if case["kind"] == "beam_1d":
        x, v, _, _ = ctx.download(s["sids"][0])
        out.update(x=x, v=v)
    return out


def _run_discharge(s):
    ctx = s["ctx"]
    ctx.step(s["dt"], s["case"]["steps"])
    ke, fe, l1, _ = ctx.energy(s["dt"])
    rho, phi, E = ctx.fields()
    out = dict(rho=rho, phi=phi, E=E, kinetic=ke, field_energy=fe, charge_l1=l1,
               channel_energy=ctx.mcc_stats()[1])
    out["wall_energy"] = np.array([ctx.losses(k)[1] for k in s["sids"]])
    out["work"] = np.array([ctx.power_transfer(k) for k in s["sids"]])
    if s["case"]["ion_model"]:
        out["ion_channel_energy"] = ctx.mcc_model_stats(1)[1]
    return out


def _run_ensemble(s):
    ens, M = s["ens"], s["case"]["instances"]
    ens.step(s["dt"], s["case"]["steps"])
    stats = [ens.stats(k, 3) for k in range(M)]
    fields = [ens.fields(k) for k in range(M)]
    return dict(channel_energy=np.array([t[1] for t in stats]),
                wall_energy=np.array([t[3] for t in stats]),
                rho=np.array([f[0] for f in fields]), phi=np.array([f[1] for f in fields]),
                E=np.array([f[2] for f in fields]))


def _run_collide(s):
    # one step's collisions, in place; the outputs are the program's own
    # device buffers, complete once the context is synchronised
    ctx = s["ctx"]
    s["step"] += 1
    ctx.mcc_collide_device(s["case"]["count"], s["v"].data_ptr(), s["dt"], s["step"],
                           s["counts"].data_ptr(), s["energy"].data_ptr(),
                           s["status"].data_ptr())
    ctx.sync()
    return dict(v=s["v"], energy=s["energy"][:3], status=s["status"])


def _run_swarm(s):
    ctx = s["ctx"]
    handles = [ctx.swarm_submit(r) for r in s["reqs"]]
    ctx.swarm_advance(s["case"]["steps"])
    res = [ctx.swarm_poll(h)[1] for h in handles]
    names = ("drift", "mean_energy_ev", "ionization_rate", "longitudinal_diffusion",
             "transverse_diffusion")
    out = {k: np.array([getattr(r, k) for r in res]) for k in names}
    out["rate"] = np.array([list(r.rate)[:3] for r in res])
    return out


def _run_branching(s):
    r, g = s["ctx"].swarm_branching(s["req"], s["req"].particles * 2)
    return dict(drift=r.drift, mean_energy_ev=r.mean_energy_ev, rate=np.array(list(r.rate)[:4]),
                growth=g.final_weight / g.initial_weight, net_creation=g.net_creation_rate)


_RUN = dict(beam_1d=_run_pic, plasma_2d=_run_pic, plasma_3d=_run_pic, discharge=_run_discharge,
            ensemble=_run_ensemble, collide=_run_collide, swarm=_run_swarm,
            branching=_run_branching)


def run(state):
    return _RUN[state["case"]["kind"]](state)


# ------------------------------------------------------------------- work
def _swarm_particles(case):
    if case["particles"]:
        return case["requests"] * case["particles"]
    return int(workloads.config_swarm_requests(case["requests"])["particles"].sum())


def work(case):
    """Bytes: per particle-step its cell, in-cell position and velocity read
    and written once, per node-step the charge written and read and the field
    written and read; the outputs once.  Operations: gather, push and deposit
    of a particle, a radix-2 transform's count for the solve, about fifty for
    the kick, energy and waiting time of a swarm electron's step."""
    kind = case["kind"]
    if kind == "collide":
        return dict(bytes=case["count"] * 24, flops=case["count"] * 50)
    if kind == "swarm":
        n = _swarm_particles(case)
        return dict(bytes=n * 24, flops=n * case["steps"] * 50)
    if kind == "branching":
        n = case["particles"] * case["steps"]
        return dict(bytes=case["particles"] * 24, flops=n * 60)
    e = case.get("precision", 32) // 8
    if kind in ("discharge", "ensemble"):
        nodes = case.get("nodes", 513) * case.get("instances", 1)
        parts = (2 * case["particles"] if kind == "discharge"
                 else case["particles"] * case["instances"])
        dim, per, species, ops = 1, 2 * (4 + 4 + 12) + 4, 2, 80
    else:
        n = _dims(case)
        dim, nodes = len(n), math.prod(n)
        species = len(_plasma(case)[3])
        parts = sum(sp[3] for sp in _plasma(case)[3])
        per = 2 * (4 + e * (dim + (1 if dim == 1 else 3)))
        ops = {1: 30, 2: 100, 3: 200}[dim]
    node = 16 * species + 2 * 4 * dim
    out = nodes * 8 * (2 + dim) + (parts * 32 if kind == "beam_1d" else 0)
    fft = 5.0 * nodes * math.log2(max(nodes, 2)) * (1 + dim)
    return dict(bytes=case["steps"] * (parts * per + nodes * node) + out,
                flops=case["steps"] * (parts * ops + fft))


# -------------------------------------------------------------- tolerance
def tolerance(case):
    """About four times what was measured: against exact(), and against the
    same run with its step changed by one unit of the last place (1e-7, or
    4e-16 in FP64), which moves every sum and decision by its rounding.
    Measured, worst output: FP64 particles 3e-13 (1.2e-12 against exact());
    FP32 2e-7 to 4e-6 (the beam at few particles per node 1e-4, its density
    being a sum of so few); with collisions a few decisions flip, and each
    one shifts a whole product or electron: density 5e-3, channel energies
    6e-4, swarm averages 1e-4.  A flip in a branching swarm moves every later
    resample, so its averages differ by their own statistical error; one in a
    lone collide sends a particle elsewhere (1e-3 of a million's norm)."""
    kind = case["kind"]
    if kind == "collide":
        return dict(rel=4.0e-3, max=0.99)
    if kind == "branching":
        return dict(rel=2.0e-2, max=0.5)
    if kind == "swarm":
        return dict(rel=5.0e-4)
    if kind in ("discharge", "ensemble"):
        return dict(rel=2.0e-2, max=0.3)
    if case["precision"] == 64:
        return dict(rel=5.0e-12)
    return dict(rel=5.0e-4) if kind == "beam_1d" else dict(rel=2.0e-5)


# ------------------------------------------------------------------ exact
def _spectral(rho, n, L, eps):
    """phi and E of the periodic Poisson problem, continuous wave numbers,
    Nyquist counted as +n/2, real part of the inverse; arrays [z, y, x]."""
    shape = tuple(reversed(n))
    r = torch.fft.fftn(rho.reshape(shape).to(torch.complex128))
    ks = []
    for a, (m, l) in enumerate(zip(n, L)):
        i = torch.arange(m, dtype=torch.float64, device=rho.device)
        k = 2.0 * math.pi / l * torch.where(i <= m // 2, i, i - m)
        view = [1] * len(n)
        view[len(n) - 1 - a] = m
        ks.append(k.reshape(view))
    k2 = sum(k * k for k in ks)
    k2.reshape(-1)[0] = 1.0
    p = r / (eps * k2)
    p.reshape(-1)[0] = 0.0
    phi = torch.fft.ifftn(p).real.reshape(-1)
    return phi, torch.stack([torch.fft.ifftn(-1j * k * p).real.reshape(-1) for k in ks])


def _corners(x, n, d):
    """Corner nodes and weights of every particle (lists over 2^dim)."""
    dim = len(n)
    g = x / torch.tensor(d, dtype=torch.float64, device=x.device)
    c = torch.floor(g)
    o = g - c
    c = c.to(torch.int64)
    nodes, weights = [], []
    for corner in range(2 ** dim):
        node, w, stride = 0, 1.0, 1
        for a in range(dim):
            up = (corner >> a) & 1
            node = node + torch.remainder(c[:, a] + up, n[a]) * stride
            w = w * (o[:, a] if up else 1.0 - o[:, a])
            stride *= n[a]
        nodes.append(node)
        weights.append(w)
    return nodes, weights


def _rotate(v, E, B, h):
    """Boris: half kick, rotation, half kick, with h = q dt / 2 m."""
    vm = v + E * h
    t = B * h
    s = 2.0 * t / (1.0 + (t * t).sum(1, keepdim=True))
    return vm + torch.linalg.cross(vm + torch.linalg.cross(vm, t), s) + E * h


def exact(case, seed):
    if case["kind"] not in ("beam_1d", "plasma_2d", "plasma_3d") or _big(case):
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    n = _dims(case)
    dim = len(n)
    L, eps, dt, species = _plasma(case)
    d = [l / m for l, m in zip(L, n)]
    nodes, volume = math.prod(n), math.prod(d)
    field = _field_b(case, L)
    state = [(torch.from_numpy(x).to(dev), torch.from_numpy(v).to(dev))
             for x, v in _particles(case, seed)]
    Lt = torch.tensor(L, dtype=torch.float64, device=dev)

    def solve():
        rho = torch.zeros(nodes, dtype=torch.float64, device=dev)
        for (q, _, w, _, _), (x, _) in zip(species, state):
            for node, wt in zip(*_corners(x, n, d)):
                rho.index_add_(0, node, wt * (q * w / volume))
        return (rho, *_spectral(rho, n, L, eps))

    def at(E, x):
        out = torch.zeros(x.shape[0], 3, dtype=torch.float64, device=dev)
        for node, wt in zip(*_corners(x, n, d)):
            for a in range(dim):
                out[:, a] += E[a][node] * wt
        return out

    def magnetic(x):
        if isinstance(field, list):
            return torch.tensor(field, dtype=torch.float64, device=dev).expand(x.shape[0], 3)
        c, val = (torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in field)
        r = torch.searchsorted(c, x[:, 0].contiguous(), right=True).clamp(1, len(c) - 1)
        f = ((x[:, 0] - c[r - 1]) / (c[r] - c[r - 1]))[:, None]
        return val[r - 1] + f * (val[r] - val[r - 1])

    def kick(v, x, E, q_m, step):
        e = at(E, x)
        if field is None:
            return v + q_m * step * e
        return _rotate(v, e, magnetic(x), 0.5 * q_m * step)

    rho, phi, E = solve()
    state = [(x, kick(v, x, E, q / m, -0.5 * dt))
             for (q, m, _, _, _), (x, v) in zip(species, state)]
    for _ in range(case["steps"]):
        moved = []
        for (q, m, _, _, _), (x, v) in zip(species, state):
            v = kick(v, x, E, q / m, dt)
            moved.append((torch.remainder(x + dt * v[:, :dim], Lt), v))
        state = moved
        rho, phi, E = solve()
    kinetic = [float((0.5 * m * w * kick(v, x, E, q / m, 0.5 * dt).square()).sum())
               for (q, m, w, _, _), (x, v) in zip(species, state)]
    out = dict(rho=rho.cpu().numpy(), phi=phi.cpu().numpy(), E=E.cpu().numpy(),
               kinetic=np.array(kinetic),
               field_energy=float(0.5 * eps * volume * E.square().sum()),
               charge_l1=float(volume * rho.abs().sum()))
    if case["kind"] == "beam_1d":
        out.update(x=state[0][0].cpu().numpy(), v=state[0][1].cpu().numpy())
    return out
