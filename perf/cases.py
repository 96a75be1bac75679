"""The calls the simulator's speed is judged on, over the range of real use.

Four ways a program calls the framework, each through its public entry point:

  run      CuTauLeaping().run(args) / CuGillespie().run(args): host arguments
           in, host trajectories out (what a script of the reference calls)
  sweep    CuTauLeaping().run_batch(list of TlArgs): a parameter sweep built
           the way sim_maker builds one, host to host
  plan     _native.Plan: tables resident on the device, trajectories left in
           device memory
  batch    _native.BatchPlan: several jobs in one plan
  noalloc  _native.run_noalloc: the table-driven kernel on caller memory

on the networks of py_stoch_amd.models (birth-death, Lotka-Volterra, Schlogl,
Michaelis-Menten turnover, random mass-action networks), in both precisions,
by tau-leaping, forced SSA and pure SSA, with either trajectory layout.
Initial counts and rate constants are jittered by the seed, which also keys
the random stream.  Outputs are the trajectories and the per-simulation
flags, whole.
"""
import math

import numpy as np
import torch

from py_stoch_amd import _native, models, workloads
from py_stoch_amd.mod.parser import GArgs, GParser, TlArgs, TlParser
from py_stoch_amd.mod.parser.tl_parser import tables_of
from py_stoch_amd.mod.simulator.cuGillespie import CuGillespie
from py_stoch_amd.mod.simulator.cuTauLeaping import CuTauLeaping

TL, FORCED, SSA = _native.METHOD_TAU_LEAPING, _native.METHOD_FORCED_SSA, _native.METHOD_PURE_SSA
RECORDED = {"birth_death": [0], "lotka_volterra": [0, 1], "schlogl": [0], "michaelis_menten": [0]}


def listed():
    return [
        # the smallest call a script makes: a first look at a model, defaults throughout
        dict(name="run_lv_small", entry="run", model="lotka_volterra", method=TL, mixed=False, t=1.0, ita=101, sims=100),
        # exact SSA of a small ensemble through the drop-in class (1024 birth-death simulations)
        dict(name="run_birth_death_ssa", entry="run", model="birth_death", method=SSA, mixed=False, t=100.0, ita=101,
             sims=1024),
        # a medium ensemble, host to host, with the copy back a script waits for
        dict(name="run_schlogl_medium", entry="run", model="schlogl", method=TL, mixed=True, t=10.0, ita=101,
             sims=20000),
        # a sweep over initial amounts and parameters, one call for all of it
        dict(name="sweep_lv", entry="sweep", model="lotka_volterra", method=TL, mixed=False, t=2.0, ita=101, sims=256,
             sets=24),
        # the benchmark's workload: device-resident, mixed precision, blocked layout, its tuned launch shape
        dict(name="plan_lv_mixed", entry="plan", model="lotka_volterra", method=TL, mixed=True, t=10.0, ita=1000,
             sims=65536, blocks=True, burst_waves=True),
        # the same method in plain FP64 at an odd ensemble size, rows layout, default launch
        dict(name="plan_lv_fp64", entry="plan", model="lotka_volterra", method=TL, mixed=False, t=10.0, ita=1000,
             sims=16411, blocks=False),
        # the largest ensemble: bistable Schlogl by tau-leaping with SSA bursts
        dict(name="plan_schlogl_tl_mixed", entry="plan", model="schlogl", method=TL, mixed=True, t=10.0, ita=100,
             sims=262144, blocks=False),
        # exact SSA at scale, mixed precision
        dict(name="plan_schlogl_ssa_mixed", entry="plan", model="schlogl", method=SSA, mixed=True, t=10.0, ita=100,
             sims=100003, blocks=True),
        # a serving loop on caller memory: table-driven kernel, plain FP64
        dict(name="noalloc_lv_fp64", entry="noalloc", model="lotka_volterra", method=TL, mixed=False, t=3.0, ita=301,
             sims=4099),
        # a device-resident sweep over both families, rates over two decades each way of use
        dict(name="batch_sweep_mixed", entry="batch", mixed=True, t=10.0, ita=100, sets=256, sims=64, spread=0.5),
        # networks beyond the lane kernels: one wavefront per simulation, step budget
        dict(name="batch_large_networks", entry="batch", networks=16, net_seed=5, min_species=20, max_species=50,
             min_reactions=40, max_reactions=200, mixed=True, t=5.0, ita=50, sims=300, steps=6000),
        # a network of middle size, compiled in
        dict(name="plan_middle_network", entry="plan", model="random", net_seed=3, species=6, reactions=10, method=TL,
             mixed=True, t=5.0, ita=50, sims=20011, steps=4000, blocks=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "sweep", "plan", "plan", "plan", "noalloc", "batch", "large", "middle"])
    mixed = rng.random() < 0.5
    if kind == "large":
        return dict(entry="batch", networks=rng.randint(1, 16), net_seed=rng.randint(1, 10 ** 6), min_species=20,
                    max_species=50, min_reactions=40, max_reactions=200, mixed=True, t=5.0, ita=rng.choice([11, 50, 73]), sims=_log_int(rng, 16, 300),
                    steps=_log_int(rng, 500, 6000))
    if kind == "middle":
        return dict(entry="plan", model="random", net_seed=rng.randint(1, 10 ** 6), species=rng.randint(5, 8),
                    reactions=rng.randint(7, 12), method=TL, mixed=mixed, t=5.0, ita=rng.choice([11, 50, 101]),
                    sims=_log_int(rng, 500, 20011), steps=_log_int(rng, 500, 4000), blocks=rng.random() < 0.5,
                    specialize=rng.random() < 0.5)
    if kind == "batch":
        return dict(entry="batch", mixed=mixed, t=rng.choice([2.0, 5.0]), ita=rng.choice([33, 100, 257]),
                    sets=2 * rng.randint(4, 128), sims=_log_int(rng, 3, 64), spread=rng.choice([0.1, 0.3, 0.5]))
    model = rng.choice(["birth_death", "lotka_volterra", "lotka_volterra", "schlogl", "michaelis_menten"])
    method = rng.choice([TL, TL, SSA, FORCED])
    if model == "lotka_volterra":
        method = TL  # its exact SSA takes 30,000 steps per unit of time: not what it is run by
    if model == "michaelis_menten":
        method = SSA  # a rational hazard has no tau-leaping table
    if kind == "sweep":
        return dict(entry="sweep", model="lotka_volterra", method=TL, mixed=mixed, t=rng.uniform(0.5, 3.0),
                    ita=rng.choice([11, 64, 101]), sims=_log_int(rng, 2, 300), sets=rng.randint(2, 32))
    t = rng.uniform(20.0, 100.0) if model in ("birth_death", "michaelis_menten") else rng.uniform(1.0, 8.0)
    c = dict(entry=kind, model=model, method=method, mixed=mixed, t=t, ita=rng.choice([11, 101, 250, 333]))
    if kind == "run":
        return dict(c, sims=_log_int(rng, 1, 20000))
    if kind == "noalloc":
        if model == "michaelis_menten":
            c["model"] = "birth_death"
        return dict(c, sims=_log_int(rng, 64, 6000))
    return dict(c, sims=_log_int(rng, 500, 60000), blocks=rng.random() < 0.5)


def _model(case, rng):
    """The network with this seed's initial counts and rate constants."""
    name = case["model"]
    j = lambda v: float(v * rng.uniform(0.98, 1.02))
    if name == "birth_death":
        return models.birth_death(j(10.0), j(0.1), int(rng.integers(0, 5)))
    if name == "lotka_volterra":
        return models.lotka_volterra(j(10.0), j(0.01), j(10.0), int(rng.integers(950, 1051)), int(rng.integers(950, 1051)))
    if name == "schlogl":
        return models.schlogl(x0=int(rng.integers(245, 256)))
    if name == "michaelis_menten":
        return models.michaelis_menten_birth_death(j(20.0), j(25.0), j(10.0), int(rng.integers(0, 5)))
    raise ValueError(name)


def _args(case, rng, seed):
    """A parsed TlArgs / GArgs, as a script builds it."""
    a = GArgs() if case["method"] == SSA else TlArgs()
    a.E = np.array(RECORDED[case["model"]], np.int32)
    a.t_max = case["t"]
    a.ita = case["ita"]
    a.U = case["sims"]
    a.gillespie = int(case["method"] == FORCED)
    a.precision = "mixed" if case["mixed"] else "fp64"
    a.seed = seed
    return (GParser if case["method"] == SSA else TlParser).parse(a, _model(case, rng))


def _random_job(rng, jitter, n_species, n_reactions):
    """Tables and rates of a random network (structure from rng), with jittered initial counts."""
    spn = models.random_network(rng, n_species=n_species, n_reactions=n_reactions)
    tabs, rates = workloads.mass_action_tables(spn)
    x0 = np.asarray(spn.M, np.int64) + jitter.integers(0, 5, size=n_species)
    return tabs, rates, x0.astype(np.int32)


def _jobs(case, seed):
    """(tables, rates, x0, settings) of every job of a batch."""
    jitter = np.random.default_rng(seed)
    I = np.linspace(0, case["t"], num=case["ita"]).astype(np.float32)
    out = []
    if "networks" in case:
        rng = np.random.default_rng(case["net_seed"])
        for _ in range(case["networks"]):
            N = int(rng.integers(case["min_species"], case["max_species"] + 1))
            M = int(rng.integers(case["min_reactions"], case["max_reactions"] + 1))
            tabs, rates, x0 = _random_job(rng, jitter, N, M)
            out.append((tabs, rates, x0, dict(method=TL, t_max=case["t"], I=I, E=np.arange(N, dtype=np.int32),
                                              n_sims=case["sims"], seed=seed, max_steps=case["steps"])))
        return out
    n = case["sets"] // 2
    for model in ("lotka_volterra", "schlogl"):
        a = _args(dict(case, model=model, method=TL), jitter, seed)
        base = np.asarray(a.c, np.float64)
        rows = [a.rate_fn(base * 10.0 ** jitter.uniform(-case["spread"], case["spread"], size=base.size))
                for _ in range(n)]
        out.append((tables_of(a), np.array(rows), np.tile(np.asarray(a.x_0).reshape(1, -1), (n, 1)),
                    dict(method=TL, t_max=case["t"], I=I, E=a.E, n_sims=n * case["sims"], sims_per_set=case["sims"],
                         seed=seed)))
    return out


def _buffers(kappa, ita, sims, blocks):
    shape = (kappa, (ita + 7) // 8, sims, 8) if blocks else (kappa, ita, sims)
    return (torch.zeros(shape, dtype=torch.int32, device="cuda"), torch.zeros(sims, dtype=torch.int32, device="cuda"))


def prepare(case, seed):
    entry = case["entry"]
    rng = np.random.default_rng(seed)
    if entry == "run":
        return dict(entry=entry, sim=CuGillespie() if case["method"] == SSA else CuTauLeaping(),
                    args=_args(case, rng, seed))
    if entry == "sweep":
        base = _args(case, rng, seed)
        args = []
        for i in range(case["sets"]):
            a = TlArgs()
            a.__dict__.update(base.__dict__)
            a.c = np.asarray(base.c) * rng.uniform(0.9, 1.1, size=len(base.c))
            a.x_0 = np.asarray(base.x_0) + rng.integers(0, 100, size=len(base.x_0)).astype(np.int32)
            a.sim_offset = i * 4096
            args.append(a)
        return dict(entry=entry, sim=CuTauLeaping(), args=args)
    precision = _native.PRECISION_MIXED if case["mixed"] else _native.PRECISION_FP64
    if entry == "batch":
        jobs = [_native.Job(t, r, x, precision=precision, specialize="networks" not in case, **kw)
                for t, r, x, kw in _jobs(case, seed)]
        bufs = [_buffers(j.kappa, j.ita, j.n_sims, False) for j in jobs]
        return dict(entry=entry, plan=_native.BatchPlan(jobs), O=[b[0] for b in bufs], F=[b[1] for b in bufs])
    if case["model"] == "random":
        tabs, rates, x0 = _random_job(np.random.default_rng(case["net_seed"]), rng, case["species"], case["reactions"])
        I = np.linspace(0, case["t"], num=case["ita"]).astype(np.float32)
        E = np.arange(case["species"], dtype=np.int32)
    else:
        a = _args(case, rng, seed)
        tabs, rates, x0, I, E = tables_of(a), a.rate_fn(a.c), a.x_0, a.I, a.E
    kw = dict(method=case["method"], precision=precision, t_max=case["t"], E=E, n_sims=case["sims"], seed=seed,
              max_steps=case.get("steps", 0))
    O, F = _buffers(len(E), case["ita"], case["sims"], case.get("blocks", False))
    if entry == "noalloc":
        dev = [torch.from_numpy(np.array(v, dt).reshape(-1)).cuda()
               for v, dt in ((rates, np.float64), (x0, np.int32), (I, np.float32))]
        return dict(entry=entry, tables=tabs, dev=dev, kw=dict(kw, ita=case["ita"]), O=O, F=F)
    plan = _native.Plan(tabs, rates, x0, I=I, specialize=case.get("specialize", True),
                        layout=_native.LAYOUT_BLOCKS if case["blocks"] else _native.LAYOUT_ROWS, **kw)
    if case.get("burst_waves"):
        plan.set_launch(0, 7, 0, 1)  # the shape the autotuner picks for this workload
    return dict(entry=entry, plan=plan, O=O, F=F, sims=case["sims"])


def run(state):
    entry = state["entry"]
    if entry == "run":
        return state["sim"].run(state["args"]), state["sim"].last_flags
    if entry == "sweep":
        return state["sim"].run_batch(state["args"]), state["sim"].last_flags
    stream = torch.cuda.current_stream().cuda_stream
    O, F = state["O"], state["F"]
    if entry == "batch":
        state["plan"].execute([o.data_ptr() for o in O], [f.numel() for f in F], [f.data_ptr() for f in F], stream)
    elif entry == "plan":
        state["plan"].execute(O.data_ptr(), state["sims"], F.data_ptr(), stream)
    else:
        d = state["dev"]
        _native.run_noalloc(state["tables"], d[0].data_ptr(), d[1].data_ptr(), 1, d[2].data_ptr(), O.data_ptr(),
                            state["kw"]["n_sims"], F.data_ptr(), stream, read_stats=False, **state["kw"])
    return O, F


def _steps(case, model):
    """(leaps, SSA steps) of one simulation, from counts of the method on each
    network (Lotka-Volterra to t = 10: 3,900 leaps and 430 SSA steps)."""
    t = case["t"]
    if model == "random":
        return 0.1 * case["steps"], 0.4 * case["steps"]  # SSA mostly; some end or leave the budget early
    if model in ("birth_death", "michaelis_menten"):
        return 0.0, 19.0 * t
    if model == "schlogl":
        return (0.0, 4400.0 * t) if case.get("method", TL) != TL else (130.0 * t, 2000.0 * t ** 0.55)
    return 60.0 * t + 33.0 * t * t, 0.43 * t ** 3


def _one(model, case, sims, kappa, reactions):
    leaps, steps = _steps(case, model)
    # per Poisson draw ~100 (uniform, inversion), per reaction of a decision ~30, per SSA step ~60 + 6 M
    flops = sims * (leaps * 130.0 * reactions + steps * (60.0 + 6.0 * reactions))
    return {"bytes": 4.0 * sims * (kappa * case["ita"] + 1) + 4.0 * case["ita"] + 64.0, "flops": flops}


def work(case):
    """Bytes and operations of one pass: the trajectories and flags written
    once, the sample times read, and the arithmetic of the steps."""
    size = {"birth_death": (1, 2), "lotka_volterra": (2, 3), "schlogl": (1, 4), "michaelis_menten": (1, 2)}
    if "networks" in case:
        n = 0.5 * (case["min_species"] + case["max_species"])
        m = 0.5 * (case["min_reactions"] + case["max_reactions"])
        parts = [_one("random", case, case["sims"], n, m)] * case["networks"]
    elif case["entry"] == "batch":
        parts = [_one(m, case, case["sets"] // 2 * case["sims"], *size[m]) for m in ("lotka_volterra", "schlogl")]
    elif case["model"] == "random":
        parts = [_one("random", case, case["sims"], case["species"], case["reactions"])]
    else:
        parts = [_one(case["model"], case, case["sims"] * case.get("sets", 1), *size[case["model"]])]
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


def exact(case, seed):
    """Every output is a sampled integer trajectory or a flag: equal or not,
    with no 64-bit value to be near to."""
    return None
