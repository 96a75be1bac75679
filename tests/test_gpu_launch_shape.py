"""A launch shape that the autotuner reports can be set on a fresh plan: it runs
there, and as the tuned plan does -- also where the default shape pairs one
network's burst wavefronts and another's cannot be paired (every test marked
gpu)."""
import numpy as np
import pytest

from devbuf import DeviceArray
from py_stoch_amd import models
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu

ITA = 11


def _jobs(native):
    """Lotka-Volterra, 72,000 simulations (much the fastest paired, as by
    default), and a network whose 200 parameters a simulation do not fit the
    hand-off slots in LDS."""
    kw = dict(method=0, precision=1, specialize=True, t_max=8.0)
    a = models.make_args(models.lotka_volterra(), E=[0, 1], t_max=8.0, ita=ITA, U=72000)
    jobs = [native.Job(tables_of(a), a.rate_fn(a.c), a.x_0, I=a.I, E=a.E, n_sims=72000, seed=2, **kw)]
    b = models.make_args(models.birth_death(), E=[0], t_max=8.0, ita=ITA, U=4000)
    tabs = dict(tables_of(b), hazard_c=["C(0)", "C(1)*X(0)"], n_params=200)
    rows = np.concatenate([b.rate_fn(b.c), np.zeros(198)])
    jobs.append(native.Job(tabs, rows, b.x_0, I=b.I, E=b.E, n_sims=4000, seed=3, **kw))
    return jobs


def test_a_reported_shape_runs_on_a_fresh_plan(native):
    results = []
    shape = None
    for step in ("default", "tuned", "set again", "library's choice"):
        print("case: two networks, %s" % step, flush=True)
        plan = native.BatchPlan(_jobs(native))
        O = [DeviceArray((j.kappa, ITA, j.n_sims)) for j in plan.jobs]
        F = [DeviceArray((j.n_sims,)) for j in plan.jobs]
        ptrs, strides = [o.ptr.value for o in O], [j.n_sims for j in plan.jobs]
        try:
            if step == "tuned":
                ch = plan.autotune(ptrs, strides)
                shape = (ch["lanes_shift"], ch["ssa_slice"], ch["waves_trim"], ch["burst_waves"])
                print("reported shape", shape, flush=True)
            elif step == "set again":
                plan.set_launch(*shape)
            elif step == "library's choice":
                plan.set_launch(0, 7, 0, 0)
                plan.set_launch(0, 7, 0, -1)
                for bad in (-2, 2):
                    with pytest.raises(native.NativeError):
                        plan.set_launch(0, 7, 0, bad)
            plan.execute(ptrs, strides, [f.ptr.value for f in F])
            plan.stats()
            results.append([b.get() for b in O + F])
        finally:
            plan.close()
            for buf in O + F:
                buf.free()
    assert shape[3] != 1  # every network of the plan can run it
    for got in results[1:]:
        assert all(np.array_equal(x, y) for x, y in zip(got, results[0]))
