"""A launch a few simulations beyond what one wavefront per SIMD holds, with a
step budget that makes every simulation as long as the others: the few are not
run after the rest, which would take twice the time (every test marked gpu)."""
import numpy as np
import pytest

from devbuf import DeviceArray
from py_stoch_amd import models, workloads
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu


def _times(native, tabs, rates, x0, kw, sizes, specialize):
    got, ms = [], []
    for n in sizes:
        plan = native.Plan(tabs, rates, x0, precision=native.PRECISION_MIXED, specialize=specialize, n_sims=n, **kw)
        O, F = DeviceArray((len(kw["E"]), len(kw["I"]), n)), DeviceArray((n,))
        try:
            times = []
            for _ in range(5):
                plan.execute(O.ptr.value, n, F.ptr.value)
                times.append(plan.stats()["kernel_ms"])
            got.append((O.get()[:, :, :sizes[0]], F.get()[:sizes[0]]))
            ms.append(min(times[1:]))
        finally:
            plan.close()
            O.free()
            F.free()
    print("kernel ms", ms, flush=True)
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    return ms


def test_network_kernel(native):
    a = models.make_args(models.lotka_volterra(), E=[0], t_max=3.0, ita=9, U=4)
    print("case: lotka_volterra, 300 steps, 16,384 and 16,400 simulations", flush=True)
    kw = dict(method=0, t_max=3.0, I=a.I, E=a.E, seed=2, max_steps=300)
    ms = _times(native, tables_of(a), a.rate_fn(a.c), a.x_0, kw, (16384, 16400), True)
    assert ms[1] < 1.5 * ms[0]


def test_table_driven(native):
    spn = models.random_network(np.random.default_rng(17), n_species=6, n_reactions=8)
    tabs, rates = workloads.mass_action_tables(spn)
    print("case: 6 species, 8 reactions, 1000 steps, 32,768 and 33,000 simulations", flush=True)
    kw = dict(method=0, t_max=5.0, I=np.linspace(0, 5, 9).astype(np.float32), E=np.arange(6, dtype=np.int32), seed=2,
              max_steps=1000)
    ms = _times(native, tabs, rates, np.asarray(spn.M, np.int32), kw, (32768, 33000), False)
    assert ms[1] < 1.5 * ms[0]
