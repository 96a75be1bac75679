"""A mixed-precision network of 10 reactions, whose kernel leaves room for one
wavefront per SIMD, with a few more simulations than that holds: the build for
such launches gives the same trajectories and does not take several times as
long (test marked gpu)."""
import numpy as np
import pytest

from devbuf import DeviceArray
from py_stoch_amd import models, workloads

pytestmark = pytest.mark.gpu


def test_a_few_more_simulations_than_one_wavefront_per_simd(native):
    spn = models.random_network(np.random.default_rng(1), n_species=6, n_reactions=10)
    tabs, rates = workloads.mass_action_tables(spn)
    got, ms = [], []
    for n in (60000, 70000):
        print("case: 6 species, 10 reactions, %d simulations" % n, flush=True)
        plan = native.Plan(tabs, rates, np.asarray(spn.M, np.int32), method=0, precision=native.PRECISION_MIXED,
                           specialize=True, t_max=5.0, I=np.linspace(0, 5, 9).astype(np.float32),
                           E=np.arange(6, dtype=np.int32), n_sims=n, seed=2, max_steps=1000)
        O, F = DeviceArray((6, 9, n)), DeviceArray((n,))
        try:
            times = []
            for _ in range(4):
                plan.execute(O.ptr.value, n, F.ptr.value)
                times.append(plan.stats()["kernel_ms"])
            got.append((O.get()[:, :, :60000], F.get()[:60000]))
            ms.append(min(times[1:]))
        finally:
            plan.close()
            O.free()
            F.free()
    print("kernel ms", ms, flush=True)
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    assert ms[1] < 2.5 * ms[0]
