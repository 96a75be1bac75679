"""Host-array batches whose outputs come back in one copy (small jobs) or in
copies of their own: sizes on both sides of each limit, jobs of different
sizes, an empty job among them.  Trajectories, flags and
counters equal the same jobs run one by one (marked gpu)."""
import numpy as np
import pytest

from py_stoch_amd import models, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sims", [
    [1],                    # a job by itself
    [1, 0, 3],              # an empty job
    [2600, 2500, 7],        # 3 jobs, just below 1 MiB a job (ita = 150)
    [3500, 1],              # 2 jobs, just above it
    [65] * 70,
])
def test_batch_output_copies(native, sims):
    spn = models.birth_death(10.0, 0.1, 3)
    tabs, rates = workloads.mass_action_tables(spn)
    I = np.linspace(0, 2.0, 150).astype(np.float32)
    jobs = [native.Job(tabs, rates, spn.M, precision=native.PRECISION_FP64, method=native.METHOD_PURE_SSA, t_max=2.0,
                       I=I, E=np.zeros(1, np.int32), n_sims=n, seed=5, sim_offset=1000 * q, specialize=False)
            for q, n in enumerate(sims)]
    O, F, stats = native.batch_simulate(jobs)
    total = 0
    for q, n in enumerate(sims):
        if n == 0:
            continue
        o, f, st = native.batch_simulate(jobs[q:q + 1])
        assert np.array_equal(O[q], o[0]) and np.array_equal(F[q], f[0])
        total += st["events"]
    assert stats["events"] == total
