"""What the lanes of a wavefront hand each other through LDS: the net changes of
a table-driven job, filled by some lanes and read by others and replaced job by
job, and the states and gathered samples of the last simulations when they are
moved to groups of lanes.  FP64 against the oracle (every test marked gpu)."""
import numpy as np
import pytest

from devbuf import DeviceArray
from py_stoch_amd import models
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu


def _ring(N, step):
    """Immigration of `step` counts into species 0, conversions round a ring that
    skips `step` species, decay of the last: every job of a plan has other net
    changes in the same places."""
    reactions = [({}, {0: step}, "parameter_0")]
    for j in range(1, N):
        reactions.append(({j - 1: 1}, {(j - 1 + step) % N: 1}, "parameter_%d*species_%d" % (j, j - 1)))
    reactions.append(({N - 1: 1}, {}, "parameter_%d*species_%d" % (N, N - 1)))
    return models._spn(N, reactions, [20] * N, [30.0] + [1.0 + 0.25 * j for j in range(1, N + 1)])


@pytest.mark.parametrize("N,method", [(3, 2), (3, 0), (7, 2), (15, 2), (15, 0)])
def test_jobs_of_one_size_class_after_one_another(native, oracle_mod, N, method):
    jobs, want = [], []
    for step in range(1, N):
        a = models.make_args(_ring(N, step), E=[0, N - 1], t_max=1.0, ita=11, U=70)
        tabs, rates = tables_of(a), a.rate_fn(a.c)
        kw = dict(method=method, t_max=1.0, I=a.I, E=a.E, n_sims=70, seed=step)
        jobs.append(native.Job(tabs, rates, a.x_0, specialize=False, **kw))
        want.append(oracle_mod.simulate(tabs, rates, a.x_0, threads=16, **kw)[:2])
    print("case: %d table jobs of %d species, method %d" % (len(jobs), N, method), flush=True)
    Os, Fs, _ = native.batch_simulate(jobs)
    for (Oc, Fc), O, F in zip(want, Os, Fs):
        assert np.array_equal(O, Oc) and np.array_equal(F, Fc)


@pytest.mark.parametrize("kappa", [1, 4])
@pytest.mark.parametrize("method,burst_waves", [(2, 0), (0, 0), (0, 1)])
def test_samples_move_with_the_last_simulations(native, oracle_mod, method, burst_waves, kappa):
    n, ita = 66003, 29
    a = models.make_args(_ring(4, 1), E=list(range(kappa)), t_max=0.5, ita=ita, U=n)
    tabs, rates = tables_of(a), a.rate_fn(a.c)
    kw = dict(method=method, t_max=0.5, I=a.I, E=a.E, n_sims=n, seed=4)
    Oc, Fc, _ = oracle_mod.simulate(tabs, rates, a.x_0, threads=16, **kw)
    print("case: samples of %d species, method %d, burst_waves %d" % (kappa, method, burst_waves), flush=True)
    plan = native.Plan(tabs, rates, a.x_0, precision=0, specialize=True, layout=native.LAYOUT_BLOCKS, **kw)
    O, F = DeviceArray((kappa, 4, n, 8)), DeviceArray((n,))
    try:
        plan.set_launch(0, 7, 0, burst_waves)
        plan.execute(O.ptr.value, n, F.ptr.value)
        plan.stats()
        Og = O.get().transpose(0, 1, 3, 2).reshape(kappa, 32, n)
        assert np.array_equal(Og[:, :ita], Oc) and not Og[:, ita:].any() and np.array_equal(F.get(), Fc)
    finally:
        plan.close()
        O.free()
        F.free()
