"""The batched SSA steps (ssa_run) where a batch of four can go wrong: bursts
and step budgets that are no multiple of four, several sample times inside one
batch, networks of one to nine reactions (one to three words of net changes),
and jobs of one plan with different seeds.  FP64 trajectories, flags and
counters equal the oracle's exactly (every test marked gpu)."""
import numpy as np
import pytest

from py_stoch_amd import models
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu

COUNTERS = ("events", "leaps", "rejected_leaps", "ssa_steps", "flagged", "flagged_events")


def _chain(n_reactions):
    """Conversions round a ring of species, the first reaction feeding it."""
    N = max(1, n_reactions - 1)
    reactions = [({}, {0: 1}, "parameter_0")]
    for j in range(1, n_reactions):
        s = (j - 1) % N
        post = {(s + 1) % N: 1} if s + 1 < N else {}
        reactions.append(({s: 1}, post, "parameter_%d*species_%d" % (j, s)))
    return models._spn(N, reactions, [7] * N, [9.0] + [0.5 + 0.25 * j for j in range(1, n_reactions)])


def _settings(spn, U, t_max=3.0, ita=41, seed=5):
    a = models.make_args(spn, E=[0], t_max=t_max, ita=ita, U=U)
    return a, tables_of(a), a.rate_fn(a.c), dict(t_max=t_max, I=a.I, E=a.E, n_sims=U, seed=seed)


@pytest.mark.parametrize("specialize", [True, False])
@pytest.mark.parametrize("n_reactions,method,burst,max_steps", [
    (1, 2, 100, 0), (2, 2, 100, 0), (4, 1, 3, 0), (5, 1, 5, 0), (5, 0, 1, 0), (9, 0, 6, 0), (9, 2, 100, 21), (5, 0, 7, 30)])
def test_batched_ssa_steps_equal_oracle(native, oracle_mod, n_reactions, method, burst, max_steps, specialize):
    spn = _chain(n_reactions)
    a, tabs, rates, kw = _settings(spn, 97)
    kw.update(method=method, ssa_burst=burst, max_steps=max_steps)
    print("case: chain M=%d method=%d burst=%d max_steps=%d specialize=%s" % (n_reactions, method, burst, max_steps,
                                                                              specialize), flush=True)
    O, F, st = native.simulate(tabs, rates, a.x_0, specialize=specialize, **kw)
    Oc, Fc, sc = oracle_mod.simulate(tabs, rates, a.x_0, **kw)
    assert np.array_equal(O, Oc) and np.array_equal(F, Fc)
    for key in COUNTERS:
        assert st[key] == sc[key], key


def test_jobs_of_one_plan_with_their_own_seeds(native, oracle_mod):
    # more simulations than one wavefront in the first job, fewer in the others:
    # lanes without a simulation must not lend their stream key to the rest
    jobs, want = [], []
    for U, seed in ((130, 11), (3, 12), (1, 13)):
        a, tabs, rates, kw = _settings(models.birth_death(), U, t_max=20.0, seed=seed)
        kw.update(method=2)
        jobs.append(native.Job(tabs, rates, a.x_0, specialize=True, **kw))
        want.append(oracle_mod.simulate(tabs, rates, a.x_0, **kw)[0])
    print("case: three pure-SSA jobs with seeds of their own", flush=True)
    Os, _, _ = native.batch_simulate(jobs)
    for O, Oc in zip(Os, want):
        assert np.array_equal(O, Oc)
