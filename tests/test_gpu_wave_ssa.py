"""SSA steps of the large-network kernel: its loop for ordinary steps (ssa_run)
against its general step, which a network takes as a whole once one of its
reactions has more than four propensity factors.  The same network with such a
reaction of rate 0 appended draws the same numbers (one block per SSA step) and
must give the same trajectories, at one to four reactions per lane, up to the
largest network, for pure and forced SSA, with and without a step budget, and
in both layouts' sample positions (every test marked gpu)."""
import numpy as np
import pytest

from py_stoch_amd import models, workloads

pytestmark = pytest.mark.gpu


def _pair(N, M, seed):
    """Tables, rates and counts of a random network, and of the same with a
    rate-0 reaction of order five appended."""
    rng = np.random.default_rng(seed)
    spn = models.random_network(rng, n_species=N, n_reactions=M - 1)
    slow = models._spn(N, [], [], [])
    slow.Pre = np.concatenate([spn.Pre, np.zeros((N, 1))], axis=1)
    slow.Post = np.concatenate([spn.Post, np.zeros((N, 1))], axis=1)
    slow.Pre[N - 1, -1], slow.Post[N - 1, -1] = 5, 4
    x0 = np.minimum(np.asarray(spn.M, np.int32), 300)
    out = []
    for s, c in ((spn, spn.c), (slow, list(spn.c) + [0.0])):
        s.c = c
        tabs, rates = workloads.mass_action_tables(s)
        out.append((tabs, rates, x0))
    return out


@pytest.mark.parametrize("method,max_steps,burst", [(2, 700, 100), (1, 333, 7), (2, 0, 100)])
@pytest.mark.parametrize("N,M", [(17, 20), (20, 64), (33, 65), (40, 129), (50, 200), (64, 256)])
def test_ordinary_steps_equal_general_steps(native, N, M, method, max_steps, burst):
    fast, slow = _pair(N, M, 100 * N + M)
    t_end = 0.05 if max_steps else 2e-4
    kw = dict(method=method, precision=1, t_max=t_end, I=np.linspace(0, t_end, 29).astype(np.float32),
              E=np.arange(N, dtype=np.int32), n_sims=70, seed=3, ssa_burst=burst, max_steps=max_steps)
    print("case: wave SSA N=%d M=%d method=%d max_steps=%d" % (N, M, method, max_steps), flush=True)
    O1, F1, s1 = native.simulate(*fast, **kw)
    O2, F2, s2 = native.simulate(*slow, **kw)
    assert s1["ssa_steps"] > 70
    assert np.array_equal(O1, O2) and np.array_equal(F1, F2)
    for key in ("events", "ssa_steps", "uniforms", "sample_rows", "flagged"):
        assert s1[key] == s2[key], key
