"""Simulations replicated over a group of lanes (launches with fewer than 64
simulations per wavefront): every group size from 2 to 64, networks whose
reactions divide evenly over a group and ones that do not, tau-leaping with
both Poisson samplers, critical reactions and SSA bursts.  FP64 trajectories,
flags and counters equal the oracle's; mixed precision gives the same bits in
every group size (every test marked gpu)."""
import numpy as np
import pytest

from devbuf import DeviceArray
from py_stoch_amd import models
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu

COUNTERS = ("events", "leaps", "rejected_leaps", "ssa_steps", "flagged", "flagged_events")
U = 16391  # 32 simulations per wavefront by default on 1024 SIMDs


def _network(n_reactions):
    """Immigration, a dimerisation and conversions down a chain: from a few
    counts (SSA, critical reactions) to thousands (PTRS draws)."""
    N = n_reactions - 1
    reactions = [({}, {0: 2}, "parameter_0")]
    x0 = [900, 12, 3000, 40, 5, 800, 60, 200][:N]
    for j in range(1, n_reactions):
        s = j - 1
        post = {s + 1: 1} if s + 1 < N else {}
        if j == 1:
            reactions.append(({0: 2}, post, "parameter_1*species_0*(species_0 - 1)"))
        else:
            reactions.append(({s: 1}, post, "parameter_%d*species_%d" % (j, s)))
    c = [400.0, 2e-3] + [1.0 + 0.5 * j for j in range(2, n_reactions)]
    return models._spn(N, reactions, x0, c)


def _plan_run(native, tabs, rates, x0, launch, U, precision, specialize, kw):
    plan = native.Plan(tabs, rates, x0, precision=precision, specialize=specialize, **kw)
    O, F = DeviceArray((len(kw["E"]), len(kw["I"]), U)), DeviceArray((U,))
    try:
        plan.set_launch(*launch)
        plan.execute(O.ptr.value, U, F.ptr.value)
        return O.get(), F.get(), plan.stats()
    finally:
        plan.close()
        O.free()
        F.free()


def _settings(n_reactions):
    spn = _network(n_reactions)
    a = models.make_args(spn, E=[0, spn.Pre.shape[0] - 1], t_max=1.0, ita=9, U=U)
    return a, tables_of(a), a.rate_fn(a.c), dict(method=0, t_max=1.0, I=a.I, E=a.E, n_sims=U, seed=9)


@pytest.mark.parametrize("specialize", [True, False])
@pytest.mark.parametrize("n_reactions", [3, 4, 6, 9])
def test_groups_equal_oracle(native, oracle_mod, n_reactions, specialize):
    a, tabs, rates, kw = _settings(n_reactions)
    Oc, Fc, sc = oracle_mod.simulate(tabs, rates, a.x_0, threads=16, **kw)
    assert sc["leaps"] > 0 and sc["ssa_steps"] > 0
    for shift in (0, 1, 2, 5):
        print("case: group M=%d specialize=%s lanes_shift=%d" % (n_reactions, specialize, shift), flush=True)
        O, F, st = _plan_run(native, tabs, rates, a.x_0, (shift, 7), U, 0, specialize, kw)
        assert np.array_equal(O, Oc) and np.array_equal(F, Fc)
        for key in COUNTERS:
            assert st[key] == sc[key], key


@pytest.mark.parametrize("specialize", [True, False])
@pytest.mark.parametrize("n_reactions", [3, 6, 9])
def test_group_size_changes_no_bit_in_mixed_precision(native, n_reactions, specialize):
    a, tabs, rates, kw = _settings(n_reactions)
    # one simulation per lane: more simulations, the same first U ids
    wide = dict(kw, n_sims=70000)
    print("case: mixed M=%d specialize=%s one lane per simulation" % (n_reactions, specialize), flush=True)
    O0, F0, _ = _plan_run(native, tabs, rates, a.x_0, (0, 7), 70000, 1, specialize, wide)
    stats = []
    for shift in (0, 1, 3):
        print("case: mixed M=%d specialize=%s lanes_shift=%d" % (n_reactions, specialize, shift), flush=True)
        O, F, st = _plan_run(native, tabs, rates, a.x_0, (shift, 7), U, 1, specialize, kw)
        assert np.array_equal(O, O0[:, :, :U]) and np.array_equal(F, F0[:U])
        st.pop("kernel_ms")
        stats.append(st)
    assert stats[0] == stats[1] == stats[2]


@pytest.mark.parametrize("method,burst_waves", [(0, 0), (0, 1), (2, 0)])
@pytest.mark.parametrize("n_reactions", [3, 6])
def test_lanes_shared_by_the_last_simulations(native, oracle_mod, n_reactions, method, burst_waves):
    """One simulation per lane, more simulations than lanes on the chip for the
    unpaired launch: wavefronts refill from the queue, then widen to groups of
    four and eight lanes; the blocked layout carries a partial block along."""
    n = 66003
    a, tabs, rates, kw = _settings(n_reactions)
    kw = dict(kw, n_sims=n, method=method, I=np.linspace(0, 0.4, 13).astype(np.float32), t_max=0.4)
    Oc, Fc, sc = oracle_mod.simulate(tabs, rates, a.x_0, threads=16, **kw)
    print("case: widening M=%d method=%d burst_waves=%d" % (n_reactions, method, burst_waves), flush=True)
    plan = native.Plan(tabs, rates, a.x_0, precision=0, specialize=True, layout=native.LAYOUT_BLOCKS, **kw)
    O, F = DeviceArray((2, 2, n, 8)), DeviceArray((n,))
    try:
        plan.set_launch(0, 7, 0, burst_waves)
        plan.execute(O.ptr.value, n, F.ptr.value)
        Og = O.get().transpose(0, 1, 3, 2).reshape(2, 16, n)
        assert np.array_equal(Og[:, :13], Oc) and not Og[:, 13:].any() and np.array_equal(F.get(), Fc)
        st = plan.stats()
        for key in COUNTERS:
            assert st[key] == sc[key], key
    finally:
        plan.close()
        O.free()
        F.free()
