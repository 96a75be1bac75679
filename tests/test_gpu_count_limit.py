"""The limit of 2^30 on a count, met inside a run of batched SSA steps.  A visit
to such a run takes up to 64 (ssa_slice + 1) steps, so how far below the limit
a count has to be for the run depends on the slice: here it starts some 8,000
below and passes the limit by steps of 1 to 127 within one visit, at the default
slice and at the largest.  The simulation ends at that step with
FLAG_OVERFLOW and zeros after it (every test marked gpu)."""
import numpy as np
import pytest

from devbuf import DeviceArray
from py_stoch_amd import models
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu

LIMIT = 1 << 30
OVERFLOW = 1
COUNTERS = ("events", "leaps", "rejected_leaps", "ssa_steps", "flagged", "flagged_events")


def _run(native, jump, slice_, method, precision, specialize):
    """A species that only grows, by `jump` a time, driven by one of about 50
    counts; some simulations pass the limit before the last sample."""
    spn = models._spn(2, [({1: 1}, {0: jump, 1: 1}, "parameter_0*species_1"), ({}, {1: 1}, "parameter_1"),
                          ({1: 1}, {}, "parameter_2*species_1")],
                      [LIMIT - 8128 - 3 * jump, 50], [20.0, 50.0, 1.0])
    t = (8128 / jump + 3) / 1000.0
    a = models.make_args(spn, E=[0, 1], t_max=1.05 * t, ita=9, U=300)
    tabs, rates = tables_of(a), a.rate_fn(a.c)
    kw = dict(method=method, t_max=1.05 * t, I=a.I, E=a.E, n_sims=300, seed=3, ssa_burst=700)
    print("case: jump %d slice %d method %d precision %d specialize %s" % (jump, slice_, method, precision, specialize),
          flush=True)
    plan = native.Plan(tabs, rates, a.x_0, precision=precision, specialize=specialize, **kw)
    O, F = DeviceArray((2, 9, 300)), DeviceArray((300,))
    try:
        plan.set_launch(0, slice_)
        plan.execute(O.ptr.value, 300, F.ptr.value)
        return (tabs, rates, a.x_0, kw), O.get(), F.get(), plan.stats()
    finally:
        plan.close()
        O.free()
        F.free()


@pytest.mark.parametrize("specialize", [True, False])
@pytest.mark.parametrize("slice_", [7, 63])
@pytest.mark.parametrize("method", [0, 1, 2])
@pytest.mark.parametrize("jump", [1, 2, 20, 127])
def test_fp64_equals_oracle(native, oracle_mod, jump, method, slice_, specialize):
    args, O, F, st = _run(native, jump, slice_, method, 0, specialize)
    Oc, Fc, sc = oracle_mod.simulate(*args[:3], **args[3])
    assert 0 < sc["flagged"] < 300
    assert np.array_equal(F, Fc) and np.array_equal(O, Oc)
    for key in COUNTERS:
        assert st[key] == sc[key], key


@pytest.mark.parametrize("specialize", [True, False])
@pytest.mark.parametrize("slice_", [7, 63])
@pytest.mark.parametrize("method", [1, 2])
@pytest.mark.parametrize("jump", [2, 20, 127])
def test_mixed_ends_at_the_limit(native, jump, method, slice_, specialize):
    _, O, F, st = _run(native, jump, slice_, method, 1, specialize)
    x = O[0]
    assert x.max() < LIMIT
    over = F == OVERFLOW
    assert 0 < over.sum() < 300 and st["flagged"] == over.sum() and np.all((F == 0) | over)
    # once a sample is zero so are those after it, and only where the limit was met
    assert np.array_equal((x[-1] == 0), over)
    grown = np.where(x == 0, LIMIT, x)
    assert np.all(np.diff(grown, axis=0) >= 0)
