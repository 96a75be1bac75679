"""A dimerisation whose monomer count is 0 has the propensity k * 0 * (0 - 1) =
-0.0.  That is an ordinary state: the batched SSA steps take it, as they take
the +0.0 of a count of 1.  The two runs compared here differ only in that sign:
same trajectories, same time (every test marked gpu)."""
import numpy as np
import pytest

from devbuf import DeviceArray
from py_stoch_amd import models
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu

U = 2048


def _run(native, precision, specialize, x):
    """Immigration and decay of species 0 beside dimerisations of species 1 and
    2, which stay at their counts; (trajectories, best kernel time of three)."""
    spn = models._spn(3, [({}, {0: 1}, "parameter_0"), ({0: 1}, {}, "parameter_1*species_0"),
                          ({1: 2}, {}, "parameter_2*species_1*(species_1 - 1)"),
                          ({2: 2}, {1: 1}, "parameter_3*species_2*(species_2 - 1)")],
                      [10, x, x], [40.0, 1.0, 0.5, 0.25])
    a = models.make_args(spn, E=[0, 1], t_max=40.0, ita=11, U=U)
    tabs = tables_of(a)
    plan = native.Plan(tabs, a.rate_fn(a.c), a.x_0, method=native.METHOD_PURE_SSA, precision=precision,
                       specialize=specialize, t_max=40.0, I=a.I, E=a.E, n_sims=U, seed=6)
    O, F = DeviceArray((2, 11, U)), DeviceArray((U,))
    try:
        ms = []
        for _ in range(4):
            plan.execute(O.ptr.value, U, F.ptr.value)
            ms.append(plan.stats()["kernel_ms"])
        assert not F.get().any()
        return O.get()[0], min(ms[1:])
    finally:
        plan.close()
        O.free()
        F.free()


@pytest.mark.parametrize("specialize", [True, False])
@pytest.mark.parametrize("precision", [0, 1])
def test_negative_zero_propensity_is_an_ordinary_step(native, precision, specialize):
    print("case: zero counts, precision %d specialize %s" % (precision, specialize), flush=True)
    O1, t1 = _run(native, precision, specialize, 1)
    O0, t0 = _run(native, precision, specialize, 0)
    print("kernel ms at count 1: %.3f, at count 0: %.3f" % (t1, t0), flush=True)
    assert np.array_equal(O0, O1)
    assert t0 < 1.5 * t1
