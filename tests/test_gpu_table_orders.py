"""Table-driven propensities of every form an entry of the factor list takes: no
factor, orders 1 to 4, falling factorials and powers, several species to a
reaction, in each size class.  FP64 equals the oracle (every test marked gpu)."""
import numpy as np
import pytest

from py_stoch_amd import models
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu


def _network(extra):
    """Reactions of all forms on three species, and `extra` plain ones on as many
    others."""
    x = lambda i, *subs: "*".join("(species_%d - %d)" % (i, s) if s else "species_%d" % i for s in subs)
    reactions = [({}, {0: 3}, "parameter_0"),
                 ({0: 2}, {1: 1}, "parameter_1*" + x(0, 0, 1)),
                 ({0: 1, 1: 3}, {1: 3, 2: 1}, "parameter_2*" + x(0, 0) + "*" + x(1, 0, 1, 2)),
                 ({1: 1, 2: 2}, {}, "parameter_3*species_1*species_2^2")]
    x0, c = [40, 30, 20], [60.0, 2e-3, 2e-6, 4e-4]
    for i in range(extra):
        j = 4 + i
        if i == 0:
            reactions.append(({2: 4}, {3: 1}, "parameter_4*" + x(2, 0, 1, 2, 3)))
            c.append(1e-6)
        else:
            reactions.append(({2 + i: 1}, {3 + i: 1}, "parameter_%d*species_%d" % (j, 2 + i)))
            c.append(0.3 + 0.1 * i)
        x0.append(5 + i)
    return models._spn(3 + extra, reactions, x0, c)


@pytest.mark.parametrize("U", [130, 3000])
@pytest.mark.parametrize("method", [0, 1, 2])
@pytest.mark.parametrize("extra", [0, 1, 4, 5, 12])
def test_every_form_equals_the_oracle(native, oracle_mod, extra, method, U):
    a = models.make_args(_network(extra), E=[0, 1, 2], t_max=2.0, ita=13, U=U)
    tabs, rates = tables_of(a), a.rate_fn(a.c)
    assert tabs["hazard_c"] is None and tabs["prop_order"].max() == (3 if extra == 0 else 4)
    kw = dict(method=method, t_max=2.0, I=a.I, E=a.E, n_sims=U, seed=13)
    print("case: %d reactions, method %d, %d simulations" % (tabs["M"], method, U), flush=True)
    O, F, st = native.simulate(tabs, rates, a.x_0, specialize=False, **kw)
    Oc, Fc, sc = oracle_mod.simulate(tabs, rates, a.x_0, threads=16, **kw)
    assert np.array_equal(O, Oc) and np.array_equal(F, Fc)
    assert st["events"] == sc["events"] > 0
