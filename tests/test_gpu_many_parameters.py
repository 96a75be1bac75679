"""Networks with as many parameters as the library takes (256, each a register
or two of a simulation): they run by every method and at every launch size, as
the same network without the unused ones does (every test marked gpu)."""
import numpy as np
import pytest

from py_stoch_amd import models
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_params", [60, 256])
@pytest.mark.parametrize("U", [100, 40001])
@pytest.mark.parametrize("method", [0, 1, 2])
@pytest.mark.parametrize("precision", [0, 1])
def test_unused_parameters_change_nothing(native, precision, method, U, n_params):
    spn = models._spn(4, [({}, {0: 1}, "parameter_0"), ({0: 1}, {1: 1}, "parameter_1*species_0"),
                          ({1: 1}, {2: 1, 3: 1}, "parameter_2*species_1"), ({2: 1}, {}, "parameter_3*species_2")],
                      [3, 40, 5, 0], [20.0, 1.0, 0.5, 2.0])
    a = models.make_args(spn, E=[0, 1, 2, 3], t_max=2.0, ita=9, U=U)
    hazards = ["C(0)", "C(1)*X(0)", "C(2)*X(1)", "C(%d)*X(2)"]
    out = []
    for n in (4, n_params):
        print("case: %d parameters, precision %d method %d U %d" % (n, precision, method, U), flush=True)
        tabs = dict(tables_of(a), hazard_c=hazards[:3] + [hazards[3] % (n - 1)], n_params=n)
        rates = np.zeros(n)
        rates[:3], rates[n - 1] = [20.0, 1.0, 0.5], 2.0
        out.append(native.simulate(tabs, rates, a.x_0, method=method, precision=precision, specialize=True, t_max=2.0,
                                   I=a.I, E=a.E, n_sims=U, seed=5))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
