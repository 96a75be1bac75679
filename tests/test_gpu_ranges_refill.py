"""Sample ranges with more simulations than lanes on the chip: the lanes of a
resumed range take simulations from the queue until every one has been visited,
also where the first ones taken had all ended in an earlier range (every test
marked gpu)."""
import ctypes

import numpy as np
import pytest

from devbuf import DeviceArray
from py_stoch_amd import models
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu

SETS, PER_SET = 20, 10007
ITA = 16


def _plan(native, method, precision, specialize, layout):
    """Immigration and decay; the first twelve parameter sets (120,084
    simulations, nearly two a lane) start and stay at 0, an absorbing state."""
    spn = models._spn(2, [({}, {0: 1}, "parameter_0"), ({0: 1}, {1: 1}, "parameter_1*species_0"),
                          ({1: 1}, {}, "parameter_2*species_1")], [0, 0], [9.0, 1.0, 0.5])
    a = models.make_args(spn, E=[0, 1], t_max=3.0, ita=ITA, U=SETS * PER_SET)
    rows = np.tile(np.asarray(a.rate_fn(a.c), np.float64), (SETS, 1))
    x0 = np.tile(np.array([[30, 20]], np.int32), (SETS, 1))
    rows[:12, 0] = 0.0
    x0[:12] = 0
    return native.Plan(tables_of(a), rows, x0, method=method, precision=precision, specialize=specialize, layout=layout,
                       t_max=3.0, I=a.I, E=a.E, n_sims=SETS * PER_SET, sims_per_set=PER_SET, seed=8)


@pytest.mark.parametrize("method,precision,specialize,burst_waves", [
    (0, 0, True, 0), (0, 0, True, 1), (0, 1, True, 1), (0, 1, False, 0), (2, 0, True, 0), (2, 1, True, 0),
    (2, 0, False, 0)])
def test_every_simulation_is_resumed(native, method, precision, specialize, burst_waves):
    U = SETS * PER_SET
    got = []
    for ends in (None, [8, ITA]):
        print("case: method %d precision %d specialize %s burst_waves %d ranges %s" % (
            method, precision, specialize, burst_waves, ends), flush=True)
        plan = _plan(native, method, precision, specialize, native.LAYOUT_BLOCKS)
        O, F = DeviceArray((2, ITA // 8, U, 8)), DeviceArray((U,))
        try:
            for buf in (O, F):  # nothing of an earlier run in them
                assert O.hip.hipMemset(buf.ptr, 0x5a, ctypes.c_size_t(buf.nbytes)) == 0
            plan.set_launch(0, 7, 7, burst_waves)  # one resident wavefront per SIMD
            if ends is None:
                plan.execute(O.ptr.value, U, F.ptr.value)
                plan.stats()
            for f in ends or []:
                plan.execute_range([O.ptr.value], [U], f, [F.ptr.value])
                plan.stats()
            got.append((O.get(), F.get()))
        finally:
            plan.close()
            O.free()
            F.free()
    assert got[0][0][0, -1, 12 * PER_SET:].any() and not got[0][0][:, :, :12 * PER_SET].any()
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
