"""pst_plan_set_stream between two sample ranges: simulations that were started
on one stream go on with it, in every kind of step, and the next run takes the
new one (every test marked gpu)."""
import numpy as np
import pytest

from devbuf import DeviceArray
from py_stoch_amd import models
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu

U, ITA = 3001, 33


@pytest.mark.parametrize("method,model,burst_waves,specialize", [
    (0, "lotka_volterra", 0, True), (0, "lotka_volterra", 1, True), (0, "lotka_volterra", 0, False),
    (0, "schlogl", 1, True), (2, "schlogl", 0, True), (1, "schlogl", 0, False)])
@pytest.mark.parametrize("precision", [0, 1])
def test_pending_ranges_keep_their_stream(native, precision, method, model, burst_waves, specialize):
    t = 3.0 if method == 0 else 0.2
    a = models.make_args(getattr(models, model)(), E=[0], t_max=t, ita=ITA, U=U)
    tabs, rates = tables_of(a), a.rate_fn(a.c)

    def run(seed, steps):
        plan = native.Plan(tabs, rates, a.x_0, method=method, precision=precision, specialize=specialize, t_max=t,
                           I=a.I, E=a.E, n_sims=U, seed=seed, sim_offset=7)
        O, F = DeviceArray((1, ITA, U)), DeviceArray((U,))
        out = []
        try:
            plan.set_launch(0, 7, 0, burst_waves)
            for step in steps:
                if step == "set_stream":
                    plan.set_stream(99, 7)
                elif step == "whole":
                    plan.execute(O.ptr.value, U, F.ptr.value)
                else:
                    plan.execute_range([O.ptr.value], [U], step, [F.ptr.value])
                if step in ("whole", ITA):
                    out.append((O.get(), F.get()))
            return out
        finally:
            plan.close()
            O.free()
            F.free()

    print("case: set_stream between ranges, %s method %d precision %d burst_waves %d specialize %s" % (
        model, method, precision, burst_waves, specialize), flush=True)
    first, = run(5, ["whole"])
    new, = run(99, ["whole"])
    assert not np.array_equal(first[0], new[0])
    ranged, after, again = run(5, [9, "set_stream", 20, ITA, "whole", 20, ITA])
    for want, got in ((first, ranged), (new, after), (new, again)):
        assert np.array_equal(want[0], got[0]) and np.array_equal(want[1], got[1])
