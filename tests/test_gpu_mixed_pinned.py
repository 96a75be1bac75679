"""Mixed-precision trajectories pinned to fixed values.

Nothing outside the kernel has the mixed engine's arithmetic (hardware log2,
exp2 and reciprocals), so a changed rounding in the leap decision shows only
against values recorded before the change.  The networks are laid out to meet
it: two species whose tau bound equals the SSA switch 10 / a0, up to the
rounding of a0, in the state where the simulations spend most time, for each of
1024 sets of rates; net changes of 3 and 5 (products that are not exact) by
reactions with and without a critical species; a hazard given as an expression;
Lotka-Volterra; a network of 6 species and 10 reactions.  The checksums are
those of a0 and the sums of CalculateTau with each product fused into its sum
(every test marked gpu)."""
import zlib

import numpy as np
import pytest

from devbuf import DeviceArray
from py_stoch_amd import models, workloads
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu

U = 65536  # one simulation per lane
SETS = 1024


def _switch_rates():
    """Rates with num^2 / sigma_0^2 = 10 / a0 at the counts (86, 120), num =
    0.03 * 86, before rounding to FP32."""
    rng = np.random.default_rng(8)
    d0 = rng.uniform(0.8, 1.25, SETS)
    b = 86.0 * d0 * rng.uniform(0.97, 1.03, SETS)
    s0 = b + 86.0 * d0
    d1 = s0 * (10.0 / (0.03 * 86.0) ** 2 - 1.0) / 120.0
    return np.stack([b, d0, d1], axis=1)


def _two_species():
    """Immigration, conversion, decay: both reactions of the second species can
    be critical, so its bound is one that may not count."""
    return models._spn(2, [({}, {0: 1}, "parameter_0"), ({0: 1}, {1: 1}, "parameter_1*species_0"),
                           ({1: 1}, {}, "parameter_2*species_1")], [86, 120], [86.0, 1.0, 0.72])


def _changes_of_three_and_five():
    return models._spn(3, [({}, {0: 3}, "parameter_0"), ({0: 1}, {1: 1}, "parameter_1*species_0"),
                           ({1: 1}, {}, "parameter_2*species_1"), ({0: 1}, {0: 1, 1: 5, 2: 5}, "parameter_3*species_0"),
                           ({2: 1}, {0: 3}, "parameter_4*species_2"),
                           ({2: 2}, {1: 3}, "parameter_5*species_2*(species_2 - 1)")],
                       [150, 160, 140], [31.0, 1.7, 1.3, 0.05, 0.37, 0.0021])


def _case(name):
    """tables, rates, x0 and settings of a run of U simulations."""
    if name == "random":
        spn = models.random_network(np.random.default_rng(3), n_species=6, n_reactions=10)
        tabs, rates = workloads.mass_action_tables(spn)
        kw = dict(t_max=2.0, I=np.linspace(0, 2.0, 9).astype(np.float32), E=np.arange(6, dtype=np.int32),
                  max_steps=1500)
        return tabs, rates, np.asarray(spn.M, np.int32), dict(kw, method=0, n_sims=U, seed=12)
    spn, E, t = {"switch": (_two_species(), [0, 1], 10.0), "hazards": (_two_species(), [0, 1], 10.0),
                 "changes": (_changes_of_three_and_five(), [0, 1, 2], 6.0),
                 "lotka_volterra": (models.lotka_volterra(), [0, 1], 4.0)}[name]
    a = models.make_args(spn, E=E, t_max=t, ita=11, U=U)
    tabs, rates, x0 = tables_of(a), a.rate_fn(a.c), a.x_0
    kw = dict(method=0, t_max=t, I=a.I, E=a.E, n_sims=U, seed=12)
    if name in ("switch", "hazards"):
        rates, x0 = _switch_rates(), np.tile(np.asarray(a.x_0).reshape(1, -1), (SETS, 1))
        kw["sims_per_set"] = U // SETS
    if name == "hazards":
        tabs = dict(tabs, hazard_c=["C(0)", "C(1)*X(0)", "C(2)*X(1)"], n_params=3)
    return tabs, rates, x0, kw


def _run(native, case, launch, n):
    """Trajectories and flags of the case's first n simulations with this launch
    shape."""
    tabs, rates, x0, kw = case
    kw = dict(kw, n_sims=n)
    plan = native.Plan(tabs, rates, x0, precision=native.PRECISION_MIXED, specialize=True, **kw)
    O, F = DeviceArray((len(kw["E"]), len(kw["I"]), n)), DeviceArray((n,))
    try:
        plan.set_launch(*launch)
        plan.execute(O.ptr.value, n, F.ptr.value)
        plan.stats()
        return O.get(), F.get()
    finally:
        plan.close()
        O.free()
        F.free()


def _crc(O, F):
    return zlib.crc32(F.tobytes(), zlib.crc32(np.ascontiguousarray(O).tobytes()))


PINNED = {"switch": 1763873137, "hazards": 1763873137, "changes": 79680652, "lotka_volterra": 1535317994,
          "random": 903482599}


@pytest.mark.parametrize("name", sorted(PINNED))
def test_mixed_trajectories_are_the_pinned_ones(native, name):
    case = _case(name)
    print("case: pinned %s, one lane per simulation" % name, flush=True)
    O, F = _run(native, case, (0, 7, 0, 0), U)
    assert _crc(O, F) == PINNED[name]
    for form, launch, n in (("a group of lanes", (0, 7, 0, 0), 8192), ("paired", (0, 7, 0, 1), U),
                            ("paired groups", (0, 7, 0, 1), 8192)):
        if name == "random" and launch[3]:
            continue  # its paired workgroup does not fit
        print("case: pinned %s, %s" % (name, form), flush=True)
        Og, Fg = _run(native, case, launch, n)
        assert np.array_equal(Og, O[:, :, :n]) and np.array_equal(Fg, F[:n]), form


def test_occupancy_build_takes_the_same_way(native):
    """More wavefronts than the plain build holds: Lotka-Volterra, 196,608
    simulations, of which the first U are the pinned ones."""
    case = _case("lotka_volterra")
    print("case: pinned lotka_volterra, occupancy build", flush=True)
    O, F = _run(native, case, (0, 7, 0, 0), 3 * U)
    assert _crc(O[:, :, :U], F[:U]) == PINNED["lotka_volterra"]


def test_a_large_launch_at_half_the_lanes(native):
    """Twice as many wavefronts as the launch needs, none of them with lanes to
    share: no groups (which took 1.6 times the time), and the same way."""
    case = _case("lotka_volterra")
    tabs, rates, x0, kw = case
    n = 4 * U
    kw = dict(kw, n_sims=n, t_max=2.0, I=np.linspace(0, 2.0, 11).astype(np.float32))
    plan = native.Plan(tabs, rates, x0, precision=native.PRECISION_MIXED, specialize=True, **kw)
    O, F = DeviceArray((2, 11, n)), DeviceArray((n,))
    try:
        got, ms = [], []
        for shift in (0, 1):
            print("case: lotka_volterra %d, lanes_shift %d" % (n, shift), flush=True)
            plan.set_launch(shift, 7, 0, 0)
            times = []
            for _ in range(4):
                plan.execute(O.ptr.value, n, F.ptr.value)
                times.append(plan.stats()["kernel_ms"])
            got.append((O.get(), F.get()))
            ms.append(min(times[1:]))
        print("kernel ms", ms, flush=True)
        assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
        assert ms[1] < 1.4 * ms[0]
    finally:
        plan.close()
        O.free()
        F.free()


def test_propensities_that_cancel_end_a_simulation(native):
    """A hazard may turn negative.  A simulation ends where the FP32 sum of the
    propensities is 0, here 1 + 1e8 - 1e8, also where the FP64 sum of the
    reaction choice is not."""
    spn = models._spn(1, [({0: 1}, {0: 2}, "parameter_0*species_0"), ({0: 1}, {0: 3}, "parameter_1*species_0"),
                          ({0: 1}, {}, "parameter_1*species_0")], [1], [1.0, 1e8])
    a = models.make_args(spn, E=[0], t_max=5.0, ita=6, U=200)
    tabs = dict(tables_of(a), hazard_c=["C(0)*X(0)", "C(1)*X(0)", "-C(1)*X(0)"], n_params=2)
    for method in (1, 2):
        print("case: cancelling propensities, method %d" % method, flush=True)
        O, F, st = native.simulate(tabs, np.array([1.0, 1e8]), a.x_0, method=method, precision=native.PRECISION_MIXED,
                                   specialize=True, t_max=5.0, I=a.I, E=a.E, n_sims=200, seed=1, max_steps=50)
        assert np.all(O == 1) and not F.any() and st["ssa_steps"] == 0
