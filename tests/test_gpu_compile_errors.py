"""A hazard that the checks let pass and the compiler refuses: the error names
the job (every test marked gpu, for a plan needs a device)."""
import pytest

from py_stoch_amd import models
from py_stoch_amd.mod.parser.tl_parser import tables_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", [0, 2])
def test_the_error_names_the_job(native, method):
    a = models.make_args(models.birth_death(), E=[0], t_max=1.0, ita=3, U=4000)
    kw = dict(method=method, specialize=True, t_max=1.0, I=a.I, E=a.E, n_sims=4000)
    good = native.Job(tables_of(a), a.rate_fn(a.c), a.x_0, **kw)
    bad = native.Job(dict(tables_of(a), hazard_c=["C(0)", "C(1)*()"], n_params=2), a.rate_fn(a.c), a.x_0, **kw)
    for jobs, which in (([bad, good], 0), ([good, bad], 1), ([good, good, bad], 2)):
        print("case: method %d, job %d of %d does not compile" % (method, which, len(jobs)), flush=True)
        with pytest.raises(native.NativeError, match=r"job %d: " % which):
            native.BatchPlan(jobs)
